// topk: the k first elements of each row in the reference's order
// (backends/cpu/cpu_math.cpp:57-67 under the plan of core/math.cpp:56-66):
// NaN before every number when the largest are asked for (after them
// otherwise), +0 == -0, ties by lower index. sorted == 0 lists the chosen
// elements in index order. Values are copied as 32-bit words, bit for bit.
//
// An element's place in that order is one unsigned integer: a 32-bit key
// (larger comes first, equal for values that tie) over the inverted index, so
// no two elements of a row compare equal and every step below is exact.
//
// Short rows with few elements asked for take a wave each (topk_wave_kernel).
// Otherwise a block works on one row at a time:
//   * rows of at most kThreads elements: every element is a candidate;
//   * k = 1, or 2 in 256 threads: a pass for each (select_rounds);
//   * k <= kThreads / 4: each thread takes the largest key of its share of the
//     row. The lower bound T of the k-th key is the smallest, over the waves,
//     of a wave's ceil(k / waves)-th largest thread maximum: at least k keys
//     are >= T. A second pass over the row collects the keys >= T, a few
//     times k of them for values in no special order;
//   * otherwise, or when too many keys are >= T (long runs of equal values,
//     ordered rows): a radix selection of the k-th key, 8 bits a pass, and a
//     compaction in index order, or for k <= kFewK a pass for each.
// Candidates in LDS are put in order by counting, for each, those before it:
// no barriers, and the counts of one candidate are shared by several lanes.
//
// What bounds it: the row is read once from HBM and once more from L2 (the
// selection reads nothing else), so a row costs two passes at the rate that
// one CU draws: 66 us for 1024 rows of 50257 with k = 50. With a workspace,
// fewer rows than CUs are cut into parts (launch_topk_parts): 22 us for 32 rows
// of 128256 with k = 50. One pass over the row for each of the k elements, as
// before, took 5.84 ms (k = 40) and 11.40.

#include <algorithm>

#include "common.hpp"

namespace tcx {
namespace {

constexpr int kCandidates = 1024;  // in LDS: 16 bytes each
// Few elements asked for have a kernel without the radix selection. It runs
// select_rounds straight away up to k = kRoundsK, by which it reads the row no
// more often than the bound and the candidates do, and where more than
// kRankedFew candidates show that the bound was a poor one: ties, rows that are
// in order already. There the radix selection (every count in one bin) and the
// ordering of a thousand candidates cost more than kFewK passes: with k = 1,
// 1024 equal rows of 50257 took 820 us and take 36, 65536 ordered rows of 1025
// took 3370 and take 185; with k = 3, 3380 and 529. Ordering more than half of
// kCandidates also costs more than the radix selection of at most kShort
// elements.
constexpr int kFewK = 12, kRankedFew = 256, kShort = 4096;
template <int kThreads>
constexpr int kRoundsK = kThreads == 256 ? 2 : 1;

struct TopkArgs {
  const std::uint32_t* x;
  std::uint32_t* values;
  std::int32_t* indices;
  std::int64_t rows, reduce, inner, k;
  int largest, sorted;
  // Rows in parts of part_len elements, where they are fewer than the CUs: the
  // places of the k first of each part go to places [rows, parts, k].
  std::int64_t parts, part_len;
  std::uint64_t* places;
};

// The elements one block selects from: n of a row from element `first` on, and
// where its choice goes (the row's outputs, or the places of a part).
struct TopkSpan {
  const std::uint32_t* x;
  std::int64_t first, n, k;
  std::uint32_t* values;
  std::int32_t* indices;
  std::uint64_t* places;
};

// Larger keys come first; equal keys are ties.
template <bool kFp>
__device__ __forceinline__ std::uint32_t topk_key(std::uint32_t word, bool largest) {
  std::uint32_t key;
  if constexpr (kFp) key = word_nan(word, true) ? 0xffffffffU : order_key(word);
  else key = word ^ 0x80000000U;
  return largest ? key : ~key;
}

__device__ __forceinline__ std::uint64_t place_of(std::uint32_t key, std::int64_t index) {
  return (static_cast<std::uint64_t>(key) << 32) | static_cast<std::uint32_t>(~static_cast<std::uint32_t>(index));
}
__device__ __forceinline__ std::int32_t index_of(std::uint64_t place) {
  return static_cast<std::int32_t>(~static_cast<std::uint32_t>(place));
}

// f(word, index) for this thread's share of a row. Contiguous rows of at least
// 4 kThreads elements (so that every thread has some) are read 16 bytes at a
// time, four or eight loads in flight, whatever the row's alignment: the
// elements in front of the first 16-byte boundary and after the last are single
// words.
template <int kThreads, typename F>
__device__ __forceinline__ void scan_row(const std::uint32_t* __restrict__ x, std::int64_t n, std::int64_t inner, F&& f) {
  using word4 = std::uint32_t __attribute__((ext_vector_type(4)));
  const int t = threadIdx.x;
  if (inner == 1 && n >= 4 * kThreads) {
    const int head = static_cast<int>((16U - (reinterpret_cast<std::uintptr_t>(x) & 15U)) & 15U) / 4;
    const std::int64_t quads = (n - head) / 4;
    const auto* body = reinterpret_cast<const word4*>(x + head);
    auto four = [&](const word4& w, std::int64_t q) {
      const std::int64_t i = head + 4 * q;
      f(w.x, i);
      f(w.y, i + 1);
      f(w.z, i + 2);
      f(w.w, i + 3);
    };
    std::int64_t q = t;
    for (; q + 7 * kThreads < quads; q += 8 * kThreads) {
      word4 w[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) w[u] = body[q + u * kThreads];
#pragma unroll
      for (int u = 0; u < 8; ++u) four(w[u], q + u * kThreads);
    }
    // What is left, four at a time too: loads past the end repeat the last.
    for (; q < quads; q += 4 * kThreads) {
      word4 w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = body[min(q + u * kThreads, quads - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (q + u * kThreads < quads) four(w[u], q + u * kThreads);
    }
    const std::int64_t tail = head + 4 * quads;
    if (t < head) f(x[t], t);
    if (tail + t < n) f(x[tail + t], tail + t);
    return;
  }
  std::int64_t i = t;
  for (; i + 3 * kThreads < n; i += 4 * kThreads) {
    std::uint32_t w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) w[u] = x[(i + u * kThreads) * inner];
#pragma unroll
    for (int u = 0; u < 4; ++u) f(w[u], i + u * kThreads);
  }
  for (; i < n; i += kThreads) f(x[i * inner], i);
}

template <int kThreads>
struct TopkShared {
  std::uint64_t place[kCandidates];
  std::uint32_t word[kCandidates];
  std::int32_t chosen[kCandidates];
  std::uint32_t histogram[256];
  std::uint32_t wave_a[kThreads / kWave], wave_b[kThreads / kWave];
  std::uint32_t count, digit, need;
};

// The wave's rank-th largest value (rank < 64), in every lane: a bitonic sort
// of the lanes, largest in lane 0.
__device__ __forceinline__ std::uint32_t wave_nth_largest(std::uint32_t v, int rank) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int size = 2; size <= 64; size <<= 1) {
#pragma unroll
    for (int stride = size / 2; stride > 0; stride >>= 1) {
      const auto other = static_cast<std::uint32_t>(__shfl_xor(static_cast<int>(v), stride, kWave));
      const bool keep_larger = ((lane & stride) == 0) == ((lane & size) == 0);
      v = (v > other) == keep_larger ? v : other;
    }
  }
  return static_cast<std::uint32_t>(__shfl(static_cast<int>(v), rank, kWave));
}

// visit(c, above) in one lane for each c < count, with above the number of
// c' < count whose value(c') is larger: lanes in groups of a power of two share
// the counting of one c, eight LDS reads in flight each (one at a time, the
// reads' latency made 750 candidates cost 30 us). Called by the whole block; no
// barriers.
template <int kThreads, typename F, typename V>
__device__ __forceinline__ void rank_each(int count, F&& value, V&& visit) {
  int group = kWave;
  while (group > 1 && count * group > kThreads) group >>= 1;
  const int g = threadIdx.x & (group - 1);
  const int step = kThreads / group;
  for (int base = 0; base < count; base += step) {
    const int c = base + threadIdx.x / group;
    const auto mine = value(c < count ? c : count - 1);
    int above = 0, j = g;
    for (; j + 7 * group < count; j += 8 * group) {
#pragma unroll
      for (int u = 0; u < 8; ++u) above += value(j + u * group) > mine ? 1 : 0;
    }
    for (; j < count; j += group) above += value(j) > mine ? 1 : 0;
    for (int offset = group / 2; offset > 0; offset >>= 1) above += __shfl_xor(above, offset, kWave);
    if (g == 0 && c < count) visit(c, above);
  }
}

// The k candidates s.chosen, written out in index order.
template <int kThreads>
__device__ __forceinline__ void emit_by_index(TopkShared<kThreads>& s, const TopkArgs& a, const TopkSpan& w) {
  rank_each<kThreads>(
      static_cast<int>(w.k),
      [&](int c) { return ~index_of(s.place[s.chosen[c]]); },  // lower indices above
      [&](int c, int before) {
        const int at = s.chosen[c];
        w.values[before * a.inner] = s.word[at];
        w.indices[before * a.inner] = index_of(s.place[at]);
      });
}

// The k first of the `count` candidates in LDS, written out.
template <int kThreads, bool kParts>
__device__ __forceinline__ void emit_candidates(TopkShared<kThreads>& s, const TopkArgs& a, const TopkSpan& w, int count) {
  const int k = static_cast<int>(w.k);  // <= count
  rank_each<kThreads>(
      count, [&](int c) { return s.place[c]; },
      [&](int c, int before) {
        if (before >= k) return;
        if constexpr (kParts) {
          w.places[before] = s.place[c];
        } else if (a.sorted) {
          w.values[before * a.inner] = s.word[c];
          w.indices[before * a.inner] = index_of(s.place[c]);
        } else {
          s.chosen[before] = c;
        }
      });
  if (kParts || a.sorted) return;
  __syncthreads();
  emit_by_index<kThreads>(s, a, w);
}

// The key of the k-th element and how many of the elements equal to it are
// among the k (s.need): 8 bits a pass from the top.
template <int kThreads, bool kFp>
__device__ std::uint32_t radix_kth(TopkShared<kThreads>& s, const TopkArgs& a, const TopkSpan& span) {
  const bool largest = a.largest != 0;
  const int t = threadIdx.x;
  std::uint32_t prefix = 0, mask = 0;
  if (t == 0) s.need = static_cast<std::uint32_t>(span.k);
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int b = t; b < 256; b += kThreads) s.histogram[b] = 0;
    __syncthreads();
    scan_row<kThreads>(span.x, span.n, a.inner, [&](std::uint32_t w, std::int64_t) {
      const std::uint32_t key = topk_key<kFp>(w, largest);
      if ((key & mask) == prefix) atomicAdd(&s.histogram[(key >> shift) & 255U], 1U);
    });
    __syncthreads();
    if (t < kWave) {
      // Lane l holds bins 255 - 4l .. 252 - 4l; the bin in which the count
      // from the top reaches `need` is the digit.
      std::uint32_t bins[4], sum = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        bins[e] = s.histogram[255 - 4 * t - e];
        sum += bins[e];
      }
      std::uint32_t upto = sum;
#pragma unroll
      for (int offset = 1; offset < kWave; offset <<= 1) {
        const auto below = static_cast<std::uint32_t>(__shfl_up(static_cast<int>(upto), offset, kWave));
        if (t >= offset) upto += below;
      }
      const std::uint32_t need = s.need;
      std::uint32_t above = upto - sum;
      if (above < need && need <= upto) {
        bool found = false;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (!found && need <= above + bins[e]) {
            s.digit = 255U - 4U * t - e;
            s.need = need - above;
            found = true;
          }
          above += bins[e];
        }
      }
    }
    __syncthreads();
    prefix |= s.digit << shift;
    mask |= 255U << shift;
  }
  return prefix;
}

// Sorts `n` output elements in place in global memory, first in order first:
// bitonic merges whose comparators all point one way, so that a length that
// is no power of two behaves as if padded with elements that come last.
template <int kThreads, bool kFp>
__device__ void sort_output(const TopkArgs& a, std::uint32_t* values, std::int32_t* indices) {
  const std::int64_t n = a.k;
  const bool largest = a.largest != 0;
  auto exchange = [&](std::int64_t i, std::int64_t j) {
    const std::uint32_t wi = values[i * a.inner], wj = values[j * a.inner];
    const std::int32_t ii = indices[i * a.inner], ij = indices[j * a.inner];
    if (place_of(topk_key<kFp>(wi, largest), ii) > place_of(topk_key<kFp>(wj, largest), ij)) return;
    values[i * a.inner] = wj;
    values[j * a.inner] = wi;
    indices[i * a.inner] = ij;
    indices[j * a.inner] = ii;
  };
  std::int64_t padded = 1;
  while (padded < n) padded <<= 1;
  for (std::int64_t size = 2; size <= padded; size <<= 1) {
    const std::int64_t half = size / 2;
    __syncthreads();
    for (std::int64_t p = threadIdx.x; p < padded / 2; p += kThreads) {
      const std::int64_t start = p / half * size, o = p % half;
      if (start + size - 1 - o < n) exchange(start + o, start + size - 1 - o);
    }
    for (std::int64_t stride = half / 2; stride > 0; stride >>= 1) {
      __syncthreads();
      for (std::int64_t p = threadIdx.x; p < padded / 2; p += kThreads) {
        const std::int64_t i = p / stride * 2 * stride + p % stride;
        if (i + stride < n) exchange(i, i + stride);
      }
    }
  }
}

// Radix selection, then the chosen elements in index order: to the output, or
// to LDS where they are still to be put in order and fit.
template <int kThreads, bool kFp, bool kParts>
__device__ void select_span(TopkShared<kThreads>& s, const TopkArgs& a, const TopkSpan& span) {
  constexpr int kWaves = kThreads / kWave;
  const bool largest = a.largest != 0;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const std::uint32_t kth = radix_kth<kThreads, kFp>(s, a, span);
  const std::int64_t ties = s.need, n = span.n;
  const bool in_lds = kParts || (a.sorted && span.k <= kCandidates);
  std::int64_t greater_run = 0, equal_run = 0;
  for (std::int64_t start = 0; start < n && greater_run + min(equal_run, ties) < span.k; start += kThreads) {
    const std::int64_t i = start + t;
    std::uint32_t w = 0;
    bool greater = false, equal = false;
    if (i < n) {
      w = span.x[i * a.inner];
      const std::uint32_t key = topk_key<kFp>(w, largest);
      greater = key > kth;
      equal = key == kth;
    }
    const unsigned long long gm = __ballot(greater), em = __ballot(equal);
    __syncthreads();  // the previous chunk's counts have been read
    if (lane == 0) {
      s.wave_a[wave] = __popcll(gm);
      s.wave_b[wave] = __popcll(em);
    }
    __syncthreads();
    const unsigned long long below = (1ULL << lane) - 1ULL;
    std::int64_t greater_before = greater_run + __popcll(gm & below), equal_before = equal_run + __popcll(em & below);
    for (int v = 0; v < kWaves; ++v) {
      const std::uint32_t g = s.wave_a[v], e = s.wave_b[v];
      if (v < wave) {
        greater_before += g;
        equal_before += e;
      }
      greater_run += g;
      equal_run += e;
    }
    if (greater || (equal && equal_before < ties)) {
      const std::int64_t at = greater_before + min(equal_before, ties);
      if (in_lds) {
        s.place[at] = place_of(topk_key<kFp>(w, largest), span.first + i);
        s.word[at] = w;
      } else {
        span.values[at * a.inner] = w;
        span.indices[at * a.inner] = static_cast<std::int32_t>(i);
      }
    }
  }
  if (!in_lds && !a.sorted) return;
  __syncthreads();
  if (in_lds) emit_candidates<kThreads, kParts>(s, a, span, static_cast<int>(span.k));
  else sort_output<kThreads, kFp>(a, span.values, span.indices);
}

// k rounds over the row for few k, each for the first element after the one
// before, whatever the values are.
template <int kThreads, bool kFp, bool kParts>
__device__ void select_rounds(TopkShared<kThreads>& s, const TopkArgs& a, const TopkSpan& span) {
  constexpr int kWaves = kThreads / kWave;
  const bool largest = a.largest != 0;
  const int t = threadIdx.x, k = static_cast<int>(span.k);
  std::uint64_t last = 0;
  for (int j = 0; j < k; ++j) {
    std::uint64_t best = 0;  // below every element's place
    scan_row<kThreads>(span.x, span.n, a.inner, [&](std::uint32_t w, std::int64_t i) {
      const std::uint64_t place = place_of(topk_key<kFp>(w, largest), span.first + i);
      if ((j == 0 || place < last) && place > best) best = place;
    });
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
      const std::uint64_t other = __shfl_xor(static_cast<unsigned long long>(best), offset, kWave);
      best = other > best ? other : best;
    }
    __syncthreads();  // the previous round's maxima have been read
    if ((t & 63) == 0) s.place[t >> 6] = best;
    __syncthreads();
    for (int v = 0; v < kWaves; ++v) best = s.place[v] > best ? s.place[v] : best;
    last = best;
    if (t == 0) {
      if constexpr (kParts) {
        span.places[j] = best;
      } else {
        const std::int32_t index = index_of(best);
        const std::uint32_t word = span.x[index * a.inner];
        if (a.sorted) {
          span.values[j * a.inner] = word;
          span.indices[j * a.inner] = index;
        } else {  // emit_by_index takes them behind the waves' maxima
          s.place[kWaves + j] = best;
          s.word[kWaves + j] = word;
          s.chosen[j] = kWaves + j;
        }
      }
    }
  }
  if (kParts || a.sorted) return;
  __syncthreads();
  emit_by_index<kThreads>(s, a, span);
}

// kFew: k <= kFewK.
template <int kThreads, bool kFp, bool kParts, bool kFew>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(kThreads == 256 && kFew ? 5 : 4, 8))) void
topk_kernel(TopkArgs a) {
  constexpr int kWaves = kThreads / kWave;
  __shared__ TopkShared<kThreads> s;
  const bool largest = a.largest != 0;
  const int t = threadIdx.x;
  const std::int64_t parts = kParts ? a.parts : 1, items = a.rows * parts;
  for (std::int64_t item = blockIdx.x; item < items; item += gridDim.x) {
    const std::int64_t row = item / parts, part = item % parts;
    const std::int64_t outer = row / a.inner, column = row % a.inner;
    TopkSpan span;
    span.first = kParts ? part * a.part_len : 0;
    span.n = kParts ? min(a.part_len, a.reduce - span.first) : a.reduce;
    span.k = kParts ? min(a.k, span.n) : a.k;
    span.x = a.x + (outer * a.reduce + span.first) * a.inner + column;
    span.values = a.values + outer * a.k * a.inner + column;
    span.indices = a.indices + outer * a.k * a.inner + column;
    span.places = kParts ? a.places + item * a.k : nullptr;
    __syncthreads();  // the previous item is done with s
    if constexpr (kParts) {  // a short last part: places below every element's
      for (std::int64_t j = span.k + t; j < a.k; j += kThreads) span.places[j] = 0;
    }
    if (span.n <= kThreads) {
      if (t < span.n) {
        const std::uint32_t w = span.x[t * a.inner];
        s.place[t] = place_of(topk_key<kFp>(w, largest), span.first + t);
        s.word[t] = w;
      }
      __syncthreads();
      emit_candidates<kThreads, kParts>(s, a, span, static_cast<int>(span.n));
      continue;
    }
    if constexpr (kFew) {
      if (span.k <= kRoundsK<kThreads>) {
        select_rounds<kThreads, kFp, kParts>(s, a, span);
        continue;
      }
    } else {
      if (span.k > kThreads / 4) {
        select_span<kThreads, kFp, kParts>(s, a, span);
        continue;
      }
    }
    std::uint32_t best = 0;
    scan_row<kThreads>(span.x, span.n, a.inner, [&](std::uint32_t w, std::int64_t) {
      best = max(best, topk_key<kFp>(w, largest));
    });
    const int per_wave = (static_cast<int>(span.k) + kWaves - 1) / kWaves;  // <= 16
    const std::uint32_t bound = wave_nth_largest(best, per_wave - 1);
    if ((t & 63) == 0) s.wave_a[t >> 6] = bound;
    if (t == 0) s.count = 0;
    __syncthreads();
    std::uint32_t least = s.wave_a[0];
#pragma unroll
    for (int v = 1; v < kWaves; ++v) least = min(least, s.wave_a[v]);
    scan_row<kThreads>(span.x, span.n, a.inner, [&](std::uint32_t w, std::int64_t i) {
      const std::uint32_t key = topk_key<kFp>(w, largest);
      if (key < least) return;
      const std::uint32_t at = atomicAdd(&s.count, 1U);
      if (at < kCandidates) {
        s.place[at] = place_of(key, span.first + i);
        s.word[at] = w;
      }
    });
    __syncthreads();
    if (s.count <= (kFew ? kRankedFew : span.n <= kShort ? kCandidates / 2 : kCandidates))
      emit_candidates<kThreads, kParts>(s, a, span, static_cast<int>(s.count));
    else if constexpr (kFew) select_rounds<kThreads, kFp, kParts>(s, a, span);
    else select_span<kThreads, kFp, kParts>(s, a, span);
  }
}

// The k first of the parts' choices (parts * k <= kCandidates), a block a row.
// Each part's places come in order, so the place of an element among all of
// them is its rank in its own part and a binary search in each other one.
__global__ __launch_bounds__(1024) void topk_join_kernel(TopkArgs a) {
  __shared__ TopkShared<1024> s;
  const int t = threadIdx.x, parts = static_cast<int>(a.parts), k = static_cast<int>(a.k), count = parts * k;
  const std::int64_t row = blockIdx.x, outer = row / a.inner, column = row % a.inner;
  TopkSpan span{};
  span.x = a.x + outer * a.reduce * a.inner + column;
  span.k = a.k;
  span.values = a.values + outer * a.k * a.inner + column;
  span.indices = a.indices + outer * a.k * a.inner + column;
  std::uint64_t mine = 0;
  if (t < count) {
    mine = a.places[row * count + t];
    s.place[t] = mine;
    s.word[t] = mine != 0 ? span.x[index_of(mine) * a.inner] : 0U;
  }
  __syncthreads();
  if (t < count && mine != 0) {
    const int own = t / k;
    int before = t % k;
#pragma unroll 4
    for (int part = 0; part < parts; ++part) {
      const std::uint64_t* const other = s.place + part * k;
      int above = 0;  // of other[0 .. k), those larger than mine
      for (int length = k; length > 0;) {
        const int half = length >> 1;
        const bool larger = other[above + half] > mine;
        above += larger ? half + 1 : 0;
        length = larger ? length - half - 1 : half;
      }
      before += part != own ? above : 0;
    }
    if (before < k) {
      if (a.sorted) {
        span.values[before * a.inner] = s.word[t];
        span.indices[before * a.inner] = index_of(mine);
      } else {
        s.chosen[before] = t;
      }
    }
  }
  if (a.sorted) return;
  __syncthreads();
  emit_by_index<1024>(s, a, span);
}

// Short rows and few of them asked for: one wave a row, the row in registers
// (kEach keys a lane), k rounds of the wave's first remaining element. Lane j
// keeps the j-th, so the stores of a row are one instruction.
constexpr std::int64_t kWaveRow = 1024, kWaveK = 8, kWaveWideK = 3;

template <int kEach, bool kFp>
__global__ __launch_bounds__(256) void topk_wave_kernel(TopkArgs a) {
  const bool largest = a.largest != 0;
  const int lane = threadIdx.x & 63;
  const int k = static_cast<int>(a.k);
  const std::int64_t step = static_cast<std::int64_t>(gridDim.x) * 4;
  for (std::int64_t row = static_cast<std::int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6); row < a.rows; row += step) {
    const std::int64_t outer = row / a.inner, column = row % a.inner;
    const std::uint32_t* __restrict__ x = a.x + outer * a.reduce * a.inner + column;
    std::uint32_t key[kEach];
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      const std::int64_t i = e * kWave + lane;
      key[e] = topk_key<kFp>(x[(i < a.reduce ? i : 0) * a.inner], largest);
    }
    std::uint64_t last = 0, mine = 0;
    for (int j = 0; j < k; ++j) {
      std::uint64_t best = 0;  // below every element's place
#pragma unroll
      for (int e = 0; e < kEach; ++e) {
        const int i = e * kWave + lane;
        const std::uint64_t place = place_of(key[e], i);
        if (i < a.reduce && (j == 0 || place < last) && place > best) best = place;
      }
#pragma unroll
      for (int offset = 32; offset > 0; offset >>= 1) {
        const std::uint64_t other = __shfl_xor(static_cast<unsigned long long>(best), offset, kWave);
        best = other > best ? other : best;
      }
      last = best;
      if (lane == j) mine = best;
    }
    int at = lane;
    const int index = index_of(mine);
    if (!a.sorted) {
      at = 0;
      for (int j = 0; j < k; ++j) at += __shfl(index, j, kWave) < index ? 1 : 0;
    }
    if (lane < k) {
      const std::int64_t to = outer * a.k * a.inner + column + at * a.inner;
      a.values[to] = x[index * a.inner];
      a.indices[to] = index;
    }
  }
}

template <int kEach, bool kFp>
void launch_topk_wave(const TopkArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((topk_wave_kernel<kEach, kFp>), dim3(grid_for(a.rows, 4, kStrideBlocks)), dim3(256), 0, s, a);
}

template <int kThreads, bool kFp>
void launch_topk(const TopkArgs& a, hipStream_t s) {
  const std::int64_t cap = kMaxLaunchWorkItems / kThreads;
  const dim3 grid(static_cast<unsigned>(a.rows < cap ? a.rows : cap));
  // Four more where many rows of a few thousand elements share the CUs: ordered,
  // 2424 x 4097 int32 with k = 13 180 us in k passes, 224 by the radix selection.
  const bool few = a.k <= kFewK || (a.k <= kFewK + 4 && a.rows >= 512 && a.reduce > 2048 && a.reduce <= 8192);
  if (few) hipLaunchKernelGGL((topk_kernel<kThreads, kFp, false, true>), grid, dim3(kThreads), 0, s, a);
  else hipLaunchKernelGGL((topk_kernel<kThreads, kFp, false, false>), grid, dim3(kThreads), 0, s, a);
}

// The number of parts to cut a row into (1: whole). Fewer rows than the 256 CUs
// and at least two parts of 8192 elements; all parts' choices are joined in LDS.
std::int64_t topk_parts(std::int64_t rows, std::int64_t reduce, std::int64_t k) {
  const std::int64_t parts = std::min({256 / rows, reduce / 8192, kCandidates / std::max<std::int64_t>(k, 1)});
  return k <= 256 && parts >= 2 ? parts : 1;
}

// The parts, each a block, and their join: 32 rows of 128256 with k = 50 in 15 +
// 6 us against 29.5 us for a block a row, whose two passes are bound by what one
// CU reads; one row of 128256 20 against 29 us.
template <bool kFp>
void launch_topk_parts(const TopkArgs& a, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(a.rows * a.parts));
  if (a.k <= kFewK) hipLaunchKernelGGL((topk_kernel<1024, kFp, true, true>), grid, dim3(1024), 0, s, a);
  else hipLaunchKernelGGL((topk_kernel<1024, kFp, true, false>), grid, dim3(1024), 0, s, a);
  hipLaunchKernelGGL(topk_join_kernel, dim3(static_cast<unsigned>(a.rows)), dim3(1024), 0, s, a);
}

// A wave a row up to kWaveRow elements and k = kWaveK: with k = 1, 14.7 us for
// 65536 rows of 32 and 5.4 us for 4096 rows of 1000, against 144 and 22.7 us
// with a block a row; with many rows up to twice k (60000 x 300 int32 with k = 13
// 262 -> 152 us, equal values 1069 -> 153) and, for kWaveWideK elements, twice the
// length (10000 x 1086 int32 with k = 1 30 -> 17 us, with k = 3 46 -> 27, equal
// values 84 -> 27). Else 256 threads, of which a CU holds four or five blocks
// (1024 rows of 50257 with k = 3 64 us, with 1024 threads 98; 8192 rows of 8193
// 90 and 322; 1024 rows of 8193 16 and 42), and 1024 where one row has a CU to
// itself and is long enough to keep them reading (one row of 50257 17 us,
// of 1000000 148; with 256 threads 22 and 306; 255 rows of 50257 the same), or
// where 256 would send k to the radix selection.
template <bool kFp>
void launch_topk_rows(const TopkArgs& a, hipStream_t s) {
  const bool short_row = a.reduce <= kWaveRow && (a.k <= kWaveK || (a.k <= 2 * kWaveK && a.rows >= (a.reduce > 256 ? 2048 : 4096)));
  if (short_row || (a.reduce <= 2 * kWaveRow && a.k <= kWaveWideK && a.rows >= 256)) {
    if (a.reduce <= 64) launch_topk_wave<1, kFp>(a, s);
    else if (a.reduce <= 256) launch_topk_wave<4, kFp>(a, s);
    else if (a.reduce <= kWaveRow) launch_topk_wave<16, kFp>(a, s);
    else launch_topk_wave<32, kFp>(a, s);
  } else if ((a.reduce > 20000 && a.rows < 256) || (a.reduce > 256 && a.k > 64)) {
    launch_topk<1024, kFp>(a, s);
  } else {
    launch_topk<256, kFp>(a, s);
  }
}

}  // namespace
}  // namespace tcx

extern "C" {

size_t tcx_hip_topk_workspace_bytes(int64_t outer, int64_t reduce, int64_t inner, int64_t k) {
  if (outer <= 0 || inner <= 0 || outer > 256 || inner > 256 || reduce > 0x7fffffff || k <= 0 || k > reduce) return 0;
  const std::int64_t rows = outer * inner;
  if (rows > 256) return 0;
  const std::int64_t parts = tcx::topk_parts(rows, reduce, k);
  return parts > 1 ? static_cast<size_t>(rows * parts * k) * sizeof(std::uint64_t) : 0;
}

int tcx_hip_topk_ws(int dtype, const void* x, void* values, int32_t* indices, int64_t outer, int64_t reduce,
                    int64_t inner, int64_t k, int largest, int sorted, void* workspace, size_t workspace_bytes,
                    tcx_stream_t stream) {
  using namespace tcx;
  if (dtype != TCX_FLOAT32 && dtype != TCX_INT32) return fail(TCX_INVALID_ARGUMENT, "math operations require float32 or int32");
  if (outer < 0 || reduce < 0 || inner < 0) return fail(TCX_INVALID_ARGUMENT, "topk extents must be non-negative");
  if (reduce > 0x7fffffff) return fail(TCX_INVALID_ARGUMENT, "topk index range exceeds int32");
  if (k < 0 || k > reduce) return fail(TCX_INVALID_ARGUMENT, "topk k must be between zero and the axis size");
  const std::int64_t rows = outer * inner;
  if (rows == 0 || k == 0) return TCX_OK;
  if (rows > 0x7fffffff) return fail(TCX_INVALID_ARGUMENT, "topk has too many rows");
  if (x == nullptr || values == nullptr || indices == nullptr) return fail(TCX_INVALID_ARGUMENT, "topk buffers are null");
  if (int rc = ready(); rc != TCX_OK) return rc;
  const auto s = static_cast<hipStream_t>(stream);
  TopkArgs a{static_cast<const std::uint32_t*>(x), static_cast<std::uint32_t*>(values), indices, rows, reduce,
             inner, k, largest, sorted, 1, reduce, nullptr};
  const size_t needed = tcx_hip_topk_workspace_bytes(outer, reduce, inner, k);
  if (needed != 0 && workspace != nullptr && workspace_bytes >= needed &&
      (reinterpret_cast<std::uintptr_t>(workspace) & 7U) == 0) {
    const std::int64_t parts = topk_parts(rows, reduce, k);
    a.part_len = ((reduce + parts - 1) / parts + 3) / 4 * 4;
    a.parts = (reduce + a.part_len - 1) / a.part_len;
    a.places = static_cast<std::uint64_t*>(workspace);
    if (dtype == TCX_FLOAT32) launch_topk_parts<true>(a, s);
    else launch_topk_parts<false>(a, s);
    return check(hipGetLastError(), "topk launch");
  }
  if (dtype == TCX_FLOAT32) launch_topk_rows<true>(a, s);
  else launch_topk_rows<false>(a, s);
  return check(hipGetLastError(), "topk launch");
}

int tcx_hip_topk(int dtype, const void* x, void* values, int32_t* indices, int64_t outer, int64_t reduce,
                 int64_t inner, int64_t k, int largest, int sorted, tcx_stream_t stream) {
  return tcx_hip_topk_ws(dtype, x, values, indices, outer, reduce, inner, k, largest, sorted, nullptr, 0, stream);
}

}  // extern "C"
