// Fused attention: out = softmax(scale * Q K^T [causal]) V without
// materialising the scores, on v_mfma_f32_16x16x4_f32.
//
// Semantics are those of the reference composite (core/inference.cpp:123-161
// over backends/cpu/cpu_inference.cpp:22-47): a score is dot(q, k) * scale
// (rounded) plus the additive mask (rounded); a key after the query under
// causal, a false entry of a bool mask or a -inf entry of an additive one is
// -inf; a row with any NaN score is NaN, a row whose maximum is -inf is 0 * V,
// otherwise exp(s - max) / sum, times V. The sums run in a different order
// (online softmax over key tiles), inside the reference test's
// allclose(rtol=2e-4, atol=2e-5).
//
// Two kernels share the work: flash_attention_kernel, below, with matrix
// instructions for 16 queries a wave, and flash_decode_kernel for up to four
// queries, which only streams K and V. Where either has too few blocks for the
// GPU, the keys are split over blocks and flash_combine_kernel joins the parts.
//
// Layout. A block owns 16 queries per wave of one batch matrix and walks the
// keys in tiles of kKeys (64, or 32 where two blocks must share a CU). K and V
// tiles go straight from HBM into LDS (buffer_load ... lds) and each tile's
// softmax overlaps the next tile's score MFMAs (details at the kernel). Each
// wave computes S^T = K Q^T for its 16 queries, so lane l holds
// S^T[key 16b + 4(l/16) + v][query l%16] (output layout of the MFMA): those
// are exactly the A operands (P[query l%16][key]) that the P V MFMAs need,
// when the k index of step (b, v) is taken as key 16b + 4(l/16) + v. The
// feature sum of S^T uses the same trick: lane l supplies features
// 16t + 4(l/16) + e of K and Q at step (t, e), read as one float4 each.
// Masked keys keep p = 0, so a non-finite V propagates as in the reference's
// P @ V: tiles the causal mask only partly covers run in full; a tile wholly
// after the block's last query skips the MFMAs and only marks the feature
// columns where its V rows hold a non-finite value (0 * inf or 0 * NaN is NaN
// in every output row of the block). Blocks start with the longest query
// tiles under causal masking.

#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace tcx {
namespace {

using mfma_acc = float __attribute__((ext_vector_type(4)));

struct FlashArgs {
  const float* q;
  const float* k;
  const float* v;
  float* out;
  std::int64_t rows, cols;
  std::int64_t features;       // of a row; the kernels' D where they are not padded
  std::int64_t qtiles, batch;  // work items: qtiles query tiles of each batch matrix
  std::int64_t first_batch;    // of this launch, in the whole call (for the mask)
  float scale;
  int causal;
  int xcd_blocks;   // group the blocks of one batch matrix on one XCD
  int heavy_first;  // causal: more blocks than fit at once, heaviest first
  // Mask: element (batch b, query i, key j) at b's offset + i mask_row + j mask_col.
  const void* mask;
  int mask_kind;  // TCX_MASK_*
  int mask_rank;
  std::int64_t mask_shape[TCX_HIP_MAX_RANK], mask_stride[TCX_HIP_MAX_RANK];
  std::int64_t mask_row, mask_col;
  // Key split: split s of a work item takes split_keys keys from s split_keys
  // (a multiple of the kernel's key tile); with splits > 1 its unnormalised
  // outputs and its maxima and sums go to part and part_ml.
  std::int64_t splits, split_keys;
  float* part;     // [splits, batch, rows, features]
  float* part_ml;  // [splits, batch, rows, 2]
};

// Offset of batch matrix b in the mask (its leading axes, row-major).
__device__ __forceinline__ std::int64_t mask_offset(const FlashArgs& a, std::int64_t b) {
  std::int64_t offset = 0;
  b += a.first_batch;
  for (int i = a.mask_rank - 1; i >= 0; --i) {
    offset += b % a.mask_shape[i] * a.mask_stride[i];
    b /= a.mask_shape[i];
  }
  return offset;
}

// The score under mask element `at`: + bias, or -inf where it is hidden.
__device__ __forceinline__ float masked_score(float score, const FlashArgs& a, std::int64_t at) {
  if (a.mask_kind == TCX_MASK_BOOL) return static_cast<const std::uint8_t*>(a.mask)[at] ? score : -__builtin_inff();
  const float bias = static_cast<const float*>(a.mask)[at];
  return bias == -__builtin_inff() ? bias : score + bias;
}

// The row length. Padded kernels (kPad) take any multiple of four features up
// to D (the entries offer multiples of eight): rows keep their own length in memory and are D features long in LDS and
// registers, where the features past the last are zero.
template <int D, bool kPad>
__device__ __forceinline__ std::int64_t row_features(const FlashArgs& a) {
  if constexpr (kPad) return a.features;
  else return D;
}

using float2_t = float __attribute__((ext_vector_type(2)));

// N contiguous floats (N = 2, 4 or 8) with 8- or 16-byte stores.
template <int N>
__device__ __forceinline__ void store_row(float* p, const float (&v)[N]) {
  if constexpr (N % 4 == 0) {
#pragma unroll
    for (int t = 0; t < N; t += 4)
      *reinterpret_cast<float4_t*>(p + t) = float4_t{v[t], v[t + 1], v[t + 2], v[t + 3]};
  } else {
    static_assert(N == 2);
    *reinterpret_cast<float2_t*>(p) = float2_t{v[0], v[1]};
  }
}

// exp(x) for x <= 0 (or NaN) as exp2(x log2 e): rounding the product costs at
// most |t| 2^-24 ln 2 relative on a term exp(-t), 1e-6 for the terms above
// 2^-24 of the largest, far inside the reference's rtol 2e-4.
__device__ __forceinline__ float exp_attention(float x) {
  constexpr float kLog2e = 1.44269502F;  // float(log2 e)
  return __builtin_amdgcn_exp2f(x * kLog2e);
}

// K/V tiles are loaded straight into LDS (buffer_load ... lds) and the loop
// is pipelined so that matrix cores stay busy through the softmax: while the
// scores of key tile j go through the softmax (VALU), the same wave's MFMAs
// already compute the scores of tile j + 1. K therefore runs
// one tile ahead of V: iteration j reads K tile j + 1 and V tile j, and loads
// K tile j + 2 and V tile j + 1 into the other halves of two-stage buffers,
// with one barrier per tile. Rows are unpadded and their 16-byte chunks
// XOR-swizzled by row (period 16), which keeps the K reads (16 rows, one
// chunk each) and the V reads (16 chunks of one row) conflict-free. Keys past
// the sequence read as zero (buffer range check).
template <int D>
__device__ __forceinline__ int kv_chunk(int row, int c) {
  if constexpr (D / 4 >= 16) return c ^ (row & 15);
  else return c ^ ((row >> 1) & 7);
}

// Output tile t of lane r holds feature output_feature(r, t): four
// consecutive features per 16-byte chunk, chunk r of each 64-feature half
// (features kT r + t for D = 32).
template <int kT>
__device__ __forceinline__ int output_feature(int r, int t) {
  if constexpr (kT >= 4) return 64 * (t / 4) + 4 * r + (t % 4);
  else return kT * r + t;
}

// Online-softmax state of a wave's 16 queries: the output accumulators in
// MFMA layout and the running maximum and sum (the lanes of query j hold its
// m and l).
template <int kT>
struct FlashState {
  mfma_acc o[kT];
  float m, l;
};

template <int kT>
__device__ __forceinline__ void flash_init(FlashState<kT>& st) {
#pragma unroll
  for (int t = 0; t < kT; ++t) st.o[t] = mfma_acc{0.F, 0.F, 0.F, 0.F};
  st.m = -__builtin_inff();
  st.l = 0.F;
}

// Key tiles [t_begin, t_end) of query tile `qtile` of batch matrix `batch`,
// folded into the state of the calling wave's 16 queries by the block's
// kWaves waves (thread tid) on two K and two V stages. kKeys keys per tile
// (64, or 32 to fit two blocks per CU), kB = kKeys / 16 MFMA blocks of keys.
// The segment opens with a barrier, so a segment may follow another on the same
// stages.
//
// kMask (TCX_MASK_*): lane (r, g) needs the mask entries of its query at keys
// 16b + 4g + v, 4 kB words a tile. They are loaded a tile ahead, behind the
// tile's DMA and ahead of the wait that ends the iteration: a load whose value
// is used in its own iteration would wait for the DMA issued before it.
template <int D, int kWaves, int kKeys, bool kCausal, int kMask, bool kPad>
__device__ __forceinline__ void flash_segment(const FlashArgs& a, float (&ks)[2][kKeys * D],
                                              float (&vs)[2][kKeys * D], int tid, std::int64_t batch,
                                              std::int64_t qtile, std::int64_t t_begin, std::int64_t t_end,
                                              FlashState<D / 16>& st) {
  constexpr int kQTile = 16 * kWaves;
  constexpr int kT = D / 16;
  constexpr int kB = kKeys / 16;
  constexpr bool kExact = kPad || kMask != TCX_MASK_NONE;
  static_assert(kKeys == 32 || kKeys == 64);
  constexpr int kChunks = D / 4;                         // 16-byte chunks per K/V row
  constexpr int kRowsPerInst = 64 / kChunks;             // rows one wave instruction fills
  constexpr int kInst = kKeys / kRowsPerInst / kWaves;   // instructions per wave per K (or V) tile
  static_assert(D % 16 == 0 && kInst >= 1 && kInst * kRowsPerInst * kWaves == kKeys);
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const std::int64_t q0 = qtile * kQTile + wave * 16;
  const std::int64_t features = row_features<D, kPad>(a);
  const float* __restrict__ qb = a.q + batch * a.rows * features;
  const float* __restrict__ kb = a.k + batch * a.cols * features;
  const float* __restrict__ vb = a.v + batch * a.cols * features;

  float4_t qf[kT];
  {
    const std::int64_t qrow = q0 + r;
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      // Unconditional loads (a row past the end reads row 0, then zero):
      // loads under a divergent branch would make the compiler wait for
      // every outstanding load inside the key loop.
      const std::int64_t qc = qrow < a.rows ? qrow : 0;
      const int f = 16 * t + 4 * g;
      const bool past = kPad && f >= features;
      qf[t] = *reinterpret_cast<const float4_t*>(qb + qc * features + (past ? 0 : f));
      if (qrow >= a.rows || past) qf[t] = float4_t{0.F, 0.F, 0.F, 0.F};
    }
  }
  mfma_acc (&o)[kT] = st.o;
  // Masked and padded kernels sum in shorter chains and take expf, so that
  // their error against 64 bits is no larger than that of the two products and
  // the softmax of the unfused route (with one chain it was up to twice that;
  // now 0.70 of it in the mean over 16 to 128 features and 5 to 2048 keys, for
  // these kernels at most 0.97): the scores in eight accumulators, four at D =
  // 32 (step (t, e) in number 4t + e), and P V of a tile apart, its steps in
  // two by turns (tile_o).
  constexpr int kParts = !kExact ? 1 : D >= 64 ? 8 : 4;
  mfma_acc s_part[kParts][kB];
  auto clear_parts = [&] {
#pragma unroll
    for (int e = 0; e < kParts; ++e)
#pragma unroll
      for (int b = 0; b < kB; ++b) s_part[e][b] = mfma_acc{0.F, 0.F, 0.F, 0.F};
  };
  auto join_parts = [&](mfma_acc (&s)[kB]) {
#pragma unroll
    for (int b = 0; b < kB; ++b) {
#pragma unroll
      for (int n = kParts / 2; n > 0; n /= 2)
#pragma unroll
        for (int e = 0; e < n; ++e) s_part[e][b] += s_part[e + n][b];
      s[b] = s_part[0][b];
    }
  };
  float& m = st.m;
  float& l = st.l;
  const float neg_inf = -__builtin_inff();
  const std::int64_t query = q0 + r;

  // DMA. Each tile is read through a buffer resource based at the tile's
  // first key row (64-bit address), whose num_records covers the keys left in
  // the sequence (at most one tile), so keys past the end read as zero and no
  // offset exceeds one tile. Instruction p of a wave fills rows
  // (p * kWaves + wave) * kRowsPerInst .. + kRowsPerInst - 1 of the tile;
  // lane i writes chunk slot i % kChunks of row i / kChunks, which holds
  // global chunk kv_chunk(row, slot).
  using int4v = int __attribute__((ext_vector_type(4)));
  auto rsrc_at = [&](const float* base, std::int64_t tile) {
    const std::int64_t j0 = tile * kKeys;
    const std::int64_t left = a.cols - j0;  // > 0 for every issued tile
    const int bytes = static_cast<int>((left < kKeys ? left : kKeys) * (features * 4));
    const auto addr = reinterpret_cast<std::uint64_t>(base + j0 * features);
    return int4v{static_cast<int>(addr), static_cast<int>(addr >> 32), bytes, 0x00020000};
  };
  int voff[kInst];
#pragma unroll
  for (int p = 0; p < kInst; ++p) {
    const int row = (p * kWaves + wave) * kRowsPerInst + lane / kChunks;
    const int f = 4 * kv_chunk<D>(row, lane % kChunks);
    // Past the last feature an offset beyond every tile, which reads as zero.
    voff[p] = kPad && f >= features ? 0x40000000 : (row * static_cast<int>(features) + f) * 4;
  }
  auto lds_of = [](const void* ptr) {
    return static_cast<unsigned>(reinterpret_cast<std::uintptr_t>((__attribute__((address_space(3))) const void*)ptr));
  };
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  auto dma16 = [](const int4v& rsrc, unsigned lds_byte, int off, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(lds_byte), "v"(off), "s"(rsrc), "s"(soff) : "memory", "m0");
  };
#pragma clang diagnostic pop
  auto issue = [&](const float* base, float* stage, std::int64_t tile) {
    const int4v rsrc = rsrc_at(base, tile);
#pragma unroll
    for (int p = 0; p < kInst; ++p) {
      const unsigned row_byte = static_cast<unsigned>((p * kWaves + wave) * kRowsPerInst * D * 4);
      dma16(rsrc, lds_of(stage) + row_byte, voff[p], 0);
    }
  };

  // Lane exchanges: xor 16 inside each half-wave (swizzle, bit-mask mode:
  // and 0x1f, xor 0x10), xor 32 and the broadcast of query 4g + v's factor
  // to lane group g through precomputed permute addresses.
  auto xor16 = [](float x) { return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(x), 0x401f)); };
  const int xor32_addr = (lane ^ 32) << 2;
  auto xor32 = [&](float x) { return __int_as_float(__builtin_amdgcn_ds_bpermute(xor32_addr, __float_as_int(x))); };
  int row_addr[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) row_addr[v] = (4 * g + v) << 2;

  // Fragment reads. K: the kB 16-key blocks of feature group t (lane (r, g)
  // reads chunk 4t + g of key 16b + r). V: key row 16b + 4g + v, features
  // output_feature(r, t): chunks r, 16 + r, ... (half of chunk r / 2 for
  // D = 32), so the 16 lanes of a row read 16 different chunks.
  auto read_k = [&](const float* __restrict__ kt_, int t, float4_t (&kf)[kB]) {
#pragma unroll
    for (int b = 0; b < kB; ++b) {
      const int row = 16 * b + r;
      kf[b] = *reinterpret_cast<const float4_t*>(&kt_[row * D + 4 * kv_chunk<D>(row, 4 * t + g)]);
    }
  };
  auto read_v = [&](const float* __restrict__ vt_, int step, float (&vv)[kT]) {
    const int row = 16 * (step / 4) + 4 * g + step % 4;
    if constexpr (kT >= 4) {
#pragma unroll
      for (int h = 0; h < kT / 4; ++h) {
        const float4_t w = *reinterpret_cast<const float4_t*>(&vt_[row * D + 4 * kv_chunk<D>(row, 16 * h + r)]);
        vv[4 * h] = w.x; vv[4 * h + 1] = w.y; vv[4 * h + 2] = w.z; vv[4 * h + 3] = w.w;
      }
    } else {
      const float2_t w =
          *reinterpret_cast<const float2_t*>(&vt_[row * D + 4 * kv_chunk<D>(row, r / 2) + 2 * (r % 2)]);
      vv[0] = w.x; vv[1] = w.y;
    }
  };

  // The online softmax of one tile as kSteps small steps, so that they can be
  // spread between the MFMAs of the next tile's scores (kB = 4 numbering):
  //   0-3       scale (and mask) of key block b, running tile maximum
  //   4         row maximum over the four lane groups, new running maximum,
  //             rescale factor alpha
  //   5         alpha of query 4g + v to lane group g
  //   6..5+kT   rescale output tile t
  //   6+kT..9+kT  p = exp(s - max) of key block b, partial row sum
  //   10+kT     row sum over the lane groups, l and m updated
  // Every key so far masked (m_new = -inf): the finite stand-in m_sub keeps
  // p = exp(-inf) = 0 without a per-score select, and alpha = 0 leaves the
  // zero rows zero (or NaN). A NaN score is skipped by fmaxf but gives p = NaN,
  // so l and the whole row turn NaN; so does a +inf score (inf - inf).
  constexpr int kSteps = 2 * kB + 3 + kT;
  float tmax = neg_inf, m_new = neg_inf, m_sub = 0.F, alpha = 1.F, psum = 0.F;
  float av[4];
  int limit = kKeys;
  using mask_word = std::conditional_t<kMask == TCX_MASK_BOOL, std::uint8_t, float>;
  mask_word mk[kMask == TCX_MASK_NONE ? 1 : 4 * kB], mk_next[kMask == TCX_MASK_NONE ? 1 : 4 * kB];
  const mask_word* __restrict__ mrow = nullptr;
  if constexpr (kMask != TCX_MASK_NONE)
    mrow = static_cast<const mask_word*>(a.mask) + mask_offset(a, batch) + min(query, a.rows - 1) * a.mask_row;
  // Keys past the sequence read the last one's entry; the limit hides them.
  auto load_mask = [&](std::int64_t tile, mask_word (&to)[kMask == TCX_MASK_NONE ? 1 : 4 * kB]) {
    if constexpr (kMask != TCX_MASK_NONE) {
      const std::int64_t j0 = tile * kKeys;
      if (j0 + kKeys <= a.cols) {
        const mask_word* __restrict__ p = mrow + (j0 + 4 * g) * a.mask_col;
#pragma unroll
        for (int b = 0; b < kB; ++b)
#pragma unroll
          for (int v = 0; v < 4; ++v) to[4 * b + v] = p[(16 * b + v) * a.mask_col];
      } else {
#pragma unroll
        for (int b = 0; b < kB; ++b)
#pragma unroll
          for (int v = 0; v < 4; ++v) to[4 * b + v] = mrow[min(j0 + 16 * b + 4 * g + v, a.cols - 1) * a.mask_col];
      }
    }
  };
  auto begin_tile = [&](std::int64_t tile) {
    const std::int64_t j0 = tile * kKeys;
    std::int64_t lim = a.cols - j0;
    if constexpr (kCausal) {
      if (query - j0 + 1 < lim) lim = query - j0 + 1;
    }
    limit = static_cast<int>(lim < 0 ? 0 : (lim > kKeys ? kKeys : lim));
    tmax = neg_inf;
    psum = 0.F;
  };
  // kLimit: the tile may hold keys past the sequence or after the query.
  auto step = [&]<int I, bool kLimit>(mfma_acc (&s)[kB]) {
    if constexpr (I < kB) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float sc = s[I][v] * a.scale;
        if constexpr (kMask == TCX_MASK_BOOL) {
          sc = mk[4 * I + v] != 0 ? sc : neg_inf;
        } else if constexpr (kMask == TCX_MASK_ADDITIVE) {
          sc = mk[4 * I + v] == neg_inf ? neg_inf : sc + mk[4 * I + v];
        }
        if constexpr (kLimit) {
          if (16 * I + 4 * g + v >= limit) sc = neg_inf;
        }
        s[I][v] = sc;
        tmax = fmaxf(tmax, sc);
      }
    } else if constexpr (I == kB) {
      tmax = fmaxf(tmax, xor16(tmax));
      tmax = fmaxf(tmax, xor32(tmax));
      m_new = fmaxf(m, tmax);
      m_sub = m_new == neg_inf ? 0.F : m_new;
      alpha = kExact ? expf(m - m_sub) : exp_attention(m - m_sub);
    } else if constexpr (I == kB + 1) {
#pragma unroll
      for (int v = 0; v < 4; ++v)
        av[v] = __int_as_float(__builtin_amdgcn_ds_bpermute(row_addr[v], __float_as_int(alpha)));
    } else if constexpr (I < kB + 2 + kT) {
#pragma unroll
      for (int v = 0; v < 4; ++v) o[I - kB - 2][v] *= av[v];
    } else if constexpr (I < 2 * kB + 2 + kT) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float x = s[I - kB - 2 - kT][v] - m_sub;
        const float p = kExact ? expf(x) : exp_attention(x);
        s[I - kB - 2 - kT][v] = p;
        psum += p;
      }
    } else {
      psum += xor16(psum);
      psum += xor32(psum);
      l = l * alpha + psum;
      m = m_new;
    }
  };
  auto all_steps = [&]<int... I>(mfma_acc (&s)[kB], std::integer_sequence<int, I...>) {
    (step.template operator()<I, true>(s), ...);
  };

  // O += P V in 4 kB steps (key 16b + 4g + v of lane group g at step 4b + v),
  // each reading the next step's V operands before its own MFMAs.
  auto accumulate = [&]<int... I>(const float* __restrict__ vt_, const mfma_acc (&p)[kB], float (&vv)[2][kT],
                                  std::integer_sequence<int, I...>) {
    mfma_acc tile_o[2][kExact ? kT : 1];
    if constexpr (kExact) {
#pragma unroll
      for (int t = 0; t < kT; ++t) tile_o[0][t] = tile_o[1][t] = mfma_acc{0.F, 0.F, 0.F, 0.F};
    }
    auto one = [&]<int J>() {
      if constexpr (J + 1 < 4 * kB) read_v(vt_, J + 1, vv[(J + 1) & 1]);
#pragma unroll
      for (int t = 0; t < kT; ++t) {
        mfma_acc& to = kExact ? tile_o[J & 1][kExact ? t : 0] : o[t];
        to = __builtin_amdgcn_mfma_f32_16x16x4f32(p[J / 4][J % 4], vv[J & 1][t], to, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    (one.template operator()<I>(), ...);
    if constexpr (kExact) {
#pragma unroll
      for (int t = 0; t < kT; ++t) o[t] += tile_o[0][t] + tile_o[1][t];
    }
  };

  // The next tile's scores in kQuads = kT kB quads of four MFMAs (feature
  // group t = J / kB, k steps 4 / kB (J % kB) .. + 4 / kB - 1, every key
  // block), with softmax step I of the current tile in quad I kQuads / kSteps
  // and the K reads of group t + 1 in the first quad of group t; the last quad
  // also reads the first P V step's V operands.
  constexpr int kQuads = kT * kB;
  auto scores_with_softmax = [&]<bool kLimit, int... Q>(const float* __restrict__ kt_, const float* __restrict__ vt_,
                                                       mfma_acc (&s_next)[kB], mfma_acc (&s)[kB],
                                                       float4_t (&kf)[2][kB], float (&vv)[2][kT],
                                                       std::bool_constant<kLimit>, std::integer_sequence<int, Q...>) {
    auto quad = [&]<int J>() {
      constexpr int t = J / kB, e0 = (J % kB) * (4 / kB);
      if constexpr (J % kB == 0 && t + 1 < kT) read_k(kt_, t + 1, kf[(t + 1) & 1]);
      if constexpr (J == kQuads - 1) read_v(vt_, 0, vv[0]);
#pragma unroll
      for (int e = e0; e < e0 + 4 / kB; ++e)
#pragma unroll
        for (int b = 0; b < kB; ++b) {
          mfma_acc& s_to = kExact ? s_part[(4 * t + e) % kParts][b] : s_next[b];
          s_to = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t & 1][b][e], qf[t][e], s_to, 0, 0, 0);
        }
      [&]<int... I>(std::integer_sequence<int, I...>) {
        ([&] {
          if constexpr (I * kQuads / kSteps == J) step.template operator()<I, kLimit>(s);
        }(), ...);
      }(std::make_integer_sequence<int, kSteps>{});
      __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (kExact) clear_parts();
    (quad.template operator()<Q>(), ...);
    if constexpr (kExact) join_parts(s_next);
  };
  // Scores of one tile without interleaving (first tile).
  auto scores = [&](const float* __restrict__ kt_, mfma_acc (&s)[kB]) {
#pragma unroll
    for (int b = 0; b < kB; ++b) s[b] = mfma_acc{0.F, 0.F, 0.F, 0.F};
    if constexpr (kExact) clear_parts();
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      float4_t kf[kB];
      read_k(kt_, t, kf);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int b = 0; b < kB; ++b) {
          mfma_acc& s_to = kExact ? s_part[(4 * t + e) % kParts][b] : s[b];
          s_to = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[b][e], qf[t][e], s_to, 0, 0, 0);
        }
    }
    if constexpr (kExact) join_parts(s);
  };

  // Every tile but the last of the segment is full unless masked causally.
  mfma_acc s_cur[kB], s_next[kB];
  float4_t kf[2][kB];
  float vv[2][kT];
  // The stages may still be read by this team's previous segment.
  __syncthreads();
  if (t_begin < t_end) {
    issue(kb, ks[0], t_begin);
    issue(vb, vs[0], t_begin);
    if (t_begin + 1 < t_end) issue(kb, ks[1], t_begin + 1);
    load_mask(t_begin, mk);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // K 0, V 0 and K 1 have landed
    scores(ks[0], s_cur);
    __syncthreads();  // every wave is done with K stage 0
  } else {
    __syncthreads();
  }
  // Iteration `tile` (stage parity counted from t_begin): K tile + 1 sits in
  // stage (tile + 1) & 1, V tile in stage tile & 1; K tile + 2 and V tile + 1
  // load into the other stages, whose last readers finished before the
  // previous barrier.
  std::int64_t tile = t_begin;
  for (; tile + 1 < t_end; ++tile) {
    const int st = static_cast<int>((tile - t_begin) & 1);
    issue(vb, vs[st ^ 1], tile + 1);
    if (tile + 2 < t_end) issue(kb, ks[st], tile + 2);
    load_mask(tile + 1, mk_next);
    begin_tile(tile);
#pragma unroll
    for (int b = 0; b < kB; ++b) s_next[b] = mfma_acc{0.F, 0.F, 0.F, 0.F};
    read_k(ks[st ^ 1], 0, kf[0]);
    // Under causal masking only tiles reaching past the block's first query
    // need the mask: a wave-uniform branch between two schedules at D = 128
    // (+2 %). At D = 64 the second schedule raised the register count from
    // 127 to 157, which costs a block per CU (-18 %), so D < 128 masks all, as do
    // the masked and padded kernels, whose registers would spill.
    if (kCausal && (D < 128 || kExact || (tile + 1) * kKeys - 1 > qtile * kQTile))
      scores_with_softmax(ks[st ^ 1], vs[st], s_next, s_cur, kf, vv, std::true_type{},
                          std::make_integer_sequence<int, kQuads>{});
    else
      scores_with_softmax(ks[st ^ 1], vs[st], s_next, s_cur, kf, vv, std::false_type{},
                          std::make_integer_sequence<int, kQuads>{});
    accumulate(vs[st], s_cur, vv, std::make_integer_sequence<int, 4 * kB>{});
#pragma unroll
    for (int b = 0; b < kB; ++b) s_cur[b] = s_next[b];
    __builtin_amdgcn_s_waitcnt(0);  // this wave's loads have landed
    if constexpr (kMask != TCX_MASK_NONE) {
#pragma unroll
      for (int e = 0; e < 4 * kB; ++e) mk[e] = mk_next[e];
    }
    __syncthreads();                // and every wave is done with this iteration's stages
  }
  if (tile < t_end) {
    const int st = static_cast<int>((tile - t_begin) & 1);
    begin_tile(tile);
    all_steps(s_cur, std::make_integer_sequence<int, kSteps>{});
    read_v(vs[st], 0, vv[0]);
    accumulate(vs[st], s_cur, vv, std::make_integer_sequence<int, 4 * kB>{});
  }
}

// Marks in bad_column the feature columns of V rows [row, end) that hold an inf
// or NaN (exponent all ones), eight independent loads in flight per thread and
// no branch in the loop (a branch on each load's value serialised the scan
// behind the load latency: 10 % of the causal kernel at D = 32).
template <int D, int kWaves, bool kPad>
__device__ __forceinline__ void scan_values(const FlashArgs& a, const float* __restrict__ vb, std::int64_t row,
                                            std::int64_t end, int* bad_column, int tid) {
  const std::int64_t features = row_features<D, kPad>(a);
  const int c = (tid % (D / 4)) * 4;
  if (kPad && c >= features) return;
  constexpr int kPass = (64 * kWaves) / (D / 4);  // rows per pass of the block
  constexpr unsigned kExp = 0x7f800000U;
  unsigned flag[4] = {0U, 0U, 0U, 0U};
  auto mark = [&](const float4_t& w) {
#pragma unroll
    for (int e = 0; e < 4; ++e) flag[e] |= (__float_as_uint(w[e]) & kExp) == kExp ? 1U : 0U;
  };
  row += tid / (D / 4);
  for (; row + 7 * kPass < end; row += 8 * kPass) {
    float4_t w[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) w[u] = *reinterpret_cast<const float4_t*>(vb + (row + u * kPass) * features + c);
#pragma unroll
    for (int u = 0; u < 8; ++u) mark(w[u]);
  }
  for (; row < end; row += kPass) mark(*reinterpret_cast<const float4_t*>(vb + row * features + c));
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (flag[e]) bad_column[c + e] = 1;
}

// The first key that a mask shared by all queries of batch matrix `batch`
// (mask_row 0) leaves visible and the one after the last; [0, 0) for none.
template <int kWaves, int kMask>
__device__ __forceinline__ void visible_keys(const FlashArgs& a, std::int64_t batch, int tid, std::int64_t& first,
                                             std::int64_t& end) {
  using mask_word = std::conditional_t<kMask == TCX_MASK_BOOL, std::uint8_t, float>;
  __shared__ long long ends[2][kWaves];
  const mask_word* __restrict__ mask = static_cast<const mask_word*>(a.mask) + mask_offset(a, batch);
  long long low = a.cols, high = 0;
  for (std::int64_t j = tid; j < a.cols; j += 64 * kWaves) {
    const mask_word w = mask[j * a.mask_col];
    const bool visible = kMask == TCX_MASK_BOOL ? w != 0 : !(w == -__builtin_inff());
    if (visible) {
      low = min(low, static_cast<long long>(j));
      high = static_cast<long long>(j) + 1;
    }
  }
#pragma unroll
  for (int offset = 32; offset > 0; offset >>= 1) {
    low = min(low, __shfl_xor(low, offset, kWave));
    high = max(high, __shfl_xor(high, offset, kWave));
  }
  if ((tid & 63) == 0) {
    ends[0][tid >> 6] = low;
    ends[1][tid >> 6] = high;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    low = min(low, ends[0][w]);
    high = max(high, ends[1][w]);
  }
  // The same in every lane: into scalar registers, as the key tiles' buffer
  // resources are.
  auto uniform = [](long long v) {
    const auto low32 = static_cast<std::uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
    return static_cast<std::int64_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v >> 32))) << 32 | low32;
  };
  end = uniform(high);
  first = end > 0 ? uniform(low) : 0;
}

// Stores the calling wave's 16 output rows of query tile `qtile` from its
// state (NaN in the columns bad_column marks, 0 * V for an all-masked row), or,
// of one split of the keys, the state itself.
template <int D, int kWaves, bool kPad>
__device__ __forceinline__ void flash_store(const FlashArgs& a, const int* bad_column, int tid, std::int64_t batch,
                                            std::int64_t qtile, std::int64_t split, const FlashState<D / 16>& st) {
  constexpr int kT = D / 16;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const std::int64_t q0 = qtile * (16 * kWaves) + wave * 16;
  const float neg_inf = -__builtin_inff();
  const bool parts = a.splits > 1;
  const std::int64_t first = (split * a.batch + batch) * a.rows;  // this split's row 0 of the batch matrix
  const std::int64_t features = row_features<D, kPad>(a);
  float* __restrict__ ob = parts ? a.part + first * features : a.out + batch * a.rows * features;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int src = 4 * g + v;
    const float lv = __shfl(st.l, src, kWave);
    const float mv = __shfl(st.m, src, kWave);
    const std::int64_t qrow = q0 + 4 * g + v;
    if (qrow >= a.rows) continue;
    // A split's outputs by the same code, over 1: a third way out of each of
    // the divisions below cost a call on 64 x 64 x 128 a microsecond of 12.
    const float over = parts ? 1.F : lv;
    const bool hidden = !parts && mv == neg_inf;
    float y[kT];
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      if (bad_column[output_feature<kT>(r, t)]) y[t] = __builtin_nanf("");
      else if (hidden) y[t] = st.o[t][v] * 0.F;
      else y[t] = st.o[t][v] / over;
    }
    if (parts && r == 0) *reinterpret_cast<float2_t*>(a.part_ml + (first + qrow) * 2) = float2_t{mv, lv};
    float* const orow = ob + qrow * features;
    if constexpr (kT >= 4) {
#pragma unroll
      for (int h = 0; h < kT / 4; ++h)
        if (!kPad || output_feature<kT>(r, 4 * h) < features)
          *reinterpret_cast<float4_t*>(orow + output_feature<kT>(r, 4 * h)) =
              float4_t{y[4 * h], y[4 * h + 1], y[4 * h + 2], y[4 * h + 3]};
    } else if (!kPad || kT * r < features) {
      store_row<kT>(orow + kT * r, y);
    }
  }
}

// One block per query tile and split of the keys.
template <int D, int kWaves, int kKeys, bool kCausal, int kMask, bool kPad>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(kWaves == 1 ? 1 : 2, 8))) void
flash_attention_kernel(FlashArgs a) {
  constexpr int kQTile = 16 * kWaves;
  __shared__ float ks[2][kKeys * D];
  __shared__ float vs[2][kKeys * D];
  __shared__ int bad_column[D];
  const int tid = threadIdx.x;
  // One block per work item on a 1-D grid of n = qtiles x batch blocks; the
  // launch id maps to an item (batch-major by default).
  // The arithmetic is in 32 bits, as a grid's size is: a block of one key tile
  // waits for each 64-bit division about as long as for its loads.
  const auto qtiles = static_cast<std::uint32_t>(a.qtiles), batches = static_cast<std::uint32_t>(a.batch);
  const std::uint32_t n = qtiles * batches;
  const std::uint32_t split = a.splits > 1 ? blockIdx.x / n : 0, id = blockIdx.x - split * n;
  std::uint32_t item_batch = id / qtiles, item_tile = id - item_batch * qtiles;
  if (a.xcd_blocks) {
    // Launch id L runs on XCD L % 8: give XCD x the consecutive (batch-major)
    // work items x * n/8 .. (x + 1) * n/8 - 1, so that the query tiles of one
    // batch matrix share its K and V in that XCD's L2 (n % 8 == 0).
    const std::uint32_t item = (id % 8) * (n / 8) + id / 8;
    item_batch = item / qtiles;
    item_tile = item - item_batch * qtiles;
    if (kMask != TCX_MASK_NONE && batches % 8 == 0) {
      // Masks can make one sequence of a batch much shorter than another, so
      // the XCDs take its matrices in turns: matrix b on XCD b % 8.
      item_batch = id % 8 + 8 * (id / 8 / qtiles);
      item_tile = id / 8 % qtiles;
    }
  }
  if constexpr (kCausal) {
    // Under causal masking the last query tiles see the most keys. Work items
    // are ranked by their key-tile count. When every block fits on the device
    // at once, the first half of the grid takes them heaviest first and the
    // second half lightest first, so the two blocks that share a CU (launch
    // ids L and L + n/2) carry about the same total work. With more blocks
    // than fit, the grid runs heaviest first throughout, so that the light
    // items fill the CUs the heavy ones leave (longest job first: 16 x 4096 x
    // 128 720 -> 658 us, 48 x 2048 x 128 536 -> 482 us on MI355X).
    const std::uint32_t half = (n + 1) / 2;
    const std::uint32_t rank = a.heavy_first || id < half ? id : n - 1 - (id - half);
    item_tile = qtiles - 1 - rank / batches;
    item_batch = rank % batches;
  }
  const std::int64_t batch = item_batch, qtile = item_tile;
  const std::int64_t q_last = min(qtile * kQTile + kQTile, a.rows) - 1;
  const std::int64_t tiles = (a.cols + kKeys - 1) / kKeys;
  // Key tiles [first, run): under causal masking tiles past the block's last
  // query are not run, and with a mask shared by all queries (the padding of a
  // batch) neither are tiles in front of its first visible key or after its
  // last: their p would be 0 and leave the state as it is, but for V rows that
  // are not finite, which are looked for instead. A call on 4 x 16 heads x 512 x
  // 64 with 1/4 to all of the keys visible: 72 -> 59 us with the matrices of one
  // sequence spread over the XCDs (no faster with them on one or two), before
  // the shorter chains of flash_segment, with which it takes 73.
  std::int64_t first = 0, run = kCausal ? min(tiles, q_last / kKeys + 1) : tiles;
  if constexpr (kMask != TCX_MASK_NONE) {
    if (a.mask_row == 0) {
      std::int64_t key = 0, end = 0;
      visible_keys<kWaves, kMask>(a, batch, tid, key, end);
      run = min(run, (end + kKeys - 1) / kKeys);
      first = min(key / kKeys, run);
    }
  }
  const std::int64_t per = a.split_keys / kKeys;
  const std::int64_t t_begin = min(first + split * per, run), t_end = min(t_begin + per, run);
  for (int d = tid; d < D; d += 64 * kWaves) bad_column[d] = 0;
  FlashState<D / 16> st;
  flash_init(st);
  flash_segment<D, kWaves, kKeys, kCausal, kMask, kPad>(a, ks, vs, tid, batch, qtile, t_begin, t_end, st);
  if (split == a.splits - 1) {
    const float* __restrict__ vb = a.v + batch * a.cols * row_features<D, kPad>(a);
    if (kMask != TCX_MASK_NONE && first > 0) scan_values<D, kWaves, kPad>(a, vb, 0, first * kKeys, bad_column, tid);
    if (run < tiles) scan_values<D, kWaves, kPad>(a, vb, run * kKeys, a.cols, bad_column, tid);
  }
  __syncthreads();
  flash_store<D, kWaves, kPad>(a, bad_column, tid, batch, qtile, split, st);
}

// Sum over the kLanes lanes (8 or 16) of a group, in every lane of it.
template <int kLanes>
__device__ __forceinline__ float group_sum(float x) {
  auto add = [&]<int kControl>() {
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kControl, 0xf, 0xf, true));
  };
  add.template operator()<0xb1>();   // lane ^ 1
  add.template operator()<0x4e>();   // lane ^ 2
  add.template operator()<0x141>();  // mirror in eight lanes
  if constexpr (kLanes == 16) add.template operator()<0x140>();  // mirror in sixteen
  return x;
}

// Joins the online-softmax state (m, l and N outputs) of two disjoint sets of keys.
template <int N>
__device__ __forceinline__ void join_state(float& m, float& l, float (&o)[N], float m2, float l2, const float (&o2)[N]) {
  const float top = fmaxf(m, m2);
  const float at = top == -__builtin_inff() ? 0.F : top;
  const float f = expf(m - at), f2 = expf(m2 - at);
  m = top;
  l = l * f + l2 * f2;
#pragma unroll
  for (int e = 0; e < N; ++e) o[e] = o[e] * f + o2[e] * f2;
}

// Attention of kRows queries (the last ones may repeat) over split_keys keys
// of one batch matrix, not causal: decoding, where a K and a V row are used
// once and the time is that of reading them. A group of lanes takes a key and
// each lane kC 16-byte chunks of its rows; kEach keys a group and pass, so that
// 16 loads a lane are in flight. Every group keeps an online softmax of its own
// (no exchange between groups in the loop); the groups are joined at the end.
// The exponentials are expf here, as in the unfused route: the loop is bound by
// memory, and the sums are as short as to keep the error below that route's too.
// 32 heads of one query and 4096 keys, D = 128 (134 MB): 21.8 us (6.2
// TB/s) and 4.0 for the combine, against 537 us for one block of flash_attention_kernel
// per head.
template <int D, int kRows, bool kPad>
__global__ __launch_bounds__(256) void flash_decode_kernel(FlashArgs a) {
  constexpr int kLanes = D >= 64 ? 16 : 8;
  constexpr int kC = D / 4 / kLanes;
  constexpr int kEach = 8 / kC;
  constexpr int kPerWave = 64 / kLanes;
  constexpr int kGroups = 4 * kPerWave;
  constexpr int kPass = kGroups * kEach;
  __shared__ float part_o[4][kRows][D];
  __shared__ float part_m[4][kRows], part_l[4][kRows];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int li = lane % kLanes, group = wave * kPerWave + lane / kLanes;
  const std::int64_t batch = blockIdx.x / a.splits, split = blockIdx.x % a.splits;
  const std::int64_t k0 = split * a.split_keys, k1 = min(k0 + a.split_keys, a.cols);
  const float neg_inf = -__builtin_inff();
  const std::int64_t features = row_features<D, kPad>(a);
  const float* __restrict__ kb = a.k + batch * a.cols * features;
  const float* __restrict__ vb = a.v + batch * a.cols * features;
  // Feature of this lane's chunk c. Chunks past the last read chunk 0 and
  // count as zero (their V is not stored).
  auto past = [&](int c) { return kPad && 4 * (c * kLanes + li) >= features; };
  auto at_chunk = [&](int c) { return past(c) ? 0 : 4 * (c * kLanes + li); };
  const std::int64_t mask0 = a.mask_kind != TCX_MASK_NONE ? mask_offset(a, batch) : 0;
  float4_t q[kRows][kC];
  float o[kRows][4 * kC], m[kRows], l[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    const std::int64_t row = min(static_cast<std::int64_t>(r), a.rows - 1);
#pragma unroll
    for (int c = 0; c < kC; ++c) {
      q[r][c] = *reinterpret_cast<const float4_t*>(a.q + (batch * a.rows + row) * features + at_chunk(c));
      if (past(c)) q[r][c] = float4_t{0.F, 0.F, 0.F, 0.F};
    }
#pragma unroll
    for (int e = 0; e < 4 * kC; ++e) o[r][e] = 0.F;
    m[r] = neg_inf;
    l[r] = 0.F;
  }
  auto pass = [&]<bool kTail>(std::int64_t j, std::bool_constant<kTail>) {
    float4_t kf[kEach][kC], vf[kEach][kC];
    std::int64_t key[kEach];
#pragma unroll
    for (int u = 0; u < kEach; ++u) {
      key[u] = j + u * kGroups + group;
      const std::int64_t at = kTail ? min(key[u], k1 - 1) : key[u];
#pragma unroll
      for (int c = 0; c < kC; ++c) {
        kf[u][c] = stream_load(reinterpret_cast<const float4_t*>(kb + at * features + at_chunk(c)));
        if (past(c)) kf[u][c] = float4_t{0.F, 0.F, 0.F, 0.F};
      }
    }
#pragma unroll
    for (int u = 0; u < kEach; ++u) {
      const std::int64_t at = kTail ? min(key[u], k1 - 1) : key[u];
#pragma unroll
      for (int c = 0; c < kC; ++c) {
        vf[u][c] = stream_load(reinterpret_cast<const float4_t*>(vb + at * features + at_chunk(c)));
        if (kTail && key[u] >= k1) vf[u][c] = float4_t{0.F, 0.F, 0.F, 0.F};
      }
    }
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      float s[kEach], top = m[r];
#pragma unroll
      for (int u = 0; u < kEach; ++u) {
        float dot = 0.F;
#pragma unroll
        for (int c = 0; c < kC; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) dot = fmaf(q[r][c][e], kf[u][c][e], dot);
        s[u] = group_sum<kLanes>(dot) * a.scale;
        if (a.mask_kind != TCX_MASK_NONE)
          s[u] = masked_score(s[u], a, mask0 + min(static_cast<std::int64_t>(r), a.rows - 1) * a.mask_row +
                                           min(key[u], a.cols - 1) * a.mask_col);
        if (kTail && key[u] >= k1) s[u] = neg_inf;
        top = fmaxf(top, s[u]);
      }
      const float at = top == neg_inf ? 0.F : top;  // as in flash_segment: every key so far hidden
      const float f = expf(m[r] - at);
      m[r] = top;
      l[r] *= f;
#pragma unroll
      for (int e = 0; e < 4 * kC; ++e) o[r][e] *= f;
#pragma unroll
      for (int u = 0; u < kEach; ++u) {
        const float p = expf(s[u] - at);
        l[r] += p;
#pragma unroll
        for (int c = 0; c < kC; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) o[r][4 * c + e] = fmaf(p, vf[u][c][e], o[r][4 * c + e]);
      }
    }
  };
  std::int64_t j = k0;
  for (; j + kPass <= k1; j += kPass) pass(j, std::false_type{});
  if (j < k1) pass(j, std::true_type{});
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
#pragma unroll
    for (int offset = kLanes; offset < 64; offset <<= 1) {
      float o2[4 * kC];
      const float m2 = __shfl_xor(m[r], offset, kWave), l2 = __shfl_xor(l[r], offset, kWave);
#pragma unroll
      for (int e = 0; e < 4 * kC; ++e) o2[e] = __shfl_xor(o[r][e], offset, kWave);
      join_state(m[r], l[r], o[r], m2, l2, o2);
    }
    if (lane < kLanes) {
#pragma unroll
      for (int c = 0; c < kC; ++c)
        *reinterpret_cast<float4_t*>(&part_o[wave][r][4 * (c * kLanes + li)]) =
            float4_t{o[r][4 * c], o[r][4 * c + 1], o[r][4 * c + 2], o[r][4 * c + 3]};
      if (lane == 0) {
        part_m[wave][r] = m[r];
        part_l[wave][r] = l[r];
      }
    }
  }
  __syncthreads();
  const std::int64_t first = (split * a.batch + batch) * a.rows;
  for (int i = t; i < kRows * D; i += 256) {
    const int r = i / D, d = i % D;
    if (r >= a.rows) break;
    if (kPad && d >= features) continue;
    float mv = part_m[0][r], lv = part_l[0][r], ov[1] = {part_o[0][r][d]};
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      const float o2[1] = {part_o[w][r][d]};
      join_state(mv, lv, ov, part_m[w][r], part_l[w][r], o2);
    }
    if (a.splits > 1) {
      a.part[(first + r) * features + d] = ov[0];
      if (d == 0) *reinterpret_cast<float2_t*>(a.part_ml + (first + r) * 2) = float2_t{mv, lv};
    } else {
      a.out[(batch * a.rows + r) * features + d] = mv == neg_inf ? ov[0] * 0.F : ov[0] / lv;
    }
  }
}

// Joins the splits of every output row, one wave a row (splits <= 64: lane s
// holds the maximum and the sum of split s), in the order of the splits.
template <int D, bool kPad>
__global__ __launch_bounds__(256) void flash_combine_kernel(FlashArgs a) {
  constexpr int kE = D >= 64 ? D / 64 : 1;
  const int lane = threadIdx.x & 63;
  const std::int64_t rows = a.batch * a.rows, features = row_features<D, kPad>(a);
  const std::int64_t step = static_cast<std::int64_t>(gridDim.x) * 4;
  const int splits = static_cast<int>(a.splits);
  const float neg_inf = -__builtin_inff();
  for (std::int64_t row = static_cast<std::int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6); row < rows; row += step) {
    float2_t ml{neg_inf, 0.F};
    if (lane < splits) ml = *reinterpret_cast<const float2_t*>(a.part_ml + (lane * rows + row) * 2);
    float top = ml.x;
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) top = fmaxf(top, __shfl_xor(top, offset, kWave));
    const float at = top == neg_inf ? 0.F : top;
    const float weight = expf(ml.x - at);
    const float sum = wave_sum(ml.y * weight);
    const int d = lane * kE;
    float y[kE] = {};
    if (d < features) {
      const float* __restrict__ p = a.part + row * features + d;
      auto add = [&]<int kN>(int s, std::integral_constant<int, kN>) {  // splits s .. s + kN - 1
        float v[kN][kE];
#pragma unroll
        for (int u = 0; u < kN; ++u)
#pragma unroll
          for (int e = 0; e < kE; ++e) v[u][e] = p[(s + u) * rows * features + e];
#pragma unroll
        for (int u = 0; u < kN; ++u) {
          const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(weight), s + u));
#pragma unroll
          for (int e = 0; e < kE; ++e) y[e] += w * v[u][e];
        }
      };
      int s = 0;
      for (; s + 8 <= splits; s += 8) add(s, std::integral_constant<int, 8>{});
      for (; s < splits; ++s) add(s, std::integral_constant<int, 1>{});
#pragma unroll
      for (int e = 0; e < kE; ++e) a.out[row * features + d + e] = top == neg_inf ? y[e] * 0.F : y[e] / sum;
    }
  }
}

// How one call runs: the kernel and its split of the keys.
struct FlashPlan {
  bool decode;      // flash_decode_kernel
  int waves, keys;  // of flash_attention_kernel
  std::int64_t splits, split_keys;
  std::size_t bytes;  // of the workspace that holds the splits' states
};

std::int64_t ceil_div(std::int64_t a, std::int64_t b) { return (a + b - 1) / b; }

constexpr std::int64_t kDecodeRows = 4;
constexpr std::int64_t kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64};  // flash_combine_kernel: a lane each

// A form of flash_attention_kernel and what a key tile costs in it, in
// microseconds of one CU: in a block that has the CU to itself, and for each
// block where two and where more share it.
struct FlashForm {
  int waves, keys;
  double alone, two, shared;
  int resident;  // blocks a CU holds
};

// What the workspace of a split costs the call, in microseconds: nothing where
// the caller has it, and a mapping of memory where it is allocated for the call
// and no pool has blocks to give (2.5 us below 2 MiB, 25 from there on).
double workspace_cost(std::size_t bytes, bool per_call) {
  if (!per_call || bytes == 0 || allocation_cached(bytes)) return 0.0;
  return bytes < (std::size_t{2} << 20) ? 2.5 : 25.0;
}

std::size_t split_bytes(std::int64_t splits, std::int64_t batch, std::int64_t rows, std::int64_t features) {
  return splits > 1 ? static_cast<std::size_t>(splits * batch * rows) * (features + 2) * sizeof(float) : 0;
}

// What a plan may use: a workspace of at most `bytes`, allocated for the one
// call or not.
struct FlashLimit {
  std::size_t bytes;
  bool per_call;
};

// The split of the keys that is expected to end first, with its time in
// microseconds. A block's time is its tiles on the busiest of 256 CUs and 4 us
// of start and end a round; a split call also runs the combine (4 us and the
// states written and read at 4 TB/s) and may have to map its workspace. Under
// causal masking almost half of the parts of a split are empty. For 1603 whole
// calls (1 to 1024 matrices, 8 to 2048 queries, 64 to 2048 keys, every form) nine
// in ten took 0.88 to 1.5 times what this says, half of them 0.97 to 1.14, and 95
// in 100 picks of a form were within 1 % of the fastest; a split has to promise
// 8 %. `cols` are the keys that the last query sees.
double best_split(const FlashForm& f, std::int64_t batch, std::int64_t rows, std::int64_t cols, std::int64_t features,
                  bool causal, FlashLimit limit, std::int64_t& splits) {
  const std::int64_t items = ceil_div(rows, 16 * f.waves) * batch, tiles = std::max<std::int64_t>(ceil_div(cols, f.keys), 1);
  double best = 0;
  splits = 1;
  for (const std::int64_t n : kSplits) {
    const std::size_t bytes = split_bytes(n, batch, rows, features);
    if (n > 1 && (n > tiles || items * n > 2048 || bytes > limit.bytes)) break;
    const std::int64_t per = ceil_div(tiles, n);
    if (n > 1 && ceil_div(tiles, per) != n) continue;  // another count cuts the tiles the same way
    const double blocks = static_cast<double>(causal && n > 1 ? items * (n + 1) : items * n) * (causal && n > 1 ? 0.6 : 1.0);
    const std::int64_t on_cu = ceil_div(static_cast<std::int64_t>(blocks), 256);
    double time = static_cast<double>(per) * (on_cu > 2 ? static_cast<double>(on_cu) * f.shared : on_cu > 1 ? 2 * f.two : f.alone);
    if (causal && n == 1 && on_cu > 1)  // the light blocks fill in beside the heavy ones
      time = std::max(static_cast<double>(per) * f.alone, 0.5 * time);
    time += 4.0 * static_cast<double>(ceil_div(on_cu, f.resident));
    if (n > 1) time += 4.0 + static_cast<double>(n * batch * rows * features) * 2e-6 + workspace_cost(bytes, limit.per_call);
    if (n == 1) best = time;
    else if (time < 0.92 * best) best = time, splits = n;
  }
  return best;
}

FlashPlan flash_plan(std::int64_t batch, std::int64_t rows, std::int64_t cols, std::int64_t features, bool causal,
                     int mask_kind, FlashLimit limit) {
  FlashPlan p{};
  const bool mostly_hidden = causal && cols > 2 * rows;
  if (causal) cols = std::min(cols, rows);  // the keys after the last query are not run
  // Decoding streams the keys; plain calls of 32 features have too few of them
  // for that up to 64, or 128 where more queries share them (their states cost
  // more to join than a tile: 1500 x 4 x 16 x 32 25 us, 8.6 in tiles).
  const bool few_keys = features == 32 && mask_kind == TCX_MASK_NONE && cols <= (rows == 1 ? 64 : 128);
  if (rows <= kDecodeRows && !causal && cols > 0 && !few_keys) {
    // Up to 256 blocks of at least 128 keys (8 splits of 32 x 4096 x 128 24.1
    // us, 32 splits 25.2, one 91.4); short sequences whole, since the combine
    // costs more than it brings (16 x 300 x 64 6.6 us, 8.2 in two).
    p.decode = true;
    std::int64_t splits = 1;
    for (const std::int64_t n : kSplits)
      if (n * batch <= 256 && n * 128 <= cols && cols >= 512 && split_bytes(n, batch, rows, features) <= limit.bytes)
        splits = n;
    p.split_keys = ceil_div(ceil_div(cols, splits), 64) * 64;
    p.splits = ceil_div(cols, p.split_keys);
  } else {
    // Tile shapes measured on MI355X. Four waves and 32-key tiles in general:
    // at D = 128 64 KB of LDS, so that two blocks share a CU, under causal
    // masking a heavy and a light one (89 TFLOP/s at 16 x 2048 x 128 against
    // 86 for a register-staged 4-wave kernel, 92 against 71 at 32 x 2048 x 64).
    // At D = 32 and 64 also 64-key tiles, with half the barriers and softmax
    // chains and half the blocks a CU: 0.83 to 0.9 of the time where a CU has one
    // block (8 x 1024 x 64 52 -> 46 us), 0.93 to 0.95 with two, 0.97 (D = 32) and
    // 1.03 (D = 64; causal 1.1) with more (512 x 512 x 64 294 against 314), times
    // what the last tile adds (200 keys: 256 for 224). Where most keys lie behind
    // the causal mask, 32-key tiles: 128 x 200 x 8000 at D = 32 64 us against 69.
    // Unmasked at D = 128 eight waves and 64-key tiles, one block per CU,
    // where there are enough (16 x 2048 281 against 291 us). Up to 16 queries
    // one wave holds them all where blocks share a CU: 60 us against 81 for 512
    // matrices of 16 queries and 512 keys at D = 128 (alone 35.5 against 33.4 for
    // 1000 keys at D = 32).
    static constexpr FlashForm kFour[] = {
        {4, 32, 1.0, 0.76, 0.76, 5}, {4, 32, 1.53, 1.27, 1.27, 4}, {4, 32, 2.65, 2.27, 2.27, 2}};
    static constexpr FlashForm kLong[] = {{4, 64, 1.66, 1.42, 1.49, 5}, {4, 64, 2.71, 2.41, 2.64, 4}};
    static constexpr FlashForm kOne[] = {
        {1, 32, 1.06, 0.4, 0.4, 8}, {1, 32, 1.7, 0.6, 0.6, 4}, {1, 32, 2.85, 1.9, 1.9, 2}};
    static constexpr FlashForm kEight128{8, 64, 8.7, 8.7, 8.7, 1};
    // Masked and padded kernels have the general form only, and are planned by
    // the plain kernels' costs: theirs are 1.1 to 2 times as much a tile, with two
    // or three blocks a CU, but with constants of their own 657 calls took the
    // same time in the mean (0.77 to 1.23 of it).
    const int d = features > 64 ? 2 : features > 32 ? 1 : 0;
    const bool padded = features != 32 << d, plain = !padded && !causal && mask_kind == TCX_MASK_NONE;
    FlashForm form = kFour[d];
    double time = best_split(form, batch, rows, cols, features, causal, limit, p.splits);
    auto consider = [&](const FlashForm& other) {
      std::int64_t splits;
      const double t = best_split(other, batch, rows, cols, features, causal, limit, splits);
      if (t >= time) return;
      time = t;
      form = other;
      p.splits = splits;
    };
    if (plain && rows <= 16) consider(kOne[d]);
    if (!padded && mask_kind == TCX_MASK_NONE && features <= 64 && form.waves == 4 && !mostly_hidden &&
        (!causal || ceil_div(rows, 64) * batch < 1024))
      consider(kLong[d]);
    if (d == 2 && plain && rows > 64) consider(kEight128);
    p.waves = form.waves;
    p.keys = form.keys;
    p.split_keys = std::max<std::int64_t>(ceil_div(ceil_div(cols, p.keys), p.splits), 1) * p.keys;
    p.splits = std::max<std::int64_t>(ceil_div(cols, p.split_keys), 1);
  }
  p.bytes = split_bytes(p.splits, batch, rows, features);
  return p;
}

template <int D, int kWaves, int kKeys, bool kCausal, int kMask, bool kPad = false>
int launch_flash(FlashArgs a, hipStream_t s) {
  constexpr int kQTile = 16 * kWaves;
  a.qtiles = ceil_div(a.rows, kQTile);
  const std::int64_t items = a.qtiles * a.batch;
  const std::int64_t blocks = items * a.splits;
  // Causal blocks keep their heavy/light order instead.
  a.xcd_blocks = !kCausal && items % 8 == 0 ? 1 : 0;
  if constexpr (kCausal) {
    thread_local int slots = 0;
    if (slots == 0) {
      int per_cu = 0, cus = 0, device = 0;
      (void)hipGetDevice(&device);
      if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < 1)
        cus = 256;
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
              &per_cu, flash_attention_kernel<D, kWaves, kKeys, kCausal, kMask, kPad>, 64 * kWaves, 0) != hipSuccess ||
          per_cu < 1)
        per_cu = 2;
      slots = per_cu * cus;
    }
    a.heavy_first = blocks > slots ? 1 : 0;
  }
  hipLaunchKernelGGL((flash_attention_kernel<D, kWaves, kKeys, kCausal, kMask, kPad>),
                     dim3(static_cast<unsigned>(blocks)), dim3(64 * kWaves), 0, s, a);
  return check(hipGetLastError(), "flash attention launch");
}

template <int D, bool kPad>
int launch_decode(const FlashArgs& a, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(a.batch * a.splits));
  if (a.rows == 1) hipLaunchKernelGGL((flash_decode_kernel<D, 1, kPad>), grid, dim3(256), 0, s, a);
  else if (a.rows == 2) hipLaunchKernelGGL((flash_decode_kernel<D, 2, kPad>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((flash_decode_kernel<D, 4, kPad>), grid, dim3(256), 0, s, a);
  return check(hipGetLastError(), "decode attention launch");
}

template <int D, bool kCausal, int kMask, bool kPad>
int launch_tiles(const FlashArgs& a, const FlashPlan& p, hipStream_t s) {
  constexpr bool kPlain = !kPad && !kCausal && kMask == TCX_MASK_NONE;
  if constexpr (kPlain) {
    if (p.waves == 1) return launch_flash<D, 1, 32, false, TCX_MASK_NONE>(a, s);
  }
  if constexpr (kPlain && D == 128) {
    if (p.waves == 8) return launch_flash<D, 8, 64, false, TCX_MASK_NONE>(a, s);
  }
  if constexpr (!kPad && kMask == TCX_MASK_NONE && D <= 64) {
    if (p.keys == 64) return launch_flash<D, 4, 64, kCausal, kMask>(a, s);
  }
  return launch_flash<D, 4, 32, kCausal, kMask, kPad>(a, s);
}

template <int D, bool kCausal, bool kPad>
int launch_mask_kind(const FlashArgs& a, const FlashPlan& p, hipStream_t s) {
  if (a.mask_kind == TCX_MASK_BOOL) return launch_tiles<D, kCausal, TCX_MASK_BOOL, kPad>(a, p, s);
  if (a.mask_kind == TCX_MASK_ADDITIVE) return launch_tiles<D, kCausal, TCX_MASK_ADDITIVE, kPad>(a, p, s);
  return launch_tiles<D, kCausal, TCX_MASK_NONE, kPad>(a, p, s);
}

template <int D, bool kPad>
int launch_features(const FlashArgs& a, const FlashPlan& p, hipStream_t s) {
  const int rc = p.decode   ? launch_decode<D, kPad>(a, s)
                 : a.causal ? launch_mask_kind<D, true, kPad>(a, p, s)
                            : launch_mask_kind<D, false, kPad>(a, p, s);
  if (rc != TCX_OK || a.splits == 1) return rc;
  hipLaunchKernelGGL((flash_combine_kernel<D, kPad>), dim3(grid_for(a.batch * a.rows, 4, kStrideBlocks)), dim3(256), 0, s, a);
  return check(hipGetLastError(), "attention combine launch");
}

}  // namespace
}  // namespace tcx

extern "C" {

int tcx_hip_flash_attention_supported(int64_t features, int64_t value_features) {
  return features == value_features && (features == 32 || features == 64 || features == 128) ? 1 : 0;
}

int tcx_hip_flash_attention_ws_supported(int64_t features, int64_t value_features) {
  // Multiples of 8 from 16: there the padded kernels' error against 64 bits was
  // at most 0.99 of the unfused route's for 5 to 2048 keys (mean 0.80); at 8
  // features 1.05. 16 x 300 x 80 97 -> 70 us, 32 x 512 x 80 causal 404 -> 100,
  // 64 x 1024 x 80 1330 -> 375, one query of 32 x 2000 x 80 80 -> 28 (calls).
  return features == value_features && features >= 16 && features <= 128 && features % 8 == 0 ? 1 : 0;
}

int tcx_hip_flash_attention_plan(const tcx_hip_flash_attention_desc_t* desc, size_t workspace_bytes, int per_call,
                                 tcx_hip_flash_attention_plan_t* plan) {
  using namespace tcx;
  if (desc == nullptr || plan == nullptr) return fail(TCX_INVALID_ARGUMENT, "attention plan or descriptor is null");
  if (desc->batch <= 0 || desc->rows <= 0 || desc->cols < 0 ||
      !tcx_hip_flash_attention_ws_supported(desc->features, desc->features))
    return fail(TCX_INVALID_ARGUMENT, "no fused attention for these extents");
  const FlashPlan p = flash_plan(desc->batch, desc->rows, desc->cols, desc->features, desc->causal != 0,
                                 desc->mask_kind, {workspace_bytes, per_call != 0});
  *plan = {p.decode ? 1 : 0, p.decode ? 4 : p.waves, p.keys, static_cast<std::int32_t>(p.splits), p.bytes};
  return TCX_OK;
}

size_t tcx_hip_flash_attention_workspace_bytes(const tcx_hip_flash_attention_desc_t* desc) {
  tcx_hip_flash_attention_plan_t plan{};
  return tcx_hip_flash_attention_plan(desc, SIZE_MAX, 0, &plan) == TCX_OK ? plan.workspace_bytes : 0;
}

int tcx_hip_flash_attention_f32_ws(const float* q, const float* k, const float* v, float* out, const void* mask,
                                   const tcx_hip_flash_attention_desc_t* desc, void* workspace,
                                   size_t workspace_bytes, tcx_stream_t stream) {
  using namespace tcx;
  if (desc == nullptr) return fail(TCX_INVALID_ARGUMENT, "attention descriptor is null");
  const auto& d = *desc;
  if (d.batch < 0 || d.rows < 0 || d.cols < 0) return fail(TCX_INVALID_ARGUMENT, "attention extents must be non-negative");
  if (!tcx_hip_flash_attention_ws_supported(d.features, d.features))
    return fail(TCX_INVALID_ARGUMENT, "fused attention supports multiples of 8 features from 16 to 128");
  if (d.mask_kind < TCX_MASK_NONE || d.mask_kind > TCX_MASK_ADDITIVE)
    return fail(TCX_INVALID_ARGUMENT, "unknown attention mask kind");
  if (d.batch == 0 || d.rows == 0) return TCX_OK;
  const bool masked = d.mask_kind != TCX_MASK_NONE && d.cols > 0;
  if (q == nullptr || out == nullptr || (d.cols > 0 && (k == nullptr || v == nullptr)) || (masked && mask == nullptr))
    return fail(TCX_INVALID_ARGUMENT, "attention buffers are null");
  for (const void* p : {static_cast<const void*>(q), static_cast<const void*>(k), static_cast<const void*>(v),
                        static_cast<const void*>(out)})
    if (p != nullptr && (reinterpret_cast<std::uintptr_t>(p) & 15U) != 0)
      return fail(TCX_INVALID_ARGUMENT, "fused attention buffers must be 16-byte aligned");
  FlashArgs a{};
  if (masked) {
    if (d.mask_rank < 0 || d.mask_rank > TCX_HIP_MAX_RANK)
      return fail(TCX_INVALID_ARGUMENT, "attention mask rank must be in [0, 8]");
    std::int64_t count = 1;
    for (int i = 0; i < d.mask_rank; ++i) {
      if (d.mask_shape[i] < 1) return fail(TCX_INVALID_ARGUMENT, "attention mask extents must be positive");
      a.mask_shape[i] = d.mask_shape[i];
      a.mask_stride[i] = d.mask_strides[i];
      count *= d.mask_shape[i];
    }
    if (count != d.batch) return fail(TCX_INVALID_ARGUMENT, "attention mask axes must multiply to the batch");
    a.mask = mask;
    a.mask_kind = d.mask_kind;
    a.mask_rank = d.mask_rank;
    a.mask_row = d.mask_row_stride;
    a.mask_col = d.mask_col_stride;
  }
  if (int rc = ready(); rc != TCX_OK) return rc;
  // The best plan that the workspace has room for.
  const bool usable = workspace != nullptr && (reinterpret_cast<std::uintptr_t>(workspace) & 15U) == 0;
  const FlashPlan p = flash_plan(d.batch, d.rows, d.cols, d.features, d.causal != 0, a.mask_kind,
                                 {usable ? workspace_bytes : 0, false});
  // Blocks of one batch matrix, and as many matrices a launch as HIP counts work-items for.
  const std::int64_t blocks = (p.decode ? 1 : ceil_div(d.rows, 16 * p.waves)) * p.splits;
  const std::int64_t per_launch = kMaxLaunchWorkItems / (p.decode ? 256 : 64 * p.waves) / blocks;
  if (per_launch == 0) return fail(TCX_INVALID_ARGUMENT, "attention grid is too large");
  a.rows = d.rows;
  a.cols = d.cols;
  a.features = d.features;
  a.scale = d.scale;
  a.causal = d.causal != 0;
  a.splits = p.splits;
  a.split_keys = p.split_keys;
  if (p.splits > 1) {
    a.part = static_cast<float*>(workspace);
    a.part_ml = a.part + p.splits * d.batch * d.rows * d.features;
  }
  const auto s = static_cast<hipStream_t>(stream);
  auto launch = [&] {
    if (d.features == 32) return launch_features<32, false>(a, p, s);
    if (d.features == 64) return launch_features<64, false>(a, p, s);
    if (d.features == 128) return launch_features<128, false>(a, p, s);
    if (d.features < 32) return launch_features<32, true>(a, p, s);
    if (d.features < 64) return launch_features<64, true>(a, p, s);
    return launch_features<128, true>(a, p, s);
  };
  // (Splits have few matrices: their states are not cut.)
  for (std::int64_t first = 0; first < d.batch; first += per_launch) {
    a.first_batch = first;
    a.batch = std::min(per_launch, d.batch - first);
    a.q = q + first * d.rows * d.features;
    a.k = k + first * d.cols * d.features;
    a.v = v + first * d.cols * d.features;
    a.out = out + first * d.rows * d.features;
    if (int rc = launch(); rc != TCX_OK) return rc;
  }
  return TCX_OK;
}

int tcx_hip_flash_attention_f32(const float* q, const float* k, const float* v, float* out, int64_t batch,
                                int64_t rows, int64_t cols, int64_t features, float scale, int causal,
                                tcx_stream_t stream) {
  if (batch >= 0 && rows >= 0 && cols >= 0 && !tcx_hip_flash_attention_supported(features, features))
    return tcx::fail(TCX_INVALID_ARGUMENT, "fused attention supports 32, 64 or 128 features");
  tcx_hip_flash_attention_desc_t d{};
  d.batch = batch;
  d.rows = rows;
  d.cols = cols;
  d.features = features;
  d.scale = scale;
  d.causal = causal != 0;
  d.mask_kind = TCX_MASK_NONE;
  return tcx_hip_flash_attention_f32_ws(q, k, v, out, nullptr, &d, nullptr, 0, stream);
}

}  // extern "C"
