// Embedding gather and attention softmax: the native primitives under the
// reference's inference composites (backends/cpu/cpu_inference.cpp:10-47,
// plans in core/inference.cpp:47-84).
//
//   embedding_kernel        row gather, copied bit for bit, that flags any index
//                           outside [0, vocabulary)
//   attention_softmax_kernel one wave per score row: masked / causal / scaled
//                           scores, NaN-first maximum, all-masked rows -> 0,
//                           exp(s - max) / sum (tree-order sum, expf)

#include <algorithm>

#include "common.hpp"

namespace tcx {
namespace {

// Every writer stores the same value.
__device__ __forceinline__ void flag_bad(std::int32_t* flag) {
  __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The check alone, for a width of 0.
__global__ __launch_bounds__(256) void embedding_check_kernel(const std::int32_t* __restrict__ indices,
                                                              std::int64_t count, std::int64_t vocabulary,
                                                              std::int32_t* __restrict__ flag) {
  const std::int64_t stride = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
  for (std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += stride) {
    const std::int32_t id = indices[i];
    if (id < 0 || id >= vocabulary) flag_bad(flag);
  }
}

// Rows of `width` units T (16 bytes, or one word), checked and copied in one
// pass: a block takes up to 256 units of a row (blockIdx.x), or several narrow
// rows, and strides over the rows, so that no index is divided; where the grid
// is too short for a row (2^28 units), it strides over the columns as well. A
// thread takes kEach rows at a time, their loads ahead of their stores: four
// where there are enough of them (a call on 10^6 rows of 36 floats 50 us with
// one, 32 with four). Out-of-range rows are never read.
template <typename T, int kEach>
__global__ __launch_bounds__(256) void embedding_kernel(const std::int32_t* __restrict__ indices,
                                                        const T* __restrict__ weight, T* __restrict__ out,
                                                        std::int64_t count, std::int64_t vocabulary, std::int64_t width,
                                                        int lanes, int per_block, std::int32_t* __restrict__ flag) {
  const int sub = threadIdx.x / lanes;
  if (sub >= per_block) return;
  const std::int64_t first = static_cast<std::int64_t>(blockIdx.x) * lanes + threadIdx.x % lanes;
  const std::int64_t column_step = static_cast<std::int64_t>(gridDim.x) * lanes;
  const std::int64_t row_step = static_cast<std::int64_t>(gridDim.y) * per_block;
  for (std::int64_t i = static_cast<std::int64_t>(blockIdx.y) * per_block + sub; i < count; i += kEach * row_step) {
    std::int32_t id[kEach];
    bool in[kEach];
#pragma unroll
    for (int u = 0; u < kEach; ++u) id[u] = indices[std::min(i + u * row_step, count - 1)];
#pragma unroll
    for (int u = 0; u < kEach; ++u) {
      in[u] = id[u] >= 0 && id[u] < vocabulary;
      if (!in[u]) flag_bad(flag);
    }
    for (std::int64_t c = first; c < width; c += column_step) {
      T v[kEach];
#pragma unroll
      for (int u = 0; u < kEach; ++u) {
        v[u] = T{};
        if (in[u]) v[u] = weight[id[u] * width + c];
      }
#pragma unroll
      for (int u = 0; u < kEach; ++u)
        if (i + u * row_step < count) out[(i + u * row_step) * width + c] = v[u];
    }
  }
}

template <typename T>
void launch_embedding(const std::int32_t* indices, const float* weight, float* out, std::int64_t count,
                      std::int64_t vocabulary, std::int64_t width, std::int32_t* flag, hipStream_t s) {
  const int lanes = static_cast<int>(std::min<std::int64_t>(width, 256)), per_block = 256 / lanes;
  const unsigned gx = grid_for(width, lanes, 1 << 20);
  auto go = [&](auto kernel, int each) {
    const unsigned gy =
        grid_for(count, per_block * each, std::min<std::int64_t>(65535, std::max<std::int64_t>(1, (1 << 20) / gx)));
    hipLaunchKernelGGL(kernel, dim3(gx, gy), dim3(256), 0, s, indices, reinterpret_cast<const T*>(weight),
                       reinterpret_cast<T*>(out), count, vocabulary, width, lanes, per_block, flag);
  };
  // Four rows a thread from 2048 blocks of them on.
  if (grid_for(count, 4 * per_block) * gx >= 2048) go(embedding_kernel<T, 4>, 4);
  else go(embedding_kernel<T, 1>, 1);
}

// The same by words where rows have no 16-byte units: a flat index over the
// output, so that stores are whole lines wherever the rows start (10^6 rows of
// 129 words 407 us by rows, 33 words 103).
template <int kEach>
__global__ __launch_bounds__(256) void embedding_words_kernel(const std::int32_t* __restrict__ indices,
                                                              const std::uint32_t* __restrict__ weight,
                                                              std::uint32_t* __restrict__ out, std::uint32_t n,
                                                              std::int64_t vocabulary, FastDiv width,
                                                              std::int32_t* __restrict__ flag) {
  const std::uint32_t first = blockIdx.x * (256U * kEach) + threadIdx.x;
  std::uint32_t column[kEach], v[kEach];
  std::int32_t id[kEach];
#pragma unroll
  for (int u = 0; u < kEach; ++u) {
    const std::uint32_t e = min(first + 256U * u, n - 1), i = width(e);
    column[u] = e - i * width.divisor;
    id[u] = indices[i];
  }
#pragma unroll
  for (int u = 0; u < kEach; ++u) {
    const bool in = id[u] >= 0 && id[u] < vocabulary;
    if (!in) flag_bad(flag);
    v[u] = 0;
    if (in) v[u] = weight[static_cast<std::int64_t>(id[u]) * width.divisor + column[u]];
  }
#pragma unroll
  for (int u = 0; u < kEach; ++u)
    if (first + 256U * u < n) out[first + 256U * u] = v[u];
}

void launch_embedding_words(const std::int32_t* indices, const float* weight, float* out, std::int64_t count,
                            std::int64_t vocabulary, std::int64_t width, std::int32_t* flag, hipStream_t s) {
  const std::int64_t n = count * width;
  auto go = [&](auto kernel, int each) {
    hipLaunchKernelGGL(kernel, dim3(grid_for(n, 256 * each, 1 << 23)), dim3(256), 0, s, indices,
                       reinterpret_cast<const std::uint32_t*>(weight), reinterpret_cast<std::uint32_t*>(out),
                       static_cast<std::uint32_t>(n), vocabulary, FastDiv(static_cast<std::uint32_t>(width)), flag);
  };
  if (n >= 256 * 1024) go(embedding_words_kernel<4>, 4);
  else go(embedding_words_kernel<1>, 1);
}

struct SoftmaxMeta {
  std::int64_t shape[TCX_HIP_MAX_RANK];
  std::int64_t s[TCX_HIP_MAX_RANK];
  std::int64_t m[TCX_HIP_MAX_RANK];
  std::int32_t rank;
  std::int32_t mask_kind;
  std::int32_t causal;
  float scale;
};

__device__ __forceinline__ float attention_score(const float* __restrict__ scores, const void* __restrict__ mask,
                                                 const SoftmaxMeta& d, std::int64_t sbase, std::int64_t mbase,
                                                 std::int64_t ss, std::int64_t ms, std::int64_t col,
                                                 std::int64_t query) {
  const float neg_inf = -__builtin_inff();
  if (d.causal && col > query) return neg_inf;
  if (d.mask_kind == TCX_MASK_BOOL && !static_cast<const std::uint8_t*>(mask)[mbase + col * ms]) return neg_inf;
  const float bias = d.mask_kind == TCX_MASK_ADDITIVE ? static_cast<const float*>(mask)[mbase + col * ms] : 0.F;
  if (bias == neg_inf) return bias;
  const float product = scores[sbase + col * ss] * d.scale;
  return product + bias;
}

__global__ __launch_bounds__(256) void attention_softmax_kernel(const float* __restrict__ scores,
                                                                const void* __restrict__ mask,
                                                                float* __restrict__ out, SoftmaxMeta d,
                                                                std::int64_t rows) {
  const int lane = threadIdx.x & 63;
  const int r = d.rank;
  const std::int64_t columns = d.shape[r - 1], queries = d.shape[r - 2];
  const std::int64_t ss = d.s[r - 1], ms = d.m[r - 1];
  const std::int64_t step = static_cast<std::int64_t>(gridDim.x) * 4;
  for (std::int64_t row = static_cast<std::int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6); row < rows; row += step) {
    std::int64_t flat = row, sbase = 0, mbase = 0;
    for (int a = r - 2; a >= 0; --a) {
      const std::int64_t c = flat % d.shape[a];
      flat /= d.shape[a];
      sbase += c * d.s[a];
      mbase += c * d.m[a];
    }
    const std::int64_t query = row % queries;
    float m = -__builtin_inff();
    bool nan = false;
    for (std::int64_t col = lane; col < columns; col += 64) {
      const float v = attention_score(scores, mask, d, sbase, mbase, ss, ms, col, query);
      if (is_nan(v)) nan = true;
      else m = v > m ? v : m;
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) m = fmaxf(m, __shfl_xor(m, offset, kWave));
    if (__any(nan)) m = __builtin_nanf("");
    float* o = out + row * columns;
    if (m == -__builtin_inff()) {
      for (std::int64_t col = lane; col < columns; col += 64) o[col] = 0.F;
      continue;
    }
    float total = 0.F;
    for (std::int64_t col = lane; col < columns; col += 64)
      total += expf(attention_score(scores, mask, d, sbase, mbase, ss, ms, col, query) - m);
    total = wave_sum(total);
    for (std::int64_t col = lane; col < columns; col += 64)
      o[col] = expf(attention_score(scores, mask, d, sbase, mbase, ss, ms, col, query) - m) / total;
  }
}

}  // namespace
}  // namespace tcx

extern "C" {

int tcx_hip_embedding_f32(const int32_t* indices, const float* weight, float* out, int64_t count,
                          int64_t vocabulary, int64_t width, int32_t* flag, tcx_stream_t stream) {
  using namespace tcx;
  if (count < 0 || vocabulary < 0 || width < 0) return fail(TCX_INVALID_ARGUMENT, "embedding extents must be non-negative");
  if (count == 0) return TCX_OK;
  if (indices == nullptr || flag == nullptr) return fail(TCX_INVALID_ARGUMENT, "embedding buffers are null");
  if (width > 0 && (weight == nullptr || out == nullptr)) return fail(TCX_INVALID_ARGUMENT, "embedding buffers are null");
  if (int rc = ready(); rc != TCX_OK) return rc;
  const auto s = static_cast<hipStream_t>(stream);
  // The check's result comes back in pinned host memory where there is some
  // (one launch in place of a clearing one, two kernels and a copy: 31.4 -> 15.1
  // us for a call on four rows of 64), else through the caller's flag.
  std::int32_t* const pinned = acquire_host_flag();
  std::int32_t host_flag = 0;
  auto run = [&]() -> int {
    std::int32_t* const where = pinned != nullptr ? pinned : flag;
    if (pinned != nullptr) *pinned = 0;
    else if (int rc = tcx_hip_fill(TCX_INT32, flag, 1, 0.0, stream); rc != TCX_OK) return rc;
    const auto at = [](const void* p) { return reinterpret_cast<std::uintptr_t>(p); };
    if (width == 0)
      hipLaunchKernelGGL(embedding_check_kernel, dim3(grid_for(count, 256, 4096)), dim3(256), 0, s, indices, count,
                         vocabulary, where);
    else if (width % 4 == 0 && ((at(weight) | at(out)) & 15U) == 0)
      launch_embedding<float4_t>(indices, weight, out, count, vocabulary, width / 4, where, s);
    else if (count < (std::int64_t{1} << 31) / width)  // FastDiv's range
      launch_embedding_words(indices, weight, out, count, vocabulary, width, where, s);
    else
      launch_embedding<std::uint32_t>(indices, weight, out, count, vocabulary, width, where, s);
    if (int rc = check(hipGetLastError(), "embedding launch"); rc != TCX_OK) return rc;
    if (pinned == nullptr)
      if (int rc = check(hipMemcpyAsync(&host_flag, flag, sizeof(host_flag), hipMemcpyDeviceToHost, s),
                         "embedding flag copy");
          rc != TCX_OK)
        return rc;
    if (int rc = check(hipStreamSynchronize(s), "embedding synchronize"); rc != TCX_OK) return rc;
    if (pinned != nullptr) host_flag = *static_cast<volatile std::int32_t*>(pinned);
    return host_flag != 0 ? fail(TCX_INVALID_ARGUMENT, "embedding index out of range") : TCX_OK;
  };
  const int rc = run();
  if (pinned != nullptr) release_host_flag(pinned);
  return rc;
}

int tcx_hip_attention_softmax_f32(const float* scores, const void* mask, float* out,
                                  const tcx_hip_attention_softmax_desc_t* desc, tcx_stream_t stream) {
  using namespace tcx;
  if (desc == nullptr) return fail(TCX_INVALID_ARGUMENT, "attention softmax descriptor is null");
  const auto& in = *desc;
  if (in.rank < 2 || in.rank > TCX_HIP_MAX_RANK) return fail(TCX_INVALID_ARGUMENT, "attention softmax rank must be in [2, 8]");
  if (in.mask_kind < TCX_MASK_NONE || in.mask_kind > TCX_MASK_ADDITIVE)
    return fail(TCX_INVALID_ARGUMENT, "unknown attention mask kind");
  SoftmaxMeta d{};
  d.rank = in.rank;
  d.mask_kind = in.mask_kind;
  d.causal = in.causal != 0;
  d.scale = in.scale;
  std::int64_t count = 1;
  for (int i = 0; i < in.rank; ++i) {
    if (in.shape[i] < 0) return fail(TCX_INVALID_ARGUMENT, "attention softmax extents must be non-negative");
    d.shape[i] = in.shape[i];
    d.s[i] = in.score_strides[i];
    d.m[i] = in.mask_kind != TCX_MASK_NONE ? in.mask_strides[i] : 0;
    count *= in.shape[i];
  }
  if (count == 0) return TCX_OK;
  if (scores == nullptr || out == nullptr || (in.mask_kind != TCX_MASK_NONE && mask == nullptr))
    return fail(TCX_INVALID_ARGUMENT, "attention softmax buffers are null");
  if (int rc = ready(); rc != TCX_OK) return rc;
  const std::int64_t rows = count / in.shape[in.rank - 1];
  hipLaunchKernelGGL(attention_softmax_kernel, dim3(grid_for(rows, 4, 256 * 16)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), scores, mask, out, d, rows);
  return check(hipGetLastError(), "attention softmax launch");
}

}  // extern "C"
