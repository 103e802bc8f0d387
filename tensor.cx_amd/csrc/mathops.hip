// log / sqrt / abs and clip of the reference's math extension
// (backends/cpu/cpu_math.cpp:27-76 under the plans of core/math.cpp:13-71).
//
// Values are handled as 32-bit words, as the reference does: abs clears the
// sign bit (float32) or negates in uint32 (int32, so INT32_MIN stays), clip
// orders words with the reference's total order (+0 == -0, NaN handled apart),
// so the results are bit-exact. log uses OCML's logf (within 1 ulp of
// glibc's logf); sqrt is IEEE correctly rounded, as std::sqrt is.
//
//   math_unary_kernel  grid-stride elementwise log / sqrt / abs
//   clip_kernel        three-way broadcast clip(x, lo, hi)

#include "common.hpp"

namespace tcx {
namespace {

template <int kCode, bool kFp>
__device__ __forceinline__ std::uint32_t math_word(std::uint32_t a) {
  if constexpr (kCode == TCX_MATH_ABS) {
    if constexpr (kFp) return a & 0x7fffffffU;
    return (a & 0x80000000U) ? 0U - a : a;
  } else {
    const float f = __builtin_bit_cast(float, a);
    const float r = kCode == TCX_MATH_LOG ? logf(f) : __builtin_sqrtf(f);
    return __builtin_bit_cast(std::uint32_t, r);
  }
}

template <int kCode, bool kFp>
__global__ __launch_bounds__(256) void math_unary_kernel(const std::uint32_t* __restrict__ x,
                                                         std::uint32_t* __restrict__ out, std::int64_t n) {
  const std::int64_t stride = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
  for (std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
    out[i] = math_word<kCode, kFp>(x[i]);
}

struct ClipMeta {
  std::int64_t shape[TCX_HIP_MAX_RANK];
  std::int64_t x[TCX_HIP_MAX_RANK];
  std::int64_t lo[TCX_HIP_MAX_RANK];
  std::int64_t hi[TCX_HIP_MAX_RANK];
  std::int32_t rank;
};

// cpu_math.cpp:45-50: a NaN value stays; a NaN bound, or a bound the value
// does not strictly exceed (lo) / stay below (hi), replaces it; lo first.
template <bool kFp>
__global__ __launch_bounds__(256) void clip_kernel(const std::uint32_t* __restrict__ x,
                                                   const std::uint32_t* __restrict__ lo,
                                                   const std::uint32_t* __restrict__ hi,
                                                   std::uint32_t* __restrict__ out, ClipMeta m, std::int64_t n) {
  const std::int64_t stride = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
  for (std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
    std::int64_t flat = i, ox = 0, ol = 0, oh = 0;
    for (int a = m.rank - 1; a >= 0; --a) {
      const std::int64_t c = flat % m.shape[a];
      flat /= m.shape[a];
      ox += c * m.x[a];
      ol += c * m.lo[a];
      oh += c * m.hi[a];
    }
    std::uint32_t v = x[ox];
    const std::uint32_t l = lo[ol], h = hi[oh];
    if (!word_nan(v, kFp)) v = (word_nan(l, kFp) || !word_less(l, v, kFp)) ? l : v;
    if (!word_nan(v, kFp)) v = (word_nan(h, kFp) || !word_less(v, h, kFp)) ? h : v;
    out[i] = v;
  }
}

template <int kCode>
void launch_unary(bool fp, const void* x, void* out, std::int64_t n, hipStream_t s) {
  const dim3 grid(grid_for(n, 256, 256 * 32));
  const auto* xi = static_cast<const std::uint32_t*>(x);
  auto* o = static_cast<std::uint32_t*>(out);
  if (fp)
    hipLaunchKernelGGL((math_unary_kernel<kCode, true>), grid, dim3(256), 0, s, xi, o, n);
  else
    hipLaunchKernelGGL((math_unary_kernel<kCode, false>), grid, dim3(256), 0, s, xi, o, n);
}

int check_dtype(int dtype) {
  if (dtype != TCX_FLOAT32 && dtype != TCX_INT32) return fail(TCX_INVALID_ARGUMENT, "math operations require float32 or int32");
  return TCX_OK;
}

}  // namespace
}  // namespace tcx

extern "C" {

int tcx_hip_math_unary(int op, int dtype, const void* x, void* out, int64_t n, tcx_stream_t stream) {
  using namespace tcx;
  if (int rc = check_dtype(dtype); rc != TCX_OK) return rc;
  if (op != TCX_MATH_LOG && op != TCX_MATH_SQRT && op != TCX_MATH_ABS)
    return fail(TCX_INVALID_ARGUMENT, "unknown math unary operation");
  if (op != TCX_MATH_ABS && dtype != TCX_FLOAT32) return fail(TCX_INVALID_ARGUMENT, "log/sqrt only support float32 tensors");
  if (n < 0) return fail(TCX_INVALID_ARGUMENT, "element count must be non-negative");
  if (n == 0) return TCX_OK;
  if (x == nullptr || out == nullptr) return fail(TCX_INVALID_ARGUMENT, "math buffers are null");
  if (int rc = ready(); rc != TCX_OK) return rc;
  const auto s = static_cast<hipStream_t>(stream);
  const bool fp = dtype == TCX_FLOAT32;
  if (op == TCX_MATH_LOG) launch_unary<TCX_MATH_LOG>(fp, x, out, n, s);
  else if (op == TCX_MATH_SQRT) launch_unary<TCX_MATH_SQRT>(fp, x, out, n, s);
  else launch_unary<TCX_MATH_ABS>(fp, x, out, n, s);
  return check(hipGetLastError(), "math unary launch");
}

int tcx_hip_clip(int dtype, const void* x, const void* lo, const void* hi, void* out, int32_t rank,
                 const int64_t* out_shape, const int64_t* x_strides, const int64_t* lo_strides,
                 const int64_t* hi_strides, tcx_stream_t stream) {
  using namespace tcx;
  if (int rc = check_dtype(dtype); rc != TCX_OK) return rc;
  if (rank < 0 || rank > TCX_HIP_MAX_RANK) return fail(TCX_INVALID_ARGUMENT, "clip rank must be in [0, 8]");
  if (rank > 0 && (out_shape == nullptr || x_strides == nullptr || lo_strides == nullptr || hi_strides == nullptr))
    return fail(TCX_INVALID_ARGUMENT, "clip metadata is null");
  ClipMeta m{};
  m.rank = rank;
  std::int64_t n = 1;
  for (int i = 0; i < rank; ++i) {
    if (out_shape[i] < 0) return fail(TCX_INVALID_ARGUMENT, "clip extents must be non-negative");
    m.shape[i] = out_shape[i];
    m.x[i] = x_strides[i];
    m.lo[i] = lo_strides[i];
    m.hi[i] = hi_strides[i];
    n *= out_shape[i];
  }
  if (n == 0) return TCX_OK;
  if (x == nullptr || lo == nullptr || hi == nullptr || out == nullptr)
    return fail(TCX_INVALID_ARGUMENT, "clip buffers are null");
  if (int rc = ready(); rc != TCX_OK) return rc;
  const auto s = static_cast<hipStream_t>(stream);
  const dim3 grid(grid_for(n, 256, 256 * 32));
  const auto* xi = static_cast<const std::uint32_t*>(x);
  const auto* li = static_cast<const std::uint32_t*>(lo);
  const auto* hi_words = static_cast<const std::uint32_t*>(hi);
  auto* o = static_cast<std::uint32_t*>(out);
  if (dtype == TCX_FLOAT32)
    hipLaunchKernelGGL((clip_kernel<true>), grid, dim3(256), 0, s, xi, li, hi_words, o, m, n);
  else
    hipLaunchKernelGGL((clip_kernel<false>), grid, dim3(256), 0, s, xi, li, hi_words, o, m, n);
  return check(hipGetLastError(), "clip launch");
}

}  // extern "C"
