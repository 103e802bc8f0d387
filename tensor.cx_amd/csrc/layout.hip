// Data movement and conversion: strided gathers (kTranspose / kSlice), block
// copies (kConcat), kCast and the scalar arithmetic family (kNegate,
// k*Scalar). Semantics are the reference CPU backend's
// (backends/cpu/cpu_backend.cpp:801-930, plans in core/shape.cpp:87-200):
// movement is bit-preserving for 1- and 4-byte elements (NaN payloads and
// signed zeros included); float32 -> int32 truncates toward zero after every
// source was checked finite and inside [-2^31, 2^31); bool conversions test
// value != 0; float32 scalar arithmetic rounds the scalar to float32 once and
// each result once; int32 scalar arithmetic wraps in uint32.

#include "common.hpp"

namespace tcx {
namespace {

struct GatherMeta {
  std::int64_t shape[TCX_HIP_MAX_RANK];
  std::int64_t strides[TCX_HIP_MAX_RANK];
  std::int64_t offset;
  std::int32_t rank;
};

template <typename T>
__global__ __launch_bounds__(256) void gather_kernel(const T* __restrict__ in, T* __restrict__ out, GatherMeta m,
                                                     std::int64_t n) {
  const std::int64_t stride = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
  for (std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
    std::int64_t rest = i, src = m.offset;
    for (int a = m.rank - 1; a >= 0; --a) {
      src += (rest % m.shape[a]) * m.strides[a];
      rest /= m.shape[a];
    }
    out[i] = in[src];
  }
}

// The same gather in 32-bit arithmetic, for fewer than 2^31 units T: whole
// elements, or 16 bytes (4 for 1-byte elements) of an innermost run. A thread
// takes kEach units, their loads ahead of their stores. Bound by memory, where the
// 64-bit division per axis and element of gather_kernel was not: the heads of
// [2, 512, 16, 64] (8 MB read and written) 6.6 -> 4.5 us.
struct FastGather {
  FastDiv shape[TCX_HIP_MAX_RANK];
  std::int64_t strides[TCX_HIP_MAX_RANK];
  std::int64_t offset;
  std::int32_t rank;
};

template <typename T, int kEach>
__global__ __launch_bounds__(256) void fast_gather_kernel(const T* __restrict__ in, T* __restrict__ out, FastGather m,
                                                          std::uint32_t n) {
  const std::uint32_t first = blockIdx.x * (256U * kEach) + threadIdx.x;
  T v[kEach];
#pragma unroll
  for (int u = 0; u < kEach; ++u) {
    std::uint32_t rest = min(first + 256U * u, n - 1);
    std::int64_t src = m.offset;
    for (int a = m.rank - 1; a > 0; --a) {
      const std::uint32_t q = m.shape[a](rest);
      src += static_cast<std::int64_t>(rest - q * m.shape[a].divisor) * m.strides[a];
      rest = q;
    }
    if (m.rank > 0) src += static_cast<std::int64_t>(rest) * m.strides[0];
    v[u] = in[src];
  }
#pragma unroll
  for (int u = 0; u < kEach; ++u)
    if (first + 256U * u < n) out[first + 256U * u] = v[u];
}

// Inputs of a concat: of each a contiguous [outer, block] rectangle, in units of
// 16 bytes or of one element, copied into out at o * out_block + dst + j.
constexpr int kConcatInputs = 8;
struct ConcatArgs {
  const void* in[kConcatInputs];
  FastDiv block[kConcatInputs];
  std::uint32_t units[kConcatInputs];       // outer * block
  std::uint32_t first_block[kConcatInputs]; // of the grid
  std::int64_t dst[kConcatInputs];
  std::int64_t out_block;
  int count;
};

// All inputs in one launch, kEach units a thread. One launch for each input
// with a 64-bit division for each element took 19 us for 33 MB of cached keys
// and 3 more for the new token's; this takes 14.4 (4.7 TB/s).
template <typename T, int kEach>
__global__ __launch_bounds__(256) void concat_kernel(ConcatArgs a, T* __restrict__ out) {
  int k = 0;
  for (int i = 1; i < a.count; ++i)
    if (blockIdx.x >= a.first_block[i]) k = i;
  const T* __restrict__ in = static_cast<const T*>(a.in[k]);
  const std::uint32_t n = a.units[k];
  const std::uint32_t first = (blockIdx.x - a.first_block[k]) * (256U * kEach) + threadIdx.x;
  T v[kEach];
#pragma unroll
  for (int u = 0; u < kEach; ++u) v[u] = in[min(first + 256U * u, n - 1)];
#pragma unroll
  for (int u = 0; u < kEach; ++u) {
    const std::uint32_t i = first + 256U * u;
    if (i >= n) break;
    const std::uint32_t row = a.block[k](i);
    out[static_cast<std::int64_t>(row) * a.out_block + a.dst[k] + (i - row * a.block[k].divisor)] = v[u];
  }
}

template <typename T>
__global__ __launch_bounds__(256) void block_copy_kernel(const T* __restrict__ in, T* __restrict__ out,
                                                         std::int64_t outer, std::int64_t block,
                                                         std::int64_t out_block, std::int64_t dst_offset) {
  const std::int64_t n = outer * block;
  const std::int64_t stride = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
  for (std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
    out[(i / block) * out_block + dst_offset + i % block] = in[i];
}

// float32 values a cast to int32 cannot represent: NaN, +-inf, outside
// [-2^31, 2^31) (cpu_backend.cpp:857-863).
__global__ __launch_bounds__(256) void cast_check_kernel(const float* __restrict__ in, std::int64_t n,
                                                         std::int32_t* __restrict__ flag) {
  const std::int64_t stride = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
  for (std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float v = in[i];
    if (!__builtin_isfinite(v) || v < -2147483648.0F || v >= 2147483648.0F) *flag = 1;  // one value from all writers
  }
}

template <int kFrom, int kTo>
__global__ __launch_bounds__(256) void cast_kernel(const void* __restrict__ in, void* __restrict__ out,
                                                   std::int64_t n) {
  const std::int64_t stride = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
  for (std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
    if constexpr (kTo == TCX_BOOL || kFrom == TCX_BOOL) {
      bool v;
      if constexpr (kFrom == TCX_FLOAT32) v = static_cast<const float*>(in)[i] != 0.F;
      else if constexpr (kFrom == TCX_INT32) v = static_cast<const std::int32_t*>(in)[i] != 0;
      else v = static_cast<const std::uint8_t*>(in)[i] != 0;
      if constexpr (kTo == TCX_BOOL) static_cast<std::uint8_t*>(out)[i] = v ? 1 : 0;
      else if constexpr (kTo == TCX_FLOAT32) static_cast<float*>(out)[i] = v ? 1.F : 0.F;
      else static_cast<std::int32_t*>(out)[i] = v ? 1 : 0;
    } else if constexpr (kFrom == TCX_FLOAT32 && kTo == TCX_INT32) {
      static_cast<std::int32_t*>(out)[i] = static_cast<std::int32_t>(static_cast<const float*>(in)[i]);
    } else if constexpr (kFrom == TCX_INT32 && kTo == TCX_FLOAT32) {
      static_cast<float*>(out)[i] = static_cast<float>(static_cast<const std::int32_t*>(in)[i]);
    } else {  // same dtype: word copy
      static_cast<std::uint32_t*>(out)[i] = static_cast<const std::uint32_t*>(in)[i];
    }
  }
}

template <int kOp>
__global__ __launch_bounds__(256) void scalar_f32_kernel(const float* __restrict__ in, float* __restrict__ out,
                                                         std::int64_t n, float scalar, int scalar_left) {
  const std::int64_t stride = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
  for (std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
    const float v = in[i];
    const float l = scalar_left ? scalar : v, r = scalar_left ? v : scalar;
    float y;
    if constexpr (kOp == TCX_SCALAR_NEGATE) y = -v;
    else if constexpr (kOp == TCX_SCALAR_ADD) y = l + r;
    else if constexpr (kOp == TCX_SCALAR_SUBTRACT) y = l - r;
    else if constexpr (kOp == TCX_SCALAR_MULTIPLY) y = l * r;
    else y = l / r;
    out[i] = y;
  }
}

template <int kOp>
__global__ __launch_bounds__(256) void scalar_i32_kernel(const std::uint32_t* __restrict__ in,
                                                         std::uint32_t* __restrict__ out, std::int64_t n,
                                                         std::uint32_t scalar, int scalar_left) {
  const std::int64_t stride = static_cast<std::int64_t>(gridDim.x) * blockDim.x;
  for (std::int64_t i = static_cast<std::int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
    const std::uint32_t v = in[i];
    const std::uint32_t l = scalar_left ? scalar : v, r = scalar_left ? v : scalar;
    std::uint32_t y;
    if constexpr (kOp == TCX_SCALAR_NEGATE) y = 0U - v;
    else if constexpr (kOp == TCX_SCALAR_ADD) y = l + r;
    else if constexpr (kOp == TCX_SCALAR_SUBTRACT) y = l - r;
    else y = l * r;
    out[i] = y;
  }
}

dim3 grid_of(std::int64_t n) { return dim3(grid_for(n, 256, 256 * 32)); }

int check_bytes(int elem_bytes) {
  if (elem_bytes != 1 && elem_bytes != 4) return fail(TCX_INVALID_ARGUMENT, "element size must be 1 or 4 bytes");
  return TCX_OK;
}

constexpr std::int64_t kFastUnits = std::int64_t{1} << 31;
// Units from which a thread takes four (with fewer, more threads with one each
// fill the GPU).
constexpr std::int64_t kEachUnits = 256 * 1024;

bool aligned_to(const void* p, int bytes) { return reinterpret_cast<std::uintptr_t>(p) % bytes == 0; }

template <typename T>
int launch_fast_gather(const void* in, void* out, const GatherMeta& m, std::int64_t n, int widen, hipStream_t s) {
  FastGather f;
  f.rank = m.rank;
  f.offset = m.offset / widen;
  for (int a = 0; a < m.rank; ++a) {
    const bool last = a == m.rank - 1;
    f.shape[a] = FastDiv(static_cast<std::uint32_t>(last ? m.shape[a] / widen : m.shape[a]));
    f.strides[a] = last ? m.strides[a] : m.strides[a] / widen;
  }
  const std::int64_t units = n / widen;
  const auto* x = static_cast<const T*>(in);
  auto* y = static_cast<T*>(out);
  if (units < kEachUnits)
    hipLaunchKernelGGL((fast_gather_kernel<T, 1>), dim3(grid_for(units, 256, kFastUnits)), dim3(256), 0, s, x, y, f,
                       static_cast<std::uint32_t>(units));
  else
    hipLaunchKernelGGL((fast_gather_kernel<T, 4>), dim3(grid_for(units, 1024, kFastUnits)), dim3(256), 0, s, x, y, f,
                       static_cast<std::uint32_t>(units));
  return check(hipGetLastError(), "gather launch");
}

// How many elements of a gather one unit of `unit` bytes can take: the innermost
// axis contiguous and every start a multiple of it; else 1.
int gather_widen(const GatherMeta& m, int elem_bytes, int unit, const void* in, const void* out) {
  const int w = unit / elem_bytes;
  if (m.rank == 0 || m.strides[m.rank - 1] != 1 || m.shape[m.rank - 1] % w != 0 || m.offset % w != 0 ||
      !aligned_to(in, unit) || !aligned_to(out, unit))
    return 1;
  for (int a = 0; a < m.rank - 1; ++a)
    if (m.strides[a] % w != 0) return 1;
  return w;
}

template <typename T>
int launch_concat(ConcatArgs& a, void* out, hipStream_t s) {
  std::int64_t units = 0, blocks = 0;
  for (int i = 0; i < a.count; ++i) units += a.units[i];
  const int each = units < kEachUnits ? 1 : 4;
  for (int i = 0; i < a.count; ++i) {
    a.first_block[i] = static_cast<std::uint32_t>(blocks);
    blocks += (a.units[i] + 256LL * each - 1) / (256 * each);
  }
  const dim3 grid(static_cast<unsigned>(blocks));
  if (each == 1) hipLaunchKernelGGL((concat_kernel<T, 1>), grid, dim3(256), 0, s, a, static_cast<T*>(out));
  else hipLaunchKernelGGL((concat_kernel<T, 4>), grid, dim3(256), 0, s, a, static_cast<T*>(out));
  return check(hipGetLastError(), "concat launch");
}

template <int kFrom>
void launch_cast_from(int to, const void* in, void* out, std::int64_t n, hipStream_t s) {
  if (to == TCX_FLOAT32) hipLaunchKernelGGL((cast_kernel<kFrom, TCX_FLOAT32>), grid_of(n), dim3(256), 0, s, in, out, n);
  else if (to == TCX_INT32) hipLaunchKernelGGL((cast_kernel<kFrom, TCX_INT32>), grid_of(n), dim3(256), 0, s, in, out, n);
  else hipLaunchKernelGGL((cast_kernel<kFrom, TCX_BOOL>), grid_of(n), dim3(256), 0, s, in, out, n);
}

}  // namespace
}  // namespace tcx

extern "C" {

int tcx_hip_gather_strided(int elem_bytes, const void* in, void* out, int32_t rank, const int64_t* out_shape,
                           const int64_t* in_strides, int64_t offset, tcx_stream_t stream) {
  using namespace tcx;
  if (int rc = check_bytes(elem_bytes); rc != TCX_OK) return rc;
  if (rank < 0 || rank > TCX_HIP_MAX_RANK) return fail(TCX_INVALID_ARGUMENT, "gather rank must be in [0, 8]");
  if (rank > 0 && (out_shape == nullptr || in_strides == nullptr)) return fail(TCX_INVALID_ARGUMENT, "gather metadata is null");
  GatherMeta m{};
  m.rank = rank;
  m.offset = offset;
  std::int64_t n = 1;
  for (int a = 0; a < rank; ++a) {
    if (out_shape[a] < 0) return fail(TCX_INVALID_ARGUMENT, "gather extents must be non-negative");
    m.shape[a] = out_shape[a];
    m.strides[a] = in_strides[a];
    n *= out_shape[a];
  }
  if (n == 0) return TCX_OK;
  if (in == nullptr || out == nullptr) return fail(TCX_INVALID_ARGUMENT, "gather buffers are null");
  if (int rc = ready(); rc != TCX_OK) return rc;
  const auto s = static_cast<hipStream_t>(stream);
  if (n < kFastUnits) {
    if (elem_bytes == 4) {
      if (const int w = gather_widen(m, 4, 16, in, out); w > 1) return launch_fast_gather<int4_t>(in, out, m, n, w, s);
      return launch_fast_gather<std::uint32_t>(in, out, m, n, 1, s);
    }
    if (const int w = gather_widen(m, 1, 16, in, out); w > 1) return launch_fast_gather<int4_t>(in, out, m, n, w, s);
    if (const int w = gather_widen(m, 1, 4, in, out); w > 1) return launch_fast_gather<std::uint32_t>(in, out, m, n, w, s);
    return launch_fast_gather<std::uint8_t>(in, out, m, n, 1, s);
  }
  if (elem_bytes == 4)
    hipLaunchKernelGGL((gather_kernel<std::uint32_t>), grid_of(n), dim3(256), 0, s,
                       static_cast<const std::uint32_t*>(in), static_cast<std::uint32_t*>(out), m, n);
  else
    hipLaunchKernelGGL((gather_kernel<std::uint8_t>), grid_of(n), dim3(256), 0, s,
                       static_cast<const std::uint8_t*>(in), static_cast<std::uint8_t*>(out), m, n);
  return check(hipGetLastError(), "gather launch");
}

int tcx_hip_copy_blocks(int elem_bytes, const void* in, void* out, int64_t outer, int64_t block, int64_t out_block,
                        int64_t dst_offset, tcx_stream_t stream) {
  using namespace tcx;
  if (int rc = check_bytes(elem_bytes); rc != TCX_OK) return rc;
  if (outer < 0 || block < 0 || dst_offset < 0 || out_block < dst_offset + block)
    return fail(TCX_INVALID_ARGUMENT, "block copy extents are inconsistent");
  if (outer == 0 || block == 0) return TCX_OK;
  if (in == nullptr || out == nullptr) return fail(TCX_INVALID_ARGUMENT, "block copy buffers are null");
  if (int rc = ready(); rc != TCX_OK) return rc;
  const auto s = static_cast<hipStream_t>(stream);
  if (elem_bytes == 4)
    hipLaunchKernelGGL((block_copy_kernel<std::uint32_t>), grid_of(outer * block), dim3(256), 0, s,
                       static_cast<const std::uint32_t*>(in), static_cast<std::uint32_t*>(out), outer, block,
                       out_block, dst_offset);
  else
    hipLaunchKernelGGL((block_copy_kernel<std::uint8_t>), grid_of(outer * block), dim3(256), 0, s,
                       static_cast<const std::uint8_t*>(in), static_cast<std::uint8_t*>(out), outer, block,
                       out_block, dst_offset);
  return check(hipGetLastError(), "block copy launch");
}

int tcx_hip_concat(int elem_bytes, const void* const* in, const int64_t* blocks, int32_t count, void* out, int64_t outer,
                   tcx_stream_t stream) {
  using namespace tcx;
  if (int rc = check_bytes(elem_bytes); rc != TCX_OK) return rc;
  if (outer < 0 || count < 0 || (count > 0 && (in == nullptr || blocks == nullptr)))
    return fail(TCX_INVALID_ARGUMENT, "concat extents are inconsistent");
  std::int64_t out_block = 0;
  for (int i = 0; i < count; ++i) {
    if (blocks[i] < 0) return fail(TCX_INVALID_ARGUMENT, "concat extents are inconsistent");
    out_block += blocks[i];
  }
  if (outer == 0 || out_block == 0) return TCX_OK;
  if (out == nullptr) return fail(TCX_INVALID_ARGUMENT, "concat buffers are null");
  for (int i = 0; i < count; ++i)
    if (blocks[i] > 0 && in[i] == nullptr) return fail(TCX_INVALID_ARGUMENT, "concat buffers are null");
  if (int rc = ready(); rc != TCX_OK) return rc;
  const auto s = static_cast<hipStream_t>(stream);
  // 16-byte units where every input's runs start and end at one, in both
  // buffers; results of 2^31 units and more are copied input by input.
  const int w16 = 16 / elem_bytes;
  bool wide = aligned_to(out, 16);
  for (int i = 0; i < count; ++i) wide = wide && (blocks[i] == 0 || (blocks[i] % w16 == 0 && aligned_to(in[i], 16)));
  const int w = wide ? w16 : 1;
  const bool small = outer * (out_block / w) < kFastUnits;
  std::int64_t dst = 0;
  ConcatArgs a{};
  a.out_block = out_block / w;
  for (int i = 0; i < count; ++i) {
    if (blocks[i] > 0) {
      if (!small) {
        if (int rc = tcx_hip_copy_blocks(elem_bytes, in[i], out, outer, blocks[i], out_block, dst, stream); rc != TCX_OK)
          return rc;
      } else {
        a.in[a.count] = in[i];
        a.block[a.count] = FastDiv(static_cast<std::uint32_t>(blocks[i] / w));
        a.units[a.count] = static_cast<std::uint32_t>(outer * (blocks[i] / w));
        a.dst[a.count] = dst / w;
        ++a.count;
      }
    }
    dst += blocks[i];
    if (a.count > 0 && (a.count == kConcatInputs || i == count - 1)) {
      const int rc = wide              ? launch_concat<int4_t>(a, out, s)
                     : elem_bytes == 4 ? launch_concat<std::uint32_t>(a, out, s)
                                       : launch_concat<std::uint8_t>(a, out, s);
      if (rc != TCX_OK) return rc;
      a.count = 0;
    }
  }
  return TCX_OK;
}

int tcx_hip_cast(int from, int to, const void* in, void* out, int64_t n, int32_t* flag, tcx_stream_t stream) {
  using namespace tcx;
  const auto valid = [](int d) { return d == TCX_FLOAT32 || d == TCX_INT32 || d == TCX_BOOL; };
  if (!valid(from) || !valid(to)) return fail(TCX_INVALID_ARGUMENT, "unsupported cast dtype");
  if (n < 0) return fail(TCX_INVALID_ARGUMENT, "cast extent must be non-negative");
  if (n == 0) return TCX_OK;
  if (in == nullptr || out == nullptr) return fail(TCX_INVALID_ARGUMENT, "cast buffers are null");
  if (int rc = ready(); rc != TCX_OK) return rc;
  const auto s = static_cast<hipStream_t>(stream);
  if (from == TCX_FLOAT32 && to == TCX_INT32) {
    // Every source is checked before any conversion result is used.
    if (flag == nullptr) return fail(TCX_INVALID_ARGUMENT, "float32 to int32 casts need a check flag");
    if (int rc = tcx_hip_fill(TCX_INT32, flag, 1, 0.0, stream); rc != TCX_OK) return rc;
    hipLaunchKernelGGL(cast_check_kernel, grid_of(n), dim3(256), 0, s, static_cast<const float*>(in), n, flag);
    if (int rc = check(hipGetLastError(), "cast check launch"); rc != TCX_OK) return rc;
    std::int32_t bad = 0;
    if (int rc = check(hipMemcpyAsync(&bad, flag, sizeof(bad), hipMemcpyDeviceToHost, s), "cast flag copy");
        rc != TCX_OK)
      return rc;
    if (int rc = check(hipStreamSynchronize(s), "cast synchronize"); rc != TCX_OK) return rc;
    if (bad) return fail(TCX_INVALID_ARGUMENT, "float32 value is out of range for int32 cast");
  }
  if (from == TCX_FLOAT32) launch_cast_from<TCX_FLOAT32>(to, in, out, n, s);
  else if (from == TCX_INT32) launch_cast_from<TCX_INT32>(to, in, out, n, s);
  else launch_cast_from<TCX_BOOL>(to, in, out, n, s);
  return check(hipGetLastError(), "cast launch");
}

int tcx_hip_scalar_op(int op, int dtype, const void* in, void* out, int64_t n, double scalar, int scalar_left,
                      tcx_stream_t stream) {
  using namespace tcx;
  if (op < TCX_SCALAR_NEGATE || op > TCX_SCALAR_DIVIDE) return fail(TCX_INVALID_ARGUMENT, "unknown scalar operation");
  if (dtype != TCX_FLOAT32 && dtype != TCX_INT32) return fail(TCX_INVALID_ARGUMENT, "numeric operations do not support bool");
  if (dtype == TCX_INT32 && op == TCX_SCALAR_DIVIDE) return fail(TCX_INVALID_ARGUMENT, "division only supports float32 tensors");
  if (dtype == TCX_INT32 && op != TCX_SCALAR_NEGATE &&
      !(scalar >= -2147483648.0 && scalar <= 2147483647.0 && scalar == static_cast<double>(static_cast<std::int64_t>(scalar))))
    return fail(TCX_INVALID_ARGUMENT, "arithmetic scalar must be an integer in int32 range");
  if (n < 0) return fail(TCX_INVALID_ARGUMENT, "extent must be non-negative");
  if (n == 0) return TCX_OK;
  if (in == nullptr || out == nullptr) return fail(TCX_INVALID_ARGUMENT, "scalar operation buffers are null");
  if (int rc = ready(); rc != TCX_OK) return rc;
  const auto s = static_cast<hipStream_t>(stream);
  if (dtype == TCX_FLOAT32) {
    const auto* x = static_cast<const float*>(in);
    auto* y = static_cast<float*>(out);
    const float v = static_cast<float>(scalar);
    switch (op) {
      case TCX_SCALAR_NEGATE: hipLaunchKernelGGL((scalar_f32_kernel<TCX_SCALAR_NEGATE>), grid_of(n), dim3(256), 0, s, x, y, n, v, scalar_left); break;
      case TCX_SCALAR_ADD: hipLaunchKernelGGL((scalar_f32_kernel<TCX_SCALAR_ADD>), grid_of(n), dim3(256), 0, s, x, y, n, v, scalar_left); break;
      case TCX_SCALAR_SUBTRACT: hipLaunchKernelGGL((scalar_f32_kernel<TCX_SCALAR_SUBTRACT>), grid_of(n), dim3(256), 0, s, x, y, n, v, scalar_left); break;
      case TCX_SCALAR_MULTIPLY: hipLaunchKernelGGL((scalar_f32_kernel<TCX_SCALAR_MULTIPLY>), grid_of(n), dim3(256), 0, s, x, y, n, v, scalar_left); break;
      default: hipLaunchKernelGGL((scalar_f32_kernel<TCX_SCALAR_DIVIDE>), grid_of(n), dim3(256), 0, s, x, y, n, v, scalar_left); break;
    }
  } else {
    const auto* x = static_cast<const std::uint32_t*>(in);
    auto* y = static_cast<std::uint32_t*>(out);
    const auto v = op == TCX_SCALAR_NEGATE ? 0U : static_cast<std::uint32_t>(static_cast<std::int32_t>(scalar));
    switch (op) {
      case TCX_SCALAR_NEGATE: hipLaunchKernelGGL((scalar_i32_kernel<TCX_SCALAR_NEGATE>), grid_of(n), dim3(256), 0, s, x, y, n, v, scalar_left); break;
      case TCX_SCALAR_ADD: hipLaunchKernelGGL((scalar_i32_kernel<TCX_SCALAR_ADD>), grid_of(n), dim3(256), 0, s, x, y, n, v, scalar_left); break;
      case TCX_SCALAR_SUBTRACT: hipLaunchKernelGGL((scalar_i32_kernel<TCX_SCALAR_SUBTRACT>), grid_of(n), dim3(256), 0, s, x, y, n, v, scalar_left); break;
      default: hipLaunchKernelGGL((scalar_i32_kernel<TCX_SCALAR_MULTIPLY>), grid_of(n), dim3(256), 0, s, x, y, n, v, scalar_left); break;
    }
  }
  return check(hipGetLastError(), "scalar operation launch");
}

}  // extern "C"
