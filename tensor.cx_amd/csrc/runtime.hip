// C ABI runtime layer: status mapping, device discovery, per-thread streams,
// device allocation through the bounded pool, copies and events.

#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "common.hpp"

namespace tcx {
namespace {
thread_local std::string last_error;
std::once_flag init_once;
int init_status = TCX_UNAVAILABLE;
std::string init_message;
// The process that loaded the library. A forked child inherits the parent's
// runtime state without its threads or device contexts, so every entry point
// refuses to run there, before any HIP call (the reference's CUDA backend
// refuses the same way, cuda_context.cpp:16-20).
const pid_t load_pid = getpid();
thread_local hipStream_t thread_stream = nullptr;
}  // namespace

void set_error(std::string message) { last_error = std::move(message); }

int fail(int code, std::string message) {
  last_error = std::move(message);
  return code;
}

int check(hipError_t error, const char* what) {
  if (error == hipSuccess) return TCX_OK;
  std::string message = std::string(what) + ": " + hipGetErrorString(error);
  switch (error) {
    case hipErrorNoDevice:
    case hipErrorInvalidDevice:
    case hipErrorInsufficientDriver:
      return fail(TCX_UNAVAILABLE, message);
    case hipErrorInvalidValue:
      return fail(TCX_INVALID_ARGUMENT, message);
    default:
      return fail(TCX_INTERNAL, message);
  }
}

bool forked() { return getpid() != load_pid; }

int refuse_forked() { return fail(TCX_UNAVAILABLE, "HIP requires a fresh process after fork"); }

int ready() { return tcx_hip_init(); }

namespace {
std::mutex flags_mutex;
// Flags not in use; as many exist as calls have ever run at once. Never
// destroyed: at process end the runtime that would free them may be gone already.
std::vector<std::int32_t*>& free_flags() {
  static auto* flags = new std::vector<std::int32_t*>;
  return *flags;
}
}  // namespace

std::int32_t* acquire_host_flag() {
  {
    std::lock_guard lock(flags_mutex);
    if (!free_flags().empty()) {
      std::int32_t* const flag = free_flags().back();
      free_flags().pop_back();
      return flag;
    }
  }
  void* flag = nullptr;
  if (hipHostMalloc(&flag, sizeof(std::int32_t), hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  return static_cast<std::int32_t*>(flag);
}

void release_host_flag(std::int32_t* flag) {
  try {
    std::lock_guard lock(flags_mutex);
    free_flags().push_back(flag);
  } catch (...) {
    (void)hipHostFree(flag);
  }
}

}  // namespace tcx

// ------------------------------------------------------------ bounded pool

// Exported storage after its release, kept by the pool it came from. Another
// framework may still read it by work that is queued on streams this library
// cannot see, so a block is handed out again only after hipDeviceSynchronize,
// which hipFree would have made its releaser wait for as well. Mapping and
// unmapping a result of 2 MiB and more for each exchange cost 40 to 280 us of a
// call.
struct Exported {
  void* ptr;
  size_t bytes;
  int device;
  std::uint64_t number;  // of its release
  bool idle;             // the device has been waited for since
};

struct tcx_hip_pool {
  std::mutex mutex;
  std::atomic<long> refs{1};
  tcx_hip_pool_runtime_t runtime{};
  bool default_runtime{true};
  tcx_hip_pool_stats_t stats{};
  std::vector<std::pair<void*, size_t>> cached;
  // Exact sizes, the newest last; they count towards the pool's limits beside
  // the cached blocks and make room for those, the oldest first.
  std::vector<Exported> exported;
  size_t exported_bytes{0};
  std::uint64_t exports{0};  // released so far
  bool used{false};
};

namespace {
thread_local tcx_hip_pool* active_pool = nullptr;

int hip_allocate(void** ptr, size_t bytes) {
  if (tcx::forked()) return tcx::refuse_forked();
  const hipError_t error = hipMalloc(ptr, bytes);
  if (error == hipErrorOutOfMemory) {
    tcx::set_error("hipMalloc: out of memory");
    return TCX_POOL_OOM;
  }
  return tcx::check(error, "hipMalloc");
}
int hip_free(void* ptr) { return tcx::forked() ? tcx::refuse_forked() : tcx::check(hipFree(ptr), "hipFree"); }
int hip_clear_error() {
  if (tcx::forked()) return tcx::refuse_forked();
  const hipError_t error = hipGetLastError();
  if (error == hipErrorOutOfMemory) return TCX_POOL_OOM;
  return tcx::check(error, "pending HIP error");
}

void pool_unref(tcx_hip_pool* pool) {
  if (pool->refs.fetch_sub(1) == 1) {
    for (auto& [ptr, bytes] : pool->cached) pool->runtime.free(ptr);
    for (const Exported& b : pool->exported) pool->runtime.free(b.ptr);
    delete pool;
  }
}

// Gives a block back to the runtime; a failure is counted and reported.
int pool_free_locked(tcx_hip_pool* pool, void* ptr, size_t bytes) {
  ++pool->stats.free_calls;
  const int rc = pool->runtime.free(ptr);
  if (rc != TCX_OK) {
    ++pool->stats.free_failures;
    pool->stats.failed_free_bytes += bytes;
  }
  return rc;
}

// True when `bytes` more fit the pool's limits, once the oldest exported blocks
// have been freed as far as that takes.
bool pool_room_locked(tcx_hip_pool* pool, size_t bytes) {
  const auto& s = pool->stats;
  if (!s.active || pool->cached.size() >= s.max_cached_blocks || bytes > s.max_cached_bytes - s.cached_bytes) return false;
  while (!pool->exported.empty() && (pool->cached.size() + pool->exported.size() >= s.max_cached_blocks ||
                                     bytes > s.max_cached_bytes - s.cached_bytes - pool->exported_bytes)) {
    const Exported oldest = pool->exported.front();
    pool->exported.erase(pool->exported.begin());
    pool->exported_bytes -= oldest.bytes;
    (void)pool_free_locked(pool, oldest.ptr, oldest.bytes);
  }
  return true;
}

// Takes a released exported block over; false where it has to be freed instead.
bool pool_keep_exported_locked(tcx_hip_pool* pool, void* ptr, size_t bytes) {
  int device = 0;
  hipPointerAttribute_t attributes{};
  if (!pool->default_runtime || !pool_room_locked(pool, bytes)) return false;
  if (hipGetDevice(&device) != hipSuccess || hipPointerGetAttributes(&attributes, ptr) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  if (attributes.device != device) return false;
  pool->exported.push_back({ptr, bytes, device, ++pool->exports, false});  // within the room reserved for max_cached_blocks
  pool->exported_bytes += bytes;
  return true;
}

// An exported block of this size, once the device has finished all work queued
// before now; null when there is none, or when the device cannot be waited for
// (during a stream capture). The lock is given up for the wait: other threads
// may release blocks meanwhile, which stay marked as not waited for.
void* pool_take_exported(tcx_hip_pool* pool, size_t bytes, std::unique_lock<std::mutex>& lock) {
  auto& blocks = pool->exported;
  int device = 0;
  if (blocks.empty() || tcx::forked() || hipGetDevice(&device) != hipSuccess) return nullptr;
  const auto found = std::find_if(blocks.rbegin(), blocks.rend(),
                                  [&](const Exported& b) { return b.bytes == bytes && b.device == device; });
  if (found == blocks.rend()) return nullptr;
  const std::uint64_t number = found->number, until = pool->exports;
  if (!found->idle) {
    // Meanwhile the block stays listed: only this thread, the pool's owner,
    // takes blocks, but a release on another may free it to make room.
    lock.unlock();
    const bool waited = hipDeviceSynchronize() == hipSuccess;
    if (!waited) (void)hipGetLastError();
    lock.lock();
    if (!waited) return nullptr;
    for (Exported& b : blocks) b.idle = b.idle || (b.device == device && b.number <= until);
  }
  // (Freed meanwhile to make room, or with the whole pool.)
  const auto at = std::find_if(blocks.begin(), blocks.end(), [&](const Exported& b) { return b.number == number; });
  if (at == blocks.end()) return nullptr;
  void* const ptr = at->ptr;
  blocks.erase(at);
  pool->exported_bytes -= bytes;
  return ptr;
}

// Frees every cached and every exported block; keeps going after a failure and reports it.
int pool_trim_locked(tcx_hip_pool* pool) {
  int status = TCX_OK;
  for (auto& [ptr, bytes] : pool->cached)
    if (pool_free_locked(pool, ptr, bytes) != TCX_OK) status = TCX_INTERNAL;
  for (const Exported& b : pool->exported)
    if (pool_free_locked(pool, b.ptr, b.bytes) != TCX_OK) status = TCX_INTERNAL;
  pool->cached.clear();
  pool->exported.clear();
  pool->exported_bytes = 0;
  pool->stats.cached_bytes = 0;
  pool->stats.cached_blocks = 0;
  if (status != TCX_OK) return tcx::fail(status, "HIP pool failed to free cached blocks");
  return TCX_OK;
}

int pool_allocate_locked(tcx_hip_pool* pool, size_t bytes, void** ptr, std::unique_lock<std::mutex>& lock) {
  if (!pool->stats.active || !bytes)
    return tcx::fail(TCX_INVALID_ARGUMENT, "inactive pool or zero-byte allocation");
  auto found = std::find_if(pool->cached.begin(), pool->cached.end(),
                            [=](const auto& b) { return b.second == bytes; });
  if (found != pool->cached.end()) {
    *ptr = found->first;
    pool->cached.erase(found);
    pool->stats.cached_bytes -= bytes;
    ++pool->stats.hits;
  } else if (void* const again = pool_take_exported(pool, bytes, lock)) {
    *ptr = again;
    ++pool->stats.hits;
  } else if (!pool->stats.active) {  // left while the lock was given up
    return tcx::fail(TCX_INVALID_ARGUMENT, "inactive pool or zero-byte allocation");
  } else {
    ++pool->stats.misses;
    ++pool->stats.allocation_calls;
    int rc = pool->runtime.allocate(ptr, bytes);
    if (rc == TCX_POOL_OOM && !(pool->cached.empty() && pool->exported.empty())) {
      // Recover only from out-of-memory: drain the pool and retry once.
      const int pending = pool->runtime.clear_error();
      if (pending != TCX_OK && pending != TCX_POOL_OOM) {
        ++pool->stats.allocation_failures;
        return tcx::fail(TCX_INTERNAL, "HIP pool allocation found a prior device error");
      }
      const int drained = pool_trim_locked(pool);
      if (drained != TCX_OK) {
        ++pool->stats.allocation_failures;
        return drained;
      }
      ++pool->stats.oom_retries;
      ++pool->stats.allocation_calls;
      rc = pool->runtime.allocate(ptr, bytes);
    }
    if (rc != TCX_OK) {
      ++pool->stats.allocation_failures;
      return tcx::fail(rc == TCX_POOL_OOM ? TCX_INTERNAL : rc, "HIP pool allocation failed: out of memory");
    }
  }
  pool->stats.cached_blocks = pool->cached.size();
  pool->stats.in_use_bytes += bytes;
  pool->stats.peak_in_use_bytes = std::max(pool->stats.peak_in_use_bytes, pool->stats.in_use_bytes);
  return TCX_OK;
}

int pool_allocate(tcx_hip_pool* pool, size_t bytes, void** ptr) {
  pool->refs.fetch_add(1);  // the block's; it also holds the pool while its lock is given up
  std::unique_lock lock(pool->mutex);
  const int rc = pool_allocate_locked(pool, bytes, ptr, lock);
  lock.unlock();
  if (rc != TCX_OK) pool_unref(pool);
  return rc;
}

void pool_release(tcx_hip_pool* pool, void* ptr, size_t bytes, bool allow_cache) {
  {
    std::lock_guard lock(pool->mutex);
    pool->stats.in_use_bytes -= bytes;
    bool cache = allow_cache && pool_room_locked(pool, bytes);
    if (cache && pool->default_runtime && tcx::thread_stream != nullptr &&
        hipStreamQuery(tcx::thread_stream) != hipSuccess) {
      // Never cache a block that queued work may still touch.
      ++pool->stats.readiness_failures;
      cache = false;
    }
    if (cache) {
      pool->cached.emplace_back(ptr, bytes);
      pool->stats.cached_bytes += bytes;
      pool->stats.cached_blocks = pool->cached.size();
      pool->stats.peak_cached_bytes = std::max(pool->stats.peak_cached_bytes, pool->stats.cached_bytes);
    } else {
      ++pool->stats.uncached_returns;
      if (allow_cache || !pool_keep_exported_locked(pool, ptr, bytes)) (void)pool_free_locked(pool, ptr, bytes);
    }
  }
  pool_unref(pool);
}
}  // namespace

bool tcx::allocation_cached(std::size_t bytes) {
  return active_pool != nullptr && active_pool->stats.max_cached_blocks > 0 && bytes <= active_pool->stats.max_cached_bytes;
}

extern "C" {

const char* tcx_hip_last_error(void) { return tcx::last_error.c_str(); }

int tcx_hip_init(void) {
  if (tcx::forked()) return tcx::refuse_forked();
  std::call_once(tcx::init_once, [] {
    hipError_t error = hipInit(0);
    int count = 0;
    if (error == hipSuccess) error = hipGetDeviceCount(&count);
    if (error != hipSuccess) {
      tcx::init_status = error == hipErrorNoDevice ? TCX_UNAVAILABLE : tcx::check(error, "hipInit");
      if (tcx::init_status == TCX_INTERNAL) tcx::init_status = TCX_UNAVAILABLE;
      tcx::init_message = std::string("HIP runtime unavailable: ") + hipGetErrorString(error);
    } else if (count == 0) {
      tcx::init_status = TCX_UNAVAILABLE;
      tcx::init_message = "no HIP device is visible";
    } else {
      tcx::init_status = TCX_OK;
    }
  });
  if (tcx::init_status != TCX_OK) return tcx::fail(tcx::init_status, tcx::init_message);
  return TCX_OK;
}

int tcx_hip_device_count(int* count) {
  *count = 0;
  const int status = tcx::ready();
  if (status != TCX_OK) return status;
  return tcx::check(hipGetDeviceCount(count), "hipGetDeviceCount");
}

int tcx_hip_device_info(int device, tcx_hip_device_info_t* info) {
  const int status = tcx::ready();
  if (status != TCX_OK) return status;
  std::memset(info, 0, sizeof(*info));
  hipDeviceProp_t prop;
  int rc = tcx::check(hipGetDeviceProperties(&prop, device), "hipGetDeviceProperties");
  if (rc != TCX_OK) return rc;
  std::snprintf(info->name, sizeof(info->name), "%s", prop.name);
  std::snprintf(info->arch, sizeof(info->arch), "%s", prop.gcnArchName);
  info->compute_units = prop.multiProcessorCount;
  info->clock_khz = prop.clockRate;
  info->memory_clock_khz = prop.memoryClockRate;
  info->memory_bus_width = prop.memoryBusWidth;
  info->l2_bytes = prop.l2CacheSize;
  info->total_bytes = prop.totalGlobalMem;
  (void)hipRuntimeGetVersion(&info->runtime_version);
  (void)hipDriverGetVersion(&info->driver_version);
  int current = 0;
  (void)hipGetDevice(&current);
  if (current == device) {
    size_t free_bytes = 0, total = 0;
    if (hipMemGetInfo(&free_bytes, &total) == hipSuccess) info->free_bytes = free_bytes;
  }
  return TCX_OK;
}

int tcx_hip_stream(tcx_stream_t* stream) {
  const int status = tcx::ready();
  if (status != TCX_OK) return status;
  if (tcx::thread_stream == nullptr) {
    hipStream_t s = nullptr;
    const int rc = tcx::check(hipStreamCreateWithFlags(&s, hipStreamNonBlocking), "hipStreamCreate");
    if (rc != TCX_OK) return rc;
    tcx::thread_stream = s;
  }
  *stream = tcx::thread_stream;
  return TCX_OK;
}

int tcx_hip_stream_synchronize(tcx_stream_t stream) {
  if (tcx::forked()) return tcx::refuse_forked();
  return tcx::check(hipStreamSynchronize(static_cast<hipStream_t>(stream)), "hipStreamSynchronize");
}

int tcx_hip_allocate(size_t bytes, void** ptr, tcx_hip_pool_t** owner) {
  *ptr = nullptr;
  *owner = nullptr;
  if (bytes == 0) return TCX_OK;
  if (active_pool != nullptr) {
    const int rc = pool_allocate(active_pool, bytes, ptr);
    if (rc == TCX_OK) *owner = active_pool;
    return rc;
  }
  const int status = tcx::ready();
  if (status != TCX_OK) return status;
  return tcx::check(hipMalloc(ptr, bytes), "hipMalloc");
}

void tcx_hip_release(void* ptr, size_t bytes, tcx_hip_pool_t* owner) {
  if (ptr == nullptr || tcx::forked()) return;  // a child does not own the parent's memory
  if (owner != nullptr) {
    pool_release(owner, ptr, bytes, true);
    return;
  }
  (void)hipFree(ptr);
}

void tcx_hip_release_uncached(void* ptr, size_t bytes, tcx_hip_pool_t* owner) {
  if (ptr == nullptr || tcx::forked()) return;
  if (owner != nullptr) {
    pool_release(owner, ptr, bytes, false);
    return;
  }
  (void)hipFree(ptr);
}

int tcx_hip_borrow_check(const void* ptr, size_t bytes) {
  const int status = tcx::ready();
  if (status != TCX_OK) return status;
  if (bytes != 0) {
    if (ptr == nullptr) return tcx::fail(TCX_INVALID_ARGUMENT, "borrowed HIP storage requires data");
    hipPointerAttribute_t attributes{};
    if (hipPointerGetAttributes(&attributes, ptr) != hipSuccess) {
      (void)hipGetLastError();  // an unknown pointer is an argument error, not a sticky one
      return tcx::fail(TCX_INVALID_ARGUMENT, "invalid borrowed HIP pointer");
    }
    if (attributes.type != hipMemoryTypeDevice || attributes.device != 0)
      return tcx::fail(TCX_INVALID_ARGUMENT, "borrowed HIP pointer must be device memory of device 0");
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if (hipMemGetAddressRange(&base, &size, const_cast<void*>(ptr)) != hipSuccess) {
      (void)hipGetLastError();
      return tcx::fail(TCX_INVALID_ARGUMENT, "borrowed HIP pointer has no allocation range");
    }
    const auto begin = reinterpret_cast<std::uintptr_t>(base), at = reinterpret_cast<std::uintptr_t>(ptr);
    if (at < begin || at - begin > size || bytes > size - (at - begin))
      return tcx::fail(TCX_INVALID_ARGUMENT, "borrowed HIP range exceeds its allocation");
  }
  // The producer may have queued its writes on any of its streams.
  return tcx::check(hipDeviceSynchronize(), "borrowed HIP readiness");
}

static int copy(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, tcx_stream_t stream,
                const char* what) {
  if (bytes == 0) return TCX_OK;
  const int status = tcx::ready();
  if (status != TCX_OK) return status;
  const auto s = static_cast<hipStream_t>(stream);
  int rc = tcx::check(hipMemcpyAsync(dst, src, bytes, kind, s), what);
  if (rc != TCX_OK) return rc;
  return tcx::check(hipStreamSynchronize(s), what);
}

int tcx_hip_memcpy_h2d(void* dst, const void* src, size_t bytes, tcx_stream_t stream) {
  return copy(dst, src, bytes, hipMemcpyHostToDevice, stream, "hipMemcpy host to device");
}
int tcx_hip_memcpy_d2h(void* dst, const void* src, size_t bytes, tcx_stream_t stream) {
  return copy(dst, src, bytes, hipMemcpyDeviceToHost, stream, "hipMemcpy device to host");
}
int tcx_hip_memcpy_d2d(void* dst, const void* src, size_t bytes, tcx_stream_t stream) {
  return copy(dst, src, bytes, hipMemcpyDeviceToDevice, stream, "hipMemcpy device to device");
}

int tcx_hip_pool_create(size_t max_cached_bytes, size_t max_cached_blocks,
                        const tcx_hip_pool_runtime_t* runtime, tcx_hip_pool_t** pool) {
  *pool = nullptr;
  if (max_cached_blocks == 0 || max_cached_blocks > 4096)
    return tcx::fail(TCX_INVALID_ARGUMENT, "max_cached_blocks must be in [1, 4096]");
  if (runtime && (!runtime->allocate || !runtime->free || !runtime->clear_error))
    return tcx::fail(TCX_INVALID_ARGUMENT, "invalid pool runtime");
  auto* p = new (std::nothrow) tcx_hip_pool();
  if (!p) return tcx::fail(TCX_INTERNAL, "pool allocation failed");
  if (runtime) {
    p->runtime = *runtime;
    p->default_runtime = false;
  } else {
    p->runtime = {hip_allocate, hip_free, hip_clear_error};
  }
  p->stats.max_cached_bytes = max_cached_bytes;
  p->stats.max_cached_blocks = max_cached_blocks;
  p->cached.reserve(max_cached_blocks);  // keeping a block never allocates host memory
  if (p->default_runtime) p->exported.reserve(max_cached_blocks);
  *pool = p;
  return TCX_OK;
}

int tcx_hip_pool_enter(tcx_hip_pool_t* pool) {
  std::lock_guard lock(pool->mutex);
  if (active_pool != nullptr)
    return tcx::fail(TCX_INVALID_ARGUMENT, "memory pools cannot be nested on the same thread");
  if (pool->used) return tcx::fail(TCX_INVALID_ARGUMENT, "memory pool contexts are single-use");
  if (pool->default_runtime) {
    const int status = tcx::ready();
    if (status != TCX_OK) return status;
  }
  pool->used = true;
  pool->stats.active = 1;
  active_pool = pool;
  return TCX_OK;
}

int tcx_hip_pool_exit(tcx_hip_pool_t* pool) {
  if (active_pool != pool)
    return tcx::fail(TCX_INVALID_ARGUMENT, "memory pool must exit on its owning thread");
  active_pool = nullptr;
  std::lock_guard lock(pool->mutex);
  pool->stats.active = 0;
  return pool_trim_locked(pool);
}

int tcx_hip_pool_trim(tcx_hip_pool_t* pool) {
  std::lock_guard lock(pool->mutex);
  return pool_trim_locked(pool);
}

int tcx_hip_pool_stats(const tcx_hip_pool_t* pool, tcx_hip_pool_stats_t* stats) {
  auto* p = const_cast<tcx_hip_pool_t*>(pool);
  std::lock_guard lock(p->mutex);
  *stats = p->stats;
  return TCX_OK;
}

void tcx_hip_pool_destroy(tcx_hip_pool_t* pool) {
  if (pool == nullptr) return;
  if (active_pool == pool) (void)tcx_hip_pool_exit(pool);
  {
    std::lock_guard lock(pool->mutex);
    pool->stats.active = 0;
    (void)pool_trim_locked(pool);
  }
  pool_unref(pool);
}

int tcx_hip_event_create(void** event) {
  const int status = tcx::ready();
  if (status != TCX_OK) return status;
  hipEvent_t e = nullptr;
  const int rc = tcx::check(hipEventCreate(&e), "hipEventCreate");
  *event = e;
  return rc;
}
int tcx_hip_event_record(void* event, tcx_stream_t stream) {
  if (tcx::forked()) return tcx::refuse_forked();
  return tcx::check(hipEventRecord(static_cast<hipEvent_t>(event), static_cast<hipStream_t>(stream)),
                    "hipEventRecord");
}
int tcx_hip_event_synchronize(void* event) {
  if (tcx::forked()) return tcx::refuse_forked();
  return tcx::check(hipEventSynchronize(static_cast<hipEvent_t>(event)), "hipEventSynchronize");
}
int tcx_hip_event_elapsed_ms(void* start, void* stop, float* ms) {
  if (tcx::forked()) return tcx::refuse_forked();
  return tcx::check(hipEventElapsedTime(ms, static_cast<hipEvent_t>(start), static_cast<hipEvent_t>(stop)),
                    "hipEventElapsedTime");
}
int tcx_hip_event_destroy(void* event) {
  if (tcx::forked()) return tcx::refuse_forked();
  return tcx::check(hipEventDestroy(static_cast<hipEvent_t>(event)), "hipEventDestroy");
}

}  // extern "C"
