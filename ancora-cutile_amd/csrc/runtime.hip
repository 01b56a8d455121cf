// Device, memory, stream and event plumbing behind the C ABI, plus the two tiny
// utility kernels (fill, copy). Replaces the cuda.bindings driver calls the reference
// makes from Python (ancora/optim/adamw.py:51-60, ancora/model/resident.py:52-94).
#include "common.h"
#include <stdarg.h>
#include <string.h>

static thread_local char g_err[512] = "";

void anc_set_error(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

int anc_hip_fail(hipError_t e, const char *what, const char *file, int line) {
  anc_set_error("HIP error %d (%s) at %s:%d in %s", (int)e, hipGetErrorString(e), file, line, what);
  return ANC_ERR_HIP;
}

extern "C" const char *anc_last_error(void) { return g_err; }

// ---- per-launch profiler -------------------------------------------------------------
#include <chrono>
#include <mutex>
#include <exception>
#include <thread>
#include <vector>
namespace {
struct ProfRec { int kind; hipEvent_t start, stop; };
std::mutex g_prof_mu;
bool g_prof_on = false;
std::vector<ProfRec> g_prof_recs;
std::vector<hipEvent_t> g_prof_pool;
hipEvent_t prof_event() {
  if (!g_prof_pool.empty()) { hipEvent_t e = g_prof_pool.back(); g_prof_pool.pop_back(); return e; }
  hipEvent_t e = nullptr;
  if (hipEventCreate(&e) != hipSuccess) return nullptr;
  return e;
}
}  // namespace

void anc_prof_begin(int kind, hipStream_t s) {
  if (!g_prof_on) return;
  std::lock_guard<std::mutex> lk(g_prof_mu);
  ProfRec r{kind, prof_event(), prof_event()};
  if (r.start == nullptr || r.stop == nullptr) return;
  (void)hipEventRecord(r.start, s);
  g_prof_recs.push_back(r);
}
void anc_prof_end(hipStream_t s) {
  if (!g_prof_on) return;
  std::lock_guard<std::mutex> lk(g_prof_mu);
  if (!g_prof_recs.empty()) (void)hipEventRecord(g_prof_recs.back().stop, s);
}
extern "C" int anc_profile_enable(int on) {
  std::lock_guard<std::mutex> lk(g_prof_mu);
  g_prof_on = on != 0;
  return ANC_OK;
}
extern "C" int anc_profile_read(float *ms, int64_t *launches) {
  ANC_REQUIRE(ms != nullptr && launches != nullptr, "anc_profile_read: null output");
  ANC_HIP(hipDeviceSynchronize());
  std::lock_guard<std::mutex> lk(g_prof_mu);
  for (int k = 0; k < ANC_PROF_KINDS; ++k) { ms[k] = 0.0f; launches[k] = 0; }
  for (const ProfRec &r : g_prof_recs) {
    float t = 0.0f;
    if (hipEventElapsedTime(&t, r.start, r.stop) == hipSuccess && r.kind >= 0 && r.kind < ANC_PROF_KINDS) {
      ms[r.kind] += t;
      launches[r.kind] += 1;
    }
    g_prof_pool.push_back(r.start);
    g_prof_pool.push_back(r.stop);
  }
  g_prof_recs.clear();
  return ANC_OK;
}
extern "C" int anc_abi_version(void) { return 3; }

int anc_gradnorm_static_init(void);   // gradnorm.hip: per-device address of its built-in scratch

extern "C" int anc_init(int device) {
  int n = 0;
  ANC_HIP(hipGetDeviceCount(&n));
  ANC_REQUIRE(device >= 0 && device < n, "anc_init: device %d out of range (%d visible)", device, n);
  ANC_HIP(hipSetDevice(device));
  hipDeviceProp_t p;
  ANC_HIP(hipGetDeviceProperties(&p, device));
  if (strncmp(p.gcnArchName, "gfx950", 6) != 0) {
    anc_set_error("anc_init: device %d is %s; this library carries gfx950 code only", device,
                  p.gcnArchName);
    return ANC_ERR_UNSUPPORTED;
  }
  return anc_gradnorm_static_init();
}

extern "C" int anc_current_device(int32_t *device) {
  ANC_REQUIRE(device != nullptr, "anc_current_device: null output");
  ANC_HIP(hipGetDevice(device));
  return ANC_OK;
}

extern "C" int anc_device_info(anc_device_info_t *out) {
  ANC_REQUIRE(out != nullptr, "anc_device_info: null output");
  int dev = 0;
  ANC_HIP(hipGetDevice(&dev));
  hipDeviceProp_t p;
  ANC_HIP(hipGetDeviceProperties(&p, dev));
  memset(out, 0, sizeof(*out));
  out->cu_count = p.multiProcessorCount;
  out->clock_khz = p.clockRate;
  out->mem_clock_khz = p.memoryClockRate;
  out->mem_bus_bits = p.memoryBusWidth;
  out->wavefront = p.warpSize;
  out->lds_bytes_per_block = (int32_t)p.sharedMemPerBlock;
  out->hbm_bytes = (int64_t)p.totalGlobalMem;
  out->l2_bytes = (int64_t)p.l2CacheSize;
  strncpy(out->name, p.name, sizeof(out->name) - 1);
  strncpy(out->arch, p.gcnArchName, sizeof(out->arch) - 1);
  return ANC_OK;
}

extern "C" int anc_malloc(uint64_t *dptr, int64_t bytes) {
  ANC_REQUIRE(dptr != nullptr && bytes > 0, "anc_malloc: bad arguments (bytes=%lld)", (long long)bytes);
  void *p = nullptr;
  ANC_HIP(hipMalloc(&p, (size_t)bytes));
  *dptr = (uint64_t)p;
  return ANC_OK;
}
extern "C" int anc_free(uint64_t dptr) {
  ANC_REQUIRE(dptr != 0, "anc_free: null pointer");
  ANC_HIP(hipFree((void *)dptr));
  return ANC_OK;
}
extern "C" int anc_host_alloc(void **hptr, int64_t bytes) {
  ANC_REQUIRE(hptr != nullptr && bytes > 0, "anc_host_alloc: bad arguments");
  ANC_HIP(hipHostMalloc(hptr, (size_t)bytes, hipHostMallocDefault));
  return ANC_OK;
}
extern "C" int anc_host_free(void *hptr) {
  ANC_REQUIRE(hptr != nullptr, "anc_host_free: null pointer");
  ANC_HIP(hipHostFree(hptr));
  return ANC_OK;
}
extern "C" int anc_mem_info(int64_t *free_bytes, int64_t *total_bytes) {
  size_t f = 0, t = 0;
  ANC_HIP(hipMemGetInfo(&f, &t));
  if (free_bytes) *free_bytes = (int64_t)f;
  if (total_bytes) *total_bytes = (int64_t)t;
  return ANC_OK;
}

__global__ void __launch_bounds__(256) k_fill_u32(uint32_t *__restrict__ p, uint32_t v, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (; i < n; i += stride) p[i] = v;
}
extern "C" int anc_fill_u32(uint64_t dptr, uint32_t value, int64_t n_words, uint64_t stream) {
  ANC_REQUIRE(dptr != 0 && n_words >= 0 && (dptr & 3) == 0, "anc_fill_u32: bad arguments");
  if (n_words == 0) return ANC_OK;
  int64_t blocks = (n_words + 255) / 256;
  if (blocks > 16384) blocks = 16384;
  AncProfScope prof(ANC_PROF_MISC, anc_stream(stream));
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, anc_stream(stream),
                     (uint32_t *)dptr, value, n_words);
  ANC_LAUNCH_CHECK();
  return ANC_OK;
}

// A word in pinned memory that the host reads while the kernel may still run. It says that a block has read its part of
// a slot, no more: nothing that it wrote has to be visible, so the store is not ordered behind it.
__device__ __forceinline__ void stage_mark(uint32_t *mark) {
  __hip_atomic_store(mark, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// From pinned memory into place, 16 bytes per lane and access; what is left over 16 bytes by bytes. The link bounds it
// (50 GB/s of a large copy), or the launch. For uploads that are ordered on a caller's stream: it shares a hardware queue and
// the compute units with other streams' kernels. Against the runtime's copy, which hands over to another engine and back:
// between two kernels 28 KB 22.5 -> 9.4 us, 128 KB 24.9 -> 11.3, 512 KB 31.5 -> 18.2; in a row 512 KB 23.8 -> 14.5.
template <int U>
__global__ void __launch_bounds__(256) k_stage_in(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, int64_t bytes, uint32_t *mark) {
  const int64_t n = bytes / 16, i = (int64_t)blockIdx.x * (256 * U) + threadIdx.x;
  anc_u32x4 v[U];
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (i + u * 256 < n) v[u] = anc_ld_stream((const anc_u32x4 *)src + i + u * 256);
#pragma unroll
  for (int u = 0; u < U; ++u)
    if (i + u * 256 < n) *((anc_u32x4 *)dst + i + u * 256) = v[u];
  const int64_t j = n * 16 + threadIdx.x;
  if (blockIdx.x == 0 && j < bytes) dst[j] = src[j];
  __syncthreads();                          // (what went into a store has been read)
  if (threadIdx.x == 0) stage_mark(mark + blockIdx.x);
}
// The same mark behind a copy of the runtime's.
__global__ void __launch_bounds__(64) k_stage_mark(uint32_t *mark) {
  if (threadIdx.x == 0) stage_mark(mark);
}

// ---- uploads through a ring of pinned slots ------------------------------------------------------
// A pageable upload runs at 31 GB/s (and some sizes at 3: 1 MiB took 368 us) where pinned memory reaches
// 57, and blocks until everything before it on the stream is done. So a source is copied slot by slot into pinned
// memory, the transfer of one slot (k_stage_in) under the copy into the next, and the call can return as soon as the last
// slot is filled. 4 MiB: 132 -> 95 us (with the runtime's copies, k_stage_in is quicker still). A source beyond the caches is read at 32 GB/s by one thread, so from 8 MiB on
// four threads copy. A slot is taken again once its last transfer has read it, which the transfer itself marks in the slot's
// memory: an event keeps the address of the stream it was recorded on, and a query looks there, but a caller's stream
// may be gone by then. (On the ring's own stream, where no kernel runs, an event it is.) An upload waits for
// slots in use on its own stream, where its data queue up behind the same work anyway, and never for those of
// another: if those hold all of them it goes the pageable way. No lock is held while anyone waits or copies.
// Events and streams belong to a device, so every device has a ring of its own, shared by all threads and streams
// (4 MiB, pinned slot by slot on first use, given back by anc_staging_release).
namespace {
constexpr int kSlots = 8, kCopyThreads = 4, kMaxDevices = 32;
constexpr int64_t kSlotBytes = 512 << 10, kThreadedBytes = 8 << 20, kFewBytes = 128 << 10;
constexpr int kMarks = 64;         // words behind a slot's bytes
constexpr int64_t stage_blocks(int64_t bytes) { return bytes <= kFewBytes ? bytes / 4096 + 1 : bytes / 16384 + 1; }
static_assert(stage_blocks(kFewBytes) <= kMarks && stage_blocks(kSlotBytes) <= kMarks, "a mark per block");
struct StageSlot {
  void *mem = nullptr;
  hipEvent_t done = nullptr;
  int marks = 0;                 // the marks that the transfer under way sets; 0: it has the event
  hipStream_t user = nullptr;    // the stream of its last transfer,
  uint64_t turn = 0;             // the older the smaller
  bool busy = false;             // that transfer was not seen to end yet
  bool taken = false;            // a call is filling it, or waiting to
};
struct StageRing {
  std::mutex mu;                 // guards the flags, not the copies
  StageSlot slot[kSlots];
  uint64_t turn = 0;
  hipStream_t own = nullptr;     // for uploads that are complete on return without waiting for anybody's work
  int own_users = 0;
};
StageRing g_ring[kMaxDevices];

// A graph would read host memory, or a slot, whose contents have changed.
int refuse_capture(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  ANC_HIP(hipStreamIsCapturing(s, &st));
  ANC_REQUIRE(st == hipStreamCaptureStatusNone, "upload: the stream is being captured, and host memory is read once, at the call");
  return ANC_OK;
}
// While this lives the device `s` belongs to is current (the null stream's is the current one already), and a capture
// of another stream by this or another thread leaves events and pinned memory usable.
struct StageScope {
  int dev = 0, before = -1;
  bool relaxed = false;
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  int enter(hipStream_t s) {
    int cur = 0;
    ANC_HIP(hipGetDevice(&cur));
    dev = cur;
    if (s != nullptr && s != hipStreamLegacy && s != hipStreamPerThread) ANC_HIP(hipStreamGetDevice(s, &dev));
    ANC_REQUIRE(dev >= 0 && dev < kMaxDevices, "upload: device %d beyond %d", dev, kMaxDevices - 1);
    ANC_HIP(hipThreadExchangeStreamCaptureMode(&mode));
    relaxed = true;
    if (dev == cur) return ANC_OK;
    ANC_HIP(hipSetDevice(dev));
    before = cur;
    return ANC_OK;
  }
  ~StageScope() {
    if (before >= 0) (void)hipSetDevice(before);
    if (relaxed) (void)hipThreadExchangeStreamCaptureMode(&mode);
  }
};

// Does k_stage_in on device `dev` reach `bytes` bytes from `dst`? The runtime's copy finds the owner of an address and refuses
// what does not fit into the allocation; a kernel writes from the stream's device whatever it is given, and memory of
// another device, or past an end, is a fault there.
bool kernel_reaches(uint64_t dst, int64_t bytes, int dev) {
  hipPointerAttribute_t at{};
  hipDeviceptr_t base = nullptr;
  size_t size = 0;
  hipError_t e = hipPointerGetAttributes(&at, (const void *)dst);
  if (e == hipSuccess && (at.type != hipMemoryTypeDevice || at.device != dev)) return false;
  if (e == hipSuccess) e = hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)dst);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  const uint64_t before = dst - (uint64_t)base;
  return before <= size && (uint64_t)bytes <= size - before;
}

uint32_t *slot_marks(const StageSlot &slot) { return (uint32_t *)((char *)slot.mem + kSlotBytes); }
// hipErrorNotReady: the slot's transfer is under way.
hipError_t slot_ended(const StageSlot &slot) {
  if (slot.marks == 0) {
    const hipError_t e = hipEventQuery(slot.done);
    if (e == hipErrorNotReady) (void)hipGetLastError();        // (not an error: a launch check must not find it)
    return e;
  }
  for (int i = 0; i < slot.marks; ++i)
    if (__atomic_load_n(slot_marks(slot) + i, __ATOMIC_ACQUIRE) == 0u) return hipErrorNotReady;
  return hipSuccess;
}
hipError_t slot_wait(const StageSlot &slot) {
  if (slot.marks == 0) return hipEventSynchronize(slot.done);
  for (int turn = 0; slot_ended(slot) != hipSuccess; ++turn)
    if (turn < 2000) std::this_thread::yield();
    else             std::this_thread::sleep_for(std::chrono::microseconds(20));
  return hipSuccess;
}

// A slot for an upload on `s`: *out stays null if work of other streams holds them all.
int slot_take(StageRing &r, hipStream_t s, StageSlot **out) {
  *out = nullptr;
  StageSlot *mine = nullptr;
  {
    std::lock_guard<std::mutex> lk(r.mu);
    for (StageSlot &slot : r.slot) {
      if (slot.taken) continue;
      if (slot.busy) {
        const hipError_t e = slot_ended(slot);
        if (e == hipErrorNotReady) {
          if (slot.user == s && (mine == nullptr || slot.turn < mine->turn)) mine = &slot;
          continue;
        }
        ANC_HIP(e);
      }
      slot.busy = false;
      slot.taken = true;
      *out = &slot;
      return ANC_OK;
    }
    if (mine == nullptr) return ANC_OK;
    mine->taken = true;
  }
  const hipError_t e = slot_wait(*mine);
  if (e != hipSuccess) {
    std::lock_guard<std::mutex> lk(r.mu);
    mine->taken = false;
  }
  ANC_HIP(e);
  *out = mine;
  return ANC_OK;
}
// `own`: on the ring's own stream. `kernel`: k_stage_in may do the transfer, else the runtime's copy does.
int slot_fill(StageSlot &slot, uint64_t dst, const void *src, int64_t bytes, hipStream_t s, bool own, bool kernel) {
  if (slot.mem == nullptr) ANC_HIP(hipHostMalloc(&slot.mem, (size_t)kSlotBytes + 4 * kMarks, hipHostMallocCoherent));
  if (slot.done == nullptr) ANC_HIP(hipEventCreateWithFlags(&slot.done, hipEventDisableTiming));
  memcpy(slot.mem, src, (size_t)bytes);
  kernel = kernel && !own && (dst & 15) == 0;
  uint32_t *mark = slot_marks(slot);
  slot.marks = own ? 0 : kernel ? (int)stage_blocks(bytes) : 1;
  memset(mark, 0, 4 * (size_t)slot.marks);
  // (launches return their own status: an error that someone else left on this thread says nothing about them)
  hipError_t e;
  if (kernel) {
    void *args[] = {&slot.mem, &dst, &bytes, &mark};       // (few bytes: as many loads at once as there are)
    e = hipLaunchKernel(bytes <= kFewBytes ? (const void *)k_stage_in<1> : (const void *)k_stage_in<4>, dim3((unsigned)slot.marks),
                        dim3(256), args, 0, s);
  } else {
    e = hipMemcpyAsync((void *)dst, slot.mem, (size_t)bytes, hipMemcpyHostToDevice, s);
    void *args[] = {&mark};
    if (e == hipSuccess) e = own ? hipEventRecord(slot.done, s) : hipLaunchKernel((const void *)k_stage_mark, dim3(1), dim3(64), args, 0, s);
  }
  if (e != hipSuccess) {
    (void)hipStreamSynchronize(s);          // nothing marks the end of a transfer that may be under way
    return anc_hip_fail(e, "a transfer out of a slot", __FILE__, __LINE__);
  }
  return ANC_OK;
}
// Up to a slot's worth: on return `src` may be reused and the copy into place is queued on `s`, or done.
int stage_piece(StageRing &r, uint64_t dst, const void *src, int64_t bytes, hipStream_t s, bool own, bool kernel) {
  StageSlot *slot;
  if (int rc = slot_take(r, s, &slot)) return rc;
  if (slot == nullptr) {
    ANC_HIP(hipMemcpyAsync((void *)dst, src, (size_t)bytes, hipMemcpyHostToDevice, s));
    ANC_HIP(hipStreamSynchronize(s));
    return ANC_OK;
  }
  const int rc = slot_fill(*slot, dst, src, bytes, s, own, kernel);
  std::lock_guard<std::mutex> lk(r.mu);
  slot->busy = rc == ANC_OK;
  slot->user = s;
  slot->turn = ++r.turn;
  slot->taken = false;
  return rc;
}
// The ring's device is current. On the ring's own stream (anc_upload_now) nothing may wait for other streams' kernels, as
// k_stage_in would in a hardware queue it shares with them, or on a chip that they fill.
int stage_upload(StageRing &r, int dev, uint64_t dst, const void *src, int64_t bytes, hipStream_t s, bool own) {
  const int64_t pieces = (bytes + kSlotBytes - 1) / kSlotBytes;
  const bool kernel = !own && kernel_reaches(dst, bytes, dev);
  auto piece = [&](int64_t c) {
    const int64_t at = c * kSlotBytes, left = bytes - at;
    return stage_piece(r, dst + (uint64_t)at, (const char *)src + at, left < kSlotBytes ? left : kSlotBytes, s, own, kernel);
  };
  if (bytes < kThreadedBytes) {
    for (int64_t c = 0; c < pieces; ++c)
      if (int rc = piece(c)) return rc;
    return ANC_OK;
  }
  int rcs[kCopyThreads] = {};
  char errs[kCopyThreads][sizeof(g_err)] = {};
  auto work = [&](int k) {
    for (int64_t c = k; c < pieces && rcs[k] == 0; c += kCopyThreads) rcs[k] = piece(c);
    if (rcs[k] != 0) memcpy(errs[k], g_err, sizeof(g_err));       // (the message is the thread's own)
  };
  std::thread th[kCopyThreads - 1];
  int started = 0;
  try {
    for (; started < kCopyThreads - 1; ++started)
      th[started] = std::thread([&, k = started + 1]() {
        hipStreamCaptureMode relaxed = hipStreamCaptureModeRelaxed;
        (void)hipThreadExchangeStreamCaptureMode(&relaxed);
        (void)hipSetDevice(dev);
        work(k);
      });
  } catch (const std::exception &) {
    // no thread to be had: this one copies the remaining shares too
  }
  work(0);
  for (int k = started + 1; k < kCopyThreads; ++k) work(k);
  for (int k = 0; k < started; ++k) th[k].join();
  for (int k = 0; k < kCopyThreads; ++k)
    if (rcs[k] != 0) { memcpy(g_err, errs[k], sizeof(g_err)); return rcs[k]; }
  return ANC_OK;
}
}  // namespace
extern "C" int anc_upload_async(uint64_t dst, const void *src, int64_t bytes, uint64_t stream) {
  ANC_REQUIRE(dst != 0 && src != nullptr && bytes >= 0, "anc_upload_async: bad arguments");
  if (bytes == 0) return ANC_OK;
  if (int rc = refuse_capture(anc_stream(stream))) return rc;
  StageScope on;
  if (int rc = on.enter(anc_stream(stream))) return rc;
  StageRing &r = g_ring[on.dev];
  return stage_upload(r, on.dev, dst, src, bytes, anc_stream(stream), false);
}
extern "C" int anc_upload_now(uint64_t dst, const void *src, int64_t bytes) {
  ANC_REQUIRE(dst != 0 && src != nullptr && bytes >= 0, "anc_upload_now: bad arguments");
  if (bytes == 0) return ANC_OK;
  StageScope on;
  if (int rc = on.enter(nullptr)) return rc;
  StageRing &r = g_ring[on.dev];
  {
    std::lock_guard<std::mutex> lk(r.mu);
    if (r.own == nullptr) ANC_HIP(hipStreamCreateWithFlags(&r.own, hipStreamNonBlocking));
    ++r.own_users;
  }
  int rc = stage_upload(r, on.dev, dst, src, bytes, r.own, true);
  if (rc == ANC_OK)
    if (hipError_t e = hipStreamSynchronize(r.own)) rc = anc_hip_fail(e, "hipStreamSynchronize", __FILE__, __LINE__);
  std::lock_guard<std::mutex> lk(r.mu);
  --r.own_users;
  return rc;
}
extern "C" int anc_staging_release(void) {
  for (StageRing &r : g_ring) {
    for (StageSlot &slot : r.slot) {
      {
        std::lock_guard<std::mutex> lk(r.mu);
        if (slot.taken || slot.mem == nullptr) continue;       // (in use by a call: it stays)
        slot.taken = true;
      }
      hipError_t e = slot.busy ? slot_wait(slot) : hipSuccess;
      if (e == hipSuccess && slot.done != nullptr) e = hipEventDestroy(slot.done);
      if (e == hipSuccess) e = hipHostFree(slot.mem);
      std::lock_guard<std::mutex> lk(r.mu);
      if (e == hipSuccess) slot = StageSlot{}; else slot.taken = false;
      ANC_HIP(e);
    }
    std::lock_guard<std::mutex> lk(r.mu);
    if (r.own == nullptr || r.own_users != 0) continue;
    // (a slot that a call held above may have its event from this stream: that call has waited for its transfer)
    for (StageSlot &slot : r.slot)
      if (!slot.taken && slot.user == r.own) slot.busy = false;
    ANC_HIP(hipStreamDestroy(r.own));
    r.own = nullptr;
  }
  return ANC_OK;
}
extern "C" int anc_memcpy_h2d(uint64_t dst, const void *src, int64_t bytes, uint64_t stream) {
  ANC_REQUIRE(dst != 0 && src != nullptr && bytes >= 0, "anc_memcpy_h2d: bad arguments");
  if (bytes == 0) return ANC_OK;
  if (int rc = refuse_capture(anc_stream(stream))) return rc;
  if (bytes <= 2 * kSlotBytes) {
    StageScope on;
    if (int rc = on.enter(anc_stream(stream))) return rc;
    StageRing &r = g_ring[on.dev];
    if (int rc = stage_upload(r, on.dev, dst, src, bytes, anc_stream(stream), false)) return rc;
  } else {
    // a state as it is set up, often memory that no one has touched yet: the runtime's own path takes its page
    // faults in larger pieces (622 MB of fresh zeros: 18 ms against 80 through the slots, 5 MB 0.1 ms less)
    ANC_HIP(hipMemcpyAsync((void *)dst, src, (size_t)bytes, hipMemcpyHostToDevice, anc_stream(stream)));
  }
  // complete on return: a kernel on any stream may read it
  ANC_HIP(hipStreamSynchronize(anc_stream(stream)));
  return ANC_OK;
}
extern "C" int anc_memcpy_d2h(void *dst, uint64_t src, int64_t bytes, uint64_t stream) {
  ANC_REQUIRE(dst != nullptr && src != 0 && bytes >= 0, "anc_memcpy_d2h: bad arguments");
  if (bytes == 0) return ANC_OK;
  ANC_HIP(hipMemcpyAsync(dst, (const void *)src, (size_t)bytes, hipMemcpyDeviceToHost, anc_stream(stream)));
  ANC_HIP(hipStreamSynchronize(anc_stream(stream)));
  return ANC_OK;
}
extern "C" int anc_memcpy_d2d(uint64_t dst, uint64_t src, int64_t bytes, uint64_t stream) {
  ANC_REQUIRE(dst != 0 && src != 0 && bytes >= 0, "anc_memcpy_d2d: bad arguments");
  if (bytes == 0) return ANC_OK;
  ANC_HIP(hipMemcpyAsync((void *)dst, (const void *)src, (size_t)bytes, hipMemcpyDeviceToDevice,
                         anc_stream(stream)));
  return ANC_OK;
}

extern "C" int anc_stream_create(uint64_t *stream) {
  ANC_REQUIRE(stream != nullptr, "anc_stream_create: null output");
  hipStream_t s;
  ANC_HIP(hipStreamCreate(&s));   // default priority only
  *stream = (uint64_t)s;
  return ANC_OK;
}
extern "C" int anc_stream_create_nonblocking(uint64_t *stream) {
  ANC_REQUIRE(stream != nullptr, "anc_stream_create_nonblocking: null output");
  hipStream_t s;
  ANC_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));   // not ordered against the null stream
  *stream = (uint64_t)s;
  return ANC_OK;
}
extern "C" int anc_stream_destroy(uint64_t stream) {
  ANC_REQUIRE(stream != 0, "anc_stream_destroy: the null stream is not destroyable");
  ANC_HIP(hipStreamDestroy(anc_stream(stream)));
  return ANC_OK;
}
extern "C" int anc_stream_is_capturing(uint64_t stream, int32_t *capturing) {
  ANC_REQUIRE(capturing != nullptr, "anc_stream_is_capturing: null output");
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  ANC_HIP(hipStreamIsCapturing(anc_stream(stream), &st));
  *capturing = st != hipStreamCaptureStatusNone;
  return ANC_OK;
}
extern "C" int anc_stream_sync(uint64_t stream) {
  ANC_HIP(hipStreamSynchronize(anc_stream(stream)));
  return ANC_OK;
}
extern "C" int anc_device_sync(void) {
  ANC_HIP(hipDeviceSynchronize());
  return ANC_OK;
}
extern "C" int anc_event_create(uint64_t *event) {
  ANC_REQUIRE(event != nullptr, "anc_event_create: null output");
  hipEvent_t e;
  ANC_HIP(hipEventCreate(&e));
  *event = (uint64_t)e;
  return ANC_OK;
}
extern "C" int anc_event_destroy(uint64_t event) {
  ANC_REQUIRE(event != 0, "anc_event_destroy: null event");
  ANC_HIP(hipEventDestroy((hipEvent_t)event));
  return ANC_OK;
}
extern "C" int anc_event_record(uint64_t event, uint64_t stream) {
  ANC_REQUIRE(event != 0, "anc_event_record: null event");
  ANC_HIP(hipEventRecord((hipEvent_t)event, anc_stream(stream)));
  return ANC_OK;
}
extern "C" int anc_event_sync(uint64_t event) {
  ANC_REQUIRE(event != 0, "anc_event_sync: null event");
  ANC_HIP(hipEventSynchronize((hipEvent_t)event));
  return ANC_OK;
}
extern "C" int anc_stream_wait_event(uint64_t stream, uint64_t event) {
  ANC_REQUIRE(event != 0, "anc_stream_wait_event: null event");
  ANC_HIP(hipStreamWaitEvent(anc_stream(stream), (hipEvent_t)event, 0));
  return ANC_OK;
}
extern "C" int anc_event_elapsed_ms(uint64_t start, uint64_t stop, float *ms) {
  ANC_REQUIRE(start != 0 && stop != 0 && ms != nullptr, "anc_event_elapsed_ms: bad arguments");
  ANC_HIP(hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop));
  return ANC_OK;
}

// Streaming copy: 16 bytes per lane per access, four accesses in flight per lane.
__global__ void __launch_bounds__(256) k_copy16(const anc_u32x4 *__restrict__ src,
                                                anc_u32x4 *__restrict__ dst, int64_t n_vec) {
  const int64_t base = (int64_t)blockIdx.x * 1024 + threadIdx.x;
  anc_u32x4 r[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    int64_t i = base + j * 256;
    if (i < n_vec) r[j] = __builtin_nontemporal_load(&src[i]);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    int64_t i = base + j * 256;
    if (i < n_vec) __builtin_nontemporal_store(r[j], &dst[i]);
  }
}
extern "C" int anc_copy_kernel(uint64_t dst, uint64_t src, int64_t n_bytes, uint64_t stream) {
  ANC_REQUIRE(dst != 0 && src != 0 && n_bytes > 0 && n_bytes % 16 == 0 && (dst & 15) == 0 &&
                  (src & 15) == 0,
              "anc_copy_kernel: pointers and size must be 16-byte aligned");
  int64_t n_vec = n_bytes / 16;
  int64_t blocks = (n_vec + 1023) / 1024;
  ANC_REQUIRE(blocks < (1ll << 31), "anc_copy_kernel: size too large");
  AncProfScope prof(ANC_PROF_COPY, anc_stream(stream));
  hipLaunchKernelGGL(k_copy16, dim3((unsigned)blocks), dim3(256), 0, anc_stream(stream),
                     (const anc_u32x4 *)src, (anc_u32x4 *)dst, n_vec);
  ANC_LAUNCH_CHECK();
  return ANC_OK;
}
