// The upload entry points of the library (runtime.hip, compiled for the host alone) on a stand-in for the HIP runtime:
// devices, streams that can be held, events, pageable and pinned memory. Each case checks one property and
// prints "ok"; a failed check or a call the stand-in refuses ends the program with a message.
#include <hip/hip_runtime_api.h>

#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <future>
#include <map>
#include <memory>
#include <mutex>
#include <set>
#include <string>
#include <vector>

#include <unistd.h>

extern "C" {
int anc_upload_async(uint64_t dst, const void *src, int64_t bytes, uint64_t stream);
int anc_upload_now(uint64_t dst, const void *src, int64_t bytes);
int anc_memcpy_h2d(uint64_t dst, const void *src, int64_t bytes, uint64_t stream);
int anc_staging_release(void);
int anc_stream_create(uint64_t *stream);
int anc_stream_destroy(uint64_t stream);
const char *anc_last_error(void);
}

#define CHECK(c) do { if (!(c)) { printf("line %d: %s (%s)\n", __LINE__, #c, anc_last_error()); fflush(stdout); _exit(1); } } while (0)

// ---- the stand-in
struct Stream {
  int dev;
  bool held = false, capturing = false;
  std::deque<std::function<void()>> queue;
};
struct Event { int dev; bool done = true, captured = false; Stream *on = nullptr; };
static std::mutex mu;
static std::condition_variable cv;
static Stream null_stream[4] = {{0}, {1}, {2}, {3}};
static std::set<Event *> events;
static std::map<char *, size_t> pinned;
static int live_streams = 0;
struct Region { size_t size; int dev; };
static std::map<char *, Region> device_memory;       // allocations; any other address is memory of the current device, without an end
static std::function<void()> at_copy, at_host_free;       // called on entry, where set
static bool chip_full = false;         // kernels do not start: their streams are held
static std::set<Stream *> gone;        // destroyed streams (their memory is kept, so that no new one has their address)
static thread_local int cur = 0;
static thread_local hipError_t last = hipSuccess;

static hipError_t ret(hipError_t e) { if (e != hipSuccess) last = e; return e; }
static Stream *str(hipStream_t s) { return s == nullptr ? &null_stream[cur] : (Stream *)s; }
static void push(Stream *s, std::function<void()> f) {       // mu held
  if (s->held) s->queue.push_back(f); else f();
}
static void release(Stream *s) {
  std::lock_guard<std::mutex> lk(mu);
  s->held = false;
  while (!s->queue.empty()) { s->queue.front()(); s->queue.pop_front(); }
  cv.notify_all();
}
static void look_at(Stream *s) {              // (in the runtime: at memory that is freed, or another stream's)
  if (gone.count(s) == 0) return;
  printf("a stream that is gone is looked at\n");
  fflush(stdout);
  _exit(1);
}
static bool is_pinned(const void *p) {
  auto it = pinned.upper_bound((char *)p);
  return it != pinned.begin() && (--it, (char *)p < it->first + it->second);
}
static const Region *region_of(const void *p, char **base) {
  auto it = device_memory.upper_bound((char *)p);
  if (it == device_memory.begin() || (--it, (char *)p >= it->first + it->second.size)) return nullptr;
  *base = it->first;
  return &it->second;
}
static std::string &kernel_of(const void *f) {       // (registered before this file's globals are made)
  static std::map<const void *, std::string> *names = new std::map<const void *, std::string>;
  return (*names)[f];
}
static uint64_t handle(Stream *s) { return (uint64_t)s; }

extern "C" {
hipError_t hipGetDevice(int *d) { *d = cur; return hipSuccess; }
hipError_t hipSetDevice(int d) { cur = d; return hipSuccess; }
hipError_t hipGetLastError(void) { hipError_t e = last; last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t) { return "refused by the stand-in"; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  std::lock_guard<std::mutex> lk(mu);
  *p = malloc(n);
  pinned[(char *)*p] = n;
  return hipSuccess;
}
hipError_t hipHostFree(void *p) { if (at_host_free) at_host_free(); std::lock_guard<std::mutex> lk(mu); pinned.erase((char *)p); free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  std::lock_guard<std::mutex> lk(mu);
  Event *n = new Event{cur};
  events.insert(n);
  *e = (hipEvent_t)n;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { std::lock_guard<std::mutex> lk(mu); events.erase((Event *)e); delete (Event *)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::lock_guard<std::mutex> lk(mu);
  Event *ev = (Event *)e;
  Stream *st = str(s);
  if (ev->dev != st->dev) return ret(hipErrorInvalidHandle);       // as the runtime does
  ev->captured = st->capturing;
  ev->on = st;
  ev->done = false;
  push(st, [ev] { ev->done = true; });
  return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
  std::lock_guard<std::mutex> lk(mu);
  look_at(((Event *)e)->on);
  if (((Event *)e)->captured) return ret(hipErrorCapturedEvent);
  return ((Event *)e)->done ? hipSuccess : ret(hipErrorNotReady);
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  std::unique_lock<std::mutex> lk(mu);
  look_at(((Event *)e)->on);
  if (((Event *)e)->captured) return ret(hipErrorCapturedEvent);
  cv.wait(lk, [e] { return ((Event *)e)->done; });
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  std::lock_guard<std::mutex> lk(mu);
  char *base;
  const Region *r = region_of(p, &base);
  *a = hipPointerAttribute_t{};
  a->type = hipMemoryTypeDevice;
  a->device = r != nullptr ? r->dev : cur;
  return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t *b, size_t *size, hipDeviceptr_t p) {
  std::lock_guard<std::mutex> lk(mu);
  char *base = nullptr;
  const Region *r = region_of(p, &base);
  *b = r != nullptr ? base : nullptr;
  *size = r != nullptr ? r->size : SIZE_MAX;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t s) {
  if (at_copy) at_copy();
  std::unique_lock<std::mutex> lk(mu);
  Stream *st = str(s);
  if (st->capturing) return hipSuccess;                            // (recorded)
  char *base;
  const Region *r = region_of(dst, &base);
  if (r != nullptr && (char *)dst + n > base + r->size) return ret(hipErrorInvalidValue);
  if (is_pinned(src)) { push(st, [=] { memcpy(dst, src, n); }); return hipSuccess; }
  cv.wait(lk, [st] { return !st->held; });                         // pageable: in the stream's turn, and blocking
  memcpy(dst, src, n);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  std::unique_lock<std::mutex> lk(mu);
  Stream *st = str(s);
  if (st->capturing) return ret(hipErrorStreamCaptureUnsupported);
  cv.wait(lk, [st] { return !st->held; });
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)new Stream{cur}; ++live_streams; return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t *s) { return hipStreamCreateWithFlags(s, 0); }
hipError_t hipStreamDestroy(hipStream_t s) { std::lock_guard<std::mutex> lk(mu); gone.insert((Stream *)s); --live_streams; return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t *d) { *d = str(s)->dev; return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c) {
  *c = str(s)->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
// (the kernels of these entry points: k_stage_in copies, source, destination, bytes, and then sets a mark per block; k_stage_mark
// sets one)
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **args, size_t, hipStream_t s) {
  const bool copies = kernel_of(f).find("k_stage_in") != std::string::npos;
  uint32_t *mark = *(uint32_t **)args[copies ? 3 : 0];
  const void *src = copies ? *(const void **)args[0] : nullptr;
  char *dst = copies ? *(char **)args[1] : nullptr;
  const int64_t n = copies ? *(int64_t *)args[2] : 0;
  std::lock_guard<std::mutex> lk(mu);
  Stream *st = str(s);
  if (!is_pinned(mark + grid.x - 1) || (copies && !is_pinned(src))) return ret(hipErrorInvalidValue);
  char *base;
  const Region *r = region_of(dst, &base);
  const char *fault = r == nullptr ? nullptr : r->dev != st->dev ? "a kernel writes another device's memory"
                                             : dst + n > base + r->size ? "a kernel writes past an allocation" : nullptr;
  if (fault != nullptr) { printf("%s\n", fault); fflush(stdout); _exit(1); }
  if (chip_full) st->held = true;
  push(st, [=] {
    if (copies) memcpy(dst, src, (size_t)n);
    for (unsigned i = 0; i < grid.x; ++i) mark[i] = 1;
  });
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *, int *) { kernel_of(f) = name; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipErrorInvalidValue; }        // (stubs of kernels launched otherwise)
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipErrorInvalidValue; }
}

// ---- the cases
static std::vector<char> bytes(size_t n, int seed) {
  std::vector<char> v(n);
  for (size_t i = 0; i < n; ++i) v[i] = (char)(i * 7 + i / 251 + (size_t)seed);
  return v;
}

// Uploads of every kind with each device current in turn, and on a stream of another device than the current one:
// all arrive, and the caller's device stays current.
static void two_devices() {
  Stream s[2] = {{0}, {1}};
  for (int round = 0; round < 2; ++round)
    for (int dev = 0; dev < 2; ++dev) {
      cur = dev;
      for (size_t n : {100u, 600u << 10, 9u << 20}) {
        const std::vector<char> want = bytes(n, dev + round);
        for (Stream *on : {&s[0], &s[1], (Stream *)nullptr}) {
          std::vector<char> src = want, a(n), b(n), c(n);
          CHECK(anc_upload_async((uint64_t)a.data(), src.data(), (int64_t)n, handle(on)) == 0);
          CHECK(anc_memcpy_h2d((uint64_t)b.data(), src.data(), (int64_t)n, handle(on)) == 0);
          CHECK(anc_upload_now((uint64_t)c.data(), src.data(), (int64_t)n) == 0);
          CHECK(a == want && b == want && c == want && cur == dev);
        }
      }
    }
  CHECK(pinned.size() <= 16 && events.size() == pinned.size() && live_streams == 2);       // 8 slots per device and no more
  CHECK(anc_staging_release() == 0);
  CHECK(pinned.empty() && events.empty() && live_streams == 0);
}

static bool soon(std::future<int> &f) { return f.wait_for(std::chrono::seconds(5)) == std::future_status::ready; }

// Work that holds stream A, and with it every slot, holds no upload on stream B, nor one that is complete on return,
// from the same thread or while another thread waits for A.
static void other_streams_do_not_wait() {
  Stream A{0}, B{0};
  const size_t n = 100;
  const std::vector<char> want = bytes(n, 1);
  std::vector<std::vector<char>> onA(9, std::vector<char>(n));
  std::future<int> ninth;
  A.held = true;
  for (int i = 0; i < 8; ++i) CHECK(anc_upload_async((uint64_t)onA[(size_t)i].data(), want.data(), (int64_t)n, handle(&A)) == 0);
  for (int blocked = 0; blocked < 2; ++blocked) {
    std::future<int> onB = std::async(std::launch::async, [&]() -> int {
      std::vector<char> src = want, a(n), b(n), c(n);
      const int rc = anc_upload_async((uint64_t)a.data(), src.data(), (int64_t)n, handle(&B)) |
                     anc_upload_now((uint64_t)b.data(), src.data(), (int64_t)n) |
                     anc_memcpy_h2d((uint64_t)c.data(), src.data(), (int64_t)n, handle(&B));
      return rc != 0 || a != want || b != want || c != want || hipGetLastError() != hipSuccess;
    });
    CHECK(soon(onB) && onB.get() == 0);
    if (blocked == 0) {
      ninth = std::async(std::launch::async, [&]() -> int {
        return anc_upload_async((uint64_t)onA[8].data(), want.data(), (int64_t)n, handle(&A));
      });
      CHECK(ninth.wait_for(std::chrono::milliseconds(200)) == std::future_status::timeout);       // A's own turn
    }
  }
  release(&A);
  CHECK(ninth.get() == 0);
  for (const auto &a : onA) CHECK(a == want);
  CHECK(anc_staging_release() == 0);
  CHECK(pinned.empty() && events.empty() && live_streams == 0);
}

// Several threads on streams of their own, sizes on both sides of a slot and of the threaded copy.
static void many_threads() {
  std::vector<std::future<int>> all;
  for (int t = 0; t < 6; ++t)
    all.push_back(std::async(std::launch::async, [t] {
      Stream s{t & 1};
      for (int i = 0; i < 20; ++i)
        for (size_t n : {64u, (512u << 10) + 1, 9u << 20}) {
          if (n > (8u << 20) && i % 8 != 0) continue;
          const std::vector<char> want = bytes(n, t * 31 + i);
          std::vector<char> src = want, a(n);
          if (anc_upload_async((uint64_t)a.data(), src.data(), (int64_t)n, handle(&s)) != 0) return 1;
          memset(src.data(), 0, n);
          if (a != want) return 2;
        }
      return 0;
    }));
  for (auto &f : all) CHECK(f.get() == 0);
  CHECK(anc_staging_release() == 0);
  CHECK(pinned.empty() && events.empty());
}

// Uploads on a stream under capture are refused and leave no slot behind whose event belongs to the graph; those that
// are complete on return go through meanwhile, and so does everything afterwards.
static void capture() {
  Stream s{0}, other{0};
  const size_t n = 100;
  const std::vector<char> want = bytes(n, 1);
  s.capturing = true;
  for (size_t big : {n, (size_t)2 << 20}) {
    std::vector<char> src(big), a(big);
    CHECK(anc_upload_async((uint64_t)a.data(), src.data(), (int64_t)big, handle(&s)) != 0);
    CHECK(anc_memcpy_h2d((uint64_t)a.data(), src.data(), (int64_t)big, handle(&s)) != 0);
  }
  for (int captured = 1; captured >= 0; --captured) {
    s.capturing = captured != 0;
    for (int i = 0; i < 10; ++i) {
      std::vector<char> a(n), b(n);
      CHECK(anc_upload_now((uint64_t)a.data(), want.data(), (int64_t)n) == 0);
      CHECK(anc_upload_async((uint64_t)b.data(), want.data(), (int64_t)n, handle(captured ? &other : &s)) == 0);
      CHECK(a == want && b == want && hipGetLastError() == hipSuccess);
    }
  }
}

// Streams come and go with the objects that made them: uploads afterwards go through the same slots, whatever the
// events of those streams would say by then.
static void streams_that_end() {
  const size_t n = 100;
  const std::vector<char> want = bytes(n, 1);
  Stream stays{0};
  for (int round = 0; round < 4; ++round) {
    uint64_t s = 0;
    CHECK(anc_stream_create(&s) == 0);
    std::vector<std::vector<char>> a(12, std::vector<char>(n));
    for (auto &x : a) CHECK(anc_upload_async((uint64_t)x.data(), want.data(), (int64_t)n, s) == 0);
    CHECK(anc_stream_destroy(s) == 0);
    for (const auto &x : a) CHECK(x == want);
    for (int i = 0; i < 12; ++i) {
      std::vector<char> b(n);
      CHECK(anc_upload_async((uint64_t)b.data(), want.data(), (int64_t)n, handle(&stays)) == 0);
      CHECK(b == want && hipGetLastError() == hipSuccess);
    }
  }
  // a stream that ends without the library's knowledge
  Stream other{0};
  for (int i = 0; i < 3; ++i) {
    std::vector<char> b(n);
    CHECK(anc_upload_async((uint64_t)b.data(), want.data(), (int64_t)n, handle(&other)) == 0);
  }
  gone.insert(&other);
  for (int i = 0; i < 12; ++i) {
    std::vector<char> b(n);
    CHECK(anc_upload_async((uint64_t)b.data(), want.data(), (int64_t)n, handle(&stays)) == 0);
    CHECK(b == want && hipGetLastError() == hipSuccess);
  }
  CHECK(pinned.size() <= 8 && events.size() <= 8);
  CHECK(anc_staging_release() == 0);
  CHECK(pinned.empty() && events.empty() && live_streams == 0);
}

// Kernels of other streams that hold every compute unit, or the hardware queue, do not hold uploads that are complete on return.
static void now_waits_for_no_kernel() {
  chip_full = true;
  for (size_t n : {100u, 600u << 10, 9u << 20}) {
    const std::vector<char> want = bytes(n, 1);
    std::vector<char> a(n);
    std::future<int> f = std::async(std::launch::async, [&] { return anc_upload_now((uint64_t)a.data(), want.data(), (int64_t)n); });
    CHECK(soon(f) && f.get() == 0 && a == want);
  }
  CHECK(anc_staging_release() == 0);
  CHECK(pinned.empty() && events.empty() && live_streams == 0);
}

// Memory of another device than the stream's (or, without a stream, the current one): no kernel writes there.
static void memory_of_another_device() {
  Stream s{0};
  for (size_t n : {112u, 600u << 10, 9u << 20}) {
    const std::vector<char> want = bytes(n, 1);
    std::vector<char> a(n), b(n), c(n), d(n);
    for (std::vector<char> *v : {&a, &b, &c, &d}) device_memory[v->data()] = Region{n, 1};
    CHECK(anc_upload_async((uint64_t)a.data(), want.data(), (int64_t)n, handle(&s)) == 0);
    CHECK(anc_memcpy_h2d((uint64_t)b.data(), want.data(), (int64_t)n, handle(&s)) == 0);
    CHECK(anc_upload_now((uint64_t)c.data(), want.data(), (int64_t)n) == 0);
    CHECK(anc_upload_async((uint64_t)d.data(), want.data(), (int64_t)n, 0) == 0);
    CHECK(a == want && b == want && c == want && d == want && cur == 0);
    device_memory.clear();
  }
}

// An error that someone else left on the thread is not an upload's: it succeeds, and its slot is not taken again before its
// transfer has ended.
static void errors_of_others() {
  for (size_t n : {112u, 300u << 10}) {
    Stream A{0};
    const std::vector<char> first = bytes(n, 1), second = bytes(n, 2);
    std::vector<char> a(n), b(n);
    A.held = true;
    last = hipErrorInvalidValue;
    CHECK(anc_upload_async((uint64_t)a.data(), first.data(), (int64_t)n, handle(&A)) == 0);
    CHECK(anc_upload_async((uint64_t)b.data(), second.data(), (int64_t)n, handle(&A)) == 0);
    release(&A);
    CHECK(a == first && b == second);
  }
}

// What does not fit into its allocation is refused, and nothing behind it is touched; anywhere inside it fits.
static void past_the_end() {
  Stream s{0};
  for (size_t n : {112u, 600u << 10, (9u << 20) - 4080})
    for (size_t at : {0u, 16u, 32u}) {
      const std::vector<char> want = bytes(n, 1), rest = bytes(64, 2);
      std::vector<char> a(n + 64);
      memcpy(a.data() + n, rest.data(), 64);
      device_memory[a.data()] = Region{n, 0};
      const uint64_t dst = (uint64_t)a.data() + at;
      CHECK(anc_upload_async(dst, want.data(), (int64_t)(n - at), handle(&s)) == 0);
      CHECK(memcmp(a.data() + at, want.data(), n - at) == 0);
      CHECK(anc_upload_async(dst, want.data(), (int64_t)(n - at + 1), handle(&s)) != 0);
      CHECK(anc_memcpy_h2d(dst, want.data(), (int64_t)(n - at + 64), handle(&s)) != 0);
      CHECK(anc_upload_now(dst, want.data(), (int64_t)(n - at + 1)) != 0);
      CHECK(memcmp(a.data() + n, rest.data(), 64) == 0);
      device_memory.clear();
    }
}

// Streams that others made and destroyed leave every slot usable, also where a transfer was under way: nobody looks at
// them again, and eight uploads on a stream that is held still find a slot each.
static void streams_of_others() {
  const size_t n = 100;
  const std::vector<char> want = bytes(n, 1);
  for (int round = 0; round < 3; ++round) {
    std::vector<std::unique_ptr<Stream>> s;
    std::vector<std::vector<char>> a(8, std::vector<char>(n + 4));
    for (size_t i = 0; i < 8; ++i) {
      s.emplace_back(new Stream{0});
      s[i]->held = i % 2 != 0;
      CHECK(anc_upload_async((uint64_t)a[i].data() + i / 2, want.data(), (int64_t)n, handle(s[i].get())) == 0);
      gone.insert(s[i].get());
    }
    for (auto &x : s) release(x.get());
    for (size_t i = 0; i < 8; ++i) CHECK(memcmp(a[i].data() + i / 2, want.data(), n) == 0);
    Stream A{0};
    A.held = true;
    std::vector<std::vector<char>> b(8, std::vector<char>(n));
    std::future<int> f = std::async(std::launch::async, [&] {
      int rc = 0;
      for (auto &x : b) rc |= anc_upload_async((uint64_t)x.data(), want.data(), (int64_t)n, handle(&A));
      return rc;
    });
    CHECK(soon(f) && f.get() == 0);
    release(&A);
    for (auto &x : b) CHECK(x == want);
    gone.clear();
  }
  CHECK(anc_staging_release() == 0);
  CHECK(pinned.empty() && events.empty() && live_streams == 0);
}

// The ring is given back while an upload that is complete on return holds a slot, and that call ends before the ring's own
// stream is destroyed: the slot stays, and nobody looks at that stream again.
static void released_beside_an_upload() {
  const size_t n = 100;
  const std::vector<char> want = bytes(n, 1);
  std::vector<char> a(n), b(n), c(n);
  Stream A{0};
  A.held = true;                       // two slots in use, so that there is one to be freed beside the call's
  CHECK(anc_upload_async((uint64_t)a.data(), want.data(), (int64_t)n, handle(&A)) == 0);
  CHECK(anc_upload_async((uint64_t)b.data(), want.data(), (int64_t)n, handle(&A)) == 0);
  release(&A);
  std::promise<void> copying, freeing;
  at_copy = [&] { copying.set_value(); freeing.get_future().wait(); };
  std::future<int> now = std::async(std::launch::async, [&] { return anc_upload_now((uint64_t)c.data(), want.data(), (int64_t)n); });
  copying.get_future().wait();
  int ended = -1;
  at_host_free = [&] { freeing.set_value(); ended = now.get(); };
  CHECK(anc_staging_release() == 0);
  at_copy = at_host_free = nullptr;
  CHECK(ended == 0 && c == want && pinned.size() == 1 && live_streams == 0);
  for (int i = 0; i < 12; ++i) {
    std::vector<char> x(n), y(n);
    CHECK(anc_upload_async((uint64_t)x.data(), want.data(), (int64_t)n, handle(&A)) == 0);
    CHECK(anc_upload_now((uint64_t)y.data(), want.data(), (int64_t)n) == 0);
    CHECK(x == want && y == want);
  }
  CHECK(anc_staging_release() == 0);
  CHECK(pinned.empty() && events.empty() && live_streams == 0);
}

int main(int argc, char **argv) {
  const std::map<std::string, void (*)()> cases = {{"two_devices", two_devices}, {"other_streams_do_not_wait", other_streams_do_not_wait},
                                                   {"many_threads", many_threads}, {"capture", capture}, {"streams_that_end", streams_that_end},
                                                   {"now_waits_for_no_kernel", now_waits_for_no_kernel},
                                                   {"memory_of_another_device", memory_of_another_device}, {"errors_of_others", errors_of_others}, {"past_the_end", past_the_end},
                                                   {"streams_of_others", streams_of_others}, {"released_beside_an_upload", released_beside_an_upload}};
  if (argc != 2 || cases.find(argv[1]) == cases.end()) return 2;
  cases.at(argv[1])();
  printf("ok\n");
  return 0;
}
