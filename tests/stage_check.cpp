// Checker for tests/test_stage_host.py: the staged host-to-device copies
// (tqsv_stage.cpp, included below) over a small imitation of HIP streams, whose
// work runs on threads of their own and can be held back.
//   stage_check <scenario>
// The imitation reports what a stream under capture or a destroyed stream must
// not see: synchronisation, event records, other work.
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <deque>
#include <functional>
#include <string>
#include <thread>
#include <vector>

#include "tqsv_stage.cpp"

namespace {

std::atomic<int> g_fault{0};
void fault(const char* what) {
  std::printf("fault: %s\n", what);
  g_fault = 1;
}
void expect(bool ok, const char* what) {
  if (!ok) fault(what);
}

struct Event {
  std::mutex m;
  std::condition_variable cv;
  int recorded = 0, reached = 0;
};

struct Stream {
  std::mutex m;
  std::condition_variable cv;
  std::deque<std::function<void()>> work;
  bool held = false, busy = false, quit = false;
  std::atomic<bool> capturing{false}, gone{false};
  std::thread t;
  Stream() : t([this] { run(); }) {}
  ~Stream() {
    hold(false);
    drain();
    {
      std::lock_guard<std::mutex> l(m);
      quit = true;
    }
    cv.notify_all();
    t.join();
  }
  void run() {
    std::unique_lock<std::mutex> l(m);
    for (;;) {
      cv.wait(l, [&] { return quit || (!held && !work.empty()); });
      if (work.empty()) return;
      auto f = std::move(work.front());
      work.pop_front();
      busy = true;
      l.unlock();
      f();
      l.lock();
      busy = false;
      cv.notify_all();
    }
  }
  void push(std::function<void()> f) {
    std::lock_guard<std::mutex> l(m);
    work.push_back(std::move(f));
    cv.notify_all();
  }
  void hold(bool on) {
    std::lock_guard<std::mutex> l(m);
    held = on;
    cv.notify_all();
  }
  void drain() {
    std::unique_lock<std::mutex> l(m);
    cv.wait(l, [&] { return work.empty() && !busy; });
  }
};

Stream* S(hipStream_t s) { return reinterpret_cast<Stream*>(s); }
hipStream_t H(Stream& s) { return reinterpret_cast<hipStream_t>(&s); }
// a call on a stream: is it allowed?
hipError_t use(hipStream_t s, const char* what) {
  if (S(s)->gone) {
    fault((std::string(what) + " on a destroyed stream").c_str());
    return hipErrorInvalidHandle;
  }
  if (S(s)->capturing) {
    fault((std::string(what) + " on a stream under capture").c_str());
    return hipErrorStreamCaptureUnsupported;
  }
  return hipSuccess;
}
std::function<void()> g_after_event_create;  // test hook
int g_device = 0;
std::atomic<int> g_allocations{0};

}  // namespace

extern "C" {
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
  *st = S(s)->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
hipError_t hipGetDevice(int* d) {
  *d = g_device;
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) {
  ++g_allocations;
  *p = std::aligned_alloc(4096, (n + 4095) / 4096 * 4096);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
  const hipError_t e = use(st, "copy");
  if (e != hipSuccess) return e;
  S(st)->push([=] { std::memcpy(d, s, n); });
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t st) {
  const hipError_t e = use(st, "synchronisation");
  if (e == hipSuccess) S(st)->drain();
  return e;
}
hipError_t hipDeviceSynchronize() {
  fault("device synchronisation");
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  Event* ev = new Event;
  if (g_after_event_create) g_after_event_create();
  *e = reinterpret_cast<hipEvent_t>(ev);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
  const hipError_t r = use(st, "event record");
  if (r != hipSuccess) return r;
  Event* ev = reinterpret_cast<Event*>(e);
  int k;
  {
    std::lock_guard<std::mutex> l(ev->m);
    k = ++ev->recorded;
  }
  S(st)->push([=] {
    std::lock_guard<std::mutex> l(ev->m);
    ev->reached = k;
    ev->cv.notify_all();
  });
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  Event* ev = reinterpret_cast<Event*>(e);
  std::unique_lock<std::mutex> l(ev->m);
  ev->cv.wait(l, [&] { return ev->reached >= ev->recorded; });
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t st, hipEvent_t e, unsigned) {
  const hipError_t r = use(st, "wait");
  if (r != hipSuccess) return r;
  Event* ev = reinterpret_cast<Event*>(e);
  int k;
  {
    std::lock_guard<std::mutex> l(ev->m);
    k = ev->recorded;
  }
  S(st)->push([=] {  // an event that was never recorded is not waited for
    std::unique_lock<std::mutex> l(ev->m);
    ev->cv.wait(l, [&] { return ev->reached >= k; });
  });
  return hipSuccess;
}
}

namespace tqsv {
int fail(int code, const std::string& msg) {
  std::printf("error: %s\n", msg.c_str());
  return code;
}
int hip_fail(hipError_t, const char* what) {
  std::printf("hip error: %s\n", what);
  return TQSV_EDEVICE;
}
hipError_t k_stage_copy(void* d, const void* s, size_t n, uint64_t* words, uint64_t nwords,
                        uint64_t number, hipStream_t st) {
  const hipError_t e = use(st, "copy");
  if (e != hipSuccess) return e;
  S(st)->push([=] {  // the pieces in no order: the last one first
    for (uint32_t p = stage_pieces(n); p-- > 0;) {
      const size_t at = p * STAGE_PIECE, len = n - at < STAGE_PIECE ? n - at : STAGE_PIECE;
      std::memcpy(static_cast<char*>(d) + at, static_cast<const char*>(s) + at, len);
      __atomic_store_n(words + (number + p) % nwords, number + p, __ATOMIC_RELEASE);
      std::this_thread::yield();
    }
  });
  return hipSuccess;
}
}  // namespace tqsv

namespace {
using tqsv::stage_copy;
using tqsv::StreamMark;

void pause_ms(int ms) { std::this_thread::sleep_for(std::chrono::milliseconds(ms)); }

// a table on the "device", an update of it queued on `s`, a use of it on `t`
struct Object {
  static constexpr size_t kWords = 9000;  // several pieces, the last one partial
  std::vector<uint32_t> dev = std::vector<uint32_t>(kWords, 0);
  StreamMark mark;
  int update(Stream& s, uint32_t v) {
    const std::vector<uint32_t> h(kWords, v);
    const int rc = stage_copy(dev.data(), h.data(), h.size() * 4, H(s));
    mark.queued(H(s));
    return rc;
  }
  // queues the use and reports what it read
  void use_on(Stream& t, std::vector<uint32_t>* got) {
    if (mark.wait(H(t)) != hipSuccess) fault("wait failed");
    t.push([this, got] { *got = dev; });
  }
};
bool all(const std::vector<uint32_t>& v, uint32_t x) {
  for (uint32_t e : v)
    if (e != x) return false;
  return v.size() == Object::kWords;
}
// lets a held stream go on after a while; joined before the streams go
struct Release {
  std::thread t;
  Release(Stream& s, int ms) : t([&s, ms] {
    pause_ms(ms);
    s.hold(false);
  }) {}
  Release(Release&&) = default;
  ~Release() {
    if (t.joinable()) t.join();
  }
};

// one updated object used by two threads on two streams
void two_threads() {
  Stream a, b, c;
  Object o;
  a.hold(true);
  o.update(a, 7);
  std::atomic<int> made{0};
  g_after_event_create = [&] {  // both threads are in it, one returns late
    const int k = ++made;
    for (int i = 0; i < 100 && made < 2; ++i) pause_ms(1);
    if (k == 2) pause_ms(30);
  };
  std::vector<uint32_t> gb, gc;
  Release r(a, 150);
  std::thread t([&] { o.use_on(b, &gb); });
  o.use_on(c, &gc);
  t.join();
  b.drain();
  c.drain();
  expect(all(gb, 7) && all(gc, 7), "a thread read the table before its copy");
  a.drain();
}

// the updating stream has begun a capture when another stream uses the object
void updater_under_capture() {
  Stream a, b;
  Object o;
  a.hold(true);
  o.update(a, 7);
  a.capturing = true;
  Release r(a, 50);
  std::vector<uint32_t> got;
  o.use_on(b, &got);
  b.drain();
  expect(all(got, 7), "the table was read before its copy");
}

// updated and captured on one stream: the graph is replayed on another
void capture_on_own_stream() {
  Stream a, b;
  Object o;
  a.hold(true);
  o.update(a, 7);
  a.capturing = true;
  Release r(a, 50);
  expect(o.mark.wait(H(a)) == hipSuccess, "wait failed");
  a.capturing = false;
  std::vector<uint32_t> got;
  b.push([&] { got = o.dev; });  // the replay
  b.drain();
  expect(all(got, 7), "the replay read the table before its copy");
}

// an object used under capture is updated, and the graph replayed elsewhere
void update_after_capture() {
  Stream a, b;
  Object o;
  o.update(a, 7);
  b.capturing = true;
  expect(o.mark.wait(H(b)) == hipSuccess, "wait failed");
  b.capturing = false;
  for (uint32_t v = 8; v < 11; ++v) {
    a.hold(true);
    Release r(a, 30);
    o.update(a, v);
    std::vector<uint32_t> got;
    b.push([&] { got = o.dev; });  // the replay
    b.drain();
    expect(all(got, v), "the replay read the table before its copy");
  }
}

// the ring comes round while a stream of earlier copies is under capture, or gone
void ring(bool gone) {
  Stream a, b;
  Object o, p;
  o.update(a, 1);
  a.drain();
  (gone ? a.gone : a.capturing) = true;
  std::vector<uint32_t> h(16384, 5);
  std::vector<uint32_t> big(16384, 0);
  for (int k = 0; k < 64; ++k) {  // 64 KiB each: four times round
    h[0] = (uint32_t)k;
    expect(stage_copy(big.data(), h.data(), h.size() * 4, H(b)) == 0, "copy refused");
  }
  b.drain();
  expect(big[0] == 63 && big[16383] == 5, "a later copy is wrong");
}

// more copies than the ring or the ticket words hold, on streams that are held
// in turn: every copy has its own bytes
void in_flight() {
  constexpr uint32_t kMost = 3000;
  Stream s[2];
  std::vector<Release> releases;
  std::vector<std::vector<uint32_t>> dev(3000, std::vector<uint32_t>(kMost, 0));
  for (int k = 0; k < 3000; ++k) {
    Stream& t = s[k % 2];
    if (k % 97 == 0) {
      t.hold(true);
      releases.emplace_back(t, 3);
    }
    const std::vector<uint32_t> h(kMost, 1000u + (uint32_t)k);
    // (sizes from one word to 12 KB: up to three pieces)
    expect(stage_copy(dev[k].data(), h.data(), 4u * (1u + (uint32_t)(37 * k) % kMost), H(t)) == 0,
           "refused");
  }
  releases.clear();
  s[0].drain();
  s[1].drain();
  for (int k = 0; k < 3000; ++k)
    for (uint32_t i = 0; i < kMost; ++i)
      if (dev[k][i] != (i < 1u + (uint32_t)(37 * k) % kMost ? 1000u + (uint32_t)k : 0u)) {
        fault("a copy's bytes are wrong");
        return;
      }
}

// the updating thread ends before the object is used elsewhere
void thread_ends() {
  Stream a, b;
  Object o;
  a.hold(true);
  std::thread t([&] { o.update(a, 9); });
  Release r(a, 50);
  t.join();
  std::vector<uint32_t> got;
  o.use_on(b, &got);
  b.drain();
  expect(all(got, 9), "the table was read before its copy");
}

// a thread that goes back and forth between devices keeps its ring
void two_devices() {
  Stream s[2];
  uint32_t dev[2] = {0, 0};
  for (uint32_t k = 1; k <= 20; ++k) {
    g_device = (int)(k % 2);
    expect(stage_copy(&dev[g_device], &k, 4, H(s[g_device])) == 0, "refused");
  }
  s[0].drain();
  s[1].drain();
  expect(dev[0] == 20 && dev[1] == 19, "a copy is wrong");
  expect(g_allocations == 1, "the ring was allocated again");
}

// refused on a stream under capture
void refused() {
  Stream a;
  a.capturing = true;
  uint32_t d = 0, h = 1;
  expect(stage_copy(&d, &h, 4, H(a)) == TQSV_EUNSUPPORTED, "accepted under capture");
  expect(d == 0, "copied under capture");
}

}  // namespace

int main(int argc, char** argv) {
  const std::string w = argc > 1 ? argv[1] : "";
  if (w == "two_threads") two_threads();
  else if (w == "updater_under_capture") updater_under_capture();
  else if (w == "capture_on_own_stream") capture_on_own_stream();
  else if (w == "update_after_capture") update_after_capture();
  else if (w == "ring_capture") ring(false);
  else if (w == "ring_gone") ring(true);
  else if (w == "in_flight") in_flight();
  else if (w == "thread_ends") thread_ends();
  else if (w == "two_devices") two_devices();
  else if (w == "refused") refused();
  else return 2;
  if (g_fault) return 1;
  std::printf("ok\n");
  return 0;
}
