// tqsv_stage.h - host-to-device copies of small tables without synchronising
// (tqsv_stage.cpp).
#ifndef TQSV_STAGE_H
#define TQSV_STAGE_H

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <memory>
#include <mutex>

namespace tqsv {

struct StageTickets;

// A place in a thread's sequence of staged copies: reached when the pieces with
// these numbers, and with them what their stream held before, have run.
struct StagePoint {
  std::shared_ptr<StageTickets> of;
  uint64_t first = 0, last = 0;
  // the host waits; no call on any stream
  void wait() const;
};

// Queues the copy of `bytes` from host memory (free to change or go on return)
// to the device.  Refused under stream capture: a replay would read what later
// copies left in the staging buffer.
int stage_copy(void* dst, const void* src, size_t bytes, hipStream_t st);
// the calling thread's last staged copy
StagePoint stage_point();

// The stream on which copies for an object were queued, and their place.  Uses
// on that stream follow them anyway; the first use on another one waits on the
// host until they have run (a device-side wait needs an event, which is a
// packet for the device at every update, or recorded later on a stream that
// may be under capture, or gone, by then).  A replay of a captured graph passes
// no such place, on whatever stream it runs: a use under capture waits on its own
// stream too, and from then on the object's copies are waited for where they are
// queued.  Several threads may use an object.
class StreamMark {
 public:
  StreamMark() = default;
  StreamMark(const StreamMark&) = delete;
  StreamMark& operator=(const StreamMark&) = delete;
  // the calling thread's staged copies so far
  void queued(hipStream_t st) {
    std::lock_guard<std::mutex> lock(m_);
    at_ = stage_point();
    st_ = st;
    if (captured_) finish();
  }
  void clear() {
    std::lock_guard<std::mutex> lock(m_);
    at_ = StagePoint{};
  }
  hipError_t wait(hipStream_t st) {
    std::lock_guard<std::mutex> lock(m_);
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    const hipError_t e = hipStreamIsCapturing(st, &cs);
    if (e != hipSuccess) return e;
    if (cs != hipStreamCaptureStatusNone) captured_ = true;
    // (each thread has a stream of its own behind hipStreamPerThread)
    if (captured_ || st != st_ || st == hipStreamPerThread) finish();
    return hipSuccess;
  }

 private:
  void finish() {
    at_.wait();
    at_ = StagePoint{};
  }

  std::mutex m_;
  StagePoint at_;
  hipStream_t st_ = nullptr;
  bool captured_ = false;
};

}  // namespace tqsv

#endif
