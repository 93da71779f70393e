// tqsv_stage.h - host-to-device copies of small tables without synchronising
// (tqsv_stage.cpp).
#ifndef TQSV_STAGE_H
#define TQSV_STAGE_H

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace tqsv {

// Queues the copy of `bytes` from host memory (free to change or go on return)
// to the device.  Refused under stream capture: a replay would read what later
// copies left in the staging buffer.
int stage_copy(void* dst, const void* src, size_t bytes, hipStream_t st);

// The stream on which copies for an object were queued.  Uses on that stream
// follow them anyway; a use on another stream waits for it, through an event
// that is recorded at the first such use (a record is a packet for the device to process).
class StreamMark {
 public:
  StreamMark() = default;
  StreamMark(const StreamMark&) = delete;
  StreamMark& operator=(const StreamMark&) = delete;
  ~StreamMark() {
    if (ev_) (void)hipEventDestroy(ev_);
  }
  void queued(hipStream_t st) {
    st_ = st;
    set_ = true;
    recorded_ = false;
  }
  void clear() { set_ = false; }
  hipError_t wait(hipStream_t st) {
    if (!set_ || st == st_) return hipSuccess;
    hipError_t e = ev_ ? hipSuccess : hipEventCreateWithFlags(&ev_, hipEventDisableTiming);
    if (e != hipSuccess) return e;
    if (!recorded_ && hipEventRecord(ev_, st_) != hipSuccess) {
      // that stream is gone
      clear();
      return hipDeviceSynchronize();
    }
    recorded_ = true;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    e = hipStreamIsCapturing(st, &cs);
    if (e != hipSuccess) return e;
    if (cs == hipStreamCaptureStatusNone) return hipStreamWaitEvent(st, ev_, 0);
    // a stream under capture cannot wait for work outside the capture: the
    // host waits, once
    e = hipEventSynchronize(ev_);
    if (e == hipSuccess) clear();
    return e;
  }

 private:
  hipEvent_t ev_ = nullptr;
  hipStream_t st_ = nullptr;
  bool set_ = false, recorded_ = false;
};

}  // namespace tqsv

#endif
