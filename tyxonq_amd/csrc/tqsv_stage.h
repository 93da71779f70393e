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

// What was queued for an object on one stream, to be waited for by uses on
// another (uses on the same stream follow it anyway).
class StreamMark {
 public:
  StreamMark() = default;
  StreamMark(const StreamMark&) = delete;
  StreamMark& operator=(const StreamMark&) = delete;
  ~StreamMark() {
    if (ev_) (void)hipEventDestroy(ev_);
  }
  hipError_t record(hipStream_t st) {
    if (!ev_) {
      const hipError_t e = hipEventCreateWithFlags(&ev_, hipEventDisableTiming);
      if (e != hipSuccess) return e;
    }
    st_ = st;
    set_ = true;
    return hipEventRecord(ev_, st);
  }
  void clear() { set_ = false; }
  // a stream under capture cannot wait for work outside the capture: the host
  // waits, once
  hipError_t wait(hipStream_t st) {
    if (!set_ || st == st_) return hipSuccess;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(st, &cs);
    if (e != hipSuccess) return e;
    if (cs == hipStreamCaptureStatusNone) return hipStreamWaitEvent(st, ev_, 0);
    e = hipEventSynchronize(ev_);
    if (e == hipSuccess) clear();
    return e;
  }

 private:
  hipEvent_t ev_ = nullptr;
  hipStream_t st_ = nullptr;
  bool set_ = false;
};

}  // namespace tqsv

#endif
