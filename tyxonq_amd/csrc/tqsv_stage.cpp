// tqsv_stage.cpp - a ring of page-locked memory per thread for the small
// host-to-device copies of plans, Hamiltonians and batches.  A copy from
// pageable memory has to be waited for before that memory changes; a parameter
// update made two such copies and waits, the reverse sweep's after the whole
// forward sweep (48 small requests: 256 copies and about 200 waits).
#include "tqsv_stage.h"

#include <cstring>
#include <deque>
#include <vector>

#include "../../include/tqsv.h"
#include "tqsv_internal.h"

namespace tqsv {

namespace {

constexpr size_t kRing = 1 << 20;        // bytes per thread, until the thread ends
constexpr size_t kLargest = kRing / 4;   // larger copies go from the caller's memory

struct Ring {
  struct Piece {
    size_t at, len;
    hipEvent_t ev;
  };
  unsigned char* base = nullptr;
  size_t head = 0;
  int dev = -1;
  std::deque<Piece> busy;  // in ring order, oldest first
  std::vector<hipEvent_t> idle;

  void drop() {
    for (Piece& p : busy) {
      (void)hipEventSynchronize(p.ev);
      (void)hipEventDestroy(p.ev);
    }
    for (hipEvent_t e : idle) (void)hipEventDestroy(e);
    if (base) (void)hipHostFree(base);
    busy.clear();
    idle.clear();
    base = nullptr;
    head = 0;
  }
  ~Ring() { drop(); }

  // the oldest copy has been made: its memory is free
  hipError_t retire() {
    const Piece p = busy.front();
    const hipError_t e = hipEventSynchronize(p.ev);
    if (e != hipSuccess) return e;
    idle.push_back(p.ev);
    busy.pop_front();
    return hipSuccess;
  }
};
thread_local Ring g_ring;

}  // namespace

int stage_copy(void* dst, const void* src, size_t bytes, hipStream_t st) {
  if (bytes == 0) return 0;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  TQSV_HIP(hipStreamIsCapturing(st, &cs));
  if (cs != hipStreamCaptureStatusNone)
    return fail(TQSV_EUNSUPPORTED, "parameters cannot be replaced under stream capture");
  if (bytes > kLargest) {
    TQSV_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st));
    TQSV_HIP(hipStreamSynchronize(st));
    return 0;
  }
  Ring& r = g_ring;
  int dev = 0;
  TQSV_HIP(hipGetDevice(&dev));
  if (!r.base || r.dev != dev) {
    r.drop();
    TQSV_HIP(hipHostMalloc(reinterpret_cast<void**>(&r.base), kRing, hipHostMallocDefault));
    r.dev = dev;
  }
  const size_t len = (bytes + 63) & ~(size_t)63;
  // pieces are taken in ring order, so those in the way are the oldest (at a
  // wrap, first those between the head and the end)
  if (r.head + len > kRing) {
    while (!r.busy.empty() && r.busy.front().at >= r.head) TQSV_HIP(r.retire());
    r.head = 0;
  }
  const size_t at = r.head;
  while (!r.busy.empty() && r.busy.front().at < at + len && at < r.busy.front().at + r.busy.front().len)
    TQSV_HIP(r.retire());
  if (r.busy.size() >= 256) TQSV_HIP(r.retire());  // bounded number of events
  hipEvent_t ev = nullptr;
  if (!r.idle.empty()) {
    ev = r.idle.back();
    r.idle.pop_back();
  } else {
    TQSV_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
  }
  std::memcpy(r.base + at, src, bytes);
  hipError_t e = hipMemcpyAsync(dst, r.base + at, bytes, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) {
    e = hipEventRecord(ev, st);
    if (e != hipSuccess) (void)hipStreamSynchronize(st);
  }
  if (e != hipSuccess) {
    (void)hipEventDestroy(ev);
    return hip_fail(e, "stage_copy");
  }
  r.busy.push_back(Ring::Piece{at, len, ev});
  r.head = at + len;
  return 0;
}

}  // namespace tqsv
