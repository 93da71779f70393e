// tqsv_stage.cpp - a ring of page-locked memory per thread for the small
// host-to-device copies of plans, Hamiltonians and batches.  A copy from
// pageable memory has to be waited for before that memory changes; a parameter
// update made two such copies and waits, the reverse sweep's after the whole
// forward sweep (48 small requests: 256 copies and about 200 waits).
#include "tqsv_stage.h"

#include <algorithm>
#include <cstring>
#include <vector>

#include "../../include/tqsv.h"
#include "tqsv_internal.h"

namespace tqsv {

namespace {

// The ring is used quarter by quarter.  Before a quarter is written again, the
// streams of its copies, three quarters ago, are waited for; no event is
// recorded per copy (an event costs the device about as much as a small copy).
constexpr size_t kRing = 1 << 20;        // bytes per thread, until the thread ends
constexpr size_t kQuarter = kRing / 4;   // larger copies go from the caller's memory

struct Ring {
  unsigned char* base = nullptr;
  size_t head = 0;
  int dev = -1;
  std::vector<hipStream_t> users[4];

  hipError_t reclaim(int q) {
    for (hipStream_t st : users[q])
      if (hipStreamSynchronize(st) != hipSuccess) {
        // that stream is gone
        const hipError_t e = hipDeviceSynchronize();
        if (e != hipSuccess) return e;
      }
    users[q].clear();
    return hipSuccess;
  }
  void drop() {
    for (int q = 0; q < 4; ++q) (void)reclaim(q);
    if (base) (void)hipHostFree(base);
    base = nullptr;
    head = 0;
  }
  ~Ring() { drop(); }
};
thread_local Ring g_ring;

}  // namespace

int stage_copy(void* dst, const void* src, size_t bytes, hipStream_t st) {
  if (bytes == 0) return 0;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  TQSV_HIP(hipStreamIsCapturing(st, &cs));
  if (cs != hipStreamCaptureStatusNone)
    return fail(TQSV_EUNSUPPORTED, "parameters cannot be replaced under stream capture");
  if (bytes > kQuarter) {
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
  // a copy lies within one quarter
  if (r.head % kQuarter + len > kQuarter || r.head == kRing)
    r.head = (r.head + kQuarter - 1) / kQuarter * kQuarter % kRing;
  const int q = (int)(r.head / kQuarter);
  if (r.head % kQuarter == 0) TQSV_HIP(r.reclaim(q));
  std::memcpy(r.base + r.head, src, bytes);
  TQSV_HIP(hipMemcpyAsync(dst, r.base + r.head, bytes, hipMemcpyHostToDevice, st));
  if (std::find(r.users[q].begin(), r.users[q].end(), st) == r.users[q].end())
    r.users[q].push_back(st);
  r.head += len;
  return 0;
}

}  // namespace tqsv
