// tqsv_stage.cpp - a ring of page-locked memory per thread for the small
// host-to-device copies of plans, Hamiltonians and batches.  A copy from
// pageable memory has to be waited for before that memory changes; a parameter
// update made two such copies and waits, the reverse sweep's after the whole
// forward sweep (48 small requests: 256 copies and about 200 waits).
#include "tqsv_stage.h"

#include <atomic>
#include <cstring>
#include <thread>

#include "../../include/tqsv.h"
#include "tqsv_internal.h"

namespace tqsv {

// The pieces (k_stage_copy) of a thread's copies are numbered.  A piece that has
// run writes its number to word (number % kWords) of page-locked memory; a word is
// used again only when its last number is there.  So "has this copy run" is a
// read of host memory, whatever has become of the copy's stream since.
struct StageTickets {
  static constexpr uint64_t kWords = 2048;
  std::mutex m;
  uint64_t* word = nullptr;  // NULL: every copy has run and the thread is done with it

  bool reached(uint64_t t) {
    std::lock_guard<std::mutex> lock(m);
    return !word || __atomic_load_n(&word[t % kWords], __ATOMIC_ACQUIRE) >= t;
  }
  void wait(uint64_t first, uint64_t last) {
    for (uint64_t t = first; t <= last; ++t)
      for (int k = 0; !reached(t); ++k)
        if (k >= 64) std::this_thread::yield();
  }
};

void StagePoint::wait() const {
  if (of) of->wait(first, last);
}

namespace {

// The ring is used quarter by quarter; before a quarter is written again, its
// copies, three quarters ago, are waited for.
constexpr size_t kRing = 1 << 20;        // bytes per thread, until the thread ends
constexpr size_t kQuarter = kRing / 4;   // larger copies go from the caller's memory

struct Ring {
  unsigned char* base = nullptr;  // the ring, then the words of the tickets
  size_t head = 0;
  std::shared_ptr<StageTickets> tickets;
  uint64_t next = 1;              // numbers start at 1: a word of 0 holds none
  uint64_t latest = 0;            // first number of the last copy
  struct {
    uint64_t first = 1, last = 0;
  } quarter[4];                   // numbers of each quarter's copies

  // (portable memory: one ring serves whichever devices the thread uses)
  int open() {
    const size_t words = StageTickets::kWords * sizeof(uint64_t);
    auto t = std::make_shared<StageTickets>();
    // (another thread may be capturing: an allocation is no part of that)
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    TQSV_HIP(hipThreadExchangeStreamCaptureMode(&mode));
    const hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&base), kRing + words,
                                       hipHostMallocCoherent | hipHostMallocPortable);
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess) {
      base = nullptr;
      return hip_fail(e, "staging ring");
    }
    t->word = reinterpret_cast<uint64_t*>(base + kRing);
    std::memset(t->word, 0, words);
    tickets = std::move(t);
    return 0;
  }
  ~Ring() {
    if (!base) return;
    tickets->wait(next > StageTickets::kWords ? next - StageTickets::kWords : 1, next - 1);
    {
      std::lock_guard<std::mutex> lock(tickets->m);
      tickets->word = nullptr;
    }
    (void)hipHostFree(base);
  }
};
thread_local Ring g_ring;

}  // namespace

StagePoint stage_point() {
  const Ring& r = g_ring;
  return r.base ? StagePoint{r.tickets, r.latest, r.next - 1} : StagePoint{};
}

int stage_copy(void* dst, const void* src, size_t bytes, hipStream_t st) {
  if (bytes == 0) return 0;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  TQSV_HIP(hipStreamIsCapturing(st, &cs));
  if (cs != hipStreamCaptureStatusNone)
    return fail(TQSV_EUNSUPPORTED, "parameters cannot be replaced under stream capture");
  if (bytes > kQuarter || bytes % 4 != 0) {
    TQSV_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st));
    TQSV_HIP(hipStreamSynchronize(st));
    return 0;
  }
  Ring& r = g_ring;
  if (!r.base) {
    const int rc = r.open();
    if (rc) return rc;
  }
  const size_t len = (bytes + 63) & ~(size_t)63;
  // a copy lies within one quarter
  if (r.head % kQuarter + len > kQuarter || r.head == kRing)
    r.head = (r.head + kQuarter - 1) / kQuarter * kQuarter % kRing;
  auto& q = r.quarter[r.head / kQuarter];
  if (r.head % kQuarter == 0) {
    r.tickets->wait(q.first, q.last);
    q.last = 0;
  }
  const uint64_t t = r.next, end = t + stage_pieces(bytes);
  // the words of these numbers
  if (end > StageTickets::kWords + 1)
    r.tickets->wait(t > StageTickets::kWords ? t - StageTickets::kWords : 1,
                    end - 1 - StageTickets::kWords);
  std::memcpy(r.base + r.head, src, bytes);
  TQSV_HIP(k_stage_copy(dst, r.base + r.head, bytes, r.tickets->word, StageTickets::kWords, t, st));
  if (!q.last) q.first = t;
  q.last = end - 1;
  r.latest = t;
  r.next = end;
  r.head += len;
  return 0;
}

}  // namespace tqsv
