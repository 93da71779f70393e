// tqsv_pass.hip - host dispatch of the tile-pass kernel variants.  The kernel
// templates are in tqsv_interp.h (gate and dual passes) and tqsv_pass_impl.h
// (expectation passes); each tqsv_pass_*.hip and tqsv_interp_*.hip
// translation unit instantiates some variants so they compile in parallel.
#include <hip/hip_runtime.h>

#include "tqsv_internal.h"
#include "tqsv_prog.h"

namespace tqsv {

template <int TB, typename IDX>
hipError_t launch_one(const PassLaunch& pl, hipStream_t st);
template <int T, int MODE, typename IDX>
hipError_t launch_interp(const PassLaunch& pl, hipStream_t st);

static size_t tile_bytes(int tb, int mode) {
  return (mode == MODE_DUAL ? 2 : 1) * ((size_t)1 << (tb + RB)) * sizeof(float2);
}

size_t pass_lds_bytes(int tb, int mode, uint32_t nred) {
  const size_t nwave = ((size_t)1 << tb) >= 64 ? ((size_t)1 << tb) / 64 : 1;
  return tile_bytes(tb, mode) + (mode == MODE_GATE ? 0 : nwave * nred * sizeof(double));
}

// four threads per 32 slots, at most 1024 (interp_threads)
size_t interp_lds_bytes(int tb, int mode, uint32_t nred) {
  const size_t nwave = (tb >= 8 ? 1024 : (size_t)4 << tb) / 64;
  return tile_bytes(tb, mode) + (mode == MODE_GATE ? 0 : nwave * nred * sizeof(double));
}

bool pass_variant_exists(int tb, int mode, bool idx64) {
  if (idx64) return (mode == MODE_GATE || mode == MODE_RED) && tb == 8;
  switch (mode) {
    case MODE_GATE: return tb >= 6 && tb <= 9;
    case MODE_RED: return tb >= 6 && tb <= 8;
    case MODE_DUAL: return tb >= 6 && tb <= 8;
    default: return false;
  }
}

hipError_t launch_pass(int tb, int mode, bool idx64, const PassLaunch& pass, hipStream_t st) {
  if (!pass_variant_exists(tb, mode, idx64)) return hipErrorInvalidValue;
  PassLaunch pl = pass;
  if (mode != MODE_RED) pl.lds_bytes = interp_lds_bytes(tb, mode, pl.nred);
  if (idx64) return mode == MODE_GATE ? launch_interp<13, MODE_GATE, uint64_t>(pl, st)
                                      : launch_one<8, uint64_t>(pl, st);
  switch (mode) {
    case MODE_GATE:
      switch (tb) {
        case 6: return launch_interp<11, MODE_GATE, uint32_t>(pl, st);
        case 7: return launch_interp<12, MODE_GATE, uint32_t>(pl, st);
        case 8: return launch_interp<13, MODE_GATE, uint32_t>(pl, st);
        default: return launch_interp<14, MODE_GATE, uint32_t>(pl, st);
      }
    case MODE_RED:
      switch (tb) {
        case 6: return launch_one<6, uint32_t>(pl, st);
        case 7: return launch_one<7, uint32_t>(pl, st);
        default: return launch_one<8, uint32_t>(pl, st);
      }
    default:
      switch (tb) {
        case 6: return launch_interp<11, MODE_DUAL, uint32_t>(pl, st);
        case 7: return launch_interp<12, MODE_DUAL, uint32_t>(pl, st);
        default: return launch_interp<13, MODE_DUAL, uint32_t>(pl, st);
      }
  }
}

}  // namespace tqsv
