// Instantiates the interpreting kernel's gate passes.
#include "tqsv_interp.h"

namespace tqsv {
template hipError_t launch_interp<11, MODE_GATE, uint32_t>(const PassLaunch& pl, hipStream_t st);
template hipError_t launch_interp<12, MODE_GATE, uint32_t>(const PassLaunch& pl, hipStream_t st);
template hipError_t launch_interp<13, MODE_GATE, uint32_t>(const PassLaunch& pl, hipStream_t st);
template hipError_t launch_interp<14, MODE_GATE, uint32_t>(const PassLaunch& pl, hipStream_t st);
template hipError_t launch_interp<13, MODE_GATE, uint64_t>(const PassLaunch& pl, hipStream_t st);
}
