// Instantiates the expectation-pass kernel for TB=7, IDX=uint32_t.
#include "tqsv_pass_impl.h"

namespace tqsv {
template hipError_t launch_one<7, uint32_t>(const PassLaunch& pl, hipStream_t st);
}
