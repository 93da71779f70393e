// Instantiates the expectation-pass kernel for TB=8, IDX=uint32_t.
#include "tqsv_pass_impl.h"

namespace tqsv {
template hipError_t launch_one<8, uint32_t>(const PassLaunch& pl, hipStream_t st);
}
