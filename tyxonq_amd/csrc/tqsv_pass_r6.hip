// Instantiates the expectation-pass kernel for TB=6, IDX=uint32_t.
#include "tqsv_pass_impl.h"

namespace tqsv {
template hipError_t launch_one<6, uint32_t>(const PassLaunch& pl, hipStream_t st);
}
