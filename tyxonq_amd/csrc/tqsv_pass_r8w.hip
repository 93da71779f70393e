// Instantiates the expectation-pass kernel for TB=8, IDX=uint64_t.
#include "tqsv_pass_impl.h"

namespace tqsv {
template hipError_t launch_one<8, uint64_t>(const PassLaunch& pl, hipStream_t st);
}
