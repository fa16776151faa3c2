// nvfp4 / mxfp4 / mxfp8 instances of the mid-row GEMM (midm_kernel.h).
#include "midm_kernel.h"

namespace mi {
namespace midm {
template hipError_t launch_fmt<100>(const MidmParams&, bool, hipStream_t);
template hipError_t launch_fmt<101>(const MidmParams&, bool, hipStream_t);
template hipError_t launch_fmt<102>(const MidmParams&, bool, hipStream_t);
}  // namespace midm
}  // namespace mi
