// 2/3/5/6-bit instances of the mid-row GEMM (midm_kernel.h).
#include "midm_kernel.h"

namespace mi {
namespace midm {
template hipError_t launch_fmt<2>(const MidmParams&, bool, hipStream_t);
template hipError_t launch_fmt<3>(const MidmParams&, bool, hipStream_t);
template hipError_t launch_fmt<5>(const MidmParams&, bool, hipStream_t);
template hipError_t launch_fmt<6>(const MidmParams&, bool, hipStream_t);
}  // namespace midm
}  // namespace mi
