// 8-bit instances of the mid-row GEMM (midm_kernel.h).
#include "midm_kernel.h"

namespace mi {
namespace midm {
template hipError_t launch_fmt<8>(const MidmParams&, bool, hipStream_t);
}  // namespace midm
}  // namespace mi
