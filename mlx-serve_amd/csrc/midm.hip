// Mid-row quantized GEMM (midm_kernel.h): plan, launch, and the 4-bit instances (the others are in
// midm_b8.hip, midm_odd.hip and midm_fp.hip).
#include "midm_kernel.h"

#include <algorithm>

namespace mi {
namespace midm {
template hipError_t launch_fmt<4>(const MidmParams&, bool, hipStream_t);
extern template hipError_t launch_fmt<8>(const MidmParams&, bool, hipStream_t);
extern template hipError_t launch_fmt<2>(const MidmParams&, bool, hipStream_t);
extern template hipError_t launch_fmt<3>(const MidmParams&, bool, hipStream_t);
extern template hipError_t launch_fmt<5>(const MidmParams&, bool, hipStream_t);
extern template hipError_t launch_fmt<6>(const MidmParams&, bool, hipStream_t);
extern template hipError_t launch_fmt<100>(const MidmParams&, bool, hipStream_t);
extern template hipError_t launch_fmt<101>(const MidmParams&, bool, hipStream_t);
extern template hipError_t launch_fmt<102>(const MidmParams&, bool, hipStream_t);
}  // namespace midm

bool midm_plan(int64_t M, int64_t N, int64_t K, int fmt, int gs, MidmPlan* out) {
  const int bits = midm::fmt_bits(fmt);
  const bool ex = fmt == 4 || fmt == 8;
  // affine groups of 64 (a bias-less mode has its own), 4-output stores, 32-bit offsets
  if ((fmt < 100 && gs != 64) || M < (ex ? 17 : 33) || M > 128 || N < 4 || N % 4 || K % 64 ||
      M * K * 2 >= ((int64_t)1 << 31) || N * (K * bits / 8) >= ((int64_t)1 << 31) ||
      N >= ((int64_t)1 << 30))
    return false;
  // Block shape (64 or 32 rows, 4 K parts) and K split by estimated
  // time: rounds of 256 blocks x (3.6 us + steps of a wave x the time of a step), plus 3 us
  // for the partials and their reduce launch when K splits over blocks. A step costs the
  // larger of its compute (measured on half-empty grids) and its bytes from L2 at the rate
  // of a full grid. Estimates against measured at 4 bits, us: [14336,4096] 32 rows 14.8 /
  // 15.8, 128 rows 24.9 / 27.5 (wide); [7168,2048] 64 rows 9.2 / 9.2, 128 rows 12.4 / 10.9
  // (narrow; wide measured 13.7 at 128); [4096,14336] 32 rows 17.8 / 18.4 (wide, 4 ranges;
  // narrow 21.7).
  // Up to 64 rows the choice does not look at M, so a row's result does not depend on how
  // many rows ride along (same K parts, same order).
  const int64_t rows = M <= 64 ? 32 : M;
  const int mt = (int)((rows + 31) / 32);
  static constexpr double kStep[2][4] = {{0.70, 0.65, 0.65, 0.80}, {0.70, 0.80, 0.95, 1.10}};
  const int64_t groups = K / 64;
  double best = 1e30;
  for (int wide = 0; wide < 2; ++wide) {
    constexpr int wk = 4;
    const int64_t tiles = (N + (wide ? 63 : 31)) / (wide ? 64 : 32);
    const double kb = (wide ? 2 : 1) * wk * 1.15 * bits / 4 + wk * rows * 0.128;
    const double rate = wide ? 50.0 : 75.0;  // KB/us of a block, grid full
    for (int64_t ks = 1; ks == 1 || (tiles * ks <= 256 && ks <= 32); ++ks) {
      const int64_t steps = (groups + wk * ks * 2 - 1) / (wk * ks * 2) * 2;
      if ((groups + wk * steps - 1) / (wk * steps) != ks) continue;  // a range without steps
      const int64_t blocks = tiles * ks;
      const double step = std::max(kStep[wide][mt - 1], kb / rate * std::min(1.0, blocks / 256.0));
      const double t = (double)((blocks + 255) / 256) * (3.6 + steps * step) + (ks > 1 ? 3.0 : 0.0);
      if (t < best - 1e-9) {
        best = t;
        *out = MidmPlan{wide != 0, (int)steps, (int)ks,
                        ks > 1 ? (size_t)ks * M * N * sizeof(float) : 0};
      }
    }
  }
  return true;
}

hipError_t launch_midm(const MidmParams& P, const MidmPlan& pl, int fmt, hipStream_t s) {
  if (P.ks > 1 && !P.part) return hipErrorInvalidValue;
  hipError_t e = hipErrorInvalidValue;
  switch (fmt) {
    case 2: e = midm::launch_fmt<2>(P, pl.wide, s); break;
    case 3: e = midm::launch_fmt<3>(P, pl.wide, s); break;
    case 4: e = midm::launch_fmt<4>(P, pl.wide, s); break;
    case 5: e = midm::launch_fmt<5>(P, pl.wide, s); break;
    case 6: e = midm::launch_fmt<6>(P, pl.wide, s); break;
    case 8: e = midm::launch_fmt<8>(P, pl.wide, s); break;
    case 100: e = midm::launch_fmt<100>(P, pl.wide, s); break;
    case 101: e = midm::launch_fmt<101>(P, pl.wide, s); break;
    case 102: e = midm::launch_fmt<102>(P, pl.wide, s); break;
  }
  if (e != hipSuccess || P.ks == 1) return e;
  return launch_split_reduce(P.part, P.y, (int64_t)P.M * P.N, P.ks, s);
}

}  // namespace mi
