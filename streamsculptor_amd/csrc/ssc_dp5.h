// Dormand-Prince 5(4) tableau, Shampine's dense-output midpoint weights and the step-control
// parameters shared by the adaptive orbit kernel and the adaptive response kernel.
#pragma once

namespace ssc {
namespace dp5 {

// Dormand & Prince (1980) tableau.
constexpr double A21 = 1.0 / 5;
constexpr double A31 = 3.0 / 40, A32 = 9.0 / 40;
constexpr double A41 = 44.0 / 45, A42 = -56.0 / 15, A43 = 32.0 / 9;
constexpr double A51 = 19372.0 / 6561, A52 = -25360.0 / 2187, A53 = 64448.0 / 6561,
                 A54 = -212.0 / 729;
constexpr double A61 = 9017.0 / 3168, A62 = -355.0 / 33, A63 = 46732.0 / 5247, A64 = 49.0 / 176,
                 A65 = -5103.0 / 18656;
constexpr double C2 = 1.0 / 5, C3 = 3.0 / 10, C4 = 4.0 / 5, C5 = 8.0 / 9;
constexpr double B1 = 35.0 / 384, B3 = 500.0 / 1113, B4 = 125.0 / 192, B5 = -2187.0 / 6784,
                 B6 = 11.0 / 84;
// b - bhat
constexpr double E1 = 71.0 / 57600, E3 = -71.0 / 16695, E4 = 71.0 / 1920,
                 E5 = -17253.0 / 339200, E6 = 22.0 / 525, E7 = -1.0 / 40;
// Shampine's midpoint weights (y at s = 1/2)
constexpr double M1 = 6025192743.0 / 30085553152.0 / 2, M3 = 51252292925.0 / 65400821598.0 / 2,
                 M4 = -2691868925.0 / 45128329728.0 / 2,
                 M5 = 187940372067.0 / 1594534317056.0 / 2,
                 M6 = -1776094331.0 / 19743644256.0 / 2, M7 = 11237099.0 / 235043384.0 / 2;

// The integral controller's step factor 0.9 (1 / e)^(1/5) before its limits [0.2 or 1, 10].  A
// library pow takes about 870 cycles on a wave by itself, every step; here the inverse fifth
// root comes from a single-precision exp2/log2 estimate (relative error below 1e-6) and one
// third-order correction, y (1 + r/5 + 3 r^2/25), r = 1 - e y^5, whose first omitted term is
// below 1e-18: about 20 instructions, within two units in the last place.  e is held to
// [1e-7, 1e5], outside of which the limits decide; NaN counts as the upper end (the lower limit
// of the factor, as with pow).
__device__ __forceinline__ double step_factor(double e) {
  const double ec = e < 1e5 ? fmax(e, 1e-7) : 1e5;
  const double y = (double)__builtin_amdgcn_exp2f(-0.2f * __builtin_amdgcn_logf((float)ec));
  const double y2 = y * y;
  const double r = fma(-ec * y, y2 * y2, 1.0);
  return 0.9 * fma(y * r, fma(0.12, r, 0.2), y);
}

struct Dp5Ctl {
  double rtol, atol, dtmin, dtmax, dt0;  // dtmin / dtmax / dt0 <= 0: none / none / heuristic
  int max_steps;
  int n_stops;
};

}  // namespace dp5
}  // namespace ssc
