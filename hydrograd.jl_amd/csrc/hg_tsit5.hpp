// hg_tsit5.hpp -- the coefficients of the adaptive integrator.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>


namespace hg {

// Tsitouras' 5(4) Runge-Kutta pair (Ch. Tsitouras, Comput. Math.
// Appl. 62 (2011) 770-775), first-same-as-last, the adaptive integrator the
// reference's examples run through OrdinaryDiffEq (Tsit5()).
namespace tsit5 {
constexpr double c[7] = {0.0, 0.161, 0.327, 0.9, 0.9800255409045097, 1.0, 1.0};
constexpr double a[7][6] = {
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.161, 0.0, 0.0, 0.0, 0.0, 0.0},
    {-0.008480655492356989, 0.335480655492357, 0.0, 0.0, 0.0, 0.0},
    {2.897153057105493, -6.359448489975075, 4.3622954328695815, 0.0, 0.0, 0.0},
    {5.325864828439257, -11.748883564062828, 7.4955393428898365, -0.09249506636175525, 0.0, 0.0},
    {5.86145544294642, -12.92096931784711, 8.159367898576159, -0.071584973281401, -0.028269050394068383, 0.0},
    {0.09646076681806523, 0.01, 0.4798896504144996, 1.379008574103742, -3.290069515436081, 2.324710524099774}};
// b = a[6] (fifth order, b7 = 0); btilde = b - bhat (bhat: the embedded fourth-order weights)
constexpr double btilde[7] = {-0.00178001105222577714, -0.0008164344596567469, 0.007880878010261995,
                              -0.1447110071732629,     0.5823571654525552,    -0.45808210592918697,
                              0.015151515151515152};
// The factor (before its limits) that the step changes by after error norm err.
__host__ __device__ __forceinline__ double step_factor(double err) {
  return err > 0.0 ? 0.9 * ::pow(err, -0.2) : 10.0;
}
}  // namespace tsit5

}  // namespace hg
