// Gaussian integrals by the McMurchie-Davidson scheme (L. E. McMurchie and E. R. Davidson, J. Comput. Phys. 26 (1978) 218;
// the recurrences as in T. Helgaker, P. Jorgensen, J. Olsen, Molecular Electronic-Structure Theory, ch. 9), for shells of
// angular momentum l <= 2 (s, p, d).  Host and device code: the GPU kernels of the SCF wrapper call these functions, and
// a host build of the same header is checked against the compiled reference on the CPU.
//
// Primitive Cartesian Gaussians x_A^i y_A^j z_A^k exp(-a r_A^2).  For a pair (a at A, b at B): p = a + b,
// P = (a A + b B) / p, mu = a b / p.  Hermite expansion coefficients per direction (E[i][j][t], t <= i + j):
//   E[0][0][0] = exp(-mu X_AB^2)
//   E[i+1][j][t] = E[i][j][t-1] / (2p) + X_PA E[i][j][t] + (t+1) E[i][j][t+1]
//   E[i][j+1][t] = E[i][j][t-1] / (2p) + X_PB E[i][j][t] + (t+1) E[i][j][t+1]
// Overlap S = E^x_0 E^y_0 E^z_0 (pi/p)^(3/2); kinetic energy from one-dimensional overlaps,
//   T_ij = -2 b^2 S_i,j+2 + b (2j+1) S_ij - j (j-1) / 2 S_i,j-2.
// Coulomb-type integrals through the Hermite integrals R_tuv(alpha, X, Y, Z):
//   R^n_000 = (-2 alpha)^n F_n(alpha |XYZ|^2),  R^n_t+1,u,v = t R^n+1_t-1,u,v + X R^n+1_t,u,v  (and so for u, v),
// with F_n the Boys function:
//   nuclear attraction  (a|1/r_C|b) = (2 pi / p) sum_tuv E_tuv R_tuv(p, P - C)
//   three-centre        (ab|c) = 2 pi^(5/2) / (p g sqrt(p + g)) sum_tuv E^ab_tuv sum_t'u'v' (-1)^(t'+u'+v') E^c_t'u'v'
//                                R_t+t',u+u',v+v'(p g / (p + g), P - C)
//   two-centre          (c|d) as the three-centre form with the pair replaced by the single Gaussian c.
// A single Gaussian's Hermite coefficients follow from the pair recurrence with b = 0 (E[0][0][0] = 1, X_PA = 0).
// The unrolled forms of these recurrences are in qs_kernels.h.
#pragma once

#include <cmath>

#ifdef __HIPCC__
#define QS_HD __host__ __device__ inline
#else
#define QS_HD inline
#endif

namespace qs {

constexpr int kMaxL = 2;                       // largest angular momentum of one shell
constexpr int kMaxR = 3 * kMaxL;               // largest t + u + v of a Hermite integral (three d shells)
constexpr int kBoysOrders = kMaxR + 1;         // F_0 .. F_6 are needed
constexpr int kBoysTaylor = 6;                 // Taylor terms beyond the tabulated order
constexpr int kBoysTable = kBoysOrders + kBoysTaylor + 1;   // tabulated orders F_0 .. F_13
constexpr double kBoysStep = 0.05;             // table spacing in T
constexpr int kBoysPoints = 801;               // T = 0 .. 40
constexpr double kBoysTMax = kBoysStep * (kBoysPoints - 1);

}  // namespace qs
