// The integral work items of the SCF wrapper (a shell pair, a fit shell pair or a shell pair with a fit shell each), as host
// and device functions: the GPU kernels of qs_integrals.hip call them, and a host build of this header checks the same
// code against the compiled reference on the CPU.  The mathematics is in qs_md.h; the Boys table comes in as an argument.
//
// The one-electron and electron-fit integrals are templates over the shells' angular momenta ("classes", la >= lb: a pair
// whose first shell has the lower one swaps the roles of its shells), so that every loop over Cartesian components and
// Hermite indices is unrolled and every intermediate (the Hermite integrals R, the sums of a block) stays in registers.
// What belongs to an orbital shell pair alone, per primitive pair its exponent, centre and Hermite coefficients, is made
// once per pair as a record; a wave of the integral kernels takes one pair, so that the records are read as scalars.
#pragma once

#include <utility>
#include <vector>

// The CPU check compiles the unrolled blocks below for correctness only.
#if defined(__GNUC__) && !defined(__HIPCC__)
#pragma GCC optimize("O1")
#endif

#include "qs_md.h"

namespace qs {

struct QPair { int x, y; };

struct QShell {                 // one angular momentum of one contracted shell (an SP shell gives two)
    double x, y, z;
    int l, nPrim, prim;         // primitives: exponents and coefficients from offset prim
    int f0, nf;                 // first function and function count (2l+1 spherical or Cartesian)
    int atom, pad;
};

struct PairEntry {              // a significant shell pair (A >= B) and its first row of electron-fit integrals
    int a, b;
    long long row;
};

struct PairItem {               // a shell pair in its class's roles (the shell of the larger l first) and its records
    int a, b, swapped;          // swapped: the roles are those of the pair B, A
    int n;                      // records
    long long first;            // offset of the first record
    long long row;              // first row of its electron-fit integrals
};

constexpr double kUnderFlow = 1.0e-12;    // electron-fit integrals dropped by the reference's storage
// Nuclei are Gaussian charge distributions of width 1e-4 bohr, exponent 4 / (w^2 pi), as the reference's electron-nuclear
// integrals take them by default (GaussianNucleus.h: _DefaultNuclearWidth, _DefaultNuclearWidthE).
constexpr double kNuclearWidth = 1.0e-4;
constexpr double kNuclearExponent = 4.0 / (kNuclearWidth * kNuclearWidth * M_PI);

QS_HD long long packed_index(int i, int j) {
    return i >= j ? static_cast<long long>(i) * (i + 1) / 2 + j : static_cast<long long>(j) * (j + 1) / 2 + i;
}

// ------------------------------------------------------------------------------------------------------------------------
// Classes.
// ------------------------------------------------------------------------------------------------------------------------
template <class F, int... I>
QS_HD void static_for_each(F f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>
QS_HD void static_for(F f) { static_for_each(f, std::make_integer_sequence<int, N>{}); }

struct Powers { int x, y, z; };
QS_HD constexpr Powers powers_of(int l, int c) {
    int n = 0;
    for (int zz = 0; zz <= l; zz++)
        for (int yy = 0; yy <= l - zz; yy++) {
            if (n == c) return Powers{l - yy - zz, yy, zz};
            n++;
        }
    return Powers{0, 0, 0};
}
QS_HD constexpr int cartesians(int l) { return (l + 1) * (l + 2) / 2; }
// Cartesian factor of component c of angular momentum l: sqrt((2l-1)!! / ((2x-1)!! (2y-1)!! (2z-1)!!)), which is sqrt(3) for
// xy, xz and yz and 1 otherwise (l <= 2).
QS_HD constexpr double cart_factor(int l, int c) { return l == 2 && (c == 1 || c == 3 || c == 4) ? 1.7320508075688772935 : 1.0; }

// Hermite coefficients of a pair of the class: component pair ab = (ia, ib) has (x + 1)(y + 1)(z + 1) of them, x, y and z
// the summed powers, from at[ab]; size is the doubles of a record (p, 1 / p, P, coefficients).  The tables are constants
// that are evaluated once per class.
template <int LA, int LB>
struct PairTable {
    static constexpr int na = cartesians(LA), nb = cartesians(LB);
    int x[na * nb] = {}, y[na * nb] = {}, z[na * nb] = {}, terms[na * nb] = {}, at[na * nb] = {}, size = 5;
    constexpr PairTable() {
        for (int k = 0; k < na * nb; k++) {
            const Powers a = powers_of(LA, k / nb), b = powers_of(LB, k % nb);
            x[k] = a.x + b.x;
            y[k] = a.y + b.y;
            z[k] = a.z + b.z;
            terms[k] = (x[k] + 1) * (y[k] + 1) * (z[k] + 1);
            at[k] = size;
            size += terms[k];
        }
    }
};
template <int LA, int LB>
struct PairClass {
    static constexpr PairTable<LA, LB> table{};
    static constexpr int na = cartesians(LA), nb = cartesians(LB), size = table.size;
};

// Primitive pairs are left out of a pair's records when their integrals with a unit charge are below about this.  An
// integral is at most the prefactor |c_a c_b| exp(-mu R^2) times 2 pi / p for a nucleus (pi^(5/2) / (p g sqrt(p + g)), c_c
// in it, for a fit function), times a power of lengths, R between the centres and p^(-1/2) of the product, that is la + lb.
constexpr double kPrimitiveScreen = 1.0e-24;

// The records of a pair (A of LA, B of LB) at out, size doubles apart; returns their number.
template <int LA, int LB>
QS_HD int pair_records(const QShell &A, const QShell &B, const double *__restrict__ exps, const double *__restrict__ coefs,
                       double *__restrict__ out) {
    using C = PairClass<LA, LB>;
    constexpr int NT = LA + LB + 1;
    const double X[3] = {A.x - B.x, A.y - B.y, A.z - B.z};
    const double r2 = X[0] * X[0] + X[1] * X[1] + X[2] * X[2];
    int n = 0;
    for (int qa = 0; qa < A.nPrim; qa++)
        for (int qb = 0; qb < B.nPrim; qb++) {
            const double a = exps[A.prim + qa], b = exps[B.prim + qb], p = a + b, ip = 1.0 / p, h = 0.5 * ip;
            const double K = coefs[A.prim + qa] * coefs[B.prim + qb] * exp(-a * b * ip * r2);
            const double q = fmax(1.0, ip);
            double bound = q * q;           // formed while the exponential is
            static_for<(LA + LB + 1) / 2>([&](auto) { bound *= r2 + q; });
            if (bound * fabs(K) < kPrimitiveScreen) continue;
            double *rec = out + static_cast<long long>(n) * C::size;
            n++;
            rec[0] = p;
            rec[1] = ip;
            rec[2] = (a * A.x + b * B.x) * ip;
            rec[3] = (a * A.y + b * B.y) * ip;
            rec[4] = (a * A.z + b * B.z) * ip;
            // E[d][i][j][t] (qs_md.h) with E[0][0][0] = 1; X_PA = -b X / p, X_PB = a X / p.
            double E[3][LA + 1][LB + 1][NT];
            static_for<3>([&](auto dd) {
                constexpr int d = dd;
                const double pa = -b * ip * X[d], pb = a * ip * X[d];
                static_for<(LA + 1) * (LB + 1)>([&](auto kk) {
                    constexpr int i = kk / (LB + 1), j = kk % (LB + 1);
                    static_for<NT>([&](auto tt) {
                        constexpr int t = tt;
                        if constexpr (i + j == 0) E[d][i][j][t] = t == 0 ? 1.0 : 0.0;
                        else if constexpr (t > i + j) E[d][i][j][t] = 0.0;
                        else {
                            constexpr int si = j > 0 ? i : i - 1, sj = j > 0 ? j - 1 : 0;   // raised from (si, sj)
                            const double *s = E[d][si][sj];
                            double e = (j > 0 ? pb : pa) * s[t];
                            if constexpr (t > 0) e += h * s[t - 1];
                            if constexpr (t + 1 < NT) e += (t + 1) * s[t + 1];
                            E[d][i][j][t] = e;
                        }
                    });
                });
            });
            static_for<C::na * C::nb>([&](auto kk) {
                constexpr int ab = kk, ia = ab / C::nb, ib = ab % C::nb;
                constexpr Powers u = powers_of(LA, ia), v = powers_of(LB, ib);
                constexpr int ny = C::table.y[ab] + 1, nz = C::table.z[ab] + 1, at = C::table.at[ab];
                const double f = K * cart_factor(LA, ia) * cart_factor(LB, ib);
                static_for<C::table.terms[ab]>([&](auto mm) {
                    constexpr int m = mm, tx = m / (ny * nz), ty = m / nz % ny, tz = m % nz;
                    rec[at + m] = f * E[0][u.x][v.x][tx] * E[1][u.y][v.y][ty] * E[2][u.z][v.z][tz];
                });
            });
        }
    return n;
}

// Boys function F_L(T) .. F_0(T) from the table F[k][n] = F_n(k step), n < kBoysTable: a Taylor expansion of F_L about the
// nearest tabulated T (|dT| <= step / 2, kBoysTaylor + 1 terms) and downward recursion F_n = (2 T F_n+1 + exp(-T)) / (2n + 1);
// beyond the table, F_0 = sqrt(pi / T) / 2 and upward recursion F_n+1 = ((2n + 1) F_n - exp(-T)) / (2T), which is stable for
// large T.
template <int L>
QS_HD void boys_of(double T, const double *__restrict__ table, double (&F)[L + 1]) {
    if (T < kBoysTMax) {
        const int k = static_cast<int>(T * (1.0 / kBoysStep) + 0.5);
        const double d = k * kBoysStep - T;
        const double *row = table + k * kBoysTable + L;
        double s = row[kBoysTaylor];
        static_for<kBoysTaylor>([&](auto jj) {
            constexpr int j = kBoysTaylor - 1 - jj;
            s = row[j] + s * (d * (1.0 / (j + 1)));
        });
        F[L] = s;
        if constexpr (L > 0) {
            const double e = exp(-T), T2 = 2.0 * T;
            static_for<L>([&](auto nn) {
                constexpr int n = L - 1 - nn;
                F[n] = (T2 * F[n + 1] + e) * (1.0 / (2 * n + 1));
            });
        }
    } else {
        const double iT = 1.0 / T;
        F[0] = 0.88622692545275801365 * sqrt(iT);   // sqrt(pi) / 2
        if constexpr (L > 0) {
            const double e = exp(-T), h = 0.5 * iT;
            static_for<L>([&](auto nn) {
                constexpr int n = nn;
                F[n + 1] = ((2 * n + 1) * F[n] - e) * h;
            });
        }
    }
}

// Hermite integrals R_tuv (t + u + v <= L; qs_md.h) times scale, at R[(t * (L + 1) + u) * (L + 1) + v].
constexpr int hermite_steps(int L) {
    int c = 0;
    for (int n = L - 1; n >= 0; n--)
        for (int s = L - n; s >= 1; s--) c += (s + 1) * (s + 2) / 2;
    return c;
}
template <int L>
struct HermitePlan {            // the steps of the in-place recursion: per level n, total orders s = L - n .. 1
    static constexpr int count = hermite_steps(L);
    int n[count + 1] = {}, t[count + 1] = {}, u[count + 1] = {}, v[count + 1] = {};
    bool last[count + 1] = {};  // the level's last step
    constexpr HermitePlan() {
        int c = 0;
        for (int k = L - 1; k >= 0; k--)
            for (int s = L - k; s >= 1; s--)
                for (int i = 0; i <= s; i++)
                    for (int j = 0; j <= s - i; j++, c++) {
                        n[c] = k;
                        t[c] = i;
                        u[c] = j;
                        v[c] = s - i - j;
                        last[c] = s == 1 && i == 1;
                    }
    }
};
template <int L>
struct HermiteSteps { static constexpr HermitePlan<L> plan{}; };
template <int L>
QS_HD constexpr int hidx(int t, int u, int v) { return (t * (L + 1) + u) * (L + 1) + v; }

template <int L>
QS_HD void hermite_of(double alpha, double X, double Y, double Z, double scale, const double *__restrict__ table,
                      double (&R)[(L + 1) * (L + 1) * (L + 1)]) {
    double F[L + 1];
    boys_of<L>(alpha * (X * X + Y * Y + Z * Z), table, F);
    double f = scale;
    static_for<L + 1>([&](auto nn) {
        F[nn] *= f;
        f *= -2.0 * alpha;
    });
    R[0] = F[L];
    static_for<hermite_steps(L)>([&](auto kk) {
        constexpr auto &plan = HermiteSteps<L>::plan;
        constexpr int t = plan.t[kk], u = plan.u[kk], v = plan.v[kk];
        double r;
        if constexpr (t > 0) {
            r = X * R[hidx<L>(t - 1, u, v)];
            if constexpr (t > 1) r += (t - 1) * R[hidx<L>(t - 2, u, v)];
        } else if constexpr (u > 0) {
            r = Y * R[hidx<L>(t, u - 1, v)];
            if constexpr (u > 1) r += (u - 1) * R[hidx<L>(t, u - 2, v)];
        } else {
            r = Z * R[hidx<L>(t, u, v - 1)];
            if constexpr (v > 1) r += (v - 1) * R[hidx<L>(t, u, v - 2)];
        }
        R[hidx<L>(t, u, v)] = r;
        if constexpr (plan.last[kk]) R[0] = F[plan.n[kk]];
    });
}

// Sums a block over the records of a pair: acc[ab] += sum_h E[ab][h] W(h) for every component pair.
template <int LA, int LB, int L, class Acc, class W>
QS_HD void add_pair(const double *__restrict__ rec, Acc acc, W w) {
    using C = PairClass<LA, LB>;
    static_for<C::na * C::nb>([&](auto kk) {
        constexpr int ny = C::table.y[kk] + 1, nz = C::table.z[kk] + 1, at = C::table.at[kk];
        double s = 0.0;
        static_for<C::table.terms[kk]>([&](auto mm) {
            constexpr int m = mm;
            s += rec[at + m] * w(std::integral_constant<int, m / (ny * nz)>{},
                                                std::integral_constant<int, m / nz % ny>{},
                                                std::integral_constant<int, m % nz>{});
        });
        acc(kk, s);
    });
}

// The real solid harmonics (m = 0, 1c, 1s, 2c, 2s) of one shell index in the place of its first 2l + 1 normalised Cartesian
// components, at(c) the component c.
template <int LQ, class At>
QS_HD void spherical_in_place(At at) {
    using std::integral_constant;
    if constexpr (LQ == 1) {
        const double x = at(integral_constant<int, 0>{}), y = at(integral_constant<int, 1>{});
        at(integral_constant<int, 0>{}) = at(integral_constant<int, 2>{});
        at(integral_constant<int, 1>{}) = x;
        at(integral_constant<int, 2>{}) = y;
    } else if constexpr (LQ == 2) {
        const double xx = at(integral_constant<int, 0>{}), xy = at(integral_constant<int, 1>{}),
                     yy = at(integral_constant<int, 2>{}), xz = at(integral_constant<int, 3>{}),
                     yz = at(integral_constant<int, 4>{}), zz = at(integral_constant<int, 5>{});
        at(integral_constant<int, 0>{}) = zz - 0.5 * (xx + yy);
        at(integral_constant<int, 1>{}) = xz;
        at(integral_constant<int, 2>{}) = yz;
        at(integral_constant<int, 3>{}) = 0.86602540378443864676 * (xx - yy);
        at(integral_constant<int, 4>{}) = xy;
    }
}

// The functions of a block acc[ab][m] in the place of its Cartesian components ab: function pair (i, j), i and j in the
// roles of the class, ends at acc[i * nb + j].
template <int LA, int LB, int NM>
QS_HD void pair_functions(int spherical, double (&acc)[PairClass<LA, LB>::na * PairClass<LA, LB>::nb][NM]) {
    constexpr int na = PairClass<LA, LB>::na, nb = PairClass<LA, LB>::nb;
    if (!spherical) return;
    static_for<na * NM>([&](auto k) {
        spherical_in_place<LB>([&](auto c) -> double & { return acc[k / NM * nb + c][k % NM]; });
    });
    static_for<nb * NM>([&](auto k) {
        spherical_in_place<LA>([&](auto c) -> double & { return acc[c * nb + k / NM][k % NM]; });
    });
}

// f(i, j, ab) for the function pairs of the class, ab their place in a block.
template <int LA, int LB, class F>
QS_HD void for_functions(int spherical, F f) {
    constexpr int nb = PairClass<LA, LB>::nb;
    const int ma = spherical ? 2 * LA + 1 : cartesians(LA), mb = spherical ? 2 * LB + 1 : nb;
    static_for<cartesians(LA) * nb>([&](auto ab) {
        constexpr int i = ab / nb, j = ab % nb;
        if (i < ma && j < mb) f(i, j, ab);
    });
}

// Fit shell components: s; x, y, z; xx, yy, zz, xy, xz, yz.  W_h of component M of a fit shell of LC from the Hermite
// integrals R of order L, without the shell's common factor c (-1 / 2g)^l; g2 = 2 g.
template <int LC, int M, int L>
QS_HD double fit_component(const double *R, int t, int u, int v, double g2) {
    constexpr double r3 = 1.7320508075688772935;      // the factor of xy, xz and yz
    constexpr int d[3] = {(L + 1) * (L + 1), L + 1, 1};
    const int o = hidx<L>(t, u, v);
    if constexpr (LC == 0) return R[o];
    else if constexpr (LC == 1) return R[o + d[M]];
    else if constexpr (M < 3) return R[o + 2 * d[M]] + g2 * R[o];
    else return r3 * R[o + (M == 5 ? d[1] : d[0]) + (M == 3 ? d[1] : d[2])];
}

// The functions of the fit shells of LC that components M0 .. M0 + NM - 1 make: their indices and values f(function, value)
// from the components x[m].  Spherical functions are in the order m = 0, 1c, 1s, 2c, 2s.
template <int LC, int M0, int NM, class F>
QS_HD void fit_functions(int spherical, const double (&x)[NM], F f) {
    if constexpr (LC == 0) f(0, x[0]);
    else if constexpr (LC == 1) static_for<3>([&](auto m) { f(spherical ? (m + 1) % 3 : static_cast<int>(m), x[m]); });
    else {
        if constexpr (M0 == 0) {
            const double xx = x[0], yy = x[1], zz = x[2];
            if (spherical) {
                f(0, zz - 0.5 * (xx + yy));
                f(3, 0.86602540378443864676 * (xx - yy));
            } else {
                f(0, xx);
                f(2, yy);
                f(5, zz);
            }
        }
        if constexpr (M0 + NM == 6) {
            f(spherical ? 4 : 1, x[3 - M0]);
            f(spherical ? 1 : 3, x[4 - M0]);
            f(spherical ? 2 : 4, x[5 - M0]);
        }
    }
}

// Cartesian block of a pair (its n records) with components M0 .. M0 + NM - 1 of one fit shell C: acc[ab][m].
template <int LA, int LB, int LC, int M0, int NM>
QS_HD void fit_block(const double *__restrict__ records, int n, const QShell &C, const double *__restrict__ fExps,
                     const double *__restrict__ fCoefs, const double *__restrict__ boysTable,
                     double (&acc)[PairClass<LA, LB>::na * PairClass<LA, LB>::nb][NM]) {
    using PC = PairClass<LA, LB>;
    constexpr int L = LA + LB + LC;
    static_for<PC::na * PC::nb>([&](auto kk) { static_for<NM>([&](auto mm) { acc[kk][mm] = 0.0; }); });
    for (int qc = 0; qc < C.nPrim; qc++) {
        const double g = fExps[C.prim + qc], ig = 1.0 / g;
        // 2 pi^(5/2) / (p g sqrt(p + g)) with the fit shell's factor folded in; pi^(5/2) = 17.493418327624862.
        double fs = 2.0 * 17.493418327624862 * ig * fCoefs[C.prim + qc];
        static_for<LC>([&](auto) { fs *= -0.5 * ig; });
        for (int r = 0; r < n; r++) {
            const double *rec = records + static_cast<long long>(r) * PC::size;
            const double p = rec[0], is = 1.0 / (p + g);
            double R[(L + 1) * (L + 1) * (L + 1)];
            hermite_of<L>(p * g * is, rec[2] - C.x, rec[3] - C.y, rec[4] - C.z, fs * rec[1] * sqrt(is), boysTable, R);
            static_for<NM>([&](auto mm) {
                constexpr int m = mm;
                add_pair<LA, LB, L>(rec, [&](auto ab, double s) { acc[ab][m] += s; }, [&](auto t, auto u, auto v) {
                    return fit_component<LC, M0 + m, L>(R, t, u, v, 2.0 * g);
                });
            });
        }
    }
}

// Components of a d fit shell that one block takes: all six, or three where a block of six would not fit in registers.
template <int LA, int LB, int LC>
constexpr int fit_group() {
    return LC < 2 ? cartesians(LC) : (cartesians(LA) * cartesians(LB) <= 9 ? 6 : 3);
}

// Overlap and kinetic energy blocks of a pair, into the packed matrices (mu >= nu).
template <int LA, int LB, class Out>
QS_HD void overlap_kinetic(const QShell &A, const QShell &B, const double *__restrict__ exps,
                           const double *__restrict__ coefs, int spherical, Out out) {
    using C = PairClass<LA, LB>;
    constexpr int NJ = LB + 3;
    double acc[C::na * C::nb][2];
    static_for<C::na * C::nb>([&](auto kk) { acc[kk][0] = acc[kk][1] = 0.0; });
    const double X[3] = {A.x - B.x, A.y - B.y, A.z - B.z};
    const double r2 = X[0] * X[0] + X[1] * X[1] + X[2] * X[2];
    for (int qa = 0; qa < A.nPrim; qa++)
        for (int qb = 0; qb < B.nPrim; qb++) {
            const double a = exps[A.prim + qa], b = exps[B.prim + qb], p = a + b, ip = 1.0 / p, h = 0.5 * ip;
            const double pip = M_PI * ip;
            const double K = coefs[A.prim + qa] * coefs[B.prim + qb] * exp(-a * b * ip * r2) * pip * sqrt(pip);
            // One-dimensional overlaps without their prefactor: S_i,j+1 = X_PB S_ij + (i S_i-1,j + j S_i,j-1) / 2p.
            double S1[3][LA + 1][NJ], T1[3][LA + 1][LB + 1];
            static_for<3>([&](auto dd) {
                constexpr int d = dd;
                const double pa = -b * ip * X[d], pb = a * ip * X[d];
                static_for<(LA + 1) * NJ>([&](auto kk) {
                    constexpr int i = kk / NJ, j = kk % NJ;
                    if constexpr (i + j == 0) S1[d][i][j] = 1.0;
                    else if constexpr (j == 0) {
                        double s = pa * S1[d][i - 1][0];
                        if constexpr (i > 1) s += (i - 1) * h * S1[d][i > 1 ? i - 2 : 0][0];
                        S1[d][i][j] = s;
                    } else {
                        double s = pb * S1[d][i][j - 1];
                        if constexpr (i > 0) s += i * h * S1[d][i > 0 ? i - 1 : 0][j - 1];
                        if constexpr (j > 1) s += (j - 1) * h * S1[d][i][j > 1 ? j - 2 : 0];
                        S1[d][i][j] = s;
                    }
                });
                static_for<(LA + 1) * (LB + 1)>([&](auto kk) {
                    constexpr int i = kk / (LB + 1), j = kk % (LB + 1);
                    double s = b * (2 * j + 1) * S1[d][i][j] - 2.0 * b * b * S1[d][i][j + 2];
                    if constexpr (j > 1) s -= 0.5 * j * (j - 1) * S1[d][i][j > 1 ? j - 2 : 0];
                    T1[d][i][j] = s;
                });
            });
            static_for<C::na * C::nb>([&](auto kk) {
                constexpr int ab = kk, ia = ab / C::nb, ib = ab % C::nb;
                constexpr Powers u = powers_of(LA, ia), v = powers_of(LB, ib);
                const double f = K * cart_factor(LA, ia) * cart_factor(LB, ib);
                const double sx = S1[0][u.x][v.x], sy = S1[1][u.y][v.y], sz = S1[2][u.z][v.z];
                acc[ab][0] += f * sx * sy * sz;
                acc[ab][1] += f * (T1[0][u.x][v.x] * sy * sz + sx * T1[1][u.y][v.y] * sz + sx * sy * T1[2][u.z][v.z]);
            });
        }
    pair_functions<LA, LB, 2>(spherical, acc);
    for_functions<LA, LB>(spherical, [&](int i, int j, auto ab) { out(i, j, acc[ab][0], acc[ab][1]); });
}

// Nuclear attraction of a pair (its n records) by the nuclei C0, C0 + step, ... of Gaussian charges Z (z/pi)^(3/2)
// exp(-z r^2), z = kNuclearExponent: -Z_C (2 pi / p) sqrt(z / (p + z)) sum_tuv E_tuv R_tuv(p z / (p + z), P - C).
template <int LA, int LB>
QS_HD void nuclear_block(const double *__restrict__ records, int n, int C0, int step, int nAtoms,
                         const double *__restrict__ atoms, const double *__restrict__ boysTable,
                         double (&acc)[PairClass<LA, LB>::na * PairClass<LA, LB>::nb][1]) {
    using PC = PairClass<LA, LB>;
    constexpr int L = LA + LB;
    static_for<PC::na * PC::nb>([&](auto kk) { acc[kk][0] = 0.0; });
    for (int C = C0; C < nAtoms; C += step) {
        const double cx = atoms[4 * C], cy = atoms[4 * C + 1], cz = atoms[4 * C + 2], q = -2.0 * M_PI * atoms[4 * C + 3];
        for (int r = 0; r < n; r++) {
            const double *rec = records + static_cast<long long>(r) * PC::size;
            const double p = rec[0], w = kNuclearExponent / (p + kNuclearExponent);
            double R[(L + 1) * (L + 1) * (L + 1)];
            hermite_of<L>(p * w, rec[2] - cx, rec[3] - cy, rec[4] - cz, q * rec[1] * sqrt(w), boysTable, R);
            add_pair<LA, LB, L>(rec, [&](auto ab, double s) { acc[ab][0] += s; },
                                [&](auto t, auto u, auto v) { return R[hidx<L>(t, u, v)]; });
        }
    }
}

// f(la, lb) as compile-time constants for the class la >= lb.
template <class F>
QS_HD void with_pair_class(int la, int lb, F f) {
    using std::integral_constant;
    switch (la * (la + 1) / 2 + lb) {
        case 0: f(integral_constant<int, 0>{}, integral_constant<int, 0>{}); break;
        case 1: f(integral_constant<int, 1>{}, integral_constant<int, 0>{}); break;
        case 2: f(integral_constant<int, 1>{}, integral_constant<int, 1>{}); break;
        case 3: f(integral_constant<int, 2>{}, integral_constant<int, 0>{}); break;
        case 4: f(integral_constant<int, 2>{}, integral_constant<int, 1>{}); break;
        default: f(integral_constant<int, 2>{}, integral_constant<int, 2>{}); break;
    }
}

// The pair A, B (A >= B) in the roles of its class, with room for its records from offset first.
inline PairItem pair_item(const QShell *shells, int a, int b, long long row, long long first) {
    const bool swapped = shells[a].l < shells[b].l;
    return PairItem{swapped ? b : a, swapped ? a : b, swapped ? 1 : 0, 0, first, row};
}
// Doubles of a pair's records, all its primitive pairs kept.
inline long long record_room(const QShell &A, const QShell &B) {
    static constexpr long long size[3][3] = {{PairClass<0, 0>::size, PairClass<1, 0>::size, PairClass<2, 0>::size},
                                             {PairClass<1, 0>::size, PairClass<1, 1>::size, PairClass<2, 1>::size},
                                             {PairClass<2, 0>::size, PairClass<2, 1>::size, PairClass<2, 2>::size}};
    return size[A.l][B.l] * A.nPrim * B.nPrim;
}

// The unit function as an s shell whose one primitive, of exponent 0 and coefficient 1, is at prim: a pair with it is the
// other shell alone.
inline QShell unit_shell(int prim) {
    QShell u{};
    u.nPrim = 1;
    u.prim = prim;
    u.nf = 1;
    return u;
}

// Row of function i of the first role and j of the second (mb functions of the pair's second shell B).
QS_HD long long pair_row(const PairItem &it, int i, int j, int ma, int mb) {
    return it.row + (it.swapped ? static_cast<long long>(j) * ma + i : static_cast<long long>(i) * mb + j);
}

// ------------------------------------------------------------------------------------------------------------------------
// One whole work item on the host, for the CPU check of the code above (not part of the GPU build).  The unnamed arguments
// are c2s transformations, which the unrolled forms have as constants.
// ------------------------------------------------------------------------------------------------------------------------
#ifndef __HIPCC__
// F_0 .. F_m (m <= kMaxR) by the fixed-order function of the kernels.
inline void boys(int m, double T, const double *table, double *F) {
    static_for<kMaxR + 1>([&](auto l) {
        if (m != l) return;
        double f[l + 1];
        boys_of<l>(T, table, f);
        for (int n = 0; n <= l; n++) F[n] = f[n];
    });
}

// Overlap, kinetic and electron-nuclear blocks of shell pair k (A >= B), written into the packed matrices (mu >= nu).
inline void one_electron_pair(int k, const QPair *pairs, const QShell *shells, const double *exps, const double *coefs,
                              int nAtoms, const double *atoms, int spherical, const double *boysTable, const double *,
                              double *S, double *T, double *V) {
    const PairItem it = pair_item(shells, pairs[k].x, pairs[k].y, 0, 0);
    const QShell &A = shells[it.a], &B = shells[it.b];
    std::vector<double> records(static_cast<size_t>(record_room(A, B)));
    with_pair_class(A.l, B.l, [&](auto la, auto lb) {
        const int n = pair_records<la, lb>(A, B, exps, coefs, records.data());
        auto at = [&](double *M, int i, int j) -> double & { return M[packed_index(A.f0 + i, B.f0 + j)]; };
        overlap_kinetic<la, lb>(A, B, exps, coefs, spherical, [&](int i, int j, double s, double t) {
            at(S, i, j) = s;
            at(T, i, j) = t;
        });
        double acc[PairClass<la, lb>::na * PairClass<la, lb>::nb][1];
        nuclear_block<la, lb>(records.data(), n, 0, 1, nAtoms, atoms, boysTable, acc);
        pair_functions<la, lb, 1>(spherical, acc);
        for_functions<la, lb>(spherical, [&](int i, int j, auto ab) { at(V, i, j) = acc[ab][0]; });
    });
}

// (C|D) of fit shell pair k (C >= D) into the packed fit matrix; the diagonal pair also writes its functions' integrals into
// row nFit.  C is taken as a pair with the unit shell.
inline void fit_matrix_pair(int k, const QPair *pairs, const QShell *shells, const double *exps, const double *coefs, int nFit,
                            int spherical, const double *boysTable, const double *, double *M) {
    QShell C = shells[pairs[k].x];
    const QShell &D = shells[pairs[k].y];
    std::vector<double> e(exps + C.prim, exps + C.prim + C.nPrim), c(coefs + C.prim, coefs + C.prim + C.nPrim);
    C.prim = 0;
    const QShell unit = unit_shell(C.nPrim);
    e.push_back(0.0);
    c.push_back(1.0);
    std::vector<double> records(static_cast<size_t>(record_room(C, unit)));
    auto left = [&](auto la) {
        const int n = pair_records<la, 0>(C, unit, e.data(), c.data(), records.data());
        auto item = [&](auto lc, auto m0) {
            constexpr int NM = fit_group<la, 0, lc>(), M0 = m0;
            double acc[PairClass<la, 0>::na][NM];
            fit_block<la, 0, lc, M0, NM>(records.data(), n, D, exps, coefs, boysTable, acc);
            pair_functions<la, 0, NM>(spherical, acc);
            for_functions<la, 0>(spherical, [&](int i, int, auto ab) {
                fit_functions<lc, M0, NM>(spherical, acc[ab], [&](int f, double x) { M[packed_index(C.f0 + i, D.f0 + f)] = x; });
            });
        };
        using std::integral_constant;
        const integral_constant<int, 0> zero;
        if (D.l == 0) item(zero, zero);
        else if (D.l == 1) item(integral_constant<int, 1>{}, zero);
        else item(integral_constant<int, 2>{}, zero);
        if (pairs[k].x == pairs[k].y)
            overlap_kinetic<la, 0>(C, unit, e.data(), c.data(), spherical,
                                   [&](int i, int, double s, double) { M[packed_index(nFit, C.f0 + i)] = s; });
    };
    if (C.l == 0) left(std::integral_constant<int, 0>{});
    else if (C.l == 1) left(std::integral_constant<int, 1>{});
    else left(std::integral_constant<int, 2>{});
}

// (mu nu|P) of item k = (significant orbital shell pair k / nFitShells, fit shell k % nFitShells) into its rows of B
// ([row][fit function]); magnitudes <= kUnderFlow are stored as zero.
inline void fit_integrals_item(long long k, int nFitShells, const PairEntry *pairs, const QShell *oShells,
                               const double *oExps, const double *oCoefs, int oSpherical, const QShell *fShells,
                               const double *fExps, const double *fCoefs, int fSpherical, int nFit, const double *boysTable,
                               const double *, double *B) {
    const PairEntry pe = pairs[k / nFitShells];
    const QShell &C = fShells[k % nFitShells];
    const PairItem it = pair_item(oShells, pe.a, pe.b, pe.row, 0);
    const QShell &A = oShells[it.a], &Bs = oShells[it.b];
    std::vector<double> records(static_cast<size_t>(record_room(A, Bs)));
    with_pair_class(A.l, Bs.l, [&](auto la, auto lb) {
        const int n = pair_records<la, lb>(A, Bs, oExps, oCoefs, records.data());
        auto item = [&](auto lc, auto m0) {
            constexpr int NM = fit_group<la, lb, lc>(), M0 = m0;
            double acc[PairClass<la, lb>::na * PairClass<la, lb>::nb][NM];
            fit_block<la, lb, lc, M0, NM>(records.data(), n, C, fExps, fCoefs, boysTable, acc);
            pair_functions<la, lb, NM>(oSpherical, acc);
            for_functions<la, lb>(oSpherical, [&](int i, int j, auto ab) {
                double *out = B + pair_row(it, i, j, A.nf, Bs.nf) * nFit + C.f0;
                fit_functions<lc, M0, NM>(fSpherical, acc[ab], [&](int f, double x) {
                    out[f] = fabs(x) > kUnderFlow ? x : 0.0;
                });
            });
        };
        using std::integral_constant;
        const integral_constant<int, 0> zero;
        if (C.l == 0) item(zero, zero);
        else if (C.l == 1) item(integral_constant<int, 1>{}, zero);
        else {
            item(integral_constant<int, 2>{}, zero);
            if constexpr (fit_group<la, lb, 2>() == 3) item(integral_constant<int, 2>{}, integral_constant<int, 3>{});
        }
    });
}

#endif

}  // namespace qs
