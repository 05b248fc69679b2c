// Grid construction on the device: Euler-Maclaurin radial shells x pruned Lebedev-Laikov spheres around every atom, Becke
// partition weights in FP64, the |w| > 1e-30 cull and per-atom blocks of at most 128 points.
//
// Follows DFTGrid_Construct (pMolecule/QCModel/__extensions__/csource/DFTGrid.c:105-263) with DFTGrid_Atom_Parameters
// (:474-523), DFTGrid_Radial_Points (:562-575), the Lebedev size <-> degree maps (pScientific/Quadrature/__extensions__/
// csource/Lebedev.c:62-193), the octahedral orbit expansion order (Lebedev.c:1565-1719) and the Becke weight
// (DFTGridWeights.c:43-80, 220-258).
//
// Device layout: a group of 16 to 64 lanes of a radial shell's (atom, radius) work-groups computes the Becke weight of one
// angular point in FP64, the atoms spread over its lanes.  Candidate points of one atom are contiguous and ordered (radial shell, angular index) exactly as the
// reference orders them, so the order-preserving cull reproduces the reference's point and block order.
//
// Becke weight: P_A / sum_i P_i with P_i = prod_{j != i} s(nu_ij).  P_A (the point's own atom) is formed first, then the
// product of the atom whose factors with the atoms done so far leave the largest bound, and so on until every remaining
// atom's bound is below 2^-64 of the largest product: each cell function lies in [0, 1], so what is left out of the sum is
// below nAtoms * 2^-64 of it.  This turns the reference's O(nAtoms^2) pair loop per point into O(nAtoms) for each of the
// few atoms whose cells matter at the point.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <hip/hip_runtime.h>

#include "lebedev_tables.h"
#include "xq_internal.h"

// No fused multiply-add in this file: the cull |w| > 1e-30 depends on Becke cell factors that cancel to exactly zero near
// nuclei, so point coordinates, distances and the cell polynomial are rounded operation by operation as in the reference.
#pragma clang fp contract(off)

namespace xq {

namespace {

// Bragg radii in Angstrom by atomic number (DFTGrid.c:29-40).
const double kBragg[120] = {
    0.75, 0.35, 0.35, 1.45, 1.05, 0.85, 0.70, 0.65, 0.60, 0.50, 0.50, 1.80, 1.50, 1.25, 1.10, 1.00, 1.00, 1.00, 1.00, 2.20,
    1.80, 1.60, 1.40, 1.35, 1.40, 1.40, 1.40, 1.35, 1.35, 1.35, 1.35, 1.30, 1.25, 1.15, 1.15, 1.15, 1.15, 2.35, 2.00, 1.80,
    1.55, 1.45, 1.45, 1.35, 1.30, 1.35, 1.40, 1.60, 1.55, 1.55, 1.45, 1.45, 1.40, 1.40, 1.40, 2.60, 2.15, 1.95, 1.85, 1.85,
    1.85, 1.85, 1.85, 1.85, 1.80, 1.75, 1.75, 1.75, 1.75, 1.75, 1.75, 1.75, 1.55, 1.45, 1.35, 1.35, 1.30, 1.35, 1.35, 1.35,
    1.50, 1.90, 1.80, 1.60, 1.90, 1.90, 1.90, 2.60, 2.15, 1.95, 1.80, 1.80, 1.75, 1.75, 1.75, 1.75, 1.75, 1.75, 1.75, 1.75,
    1.75, 1.75, 1.75, 1.75, 1.55, 1.55, 1.55, 1.55, 1.55, 1.55, 1.55, 1.55, 1.55, 1.55, 1.55, 1.55, 1.55, 1.55, 1.55, 1.55};
const double kAngstromToBohr = 1.0e-10 / 5.291772083e-11;   // Units.h:35, Constants.h:15
const double kBFTol[5] = {1.0e-8, 1.0e-9, 1.0e-10, 1.0e-12, 1.0e-15};    // DFTGrid.c:43
const double kRhoTol[5] = {1.0e-13, 1.0e-14, 1.0e-15, 1.0e-17, 1.0e-20}; // DFTGrid.c:46
constexpr int kMinL = 9;                 // DFTGrid.c:101
constexpr double kRadialCutFactor = 0.2; // DFTGrid.c:102
constexpr double kWeightTol = 1.0e-30;   // DFTGrid.c:103

void atom_parameters(int accuracy, int z, int *nR, int *lMax, double *rMax) {
    switch (accuracy) {
        case 0: *nR = z < 11 ? 21 : z < 19 ? 42 : z < 37 ? 75 : 84; *rMax = 20.0; *lMax = 23; break;
        case 1: *nR = z < 11 ? 35 : z < 19 ? 70 : z < 37 ? 95 : 104; *rMax = 25.0; *lMax = 35; break;
        case 2: *nR = z < 11 ? 49 : z < 19 ? 88 : z < 37 ? 112 : 123; *rMax = 30.0; *lMax = z < 11 ? 35 : 41; break;
        case 3:
            *nR = z < 11 ? 70 : z < 19 ? 123 : z < 37 ? 130 : 155; *rMax = 35.0;
            *lMax = z < 11 ? 41 : z < 19 ? 47 : z < 89 ? 53 : 59;
            break;
        default: *nR = z < 11 ? 100 : z < 19 ? 125 : z < 37 ? 160 : 205; *rMax = 35.0; *lMax = 65; break;
    }
}

double bragg_radius(int z) {
    if (z < 0) z = 0;
    if (z >= 120) z = 119;
    return kAngstromToBohr * kBragg[z];
}

// Number of points of the smallest rule integrating degree l (Lebedev.c:134-193).
int lebedev_size_for_l(int l) {
    static const int small[16] = {6, 6, 14, 26, 38, 50, 74, 86, 110, 146, 170, 194, 230, 266, 302, 350};
    static const int large[22] = {0, 0, 0, 0, 0, 434, 590, 770, 974, 1202, 1454, 1730, 2030, 2354, 2702, 3074, 3470,
                                  3890, 4334, 4802, 5294, 5810};
    if (l < 3) return 6;
    if (l <= 31) return small[l / 2];
    if (l <= 131) return large[l / 6];
    return 0;
}

// Degree of the smallest rule with at least n points (Lebedev.c:62-98).
int lebedev_l_for_size(int n) {
    static const int ls[XQ_LEBEDEV_NRULES] = {3, 5, 7, 9, 11, 13, 15, 17, 19, 21, 23, 25, 27, 29, 31, 35,
                                              41, 47, 53, 59, 65, 71, 77, 83, 89, 95, 101, 107, 113, 119, 125, 131};
    for (int k = 0; k < XQ_LEBEDEV_NRULES; k++)
        if (n <= xq_lebedev_npoints[k]) return ls[k];
    return 0;
}

// Expand rule k into unit vectors and weights, in the orbit order of Lebedev.c:1565-1719.  Each template row names, for x, y
// and z, the generator slot (1 = a, 2 = b, 3 = c, 0 = zero) and its sign.
int lebedev_expand(int k, double *out /* x, y, z, w per point */) {
    static const signed char T1[6][3] = {{1, 0, 0}, {-1, 0, 0}, {0, 1, 0}, {0, -1, 0}, {0, 0, 1}, {0, 0, -1}};
    static const signed char T2[12][3] = {{0, 1, 1}, {0, 1, -1}, {0, -1, 1}, {0, -1, -1}, {1, 0, 1}, {1, 0, -1},
                                          {-1, 0, 1}, {-1, 0, -1}, {1, 1, 0}, {1, -1, 0}, {-1, 1, 0}, {-1, -1, 0}};
    static const signed char T3[8][3] = {{1, 1, 1}, {1, 1, -1}, {1, -1, 1}, {1, -1, -1},
                                         {-1, 1, 1}, {-1, 1, -1}, {-1, -1, 1}, {-1, -1, -1}};
    static const signed char T4[24][3] = {{1, 1, 2}, {1, 1, -2}, {1, -1, 2}, {1, -1, -2}, {-1, 1, 2}, {-1, 1, -2},
                                          {-1, -1, 2}, {-1, -1, -2}, {1, 2, 1}, {1, -2, 1}, {1, 2, -1}, {1, -2, -1},
                                          {-1, 2, 1}, {-1, -2, 1}, {-1, 2, -1}, {-1, -2, -1}, {2, 1, 1}, {-2, 1, 1},
                                          {2, 1, -1}, {-2, 1, -1}, {2, -1, 1}, {-2, -1, 1}, {2, -1, -1}, {-2, -1, -1}};
    static const signed char T5[24][3] = {{1, 2, 0}, {1, -2, 0}, {-1, 2, 0}, {-1, -2, 0}, {2, 1, 0}, {2, -1, 0},
                                          {-2, 1, 0}, {-2, -1, 0}, {1, 0, 2}, {1, 0, -2}, {-1, 0, 2}, {-1, 0, -2},
                                          {2, 0, 1}, {2, 0, -1}, {-2, 0, 1}, {-2, 0, -1}, {0, 1, 2}, {0, 1, -2},
                                          {0, -1, 2}, {0, -1, -2}, {0, 2, 1}, {0, 2, -1}, {0, -2, 1}, {0, -2, -1}};
    static const signed char T6[48][3] = {
        {1, 2, 3}, {1, 2, -3}, {1, -2, 3}, {1, -2, -3}, {-1, 2, 3}, {-1, 2, -3}, {-1, -2, 3}, {-1, -2, -3},
        {1, 3, 2}, {1, 3, -2}, {1, -3, 2}, {1, -3, -2}, {-1, 3, 2}, {-1, 3, -2}, {-1, -3, 2}, {-1, -3, -2},
        {2, 1, 3}, {2, 1, -3}, {2, -1, 3}, {2, -1, -3}, {-2, 1, 3}, {-2, 1, -3}, {-2, -1, 3}, {-2, -1, -3},
        {2, 3, 1}, {2, 3, -1}, {2, -3, 1}, {2, -3, -1}, {-2, 3, 1}, {-2, 3, -1}, {-2, -3, 1}, {-2, -3, -1},
        {3, 1, 2}, {3, 1, -2}, {3, -1, 2}, {3, -1, -2}, {-3, 1, 2}, {-3, 1, -2}, {-3, -1, 2}, {-3, -1, -2},
        {3, 2, 1}, {3, 2, -1}, {3, -2, 1}, {3, -2, -1}, {-3, 2, 1}, {-3, 2, -1}, {-3, -2, 1}, {-3, -2, -1}};
    int m = 0;
    for (int o = xq_lebedev_first[k]; o < xq_lebedev_first[k + 1]; o++) {
        const xq_lebedev_orbit &orb = xq_lebedev_orbits[o];
        double g[4] = {0.0, 0.0, 0.0, 0.0};
        const signed char(*T)[3] = nullptr;
        int count = 0;
        switch (orb.type) {
            case 1: g[1] = 1.0; T = T1; count = 6; break;
            case 2: g[1] = 1.0 / std::sqrt(2.0); T = T2; count = 12; break;
            case 3: g[1] = 1.0 / std::sqrt(3.0); T = T3; count = 8; break;
            case 4: g[1] = orb.a; g[2] = std::sqrt(1.0 - 2.0 * orb.a * orb.a); T = T4; count = 24; break;
            case 5: g[1] = orb.a; g[2] = std::sqrt(1.0 - orb.a * orb.a); T = T5; count = 24; break;
            case 6: g[1] = orb.a; g[2] = orb.b; g[3] = std::sqrt(1.0 - orb.a * orb.a - orb.b * orb.b); T = T6; count = 48; break;
        }
        for (int n = 0; n < count; n++, m++) {
            for (int c = 0; c < 3; c++) {
                int s = T[n][c];
                out[4 * m + c] = s == 0 ? 0.0 : (s > 0 ? g[s] : -g[-s]);
            }
            out[4 * m + 3] = orb.v;
        }
    }
    return m;
}

// Becke cell-function constants (DFTGridWeights.c:21-35).
__constant__ double c_beckeC[11] = {1.000000000000000e+00, -3.333333333333333e+00, 9.000000000000000e+00,
                                    -17.142857142857142e+00, 23.333333333333332e+00, -22.909090909090910e+00,
                                    16.153846153846153e+00, -8.000000000000000e+00, 2.647058823529412e+00,
                                    -0.526315789473684e+00, 0.047619047619048e+00};
constexpr double kBeckeA = 1.850069046020527e+00;

struct RadialShell {
    int atom;
    int rule;        // first unit vector of the Lebedev rule in the device rule array
    int nAng;
    int out;         // first candidate point of the shell
    double r;
    double wr;       // 4 pi w_r
};

__device__ __forceinline__ double becke_poly(double nu) {
    double nu2 = nu * nu, term = nu, sum = 0.0;
#pragma unroll
    for (int t = 0; t <= 10; t++) {
        sum += c_beckeC[t] * term;
        term *= nu2;
    }
    return sum;
}

// Reductions over groups of GS = 16, 32 or 64 lanes, every lane receiving the result.  The lane exchanges are register
// moves (DPP within a row of 16 lanes, row and half swaps above): with shuffles through the LDS crossbar, six dependent ones
// per reduction, the weight derivatives of (H2O)64 took 24 ms instead of 20, its grid weights 14 instead of 12.
template <int kControl>
__device__ __forceinline__ unsigned row_move(unsigned x) {
    return static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(x), kControl, 0xf, 0xf, true));
}
template <int kControl>
__device__ __forceinline__ double row_move(double x) {
    return __hiloint2double(static_cast<int>(row_move<kControl>(static_cast<unsigned>(__double2hiint(x)))),
                            static_cast<int>(row_move<kControl>(static_cast<unsigned>(__double2loint(x)))));
}
// The even and the odd rows of 16 lanes (kRows = 1), or the halves of the wave (kRows = 2), each in place of both.
template <int kRows>
__device__ __forceinline__ void spread(unsigned x, unsigned &even, unsigned &odd) {
    if constexpr (kRows == 1) {
        const auto p = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        even = p[0];
        odd = p[1];
    } else {
        const auto p = __builtin_amdgcn_permlane32_swap(x, x, false, false);
        even = p[0];
        odd = p[1];
    }
}
template <int kRows>
__device__ __forceinline__ void spread(double x, double &even, double &odd) {
    unsigned eh, oh, el, ol;
    spread<kRows>(static_cast<unsigned>(__double2hiint(x)), eh, oh);
    spread<kRows>(static_cast<unsigned>(__double2loint(x)), el, ol);
    even = __hiloint2double(static_cast<int>(eh), static_cast<int>(el));
    odd = __hiloint2double(static_cast<int>(oh), static_cast<int>(ol));
}
template <int GS, class T, class Op>
__device__ __forceinline__ T group_reduce(T x, Op op) {
    static_assert(GS == 16 || GS == 32 || GS == 64, "groups of whole rows");
    x = op(x, row_move<0xB1>(x));       // lanes 1, 0, 3, 2 of each four
    x = op(x, row_move<0x4E>(x));       // lanes 2, 3, 0, 1
    x = op(x, row_move<0x141>(x));      // each eight lanes reversed
    x = op(x, row_move<0x140>(x));      // each sixteen lanes reversed
    T even, odd;
    if constexpr (GS >= 32) { spread<1>(x, even, odd); x = op(even, odd); }
    if constexpr (GS == 64) { spread<2>(x, even, odd); x = op(even, odd); }
    return x;
}
template <int GS>
__device__ __forceinline__ double group_sum(double x) { return group_reduce<GS>(x, [](double u, double v) { return u + v; }); }
template <int GS>
__device__ __forceinline__ double group_product(double x) { return group_reduce<GS>(x, [](double u, double v) { return u * v; }); }

// LDS writes of a wave are in order; this keeps the compiler from moving accesses over it.
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The group's ballot bits (group at lane bit0 of its wave), lowest first.
template <int GS>
__device__ __forceinline__ unsigned long long group_ballot(bool x, int bit0) {
    return (__ballot(x) >> bit0) & (GS == 64 ? ~0ull : ((1ull << (GS & 63)) - 1ull));
}

// The atom (lane atoms gl + GS a, not done) of the largest bound of a group by the bounds' upper words, and that bound or
// the next larger double with these upper words (0 if all are done or vanish).
template <int LA, int GS>
__device__ __forceinline__ int next_atom(const double (&b)[LA], const bool (&done)[LA], int gl, int bit0, double &top) {
    unsigned best = 0u;
    int bi = gl;
#pragma unroll
    for (int a = 0; a < LA; a++) {
        const unsigned key = done[a] ? 0u : static_cast<unsigned>(__double2hiint(b[a]));
        if (key > best) { best = key; bi = gl + GS * a; }
    }
    const unsigned most = group_reduce<GS>(best, [](unsigned u, unsigned v) { return u > v ? u : v; });
    top = most == 0u ? 0.0 : __hiloint2double(static_cast<int>(most), -1);
    const int first = __ffsll(static_cast<long long>(group_ballot<GS>(best == most, bit0))) - 1;
    if constexpr (GS == 64) return __builtin_amdgcn_readlane(bi, first);
    else return __shfl(bi, bit0 + first, 64);
}

// The pairs of atom c with the lane atoms.  With up to four atoms per lane they are loaded when c is known, before the
// reductions that end the row before; more would cost too many registers, and are read in place.
template <int LA, int GS>
struct PairRow {
    static constexpr int kAhead = LA <= 4 ? LA : 1;
    const double2 *__restrict__ row;
    double2 q[kAhead];
    __device__ __forceinline__ void load(const double2 *__restrict__ pairs, int c, int gl, int nAtoms) {
        row = pairs + static_cast<size_t>(c) * nAtoms + gl;
        if constexpr (kAhead == LA)
#pragma unroll
            for (int a = 0; a < LA; a++) q[a] = gl + GS * a < nAtoms ? row[GS * a] : make_double2(0.0, 0.0);
    }
    __device__ __forceinline__ double2 operator[](int a) const {
        if constexpr (kAhead == LA) return q[a];
        else return row[GS * a];
    }
};

// Share of the largest cell product at a point below which an atom's product does not count: in the sum of the products, and
// in the derivatives, where a factor s = c y^11 P (y = 1 - nu) near its zero has a derivative of 11 s / y, so that a dropped
// term is below 1e-16 of the point's energy over a bond length.  With 2^-80 gradients and weights are the same to 2e-15 and
// (H2O)64 gradients take 39.6 instead of 35.1 ms.
constexpr double kCellScreen = 0x1p-64;

// Candidate points of one radial shell and their Becke weights w = 4 pi w_r w_ang P_A / sum_i P_i (DFTGrid.c:158-211,
// DFTGridWeights.c:220-258).  A group of GS lanes takes a point, lane l the atoms l, l + GS, ... (at most LA).  Row c
// evaluates the pairs of atom c with every lane atom: s_ci for P_c and s_ic for the lane atoms' bounds.  Rows are taken for
// the shell's atom A, then always for the atom of the largest bound, until none passes the screen or the point's weight
// cannot pass the cull.  Each factor is the reference's cell function of the same mu and nu, rounded as the reference rounds
// it (so factors that vanish there vanish here, and the same points pass the cull); products and sums are taken in another
// order, so weights agree with the reference's to rounding.  pairs[i][j] = {1 / R_ij, a_ij} (a_ji = -a_ij: -nu and its
// polynomial are exact negatives).  The shell's points are dealt to gridDim.y work-groups.
// Bound by FP64 arithmetic (45 operations a factor).  One point per thread, whose lanes lay in all directions from A and
// so took nearly every factor of every atom between them, took 7.4 ms on (H2O)24 and 48 ms on (H2O)64; this
// takes 2.7 and 11 ms.  Each row's pairs are fetched before the product that ends the row before.
template <int LA, int GS, int WPG>
__global__ void __launch_bounds__(64 * WPG) candidate_points_kernel(const RadialShell *__restrict__ shells,
                                                                    const double *__restrict__ rules,
                                                                    const double *__restrict__ xyz, int nAtoms,
                                                                    const double2 *__restrict__ pairs,
                                                                    double *__restrict__ cx, double *__restrict__ cy,
                                                                    double *__restrict__ cz, double *__restrict__ cw,
                                                                    int *__restrict__ keep) {
    constexpr int kGroups = 64 * WPG / GS;
    extern __shared__ double lds[];
    const int t = threadIdx.x, gl = t & (GS - 1), gi = t / GS, bit0 = t & 63 & ~(GS - 1);
    double *sxyz = lds, *rL = lds + static_cast<size_t>(3 + gi) * nAtoms;
    for (int i = t; i < 3 * nAtoms; i += 64 * WPG) sxyz[i] = xyz[i];
    __syncthreads();
    const RadialShell sh = shells[blockIdx.x];
    const int A = sh.atom;
    for (int k0 = blockIdx.y * kGroups; k0 < sh.nAng; k0 += gridDim.y * kGroups) {
        const int k = k0 + gi;
        const bool active = k < sh.nAng;
        const double *u = rules + 4 * (sh.rule + (active ? k : 0));
        const double px = u[0] * sh.r + sxyz[3 * A], py = u[1] * sh.r + sxyz[3 * A + 1], pz = u[2] * sh.r + sxyz[3 * A + 2];
        const double wru = sh.wr * u[3];
        double r[LA], b[LA];
        bool done[LA];
        wave_fence();
#pragma unroll
        for (int a = 0; a < LA; a++) {
            const int i = gl + GS * a;
            r[a] = 0.0;
            if (i < nAtoms) {
                const double dx = sxyz[3 * i] - px, dy = sxyz[3 * i + 1] - py, dz = sxyz[3 * i + 2] - pz;
                r[a] = sqrt(dx * dx + dy * dy + dz * dz);
                rL[i] = r[a];
            }
            b[a] = 1.0;
            done[a] = i >= nAtoms;
        }
        wave_fence();
        bool run = active;
        int c = A;
        double PA = 0.0, sum = 0.0, most = 0.0, rc = rL[A];
        PairRow<LA, GS> row;
        row.load(pairs, c, gl, nAtoms);
        do {
            double prod = 1.0;
#pragma unroll
            for (int a = 0; a < LA; a++) {
                const int i = gl + GS * a;
                if (i >= nAtoms || i == c) continue;
                const double2 q = row[a];
                const double mu = (rc - r[a]) * q.x, nu = mu + q.y * (1.0 - mu * mu), S = kBeckeA * becke_poly(nu);
                prod *= 0.5 - S;
                b[a] *= fabs(0.5 + S);
            }
            const bool first = c == A;
#pragma unroll
            for (int a = 0; a < LA; a++) done[a] = done[a] || gl + GS * a == c;
            double top;
            c = next_atom<LA, GS>(b, done, gl, bit0, top);
            rc = rL[c];
            row.load(pairs, c, gl, nAtoms);
            prod = group_product<GS>(prod);
            if (run) {
                if (first) PA = prod;
                sum += prod;
                most = fmax(most, fabs(prod));
                // A point whose weight cannot exceed half the cull tolerance with the products so far is culled.
                run = PA != 0.0 && !(sum > 0.0 && fabs(wru) * (fabs(PA) / sum) < 0.5 * kWeightTol) &&
                      top >= kCellScreen * most && top > 0.0;
            }
        } while (__any(run));
        if (active && gl == 0) {
            const int o = sh.out + k;
            const double w = PA != 0.0 ? wru * (PA / sum) : 0.0;
            cx[o] = px;
            cy[o] = py;
            cz[o] = pz;
            cw[o] = w;
            keep[o] = fabs(w) > kWeightTol ? 1 : 0;
        }
    }
}

// Order-preserving compaction of the kept candidates: dst = exclusive prefix sum of keep.
__global__ void compact_points_kernel(int n, const int *__restrict__ keep, const int *__restrict__ dst,
                                      const double *__restrict__ cx, const double *__restrict__ cy,
                                      const double *__restrict__ cz, const double *__restrict__ cw,
                                      double *__restrict__ x, double *__restrict__ y, double *__restrict__ z,
                                      double *__restrict__ w) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && keep[i]) {
        int d = dst[i];
        x[d] = cx[i];
        y[d] = cy[i];
        z[d] = cz[i];
        w[d] = cw[i];
    }
}

// Exclusive prefix sum of keep in three passes over tiles of kScanTile entries: tile sums, a scan of the tile sums in
// one work-group, then each tile's own scan offset by its tile's prefix.
constexpr int kScanTile = 1024;

__device__ __forceinline__ int block_exclusive_scan_256(int v, int *sh, int *total) {
    // Work-group of 256: inclusive wave scans, then the four wave totals.
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    int x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) sh[wv] = x;
    __syncthreads();
    int base = 0;
    for (int k = 0; k < wv; k++) base += sh[k];
    if (total) *total = sh[0] + sh[1] + sh[2] + sh[3];
    __syncthreads();
    return base + x - v;
}

__global__ void __launch_bounds__(256) scan_tile_sums_kernel(int n, const int *__restrict__ in, int *__restrict__ sums) {
    __shared__ int sh[4];
    const int base = blockIdx.x * kScanTile + 4 * threadIdx.x;
    int v = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) v += base + k < n ? in[base + k] : 0;
    int total = 0;
    (void)block_exclusive_scan_256(v, sh, &total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

__global__ void __launch_bounds__(256) scan_sums_kernel(int nTiles, int *__restrict__ sums, int *__restrict__ total) {
    __shared__ int sh[4];
    int run = 0;
    for (int base = 0; base < nTiles; base += 256) {
        const int i = base + threadIdx.x;
        const int v = i < nTiles ? sums[i] : 0;
        int chunk = 0;
        const int ex = block_exclusive_scan_256(v, sh, &chunk);
        if (i < nTiles) sums[i] = run + ex;
        run += chunk;
    }
    if (threadIdx.x == 0) *total = run;
}

__global__ void __launch_bounds__(256) scan_apply_kernel(int n, const int *__restrict__ in, const int *__restrict__ sums,
                                                         int *__restrict__ out) {
    __shared__ int sh[4];
    const int base = blockIdx.x * kScanTile + 4 * threadIdx.x;
    int e[4], v = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) { e[k] = base + k < n ? in[base + k] : 0; v += e[k]; }
    int run = sums[blockIdx.x] + block_exclusive_scan_256(v, sh, nullptr);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if (base + k < n) out[base + k] = run;
        run += e[k];
    }
}

// start[a] = kept points before atom a's first candidate (a <= nAtoms).
__global__ void __launch_bounds__(256) atom_starts_kernel(int nAtoms, int nCand, const int *__restrict__ atomFirst,
                                                          const int *__restrict__ dst, const int *__restrict__ total,
                                                          int *__restrict__ start) {
    const int a = blockIdx.x * 256 + threadIdx.x;
    if (a <= nAtoms) start[a] = atomFirst[a] < nCand ? dst[atomFirst[a]] : *total;
}

// Becke pair data (DFTGridWeights.c:43-80): pairs[i][j] = {1 / R_ij, a_ij}, a_ij the size adjustment (a_ji = -a_ij).
std::vector<double2> becke_pairs(const xq_grid *g) {
    const size_t nA = static_cast<size_t>(g->nAtoms);
    std::vector<double2> pairs(nA * nA, make_double2(0.0, 0.0));
    for (size_t i = 0; i < nA; i++)
        for (size_t j = 0; j < i; j++) {
            const double dx = g->xyz[3 * i] - g->xyz[3 * j], dy = g->xyz[3 * i + 1] - g->xyz[3 * j + 1],
                         dz = g->xyz[3 * i + 2] - g->xyz[3 * j + 2];
            const double chi = bragg_radius(g->Z[i]) / bragg_radius(g->Z[j]);
            const double u = (chi - 1.0) / (chi + 1.0), a = u / (u * u - 1.0);
            const double invR = 1.0 / std::sqrt(dx * dx + dy * dy + dz * dz), adj = a > 0.5 ? 0.5 : (a < -0.5 ? -0.5 : a);
            pairs[i * nA + j] = make_double2(invR, adj);
            pairs[j * nA + i] = make_double2(invR, -adj);
        }
    return pairs;
}

// Largest number of atoms per lane of the weight-derivative kernel: 64 x 16 = 1024 atoms (more atoms per lane spill
// registers).
constexpr int kMaxLaneAtoms = 16;

// The cell function's small side: s = kBeckeA * integral of (1 - x^2)^10 from n to 1 for n = |nu|.  With y = 1 - n that is
// kBeckeA y^11 sum_j e_j n^j, e_j = binom(10, j) * integral of t^(10 + j) (2 - t)^(10 - j) from 0 to 1: every e_j is
// positive, so the form keeps its relative accuracy down to the smallest factors.
__device__ __forceinline__ double becke_small(double n, double y) {
    constexpr double e[11] = {0.27026018357287707, 1.9728620193016477, 6.8371721158098868, 14.627745835176176,
                                21.197110423116616, 21.591331269349844, 15.57688338493292, 7.829573934837093,
                                2.6165413533834587, 0.52380952380952384, 0.047619047619047616};
    double p = e[10];
#pragma unroll
    for (int j = 9; j >= 0; j--) p = fma(p, n, e[j]);
    const double y2 = y * y, y4 = y2 * y2;
    return kBeckeA * p * (y4 * y4 * y2 * y);
}

// 1 / x for normal x: the hardware's estimate with two Newton steps.
__device__ __forceinline__ double reciprocal(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
}

// XC gradient weight terms (DFTGridWeights_Derivatives, DFTGridWeights.c:98-215).  A group of GS lanes takes a point (grid
// atom g, weight w, energy density eXC = eps rho); lane l owns atoms l, l + GS, ... (at most LA of them) and accumulates
// their gradient in registers.  With A_i = prod_j s_ij and S = sum_i A_i the point's term is
//     eXC dw = sum_m c_m d ln A_m,   c_m = eXC w (delta_mg - A_m / S)   (w of the exact A_g),
// and every pair of atoms m, k enters it as D dmu_mk with D = g (c_k / s_km - c_m / s_mk), g = -ds_mk / dmu_mk (the same for
// both orders), mu_mk = (r_m - r_k) / R_mk.
//   Products.  Row c evaluates the factors of atom c with every lane atom: s_ci for A_c and s_ic, which multiplies lane
//   atom i's bound b_i >= A_i.  Rows are taken for g, then always for the atom of the largest bound, until no bound passes
//   the screen at the largest product found: the atoms that matter at the point, and about one row more.
//   Derivatives.  For each m whose c_m passes the screen, one row of pair terms: a pair of two such atoms is met from both
//   sides and gives each side's own atom its force; a pair with another atom k (c_k = 0) gives both forces at once.
//   The point moves with g, and its force is what makes the sum of a point's forces vanish.
// Bound by FP64 arithmetic (about 35 operations a factor, 70 a pair term, 4,300 instructions a point of (H2O)64: the vector
// units are busy for nine tenths of the time); a row's pairs are fetched while the row before is reduced.  Groups of 16
// and 32 lanes keep small molecules' lanes busy.  pairs[m][k] = {1 / R_mk, a_mk} (square, so that a row is read in order;
// a_km = -a_mk).  LDS: the coordinates, and per group each atom's distance and c.
// Against one point a wave with bounds from the 24 atoms nearest g and a screen on products without their smallest factor
// (which kept several times the atoms): (H2O)64, 2.4 million points, 102 -> 19 ms; (H2O)5, four points a wave, 2.5 -> 0.19 ms.
template <int LA, int GS, int WPG>
__global__ void __launch_bounds__(64 * WPG) weight_gradient_kernel(int nPoints,
                                                              const double *__restrict__ px, const double *__restrict__ py,
                                                              const double *__restrict__ pz, const double *__restrict__ pw,
                                                              const int *__restrict__ pointAtom,
                                                              const double *__restrict__ eXC, const double *__restrict__ xyz,
                                                              int nAtoms, const double2 *__restrict__ pairs,
                                                              double *__restrict__ grad) {
    static_assert(LA == 1 || GS == 64, "smaller groups hold one atom per lane");
    constexpr int kGroups = 64 * WPG / GS;
    extern __shared__ double lds[];
    const int t = threadIdx.x, gl = t & (GS - 1), gi = t / GS;
    double *sxyz = lds, *rL = lds + static_cast<size_t>(3 + 2 * gi) * nAtoms, *cL = rL + nAtoms;
    for (int i = t; i < 3 * nAtoms; i += 64 * WPG) sxyz[i] = xyz[i];
    __syncthreads();
    double G[LA][3];
#pragma unroll
    for (int a = 0; a < LA; a++) G[a][0] = G[a][1] = G[a][2] = 0.0;
    const int bit0 = t & 63 & ~(GS - 1);   // the group's place in its wave
    // Work-group b takes the rounds b, b + gridDim.x, ... of kGroups consecutive points (a point's cost depends on the atoms
    // whose cells matter there, so contiguous ranges would differ in cost).
    for (int base = blockIdx.x * kGroups; base < nPoints; base += gridDim.x * kGroups) {
        const int p = base + gi;
        const double e = p < nPoints ? eXC[p] : 0.0;
        const bool active = e != 0.0;
        if (!__any(active)) continue;
        const double rx = active ? px[p] : 0.0, ry = active ? py[p] : 0.0, rz = active ? pz[p] : 0.0;
        const int g = active ? pointAtom[p] : 0;
        double r[LA], b[LA], A[LA];
        bool done[LA];
        wave_fence();
#pragma unroll
        for (int a = 0; a < LA; a++) {
            const int i = gl + GS * a;
            r[a] = 0.0;
            if (i < nAtoms) {
                const double dx = sxyz[3 * i] - rx, dy = sxyz[3 * i + 1] - ry, dz = sxyz[3 * i + 2] - rz;
                r[a] = sqrt(dx * dx + dy * dy + dz * dz);
                rL[i] = r[a];
            }
            b[a] = 1.0;
            A[a] = 0.0;
            done[a] = i >= nAtoms;
        }
        wave_fence();
        PairRow<LA, GS> row;
        row.load(pairs, g, gl, nAtoms);
        // A_g from the cell factors as the weight w was made from them (candidate_points_kernel): deep in another atom's cell
        // they are rounding, and w with them.
        double made = 1.0, rc = rL[g];
#pragma unroll
        for (int a = 0; a < LA; a++) {
            const int i = gl + GS * a;
            if (i >= nAtoms || i == g) continue;
            const double2 q = row[a];
            const double mu = (rc - r[a]) * q.x;
            made *= 0.5 - kBeckeA * becke_poly(mu + q.y * (1.0 - mu * mu));
        }
        made = group_product<GS>(made);
        // Products.
        bool run = active;
        int c = g;
        double most = 0.0;
        do {
            double prod = 1.0;
#pragma unroll
            for (int a = 0; a < LA; a++) {
                const int i = gl + GS * a;
                if (i >= nAtoms || i == c) continue;
                const double2 q = row[a];
                const double mu = (rc - r[a]) * q.x, nu = fma(q.y, fma(-mu, mu, 1.0), mu), n = fabs(nu);
                const double small = becke_small(n, fmax(1.0 - n, 0.0)), large = 1.0 - small;
                prod *= nu > 0.0 ? small : large;
                b[a] *= nu > 0.0 ? large : small;
            }
            const int taken = c;
#pragma unroll
            for (int a = 0; a < LA; a++) done[a] = done[a] || gl + GS * a == taken;
            double top;
            c = next_atom<LA, GS>(b, done, gl, bit0, top);
            rc = rL[c];
            row.load(pairs, c, gl, nAtoms);
            prod = group_product<GS>(prod);
            if (run) {
                most = fmax(most, prod);
#pragma unroll
                for (int a = 0; a < LA; a++)
                    if (gl + GS * a == taken) A[a] = prod;
                run = top >= kCellScreen * most && top > 0.0;
            }
        } while (__any(run));
        // c_m; that of g from the others' share, which keeps its accuracy where g's cell holds almost all.
        double others = 0.0, own = 0.0;
#pragma unroll
        for (int a = 0; a < LA; a++) {
            if (gl + GS * a == g) own = A[a];
            else others += A[a];
        }
        others = group_sum<GS>(others);
        own = group_sum<GS>(own);
        const double ew = active ? e * pw[p] * (own / made) : 0.0, scale = active ? ew / (own + others) : 0.0;
        double cf[LA];
        unsigned long long maskK[LA], anyK = 0ull;
#pragma unroll
        for (int a = 0; a < LA; a++) {
            const int i = gl + GS * a;
            cf[a] = i == g ? scale * others : -scale * A[a];
            if (!(fabs(cf[a]) >= kCellScreen * fabs(ew)) || !active) cf[a] = 0.0;
            if (i < nAtoms) cL[i] = cf[a];
            maskK[a] = group_ballot<GS>(cf[a] != 0.0, bit0);
            anyK |= maskK[a];
        }
        if (!__any(anyK != 0ull)) continue;
        wave_fence();
        // Derivatives.  ir: 1 / distance of the lane's atoms.
        double ir[LA], gs[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int a = 0; a < LA; a++) ir[a] = gl + GS * a < nAtoms ? reciprocal(r[a]) : 0.0;
        // The next atom m of a group, -1 after the last.
        auto take = [&]() {
            int m = -1;
#pragma unroll
            for (int a = 0; a < LA; a++)
                if (m < 0 && maskK[a] != 0ull) {
                    m = GS * a + __ffsll(static_cast<long long>(maskK[a])) - 1;
                    maskK[a] &= maskK[a] - 1ull;
                }
            return m;
        };
        int next = take();
        row.load(pairs, next < 0 ? 0 : next, gl, nAtoms);
        while (__any(next >= 0)) {
            const bool some = next >= 0;
            const int m = some ? next : 0;
            const double xm = sxyz[3 * m], ym = sxyz[3 * m + 1], zm = sxyz[3 * m + 2], rm = rL[m];
            const double cm = some ? cL[m] : 0.0, irm = reciprocal(rm);
            const double ex = (xm - rx) * irm, ey = (ym - ry) * irm, ez = (zm - rz) * irm;
            double h[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int a = 0; a < LA; a++) {
                const int k = gl + GS * a;
                if (k >= nAtoms || k == m || !some) continue;
                const double2 q = row[a];
                const double mu = (rm - r[a]) * q.x, nu = fma(q.y, fma(-mu, mu, 1.0), mu), n = fabs(nu);
                const double y = fmax(1.0 - n, 0.0), small = becke_small(n, y), large = 1.0 - small;
                const double smk = nu > 0.0 ? small : large, skm = nu > 0.0 ? large : small;
                // 1 - nu^2 = y (2 - y); dnu / dmu = 1 - 2 a mu.
                const double u = y * (2.0 - y), u2 = u * u, u4 = u2 * u2;
                const double d = kBeckeA * (u4 * u4 * u2) * fma(-2.0 * q.y, mu, 1.0) * (cf[a] * smk - cm * skm) *
                                 reciprocal(fmax(small * large, 0x1p-1000));
                // d mu_mk / d r_k = -e_k / R - mu (r_k - r_m) / R^2, d mu_mk / d r_m = e_m / R + mu (r_k - r_m) / R^2.
                const double al = d * q.x, be = al * q.x * mu, ak = al * ir[a];
                const double xk = sxyz[3 * k], yk = sxyz[3 * k + 1], zk = sxyz[3 * k + 2];
                const double bx = be * (xk - xm), by = be * (yk - ym), bz = be * (zk - zm);
                const double fx = -fma(ak, xk - rx, bx), fy = -fma(ak, yk - ry, by), fz = -fma(ak, zk - rz, bz);
                G[a][0] += fx;
                G[a][1] += fy;
                G[a][2] += fz;
                gs[0] += fx;
                gs[1] += fy;
                gs[2] += fz;
                if (cf[a] == 0.0) {
                    h[0] += fma(al, ex, bx);
                    h[1] += fma(al, ey, by);
                    h[2] += fma(al, ez, bz);
                }
            }
            next = take();
            row.load(pairs, next < 0 ? 0 : next, gl, nAtoms);
#pragma unroll
            for (int x = 0; x < 3; x++) h[x] = group_sum<GS>(h[x]);
            if (some && gl == (m & (GS - 1))) {
#pragma unroll
                for (int a = 0; a < LA; a++)
                    if (a == m / GS) { G[a][0] += h[0]; G[a][1] += h[1]; G[a][2] += h[2]; }
                gs[0] += h[0];
                gs[1] += h[1];
                gs[2] += h[2];
            }
        }
#pragma unroll
        for (int x = 0; x < 3; x++) gs[x] = group_sum<GS>(gs[x]);
#pragma unroll
        for (int a = 0; a < LA; a++)
            if (active && gl + GS * a == g) { G[a][0] -= gs[0]; G[a][1] -= gs[1]; G[a][2] -= gs[2]; }
    }
    // The work-group's groups summed in LDS (the coordinates' place), then one addition per atom and component.
    __syncthreads();
    for (int i = t; i < 3 * nAtoms; i += 64 * WPG) sxyz[i] = 0.0;
    __syncthreads();
#pragma unroll
    for (int a = 0; a < LA; a++) {
        const int k = gl + GS * a;
        if (k < nAtoms)
#pragma unroll
            for (int x = 0; x < 3; x++) atomicAdd(&sxyz[3 * k + x], G[a][x]);
    }
    __syncthreads();
    for (int i = t; i < 3 * nAtoms; i += 64 * WPG) atomicAdd(&grad[i], sxyz[i]);
}

}  // namespace

int build_grid(xq_grid *g) {
    const int nA = g->nAtoms;
    g->bfTol = kBFTol[g->accuracy];
    g->rhoTol = kRhoTol[g->accuracy];
    // Lebedev rules used by this grid, expanded once.
    std::vector<int> ruleFirst(XQ_LEBEDEV_NRULES, -1);
    std::vector<double> rules;
    auto rule_of = [&](int l) -> int {
        int n = lebedev_size_for_l(l), k = 0;
        while (k < XQ_LEBEDEV_NRULES && xq_lebedev_npoints[k] != n) k++;
        if (ruleFirst[k] < 0) {
            ruleFirst[k] = static_cast<int>(rules.size() / 4);
            rules.resize(rules.size() + 4 * static_cast<size_t>(n));
            lebedev_expand(k, rules.data() + 4 * static_cast<size_t>(ruleFirst[k]));
        }
        return k;
    };
    // Radial shells, per atom in order (DFTGrid.c:138-211).
    std::vector<RadialShell> shells;
    std::vector<int> atomFirst(nA + 1, 0);
    int nCand = 0;
    for (int a = 0; a < nA; a++) {
        int nR, lMax;
        double rMax;
        atom_parameters(g->accuracy, g->Z[a], &nR, &lMax, &rMax);
        const int nAngMax = lebedev_size_for_l(lMax), nAngMin = lebedev_size_for_l(kMinL);
        const double range = bragg_radius(g->Z[a]), rCut = kRadialCutFactor * range;
        const double d = 1.0 + static_cast<double>(nR);
        atomFirst[a] = nCand;
        for (int i = 0; i < nR; i++) {
            const double x = static_cast<double>(i + 1) / d;
            const double r = range * std::pow(x / (1.0 - x), 2.0);
            const double wr = 2.0 * std::pow(range, 3.0) * std::pow(x, 5.0) / std::pow(1.0 - x, 7.0) / d;
            if (r > rMax) break;
            int l;
            if (r > rCut) l = lMax;
            else {
                int n = static_cast<int>(std::ceil(static_cast<double>(nAngMax) * r / rCut));
                l = n < nAngMin ? kMinL : lebedev_l_for_size(n);
            }
            const int k = rule_of(l);
            RadialShell s;
            s.atom = a;
            s.rule = ruleFirst[k];
            s.nAng = xq_lebedev_npoints[k];
            s.out = nCand;
            s.r = r;
            s.wr = 4.0 * M_PI * wr;
            shells.push_back(s);
            nCand += s.nAng;
        }
    }
    atomFirst[nA] = nCand;
    const std::vector<double2> pairs = becke_pairs(g);
    // Device work.
    RadialShell *d_shells = nullptr;
    double *d_rules = nullptr, *d_xyz = nullptr;
    double2 *d_pairs = nullptr;
    double *cx = nullptr, *cy = nullptr, *cz = nullptr, *cw = nullptr;
    int *keep = nullptr, *dst = nullptr, *total = nullptr, *tileSums = nullptr, *d_atomFirst = nullptr, *d_atomStart = nullptr;
    // Waves per work-group of the candidate kernel: four up to 640 atoms, two above (the coordinates and 8 bytes of LDS per
    // atom and group: 7 x 8 x 640 and 5 x 8 x 1489 bytes both fit in 64 KB).  Up to 16 atoms four points share a wave, up to
    // 32 two.
    const int wpg = nA <= 640 ? 4 : 2, group = nA <= 16 ? 16 : (nA <= 32 ? 32 : 64);
    const size_t lds = (3 + static_cast<size_t>(64 * wpg / group)) * sizeof(double) * static_cast<size_t>(nA);
    if (nA > 1489) {
        set_error("grid construction supports at most 1489 atoms");
        return kInvalidArgument;
    }
    int status = kOK;
    auto cleanup = [&]() {
        // The kernels that use these arrays must be done before the arrays are reused.
        (void)hipStreamSynchronize(g->stream);
        dev_free(g, &d_shells); dev_free(g, &d_rules); dev_free(g, &d_xyz); dev_free(g, &d_pairs);
        dev_free(g, &d_atomFirst); dev_free(g, &d_atomStart);
        dev_free(g, &cx); dev_free(g, &cy); dev_free(g, &cz); dev_free(g, &cw); dev_free(g, &keep); dev_free(g, &dst); dev_free(g, &total);
        dev_free(g, &tileSums);
    };
    do {
        if ((status = dev_alloc(g, &d_shells, shells.size())) != kOK) break;
        if ((status = dev_alloc(g, &d_rules, rules.size())) != kOK) break;
        if ((status = dev_alloc(g, &d_xyz, g->xyz.size())) != kOK) break;
        if ((status = dev_alloc(g, &d_pairs, pairs.size())) != kOK) break;
        if ((status = dev_alloc(g, &d_atomFirst, atomFirst.size())) != kOK) break;
        if ((status = dev_alloc(g, &d_atomStart, atomFirst.size())) != kOK) break;
        if ((status = dev_alloc(g, &cx, nCand)) != kOK) break;
        if ((status = dev_alloc(g, &cy, nCand)) != kOK) break;
        if ((status = dev_alloc(g, &cz, nCand)) != kOK) break;
        if ((status = dev_alloc(g, &cw, nCand)) != kOK) break;
        if ((status = dev_alloc(g, &keep, nCand)) != kOK) break;
        if ((status = dev_alloc(g, &dst, nCand)) != kOK) break;
        if ((status = dev_alloc(g, &total, 1)) != kOK) break;
        if ((status = dev_alloc(g, &tileSums, static_cast<size_t>((nCand + kScanTile - 1) / kScanTile))) != kOK) break;
        hipStream_t s = g->stream;
        if ((status = check(hipMemcpyAsync(d_shells, shells.data(), shells.size() * sizeof(RadialShell),
                                           hipMemcpyHostToDevice, s), "copy shells")) != kOK) break;
        if ((status = check(hipMemcpyAsync(d_rules, rules.data(), rules.size() * sizeof(double), hipMemcpyHostToDevice, s),
                            "copy rules")) != kOK) break;
        if ((status = check(hipMemcpyAsync(d_xyz, g->xyz.data(), g->xyz.size() * sizeof(double), hipMemcpyHostToDevice, s),
                            "copy xyz")) != kOK) break;
        if ((status = check(hipMemcpyAsync(d_pairs, pairs.data(), pairs.size() * sizeof(double2), hipMemcpyHostToDevice, s),
                            "copy pairs")) != kOK) break;
        if ((status = check(hipMemcpyAsync(d_atomFirst, atomFirst.data(), atomFirst.size() * sizeof(int),
                                           hipMemcpyHostToDevice, s), "copy atoms")) != kOK) break;
        if (!shells.empty()) {
            // A shell's points go to several work-groups (at most one per round of points), some 32768 in all: their costs
            // differ, and with 2048 the chip stood idle for a third of the kernel ((H2O)24: 4.0 ms against 2.7).
            const unsigned rounds = static_cast<unsigned>((lebedev_size_for_l(65) * group + 64 * wpg - 1) / (64 * wpg));
            const unsigned split = std::min<unsigned>(rounds, static_cast<unsigned>(32768 / shells.size()) + 1);
            auto launch = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(shells.size()), split), dim3(64 * wpg), lds, s,
                                   d_shells, d_rules, d_xyz, nA, d_pairs, cx, cy, cz, cw, keep);
            };
            // Atoms per lane: the smallest instance that covers nAtoms.
            if (nA <= 16) launch(candidate_points_kernel<1, 16, 4>);
            else if (nA <= 32) launch(candidate_points_kernel<1, 32, 4>);
            else if (nA <= 64) launch(candidate_points_kernel<1, 64, 4>);
            else if (nA <= 128) launch(candidate_points_kernel<2, 64, 4>);
            else if (nA <= 192) launch(candidate_points_kernel<3, 64, 4>);
            else if (nA <= 256) launch(candidate_points_kernel<4, 64, 4>);
            else if (nA <= 384) launch(candidate_points_kernel<6, 64, 4>);
            else if (nA <= 640) launch(candidate_points_kernel<10, 64, 4>);
            else if (nA <= 1024) launch(candidate_points_kernel<16, 64, 2>);
            else launch(candidate_points_kernel<24, 64, 2>);
            if ((status = check(hipGetLastError(), "candidate_points_kernel")) != kOK) break;
            const int nTiles = (nCand + kScanTile - 1) / kScanTile;
            hipLaunchKernelGGL(scan_tile_sums_kernel, dim3(nTiles), dim3(256), 0, s, nCand, keep, tileSums);
            hipLaunchKernelGGL(scan_sums_kernel, dim3(1), dim3(256), 0, s, nTiles, tileSums, total);
            hipLaunchKernelGGL(scan_apply_kernel, dim3(nTiles), dim3(256), 0, s, nCand, keep, tileSums, dst);
            // Each atom's first kept point: the scan at the atom boundaries (the end's is the total).
            hipLaunchKernelGGL(atom_starts_kernel, dim3((nA + 256) / 256), dim3(256), 0, s, nA, nCand, d_atomFirst, dst, total,
                               d_atomStart);
            if ((status = check(hipGetLastError(), "scan kernels")) != kOK) break;
        }
        std::vector<int> atomStart(static_cast<size_t>(nA) + 1, 0);
        if (nCand > 0) {
            // Wait for the kernels first: a pageable copy that waits for its stream holds the runtime's staging path.
            if ((status = check(hipStreamSynchronize(s), "grid sync")) != kOK) break;
            if ((status = check(hipMemcpyAsync(atomStart.data(), d_atomStart, atomStart.size() * sizeof(int),
                                               hipMemcpyDeviceToHost, s), "copy scan")) != kOK) break;
            if ((status = check(hipStreamSynchronize(s), "grid sync")) != kOK) break;
        }
        const int nKept = atomStart[nA];
        g->nPoints = nKept;
        if ((status = dev_alloc(g, &g->d_x, nKept)) != kOK) break;
        if ((status = dev_alloc(g, &g->d_y, nKept)) != kOK) break;
        if ((status = dev_alloc(g, &g->d_z, nKept)) != kOK) break;
        if ((status = dev_alloc(g, &g->d_w, nKept)) != kOK) break;
        if (nCand > 0) {
            hipLaunchKernelGGL(compact_points_kernel, dim3((nCand + 255) / 256), dim3(256), 0, s, nCand, keep, dst, cx, cy,
                               cz, cw, g->d_x, g->d_y, g->d_z, g->d_w);
            if ((status = check(hipGetLastError(), "compact_points_kernel")) != kOK) break;
        }
        // Blocks of at most kBlockSize consecutive points per atom.
        g->blocks.clear();
        for (int a = 0; a < nA; a++) {
            const int p0 = atomStart[a], p1 = atomStart[a + 1];
            for (int p = p0; p < p1; p += kBlockSize) {
                DevBlock b;
                b.atom = a;
                b.pStart = p;
                b.nPoints = (p1 - p) < kBlockSize ? (p1 - p) : kBlockSize;
                b.nKept = 0;
                b.vOffset = 0;
                b.iOffset = 0;
                b.pad = 0;
                g->blocks.push_back(b);
            }
        }
        g->nBlocks = static_cast<int>(g->blocks.size());
        if ((status = dev_alloc(g, &g->d_blocks, g->blocks.size())) != kOK) break;
        if (!g->blocks.empty() &&
            (status = check(hipMemcpyAsync(g->d_blocks, g->blocks.data(), g->blocks.size() * sizeof(DevBlock),
                                           hipMemcpyHostToDevice, s), "copy blocks")) != kOK) break;
        status = check(hipStreamSynchronize(s), "grid sync");
    } while (false);
    cleanup();   // only the kept points and the block table stay resident (and counted on the handle)
    return status;
}

// Estimated point count without the cull (DFTGrid_EstimatedPoints, DFTGrid.c:301-356).
long long estimated_points(int accuracy, int nAtoms, const int *Z) {
    long long p = 0;
    for (int a = 0; a < nAtoms; a++) {
        int nR, lMax;
        double rMax;
        atom_parameters(accuracy, Z[a], &nR, &lMax, &rMax);
        const int nAngMax = lebedev_size_for_l(lMax), nAngMin = lebedev_size_for_l(kMinL);
        const double range = bragg_radius(Z[a]), rCut = kRadialCutFactor * range, d = 1.0 + nR;
        for (int i = 0; i < nR; i++) {
            const double x = static_cast<double>(i + 1) / d;
            const double r = range * std::pow(x / (1.0 - x), 2.0);
            if (r > rMax) break;
            int l;
            if (r > rCut) l = lMax;
            else {
                int n = static_cast<int>(std::ceil(static_cast<double>(nAngMax) * r / rCut));
                l = n < nAngMin ? kMinL : lebedev_l_for_size(n);
            }
            p += lebedev_size_for_l(l);
        }
    }
    return p;
}


// XC gradient weight terms of every point with a non-zero energy density eXC (device arrays; grad is incremented).
int weight_gradients(xq_grid *g, const double *d_eXC, double *d_grad, hipStream_t s) {
    const int nA = g->nAtoms, G = g->nPoints;
    if (G <= 0 || nA < 2) return kOK;
    // Waves per work-group: four up to 640 atoms, two above (the coordinates and 16 bytes of LDS per atom and wave: 11 x 8 x
    // 640 and 7 x 8 x 1024 bytes both fit in 64 KB).  Up to 16 atoms four points share a wave, up to 32 two.
    const int wpg = nA <= 640 ? 4 : 2, group = nA <= 16 ? 16 : (nA <= 32 ? 32 : 64);
    const size_t lds = (3 + 2 * static_cast<size_t>(64 * wpg / group)) * sizeof(double) * static_cast<size_t>(nA);
    if (nA > 64 * kMaxLaneAtoms || lds > 64 * 1024) {
        set_error("XC gradients support at most " + std::to_string(64 * kMaxLaneAtoms) + " atoms");
        return kInvalidArgument;
    }
    const std::vector<double2> pairs = becke_pairs(g);
    std::vector<int> pointAtom(static_cast<size_t>(G), 0);
    for (const DevBlock &b : g->blocks)
        for (int k = 0; k < b.nPoints; k++) pointAtom[static_cast<size_t>(b.pStart) + k] = b.atom;
    double2 *d_pairs = nullptr;
    double *d_xyz = nullptr;
    int *d_pointAtom = nullptr;
    int status = kOK;
    do {
        if ((status = dev_alloc(g, &d_pairs, pairs.size())) != kOK) break;
        if ((status = dev_alloc(g, &d_xyz, g->xyz.size())) != kOK) break;
        if ((status = dev_alloc(g, &d_pointAtom, pointAtom.size())) != kOK) break;
        if ((status = check(hipMemcpyAsync(d_pairs, pairs.data(), pairs.size() * sizeof(double2), hipMemcpyHostToDevice, s),
                            "copy pairs")) != kOK) break;
        if ((status = check(hipMemcpyAsync(d_xyz, g->xyz.data(), g->xyz.size() * sizeof(double), hipMemcpyHostToDevice, s),
                            "copy xyz")) != kOK) break;
        if ((status = check(hipMemcpyAsync(d_pointAtom, pointAtom.data(), pointAtom.size() * sizeof(int),
                                           hipMemcpyHostToDevice, s), "copy point atoms")) != kOK) break;
        // Enough work-groups to even their costs out ((H2O)64: 19.9 ms with 2048, 18.9 with 8192).
        const int nGroups = std::min(8192 * 4 / wpg, (G + 63) / 64);
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(nGroups), dim3(64 * wpg), lds, s, G, g->d_x, g->d_y, g->d_z,
                               g->d_w, d_pointAtom, d_eXC, d_xyz, nA, d_pairs, d_grad);
        };
        // Atoms per lane: the smallest instance that covers nAtoms (fewer registers for small systems).
        if (nA <= 16) launch(weight_gradient_kernel<1, 16, 4>);
        else if (nA <= 32) launch(weight_gradient_kernel<1, 32, 4>);
        else if (nA <= 64) launch(weight_gradient_kernel<1, 64, 4>);
        else if (nA <= 128) launch(weight_gradient_kernel<2, 64, 4>);
        else if (nA <= 192) launch(weight_gradient_kernel<3, 64, 4>);
        else if (nA <= 256) launch(weight_gradient_kernel<4, 64, 4>);
        else if (nA <= 384) launch(weight_gradient_kernel<6, 64, 4>);
        else if (nA <= 640) launch(weight_gradient_kernel<10, 64, 4>);
        else launch(weight_gradient_kernel<kMaxLaneAtoms, 64, 2>);
        if ((status = check(hipGetLastError(), "weight_gradient_kernel")) != kOK) break;
        status = check(hipStreamSynchronize(s), "gradient sync");
    } while (false);
    (void)hipStreamSynchronize(s);
    dev_free(g, &d_pairs);
    dev_free(g, &d_xyz);
    dev_free(g, &d_pointAtom);
    return status;
}

}  // namespace xq
