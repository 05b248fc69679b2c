// Gaussian basis set-up and block-wise basis values and gradients on the device.
//
// Host side: the element specification is turned into per-atom shells with unnormalised primitive coefficients and the
// Cartesian factors of GaussianBasis_UnnormalizePrimitives / _NormalizePrimitiveCCBF (pMolecule/QCModel/GaussianBases/
// __extensions__/csource/GaussianBasis.c:448-501, 728-751), and the Cartesian -> real solid harmonic transformation of
// Schlegel & Frisch (Int. J. Quantum Chem. 54 (1995) 83, eq. 15), with the reference's function order (GaussianBasis.c:13-27).
//
// Device side, once per geometry ("in core", DFTIntegrator.c:209-210,491):
//   1. count kernel, one work-group per grid block: bounding sphere of the block's points, a rigorous per-shell upper bound on
//      |phi| over the sphere (shells that cannot reach bfTol are skipped), exact values of the remaining functions, and the
//      reference's filter max_p |phi_m(p)| > bfTol (GridFunctionDataBlock.c:130-185) -> ascending kept-function list.
//   2. eval kernel, one work-group per block: values and gradients of the kept functions (GaussianBasisIntegrals_f1Op1.c:
//      100-197 and GaussianBasisTransform.c:85-125), stored function-major in rows of 128 points (coalesced stores).
// The kept sets are exactly the reference's: screening removes only functions whose bound is below the tolerance.
#include <cmath>
#include <cstring>
#include <type_traits>
#include <hip/hip_runtime.h>

#include "xq_internal.h"
#include "xq_c2s.h"

namespace xq {

namespace {

constexpr int kMaxShellsLDS = 16384;

// Cartesian powers in the reference order (for z = 0..l, for y = 0..l-z, x = l-y-z), for l = 0..3, concatenated.
__host__ __device__ constexpr int cart_offset(int l) { return l * (l + 1) * (l + 2) / 6; }
__host__ __device__ constexpr int ncart(int l) { return (l + 1) * (l + 2) / 2; }

struct CartPow {
    int x[20], y[20], z[20];
};
__host__ __device__ constexpr CartPow make_cart_pow() {
    CartPow p{};
    int n = 0;
    for (int l = 0; l <= 3; l++)
        for (int z = 0; z <= l; z++)
            for (int y = 0; y <= l - z; y++) {
                p.x[n] = l - y - z;
                p.y[n] = y;
                p.z[n] = z;
                n++;
            }
    return p;
}
constexpr CartPow kCart = make_cart_pow();

// ------------------------------------------------------------------------------------------------------------------------
// Device evaluation of one shell at one point.  Template over (lLow, lHigh, spherical) so that every array index is a
// compile-time constant and stays in registers.
// ------------------------------------------------------------------------------------------------------------------------
template <int LL, int LH>
struct ShellDims {
    static constexpr int nCBF = cart_offset(LH + 1) - cart_offset(LL);
    static constexpr int nSph = (LH + 1) * (LH + 1) - LL * LL;
};

// f(lLow, lHigh, spherical) as compile-time constants for the shell's type.
template <typename F>
__device__ __forceinline__ void for_shell_type(const xq::DevShell &sh, bool sph, F f) {
    using std::integral_constant;
    auto type = [&](auto ll, auto lh) {
        if (sph) f(ll, lh, std::true_type{});
        else f(ll, lh, std::false_type{});
    };
    switch (sh.lLow * 4 + sh.lHigh) {
        case 0: type(integral_constant<int, 0>{}, integral_constant<int, 0>{}); break;
        case 5: type(integral_constant<int, 1>{}, integral_constant<int, 1>{}); break;
        case 1: type(integral_constant<int, 0>{}, integral_constant<int, 1>{}); break;
        case 10: type(integral_constant<int, 2>{}, integral_constant<int, 2>{}); break;
        case 15: type(integral_constant<int, 3>{}, integral_constant<int, 3>{}); break;
        default: break;
    }
}

template <int LL, int LH, bool SPH, bool GRAD>
__device__ __forceinline__ void shell_eval(const xq::DevShell &sh, const double *__restrict__ coef,
                                           const double *__restrict__ trans, double dx, double dy, double dz, double *v,
                                           double *vx, double *vy, double *vz) {
    constexpr int NC = ShellDims<LL, LH>::nCBF;
    constexpr int NB = SPH ? ShellDims<LL, LH>::nSph : NC;
    constexpr int C0 = cart_offset(LL);
    const double r2 = dx * dx + dy * dy + dz * dz;
    double e0[NC], e1[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) { e0[c] = 0.0; e1[c] = 0.0; }
    const double *ex = coef + sh.coef, *cc = coef + sh.coef + sh.nPrim;
    for (int q = 0; q < sh.nPrim; q++) {
        const double a = ex[q], e = exp(-a * r2);
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const double k = cc[q * NC + c];
            e0[c] += k * e;
            e1[c] += k * a * e;
        }
    }
    double X0[LH + 2], Y0[LH + 2], Z0[LH + 2];
    X0[0] = Y0[0] = Z0[0] = 1.0;
#pragma unroll
    for (int i = 1; i <= LH + 1; i++) { X0[i] = dx * X0[i - 1]; Y0[i] = dy * Y0[i - 1]; Z0[i] = dz * Z0[i - 1]; }
    double g0[NC], gx[NC], gy[NC], gz[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int i = kCart.x[C0 + c], j = kCart.y[C0 + c], k = kCart.z[C0 + c];
        g0[c] = X0[i] * Y0[j] * Z0[k] * e0[c];
        if (GRAD) {
            const double E1 = -2.0 * e1[c];
            const double xi1 = i > 0 ? i * X0[i > 0 ? i - 1 : 0] : 0.0;
            const double yj1 = j > 0 ? j * Y0[j > 0 ? j - 1 : 0] : 0.0;
            const double zk1 = k > 0 ? k * Z0[k > 0 ? k - 1 : 0] : 0.0;
            gx[c] = (xi1 * e0[c] + X0[i + 1] * E1) * Y0[j] * Z0[k];
            gy[c] = (yj1 * e0[c] + Y0[j + 1] * E1) * X0[i] * Z0[k];
            gz[c] = (zk1 * e0[c] + Z0[k + 1] * E1) * X0[i] * Y0[j];
        }
    }
    if (SPH) {
        const double *T = trans + sh.trans;
#pragma unroll
        for (int s = 0; s < NB; s++) {
            double a = 0.0, bx = 0.0, by = 0.0, bz = 0.0;
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const double t = T[c * NB + s];
                a += t * g0[c];
                if (GRAD) { bx += t * gx[c]; by += t * gy[c]; bz += t * gz[c]; }
            }
            v[s] = a;
            if (GRAD) { vx[s] = bx; vy[s] = by; vz[s] = bz; }
        }
    } else {
#pragma unroll
        for (int s = 0; s < NB; s++) {
            v[s] = g0[s];
            if (GRAD) { vx[s] = gx[s]; vy[s] = gy[s]; vz[s] = gz[s]; }
        }
    }
}

// Dispatch on the shell type; calls body(N, v, vx, vy, vz), N the shell's functions as a compile-time constant (so that the
// arrays stay in registers).  Supported: S, P, D, F, SP.
template <bool GRAD, typename Body>
__device__ __forceinline__ void with_shell(const xq::DevShell &sh, bool sph, const double *coef, const double *trans,
                                           double dx, double dy, double dz, Body body) {
    auto shell = [&](auto ll, auto lh, auto s) {
        constexpr int N = s ? ShellDims<ll, lh>::nSph : ShellDims<ll, lh>::nCBF;
        double v[N], vx[N], vy[N], vz[N];
        shell_eval<ll, lh, s, GRAD>(sh, coef, trans, dx, dy, dz, v, vx, vy, vz);
        body(std::integral_constant<int, N>{}, v, vx, vy, vz);
    };
    for_shell_type(sh, sph, shell);
}

__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Upper bound of max_{r >= d} r^L exp(-a r^2).
__device__ __forceinline__ double radial_bound(int L, double a, double d) {
    if (L == 0) return exp(-a * d * d);
    const double rs = sqrt(L / (2.0 * a)), r = d > rs ? d : rs;
    double p = 1.0;
    for (int i = 0; i < L; i++) p *= r;
    return p * exp(-a * r * r);
}

// Work-group of kBlockSize threads, one thread per point.  Writes the kept functions of block b to tmpIdx[b * nF ...] and
// their count to counts[b].  mask (dynamic LDS, two shells a word): per shell, bit 15 if its bound reaches bfTol on the
// block's sphere, bits 0 .. 9 its functions that pass bfTol at some point.  Each wave evaluates the candidate shells at its
// 64 points and marks the functions that pass there (one ballot each), and the marked functions are written in order after
// one barrier; a maximum over the work-group with two barriers per function took 0.61 ms on (H2O)24, this
// takes 0.30 ms.
__global__ void __launch_bounds__(kBlockSize) basis_count_kernel(
    int nBlocks, const xq::DevBlock *__restrict__ blocks, const double *__restrict__ px, const double *__restrict__ py,
    const double *__restrict__ pz, int nShells, const xq::DevShell *__restrict__ shells, const double *__restrict__ coef,
    const double *__restrict__ trans, int spherical, int nF, double bfTol, int *__restrict__ tmpIdx,
    int *__restrict__ counts) {
    extern __shared__ unsigned mask[];
    __shared__ double red[4][2];
    __shared__ int waveKept[2];
    const int b = blockIdx.x;
    const xq::DevBlock blk = blocks[b];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const bool valid = t < blk.nPoints;
    const double x = valid ? px[blk.pStart + t] : 0.0, y = valid ? py[blk.pStart + t] : 0.0,
                 z = valid ? pz[blk.pStart + t] : 0.0;
    // Bounding sphere: centroid and largest distance.
    double sx = wave_sum(x), sy = wave_sum(y), sz = wave_sum(z);
    if (lane == 0) { red[wave][0] = sx; red[wave][1] = sy; red[wave + 2][0] = sz; }
    for (int w = t; w < (nShells + 1) / 2; w += kBlockSize) mask[w] = 0u;
    __syncthreads();
    const double inv = 1.0 / blk.nPoints;
    const double cx = (red[0][0] + red[1][0]) * inv, cy = (red[0][1] + red[1][1]) * inv, cz = (red[2][0] + red[3][0]) * inv;
    __syncthreads();
    double rr = valid ? sqrt((x - cx) * (x - cx) + (y - cy) * (y - cy) + (z - cz) * (z - cz)) : 0.0;
    rr = wave_max(rr);
    if (lane == 0) red[wave][0] = rr;
    __syncthreads();
    const double radius = fmax(red[0][0], red[1][0]);
    // Candidate shells.
    for (int s = t; s < nShells; s += kBlockSize) {
        const xq::DevShell &sh = shells[s];
        const double dd = sqrt((sh.x - cx) * (sh.x - cx) + (sh.y - cy) * (sh.y - cy) + (sh.z - cz) * (sh.z - cz)) - radius;
        const double d = dd > 0.0 ? dd : 0.0;
        double bound = 0.0;
        const double *ex = coef + sh.coef;
        for (int q = 0; q < sh.nPrim; q++)
            for (int L = sh.lLow; L <= sh.lHigh; L++) bound += sh.bound[q] * radial_bound(L, ex[q], d);
        if (bound * (1.0 + 1.0e-12) > bfTol) atomicOr(&mask[s >> 1], 0x8000u << (16 * (s & 1)));
    }
    __syncthreads();
    auto bits = [&](int s) { return s < nShells ? (mask[s >> 1] >> (16 * (s & 1))) & 0xffffu : 0u; };
    for (int s0 = 0; s0 < nShells; s0 += 64)
        for (unsigned long long cand = __ballot((bits(s0 + lane) & 0x8000u) != 0u); cand != 0ull; cand &= cand - 1ull) {
            const int s = s0 + __ffsll(static_cast<long long>(cand)) - 1;
            const xq::DevShell &sh = shells[s];
            with_shell<false>(sh, spherical != 0, coef, trans, x - sh.x, y - sh.y, z - sh.z,
                              [&](auto n, const double *v, const double *, const double *, const double *) {
                                  unsigned pass = 0u;
#pragma unroll
                                  for (int k = 0; k < n; k++)
                                      if (__ballot(valid && fabs(v[k]) > bfTol) != 0ull) pass |= 1u << k;
                                  if (lane == 0 && pass != 0u) atomicOr(&mask[s >> 1], pass << (16 * (s & 1)));
                              });
        }
    __syncthreads();
    // Thread t lists the functions of the shells t * per .. + per - 1.
    const int per = (nShells + kBlockSize - 1) / kBlockSize, s1 = t * per;
    int kept = 0;
    for (int s = s1; s < s1 + per; s++) kept += __popc(bits(s) & 0x7fffu);
    int before = kept;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(before, o, 64);
        if (lane >= o) before += u;
    }
    if (lane == 63) waveKept[wave] = before;
    __syncthreads();
    int o = before - kept + (wave == 1 ? waveKept[0] : 0);
    int *out = tmpIdx + static_cast<size_t>(b) * nF;
    for (int s = s1; s < s1 + per; s++)
        for (unsigned m = bits(s) & 0x7fffu; m != 0u; m &= m - 1u) out[o++] = shells[s].fStart + __ffs(static_cast<int>(m)) - 1;
    if (t == 0) counts[b] = waveKept[0] + waveKept[1];
}

// Values and gradients of the kept functions of block b into rows [vOffset, vOffset + nKept) of f, fx, fy, fz (row stride
// kBlockSize; entries past the block's points are zero).  EB, EG (mixed precision, else null): per point, the powers of two
// above max |phi| and above max |d phi / dx_c| over the block's kept functions.
__global__ void __launch_bounds__(kBlockSize) basis_eval_kernel(
    const xq::DevBlock *__restrict__ blocks, const double *__restrict__ px, const double *__restrict__ py,
    const double *__restrict__ pz, const xq::DevShell *__restrict__ shells, const int *__restrict__ shellOf,
    const double *__restrict__ coef, const double *__restrict__ trans, int spherical, int nF,
    const int *__restrict__ tmpIdx, int *__restrict__ idx, double *__restrict__ f, double *__restrict__ fx,
    double *__restrict__ fy, double *__restrict__ fz, signed char *__restrict__ EB, signed char *__restrict__ EG) {
    const int b = blockIdx.x;
    const xq::DevBlock blk = blocks[b];
    const int t = threadIdx.x;
    const bool valid = t < blk.nPoints;
    const double x = valid ? px[blk.pStart + t] : 0.0, y = valid ? py[blk.pStart + t] : 0.0,
                 z = valid ? pz[blk.pStart + t] : 0.0;
    const int *kept = tmpIdx + static_cast<size_t>(b) * nF;
    for (int k = t; k < blk.nKept; k += blockDim.x) idx[blk.iOffset + k] = kept[k];
    double m[4] = {0.0, 0.0, 0.0, 0.0};
    int k = 0;
    while (k < blk.nKept) {
        const xq::DevShell &sh = shells[shellOf[kept[k]]];
        with_shell<true>(sh, spherical != 0, coef, trans, x - sh.x, y - sh.y, z - sh.z,
                         [&](auto n, const double *v, const double *vx, const double *vy, const double *vz) {
#pragma unroll
                             for (int j = 0; j < n; j++) {
                                 if (k < blk.nKept && kept[k] == sh.fStart + j) {
                                     const size_t o = static_cast<size_t>(blk.vOffset + k) * kBlockSize + t;
                                     f[o] = valid ? v[j] : 0.0;
                                     fx[o] = valid ? vx[j] : 0.0;
                                     fy[o] = valid ? vy[j] : 0.0;
                                     fz[o] = valid ? vz[j] : 0.0;
                                     m[0] = fmax(m[0], fabs(v[j]));
                                     m[1] = fmax(m[1], fabs(vx[j]));
                                     m[2] = fmax(m[2], fabs(vy[j]));
                                     m[3] = fmax(m[3], fabs(vz[j]));
                                     k++;
                                 }
                             }
                         });
    }
    if (EB != nullptr) {
        EB[static_cast<size_t>(b) * kBlockSize + t] = static_cast<signed char>(valid ? stored_exponent(m[0]) : 0);
        for (int c = 0; c < 3; c++)
            EG[(static_cast<size_t>(b) * 3 + c) * kBlockSize + t] =
                static_cast<signed char>(valid ? stored_exponent(m[c + 1]) : 0);
    }
}

// sum_r H_r A_r over a shell's functions r at one point, added to out: H_r the function's Hessian
// (GaussianBasisIntegrals_f1Op1.c:203-331), with e2 = 4 sum c a^2 e^{-a r^2}
//     d2/dx2 phi = (i(i-1) x^{i-2} e0 + (2i+1) x^i e1 + x^{i+2} e2) y^j z^k,
//     d2/dxdy phi = (i j x^{i-1} y^{j-1} e0 + (i x^{i-1} y^{j+1} + j x^{i+1} y^{j-1}) e1 + x^{i+1} y^{j+1} e2) z^k,
// and A_r a vector.  The vectors are transformed to the Cartesian functions (where the shell's functions are spherical), whose Hessians are then used one
// by one.
template <int LL, int LH, bool SPH>
__device__ __forceinline__ void shell_second(const xq::DevShell &sh, const double *__restrict__ coef,
                                             const double *__restrict__ trans, double dx, double dy, double dz,
                                             const double (&A)[3][SPH ? ShellDims<LL, LH>::nSph : ShellDims<LL, LH>::nCBF],
                                             double (&out)[3]) {
    constexpr int NC = ShellDims<LL, LH>::nCBF;
    constexpr int NB = SPH ? ShellDims<LL, LH>::nSph : NC;
    constexpr int C0 = cart_offset(LL);
    const double r2 = dx * dx + dy * dy + dz * dz;
    double e0[NC], e1[NC], e2[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) { e0[c] = 0.0; e1[c] = 0.0; e2[c] = 0.0; }
    const double *ex = coef + sh.coef, *cc = coef + sh.coef + sh.nPrim;
    for (int q = 0; q < sh.nPrim; q++) {
        const double a = ex[q], e = exp(-a * r2);
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const double k = cc[q * NC + c];
            e0[c] += k * e;
            e1[c] += k * a * e;
            e2[c] += k * (a * a) * e;
        }
    }
    double X0[LH + 3], Y0[LH + 3], Z0[LH + 3], X1[LH + 3], Y1[LH + 3], Z1[LH + 3], X2[LH + 3], Y2[LH + 3], Z2[LH + 3];
    X0[0] = Y0[0] = Z0[0] = 1.0;
    X1[0] = Y1[0] = Z1[0] = X2[0] = Y2[0] = Z2[0] = 0.0;
#pragma unroll
    for (int i = 1; i <= LH + 2; i++) {
        X0[i] = dx * X0[i - 1]; Y0[i] = dy * Y0[i - 1]; Z0[i] = dz * Z0[i - 1];
        X1[i] = i * X0[i - 1]; Y1[i] = i * Y0[i - 1]; Z1[i] = i * Z0[i - 1];
        X2[i] = i * X1[i - 1]; Y2[i] = i * Y1[i - 1]; Z2[i] = i * Z1[i - 1];
    }
#pragma unroll
    for (int c = 0; c < NC; c++) {
        double B[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            if (SPH) {
                const double *T = trans + sh.trans;
                B[d] = 0.0;
#pragma unroll
                for (int r = 0; r < NB; r++) B[d] += T[c * NB + r] * A[d][r];
            } else {
                B[d] = A[d][c];
            }
        }
        const int i = kCart.x[C0 + c], j = kCart.y[C0 + c], k = kCart.z[C0 + c];
        const double E0 = e0[c], E1 = -2.0 * e1[c], E2 = 4.0 * e2[c];
        const double xx = (X2[i] * E0 + (dx * X1[i] + X1[i + 1]) * E1 + X0[i + 2] * E2) * Y0[j] * Z0[k];
        const double xy = (X1[i] * Y1[j] * E0 + (X1[i] * Y0[j + 1] + X0[i + 1] * Y1[j]) * E1 + X0[i + 1] * Y0[j + 1] * E2) * Z0[k];
        const double xz = (X1[i] * Z1[k] * E0 + (X1[i] * Z0[k + 1] + X0[i + 1] * Z1[k]) * E1 + X0[i + 1] * Z0[k + 1] * E2) * Y0[j];
        const double yy = (Y2[j] * E0 + (dy * Y1[j] + Y1[j + 1]) * E1 + Y0[j + 2] * E2) * X0[i] * Z0[k];
        const double yz = (Y1[j] * Z1[k] * E0 + (Y1[j] * Z0[k + 1] + Y0[j + 1] * Z1[k]) * E1 + Y0[j + 1] * Z0[k + 1] * E2) * X0[i];
        const double zz = (Z2[k] * E0 + (dz * Z1[k] + Z1[k + 1]) * E1 + Z0[k + 2] * E2) * X0[i] * Y0[j];
        out[0] += xx * B[0] + xy * B[1] + xz * B[2];
        out[1] += xy * B[0] + yy * B[1] + yz * B[2];
        out[2] += xz * B[0] + yz * B[1] + zz * B[2];
    }
}

// The kept rows h nKept / S .. (h + 1) nKept / S - 1 of a block, S = gridDim.y and h = blockIdx.y.
__device__ __forceinline__ void row_range(int nKept, int &k0, int &k1) {
    const long long S = gridDim.y, h = blockIdx.y;
    k0 = static_cast<int>(h * nKept / S);
    k1 = static_cast<int>((h + 1) * nKept / S);
}

// Values and first derivatives of the kept functions of blocks b0 + blockIdx.x into rows [vOffset - rowBase, + nKept) of the
// planes out[0..3] (row stride kBlockSize; zero past a block's points).  A shell that straddles two work-groups' rows is
// evaluated by both.
__global__ void __launch_bounds__(kBlockSize) basis_planes_kernel(
    int b0, long long rowBase, const xq::DevBlock *__restrict__ blocks, const double *__restrict__ px,
    const double *__restrict__ py, const double *__restrict__ pz, const xq::DevShell *__restrict__ shells,
    const int *__restrict__ shellOf, const double *__restrict__ coef, const double *__restrict__ trans, int spherical,
    const int *__restrict__ idx, xq::Planes4 out) {
    const xq::DevBlock blk = blocks[b0 + static_cast<int>(blockIdx.x)];
    const int t = threadIdx.x;
    const bool valid = t < blk.nPoints;
    const double x = valid ? px[blk.pStart + t] : 0.0, y = valid ? py[blk.pStart + t] : 0.0,
                 z = valid ? pz[blk.pStart + t] : 0.0;
    const int *kept = idx + blk.iOffset;
    int k, k1;
    row_range(blk.nKept, k, k1);
    while (k < k1) {
        const xq::DevShell &sh = shells[shellOf[kept[k]]];
        with_shell<true>(sh, spherical != 0, coef, trans, x - sh.x, y - sh.y, z - sh.z,
                         [&](auto n, const auto &v, const auto &vx, const auto &vy, const auto &vz) {
#pragma unroll
            for (int j = 0; j < n; j++) {
                if (k < k1 && kept[k] == sh.fStart + j) {
                    const size_t o = static_cast<size_t>(blk.vOffset - rowBase + k) * kBlockSize + t;
                    out.p[0][o] = valid ? v[j] : 0.0;
                    out.p[1][o] = valid ? vx[j] : 0.0;
                    out.p[2][o] = valid ? vy[j] : 0.0;
                    out.p[3][o] = valid ? vz[j] : 0.0;
                    k++;
                }
            }
        });
    }
}

// The second derivatives' part of the XC gradients of blocks b0 + blockIdx.x: for each kept function r with its atom m,
// sum_p sum_s X^s_rp H_rp a^s_p (H the function's Hessian at point p, a^s the spins' coefficients coef[..][1..3]) is
// subtracted from the gradient of m and added to that of the block's atom.  The Hessians are used where they are
// evaluated, for all spins at once; a thread sums its point over an atom's functions before the wave is reduced.  Bound by
// FP64 arithmetic.  With ten planes of values and derivatives written and the second ones read by the Z pass, the two
// took 10.7 ms on (H2O)64; four planes, this kernel (3.2 ms) and the Z pass without them take 9.3 ms.
__global__ void __launch_bounds__(kBlockSize) second_terms_kernel(
    int b0, long long rowBase, const xq::DevBlock *__restrict__ blocks, const double *__restrict__ px,
    const double *__restrict__ py, const double *__restrict__ pz, const xq::DevShell *__restrict__ shells,
    const int *__restrict__ shellOf, const double *__restrict__ coef, const double *__restrict__ trans, int spherical,
    const int *__restrict__ idx, const double *__restrict__ X0, const double *__restrict__ X1, int nSpins,
    const double *__restrict__ pointCoef, const int *__restrict__ skip, int nAtoms, int nCopies, double *__restrict__ copies) {
    const int local = static_cast<int>(blockIdx.x), b = b0 + local;
    if (skip[local]) return;
    const xq::DevBlock blk = blocks[b];
    const int t = threadIdx.x, lane = t & 63;
    const bool valid = t < blk.nPoints;
    const double x = valid ? px[blk.pStart + t] : 0.0, y = valid ? py[blk.pStart + t] : 0.0,
                 z = valid ? pz[blk.pStart + t] : 0.0;
    double a0[3], a1[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double *q = pointCoef + (static_cast<size_t>(local) * 4 * nSpins + 1 + d) * kBlockSize + t;
        a0[d] = valid ? q[0] : 0.0;
        a1[d] = valid && nSpins == 2 ? q[4 * kBlockSize] : 0.0;
    }
    const int *kept = idx + blk.iOffset;
    double *grad = copies + static_cast<size_t>((b + static_cast<int>(blockIdx.y)) % nCopies) * 3 * nAtoms;
    double c[3] = {0.0, 0.0, 0.0}, total[3] = {0.0, 0.0, 0.0};
    int atom = -1;
    auto flush = [&]() {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            double e = c[d];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o, 64);
            if (lane == 0) atomicAdd(&grad[3 * atom + d], -e);
            total[d] += e;
            c[d] = 0.0;
        }
    };
    int k, k1;
    row_range(blk.nKept, k, k1);
    while (k < k1) {
        const xq::DevShell &sh = shells[shellOf[kept[k]]];
        if (sh.atom != atom) {
            if (atom >= 0) flush();
            atom = sh.atom;
        }
        for_shell_type(sh, spherical != 0, [&](auto ll, auto lh, auto s) {
            constexpr int N = s ? ShellDims<ll, lh>::nSph : ShellDims<ll, lh>::nCBF;
            double A[3][N];
#pragma unroll
            for (int j = 0; j < N; j++) {
                const bool has = k < k1 && kept[k] == sh.fStart + j;
                const size_t o = static_cast<size_t>(blk.vOffset - rowBase + k) * kBlockSize + t;
                const double x0 = has && valid ? X0[o] : 0.0, x1 = has && valid && nSpins == 2 ? X1[o] : 0.0;
#pragma unroll
                for (int d = 0; d < 3; d++) A[d][j] = x0 * a0[d] + x1 * a1[d];
                k += has ? 1 : 0;
            }
            shell_second<ll, lh, s>(sh, coef, trans, x - sh.x, y - sh.y, z - sh.z, A, c);
        });
    }
    if (atom >= 0) flush();
    if (lane == 0)
#pragma unroll
        for (int d = 0; d < 3; d++) atomicAdd(&grad[3 * blk.atom + d], total[d]);
}

}  // namespace

void free_basis(xq_grid *g) {
    free_mixed(g);
    free_f64(g);
    dev_free(g, &g->d_shells);
    dev_free(g, &g->d_coef);
    dev_free(g, &g->d_trans);
    dev_free(g, &g->d_pow);
    dev_free(g, &g->d_idx);
    dev_free(g, &g->d_shellOf);
    g->h_shellOf.clear();
    g->h_funcAtom.clear();
    void **values[4] = {&g->d_f, &g->d_fx, &g->d_fy, &g->d_fz};
    for (void **a : values) {
        g->deviceBytes -= static_cast<long long>(cache_free(*a));
        *a = nullptr;
    }
    g->hasBasis = false;
}

int set_basis(xq_grid *g, int nSpec, const double *spec, int spherical, int precision) {
    if (precision != XQ_PRECISION_FP64 && precision != XQ_PRECISION_MIXED) {
        set_error("unknown precision mode");
        return kInvalidArgument;
    }
    // Parse the element specification.
    struct Element { int z, start, nShells; };
    std::vector<Element> elements;
    for (int p = 0; p < nSpec;) {
        if (p + 2 > nSpec) { set_error("truncated basis specification"); return kInvalidArgument; }
        Element e{static_cast<int>(spec[p]), p + 2, static_cast<int>(spec[p + 1])};
        p += 2;
        for (int s = 0; s < e.nShells; s++) {
            if (p + 3 > nSpec) { set_error("truncated basis specification"); return kInvalidArgument; }
            const int lLow = static_cast<int>(spec[p]), lHigh = static_cast<int>(spec[p + 1]), np = static_cast<int>(spec[p + 2]);
            if (lLow < 0 || lHigh < lLow || lHigh > kMaxL || np < 1 || np > kMaxPrim) {
                set_error("unsupported shell in basis specification");
                return kInvalidArgument;
            }
            const int key = lLow * 4 + lHigh;
            if (!(key == 0 || key == 5 || key == 1 || key == 10 || key == 15)) {
                set_error("unsupported shell type (supported: S, P, D, F, SP)");
                return kInvalidArgument;
            }
            p += 3 + np * (1 + lHigh - lLow + 1);
        }
        if (p > nSpec) { set_error("truncated basis specification"); return kInvalidArgument; }
        elements.push_back(e);
    }
    std::vector<DevShell> shells;
    std::vector<double> coef, trans;
    std::vector<int> shellOf;
    int f = 0;
    for (int a = 0; a < g->nAtoms; a++) {
        const Element *el = nullptr;
        for (const Element &e : elements) if (e.z == g->Z[a]) el = &e;
        if (el == nullptr) { set_error("no basis for an atom's element"); return kInvalidArgument; }
        int p = el->start;
        for (int s = 0; s < el->nShells; s++) {
            DevShell sh{};
            sh.x = g->xyz[3 * a]; sh.y = g->xyz[3 * a + 1]; sh.z = g->xyz[3 * a + 2];
            sh.atom = a;
            sh.lLow = static_cast<int>(spec[p]); sh.lHigh = static_cast<int>(spec[p + 1]); sh.nPrim = static_cast<int>(spec[p + 2]);
            p += 3;
            sh.nCBF = 0; sh.nBasis = 0;
            for (int l = sh.lLow; l <= sh.lHigh; l++) { sh.nCBF += ncart(l); sh.nBasis += 2 * l + 1; }
            if (!spherical) sh.nBasis = sh.nCBF;
            sh.fStart = f;
            sh.coef = static_cast<int>(coef.size());
            sh.pow = 0;
            std::vector<double> ex(sh.nPrim), cc(static_cast<size_t>(sh.nPrim) * sh.nCBF);
            for (int q = 0; q < sh.nPrim; q++) {
                const double alpha = spec[p++];
                ex[q] = alpha;
                for (int l = sh.lLow, c = 0; l <= sh.lHigh; l++) {
                    // Unnormalise (GaussianBasis.c:728-751).
                    const double e2 = 2.0 * alpha;
                    double fac = std::pow(M_PI, 1.5) / (e2 * std::sqrt(e2));
                    for (int i = 1; i <= l; i++) fac *= static_cast<double>(2 * i - 1) / (2.0 * e2);
                    const double k = spec[p++] / std::sqrt(fac);
                    // Cartesian factors (GaussianBasis.c:448-501).
                    const int off = cart_offset(l);
                    for (int i = 0; i < ncart(l); i++, c++) {
                        const double m = std::sqrt(odd_fact(2 * l - 1) / (odd_fact(2 * kCart.x[off + i] - 1) *
                                                                         odd_fact(2 * kCart.y[off + i] - 1) *
                                                                         odd_fact(2 * kCart.z[off + i] - 1)));
                        cc[static_cast<size_t>(q) * sh.nCBF + c] = k * m;
                    }
                }
            }
            coef.insert(coef.end(), ex.begin(), ex.end());
            coef.insert(coef.end(), cc.begin(), cc.end());
            double K = 1.0;
            if (spherical) {
                sh.trans = static_cast<int>(trans.size());
                std::vector<double> T(static_cast<size_t>(sh.nCBF) * sh.nBasis, 0.0);
                for (int l = sh.lLow, r0 = 0, c0 = 0; l <= sh.lHigh; l++) {
                    c2s_block(l, T.data(), sh.nBasis, r0, c0);
                    r0 += ncart(l);
                    c0 += 2 * l + 1;
                }
                K = 0.0;
                for (int sI = 0; sI < sh.nBasis; sI++) {
                    double col = 0.0;
                    for (int c = 0; c < sh.nCBF; c++) col += std::fabs(T[static_cast<size_t>(c) * sh.nBasis + sI]);
                    K = std::max(K, col);
                }
                trans.insert(trans.end(), T.begin(), T.end());
            } else sh.trans = -1;
            for (int q = 0; q < sh.nPrim; q++) {
                double amax = 0.0;
                for (int c = 0; c < sh.nCBF; c++) amax = std::max(amax, std::fabs(cc[static_cast<size_t>(q) * sh.nCBF + c]));
                sh.bound[q] = amax * K;
            }
            for (int j = 0; j < sh.nBasis; j++) shellOf.push_back(static_cast<int>(shells.size()));
            f += sh.nBasis;
            shells.push_back(sh);
        }
    }
    if (shells.size() > static_cast<size_t>(kMaxShellsLDS)) { set_error("too many shells"); return kInvalidArgument; }
    free_basis(g);
    free_work(g);
    g->nFunctions = f;
    g->nShells = static_cast<int>(shells.size());
    g->spherical = spherical ? 1 : 0;
    g->precision = precision;
    hipStream_t s = g->stream;
    XQ_TRY(dev_alloc(g, &g->d_shells, shells.size()));
    XQ_TRY(dev_alloc(g, &g->d_coef, coef.size()));
    XQ_TRY(dev_alloc(g, &g->d_trans, trans.size()));
    XQ_CHECK(hipMemcpyAsync(g->d_shells, shells.data(), shells.size() * sizeof(DevShell), hipMemcpyHostToDevice, s));
    XQ_CHECK(hipMemcpyAsync(g->d_coef, coef.data(), coef.size() * sizeof(double), hipMemcpyHostToDevice, s));
    if (!trans.empty())
        XQ_CHECK(hipMemcpyAsync(g->d_trans, trans.data(), trans.size() * sizeof(double), hipMemcpyHostToDevice, s));
    // Pass 1: kept functions per block.
    int *tmpIdx = nullptr, *counts = nullptr, *d_shellOf = nullptr;
    int status = kOK;
    do {
        if ((status = dev_alloc(g, &tmpIdx, static_cast<size_t>(g->nBlocks) * f)) != kOK) break;
        if ((status = dev_alloc(g, &counts, g->nBlocks)) != kOK) break;
        if ((status = dev_alloc(g, &d_shellOf, shellOf.size())) != kOK) break;
        if ((status = check(hipMemcpyAsync(d_shellOf, shellOf.data(), shellOf.size() * sizeof(int), hipMemcpyHostToDevice, s),
                            "copy shellOf")) != kOK) break;
        if (g->nBlocks > 0) {
            const size_t mask = sizeof(unsigned) * ((static_cast<size_t>(g->nShells) + 1) / 2);
            hipLaunchKernelGGL(basis_count_kernel, dim3(g->nBlocks), dim3(kBlockSize), mask, s, g->nBlocks, g->d_blocks, g->d_x,
                               g->d_y, g->d_z, g->nShells, g->d_shells, g->d_coef, g->d_trans, g->spherical, f, g->bfTol,
                               tmpIdx, counts);
            if ((status = check(hipGetLastError(), "basis_count_kernel")) != kOK) break;
        }
        std::vector<int> h_counts(g->nBlocks > 0 ? g->nBlocks : 1, 0);
        // Wait for the kernels first: a pageable copy that waits for its stream holds the runtime's staging path.
        if ((status = check(hipStreamSynchronize(s), "basis sync")) != kOK) break;
        if (g->nBlocks > 0 &&
            (status = check(hipMemcpyAsync(h_counts.data(), counts, g->nBlocks * sizeof(int), hipMemcpyDeviceToHost, s),
                            "copy counts")) != kOK) break;
        if ((status = check(hipStreamSynchronize(s), "basis sync")) != kOK) break;
        long long rows = 0;
        double bfv = 0.0, bfs = 0.0, bfp = 0.0;
        for (int b = 0; b < g->nBlocks; b++) {
            bfs += static_cast<double>(h_counts[b]) * h_counts[b] * g->blocks[b].nPoints;
            const double padded = 32.0 * ((h_counts[b] + 31) / 32);
            bfp += padded * padded * kBlockSize;
            g->blocks[b].nKept = h_counts[b];
            g->blocks[b].vOffset = rows;
            g->blocks[b].iOffset = static_cast<int>(rows);
            rows += h_counts[b];
            bfv += static_cast<double>(h_counts[b]) * g->blocks[b].nPoints;
        }
        g->nValueRows = rows;
        g->bfValues = bfv;
        g->bfSquares = bfs;
        g->bfSquaresPadded = bfp;
        if ((status = check(hipMemcpyAsync(g->d_blocks, g->blocks.data(), g->nBlocks * sizeof(DevBlock), hipMemcpyHostToDevice, s),
                            "copy blocks")) != kOK) break;
        const size_t nVal = static_cast<size_t>(rows > 0 ? rows : 1) * kBlockSize;
        const size_t elt = sizeof(double);
        if ((status = dev_alloc(g, &g->d_idx, static_cast<size_t>(rows > 0 ? rows : 1))) != kOK) break;
        void **arrays[4] = {&g->d_f, &g->d_fx, &g->d_fy, &g->d_fz};
        for (void **a : arrays) {
            hipError_t e = cache_alloc(a, nVal * elt);
            if (e != hipSuccess) { set_error("hipMalloc failed for basis values"); status = kOutOfMemory; break; }
            g->deviceBytes += static_cast<long long>(nVal * elt);
        }
        if (status != kOK) break;
        if (precision == XQ_PRECISION_MIXED) {
            const size_t nB = static_cast<size_t>(g->nBlocks > 0 ? g->nBlocks : 1);
            if ((status = dev_alloc(g, &g->d_EB, nB * kBlockSize)) != kOK) break;
            if ((status = dev_alloc(g, &g->d_EG, 3 * nB * kBlockSize)) != kOK) break;
        }
        if (g->nBlocks > 0) {
            hipLaunchKernelGGL(basis_eval_kernel, dim3(g->nBlocks), dim3(kBlockSize), 0, s, g->d_blocks, g->d_x,
                               g->d_y, g->d_z, g->d_shells, d_shellOf, g->d_coef, g->d_trans, g->spherical, f, tmpIdx,
                               g->d_idx, static_cast<double *>(g->d_f), static_cast<double *>(g->d_fx),
                               static_cast<double *>(g->d_fy), static_cast<double *>(g->d_fz), g->d_EB, g->d_EG);
            if ((status = check(hipGetLastError(), "basis_eval_kernel")) != kOK) break;
        }
        // The operand-order planes of the chosen precision replace the FP64 rows.
        if (precision == XQ_PRECISION_MIXED)
            status = prepare_mixed(g, static_cast<double *>(g->d_f), static_cast<double *>(g->d_fx),
                                   static_cast<double *>(g->d_fy), static_cast<double *>(g->d_fz));
        else
            status = prepare_f64(g, static_cast<double *>(g->d_f), static_cast<double *>(g->d_fx),
                                 static_cast<double *>(g->d_fy), static_cast<double *>(g->d_fz));
        if (status != kOK) break;
        if ((status = check(hipStreamSynchronize(s), "basis sync")) != kOK) break;
        for (void **a : arrays) {
            g->deviceBytes -= static_cast<long long>(cache_free(*a));
            *a = nullptr;
        }
        status = check(hipStreamSynchronize(s), "basis sync");
    } while (false);
    (void)hipStreamSynchronize(s);   // the kernels that use the scratch arrays are done before they are reused
    dev_free(g, &tmpIdx);
    dev_free(g, &counts);
    dev_free(g, &d_shellOf);
    if (status != kOK) { free_basis(g); return status; }
    g->h_shellOf = shellOf;     // kept for the second-derivative evaluation of the XC gradients
    g->h_funcAtom.resize(shellOf.size());
    for (size_t fn = 0; fn < shellOf.size(); fn++) g->h_funcAtom[fn] = shells[shellOf[fn]].atom;
    g->hasBasis = true;
    return kOK;
}


// Work-groups per block of the two launches below, each a part of its kept rows: the blocks' rows are evaluated one shell
// after another, so a launch would otherwise last as long as its largest block.
constexpr unsigned kRowParts = 4;

static int shell_of_functions(xq_grid *g) {
    if (g->d_shellOf != nullptr) return kOK;
    XQ_TRY(dev_alloc(g, &g->d_shellOf, g->h_shellOf.size()));
    XQ_CHECK(hipMemcpyAsync(g->d_shellOf, g->h_shellOf.data(), g->h_shellOf.size() * sizeof(int), hipMemcpyHostToDevice,
                            g->stream));
    XQ_CHECK(hipStreamSynchronize(g->stream));
    return kOK;
}

// Basis values and gradients of blocks [b0, b1) into the planes (rows from the blocks' value-row offsets less rowBase), for
// the XC gradients.
int eval_planes(xq_grid *g, int b0, int b1, long long rowBase, const Planes4 &out, hipStream_t s) {
    if (b1 <= b0) return kOK;
    XQ_TRY(shell_of_functions(g));
    hipLaunchKernelGGL(basis_planes_kernel, dim3(b1 - b0, kRowParts), dim3(kBlockSize), 0, s, b0, rowBase, g->d_blocks,
                       g->d_x, g->d_y, g->d_z, g->d_shells, g->d_shellOf, g->d_coef, g->d_trans, g->spherical, g->d_idx, out);
    XQ_CHECK(hipGetLastError());
    return kOK;
}

// The second derivatives' part of the XC gradients of blocks [b0, b1), added to nCopies copies of the gradients.
int second_derivative_terms(xq_grid *g, int b0, int b1, long long rowBase, int spins, const double *X0, const double *X1,
                            const double *pointCoef, const int *skip, int nCopies, double *copies, hipStream_t s) {
    if (b1 <= b0) return kOK;
    XQ_TRY(shell_of_functions(g));
    hipLaunchKernelGGL(second_terms_kernel, dim3(b1 - b0, kRowParts), dim3(kBlockSize), 0, s, b0, rowBase, g->d_blocks,
                       g->d_x, g->d_y, g->d_z, g->d_shells, g->d_shellOf, g->d_coef, g->d_trans, g->spherical, g->d_idx,
                       X0, X1, spins, pointCoef, skip, g->nAtoms, nCopies, copies);
    XQ_CHECK(hipGetLastError());
    return kOK;
}

}  // namespace xq
