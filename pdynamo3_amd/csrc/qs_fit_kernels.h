// The electron-fit integral kernel and its launches, for the files that instantiate them (qs_fit_*.hip: one class of orbital
// shell pairs or a part of one each, so that they compile side by side).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "qs_kernels.h"

namespace qs {

// What the launches of one qs_fit_create or qs_fit_matrix share.
struct FitLaunch {
    hipStream_t stream;
    const QShell *oShells;
    int oSpherical;
    const double *records;
    const QShell *fShells;          // the fit shells by angular momentum
    int fSpherical;
    int first[kMaxL + 2];           // first fit shell and first stored column of each angular momentum
    int column[kMaxL + 2];
    const double *fExps, *fCoefs, *boys;
    int nFit;
    double cut;                     // integrals not above it in magnitude are stored as zero; negative for none
    double *B;
};

// The electron-fit integrals of n pairs of the class (la, lb) with the fit shells of lc.
template <int LA, int LB, int LC>
void launch_fit(const FitLaunch &f, const PairItem *items, int n);

#ifdef QS_FIT_KERNELS

// Waves of one launch: a launch holds less than 2^32 threads.
constexpr int kLaunchWaves = 1 << 25;

// One wave per pair and 64 fit shells of an angular momentum, components M0 .. M0 + NM - 1 of the shells.  The pair's
// records are read as scalars, and a lane holds its fit shell's Hermite integrals and its part of the block in registers
// (no private memory): the kernel is bound by FP64 arithmetic and the Boys table's gathers.  It replaces a kernel of one
// thread per pair and fit shell with loops over all angular momenta, whose tables were 8 KB of private memory per lane:
// on (H2O)16 with 624 fit functions all classes together take 0.4 ms instead of 31.6 ms.  The fit functions of an angular
// momentum are stored function by function (column function * shells + shell), so that a wave's stores are contiguous.
template <int LA, int LB, int LC, int M0, int NM>
__global__ void __launch_bounds__(256) fit_integrals_kernel(int nPairs, const PairItem *__restrict__ items,
                                                            const QShell *__restrict__ oShells, int oSpherical,
                                                            const double *__restrict__ records, int nFitShells,
                                                            const QShell *__restrict__ fShells, int fSpherical,
                                                            const double *__restrict__ fExps,
                                                            const double *__restrict__ fCoefs,
                                                            const double *__restrict__ boysTable, int column, int nFit,
                                                            double cut, double *__restrict__ B) {
    const int chunks = (nFitShells + 63) / 64;
    const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x * 4 + (threadIdx.x >> 6)));
    const int k = w / chunks, c = (w - k * chunks) * 64 + static_cast<int>(threadIdx.x & 63);
    if (k >= nPairs || c >= nFitShells) return;
    const PairItem it = items[k];
    double acc[PairClass<LA, LB>::na * PairClass<LA, LB>::nb][NM];
    fit_block<LA, LB, LC, M0, NM>(records + it.first, it.n, fShells[c], fExps, fCoefs, boysTable, acc);
    const int ma = oShells[it.a].nf, mb = oShells[it.b].nf;
    double *out = B + column + c;
    pair_functions<LA, LB, NM>(oSpherical, acc);
    for_functions<LA, LB>(oSpherical, [&](int i, int j, auto ab) {
        double *row = out + pair_row(it, i, j, ma, mb) * nFit;
        fit_functions<LC, M0, NM>(fSpherical, acc[ab], [&](int f, double x) {
            row[f * nFitShells] = cut >= 0.0 && !(fabs(x) > cut) ? 0.0 : x;
        });
    });
}

template <int LA, int LB, int LC>
void launch_fit(const FitLaunch &f, const PairItem *items, int n) {
    constexpr int NM = fit_group<LA, LB, LC>();
    const int shells = f.first[LC + 1] - f.first[LC];
    if (shells == 0 || n == 0) return;
    const int chunks = (shells + 63) / 64, most = std::max(1, kLaunchWaves / chunks);
    for (int k = 0; k < n; k += most) {
        const int m = std::min(most, n - k);
        const dim3 grid(static_cast<unsigned>((static_cast<long long>(m) * chunks + 3) / 4));
        static_for<cartesians(LC) / NM>([&](auto group) {
            hipLaunchKernelGGL((fit_integrals_kernel<LA, LB, LC, group * NM, NM>), grid, dim3(256), 0, f.stream, m, items + k,
                               f.oShells, f.oSpherical, f.records, shells, f.fShells + f.first[LC], f.fSpherical, f.fExps,
                               f.fCoefs, f.boys, f.column[LC], f.nFit, f.cut, f.B);
        });
    }
}

#endif

}  // namespace qs
