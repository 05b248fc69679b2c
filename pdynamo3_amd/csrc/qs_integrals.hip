// Integrals of the SCF wrapper on the GPU: the one-electron matrices (overlap, kinetic energy, electron-nuclear attraction)
// and the density-fitted Coulomb term, whose electron-fit integrals (mu nu|P) stay resident in device memory.
//
// Counterparts in the reference (QCModelDFT's energy closures, QCModelDFT.py:130-160, through
// GaussianBasisIntegralEvaluator.pyx):
//   qs_one_electron  <- GaussianBasisContainerIntegrals_f1KOf1i (GaussianBasisContainerIntegrals_f1Xg1.c:233-296) and
//                       GaussianBasisContainerIntegrals_f2Cm1V (GaussianBasisContainerIntegrals_f2Cp1.c:104-173), point nuclei
//   qs_fit_create    <- GaussianBasisContainerIntegrals_f1Xg2i (GaussianBasisContainerIntegrals_f1Xg2.c:43-128), Coulomb
//                       operator; values of magnitude <= 1e-12 are dropped, as its block storage drops them (:42, :67)
//   qs_fit_matrix    <- f1Xf1i_f1Oi with constraints (GaussianBasisIntegralEvaluator.pyx:260-302): (P|Q) from
//                       GaussianBasisContainerIntegrals_f1Cf1i, the last row the fit functions' integrals (f1Oi)
//   qs_fit_b, qs_fit_fock <- the two contractions of Fock_MakeFromFitIntegralsCoulomb (FockConstruction.c:31-108):
//                       b_P = sum_mn P_mn (mn|P) and F_mn += sum_P c_P (mn|P); the bordered solve between them is the caller's
// The integrals themselves are the McMurchie-Davidson forms of qs_md.h (the reference uses Rys quadrature; the values agree
// to rounding).  Functions are the reference's: contraction coefficients unnormalised as GaussianBasis_UnnormalizePrimitives,
// Cartesian factors sqrt((2l-1)!! / ((2x-1)!! (2y-1)!! (2z-1)!!)) (GaussianBasis.c:448-501, 728-751), spherical functions by
// the c2s transformation of xq_c2s.h.
//
// Layout of the electron-fit integrals: the significant orbital shell pairs (A >= B, pair prefactor above 1e-15) each own
// nA x nB consecutive rows of a row-major [rows][fit functions] FP64 array; a row's packed orbital index (mu >= nu) is in
// rowPacked, -1 for the upper-triangle duplicates of a diagonal shell pair.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/qcscf.h"
#include "qs_fit_kernels.h"
#include "qs_shells.h"
#include "xq_c2s.h"
#include "xq_internal.h"

using xq::check;
using xq::kInvalidArgument;
using xq::kOK;
using xq::kOutOfMemory;
using xq::set_error;

namespace qs {

// The Boys function table, one copy per GPU (filled once per device by the first basis created on it).
__device__ double g_boys[kBoysPoints * kBoysTable];

namespace {

constexpr int kThreads = 128;

std::mutex g_boysMutex;
bool g_boysReady[64] = {};

// The Boys table on the current GPU (once per device).
int ensure_boys() {
    int device = 0;
    XQ_CHECK(hipGetDevice(&device));
    if (device < 0 || device >= 64) { set_error("device index out of range"); return kInvalidArgument; }
    std::lock_guard<std::mutex> lock(g_boysMutex);
    if (g_boysReady[device]) return kOK;
    std::vector<double> t;
    boys_table(t);
    XQ_CHECK(hipMemcpyToSymbol(HIP_SYMBOL(g_boys), t.data(), t.size() * sizeof(double)));
    g_boysReady[device] = true;
    return kOK;
}

// The device address of the Boys table on the current GPU.
int boys_address(const double **boys) {
    void *p = nullptr;
    XQ_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(g_boys)));
    *boys = static_cast<const double *>(p);
    return kOK;
}

// ------------------------------------------------------------------------------------------------------------------------
// Shell pairs by class (qs_kernels.h): their records, one thread per pair, and the one-electron matrices.
// ------------------------------------------------------------------------------------------------------------------------
template <int LA, int LB>
__global__ void __launch_bounds__(kThreads) pair_records_kernel(int nPairs, PairItem *__restrict__ items,
                                                                const QShell *__restrict__ shells,
                                                                const double *__restrict__ exps,
                                                                const double *__restrict__ coefs,
                                                                double *__restrict__ records) {
    const int k = blockIdx.x * kThreads + threadIdx.x;
    if (k >= nPairs) return;
    const PairItem it = items[k];
    items[k].n = pair_records<LA, LB>(shells[it.a], shells[it.b], exps, coefs, records + it.first);
}

template <int LA, int LB>
__global__ void __launch_bounds__(kThreads) overlap_kinetic_kernel(int nPairs, const PairItem *__restrict__ items,
                                                                   const QShell *__restrict__ shells,
                                                                   const double *__restrict__ exps,
                                                                   const double *__restrict__ coefs, int spherical,
                                                                   double *__restrict__ S, double *__restrict__ T) {
    const int k = blockIdx.x * kThreads + threadIdx.x;
    if (k >= nPairs) return;
    const QShell A = shells[items[k].a], B = shells[items[k].b];
    overlap_kinetic<LA, LB>(A, B, exps, coefs, spherical, [&](int i, int j, double overlap, double kinetic) {
        const long long o = packed_index(A.f0 + i, B.f0 + j);
        S[o] = overlap;
        T[o] = kinetic;
    });
}

// Nuclear attraction: one wave per pair, its lanes the nuclei; the lanes' blocks are summed over the wave.  With the pair's
// integrals unrolled by class and its records shared by the lanes, S, T and V of (H2O)16 take 0.2 ms; one thread per pair
// with loops over all angular momenta and 6 KB of private memory took 12.7 ms.
template <int LA, int LB>
__global__ void __launch_bounds__(256) nuclear_kernel(int nPairs, const PairItem *__restrict__ items,
                                                      const QShell *__restrict__ shells,
                                                      const double *__restrict__ records, int nAtoms,
                                                      const double *__restrict__ atoms, int spherical,
                                                      double *__restrict__ V) {
    const int k = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x * 4 + (threadIdx.x >> 6)));
    if (k >= nPairs) return;
    const int lane = threadIdx.x & 63;
    const PairItem it = items[k];
    double acc[PairClass<LA, LB>::na * PairClass<LA, LB>::nb][1];
    nuclear_block<LA, LB>(records + it.first, it.n, lane, 64, nAtoms, atoms, g_boys, acc);
    static_for<PairClass<LA, LB>::na * PairClass<LA, LB>::nb>([&](auto ab) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) acc[ab][0] += __shfl_xor(acc[ab][0], o, 64);
    });
    const int fa = shells[it.a].f0, fb = shells[it.b].f0;
    pair_functions<LA, LB, 1>(spherical, acc);
    for_functions<LA, LB>(spherical, [&](int i, int j, auto ab) {
        if (lane == 0) V[packed_index(fa + i, fb + j)] = acc[ab][0];
    });
}

// ------------------------------------------------------------------------------------------------------------------------
// Fit matrix: its integrals are the electron-fit integrals of pairs of a fit shell with the unit shell (qs_kernels.h), dense
// with the fit functions' stored columns; here the lower triangle of the rows p0 .. p1 - 1 is packed, with the functions' own
// integrals in the last row.  One thread per entry, and per fit shell.
// ------------------------------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) fit_matrix_pack_kernel(int nFit, int p0, int p1, const double *__restrict__ dense,
                                                              const int *__restrict__ column, double *__restrict__ M) {
    const int q = blockIdx.x * 256 + threadIdx.x;
    for (int p = p0 + static_cast<int>(blockIdx.y); p < p1; p += gridDim.y)
        if (q <= p) M[packed_index(p, q)] = dense[static_cast<size_t>(p - p0) * nFit + column[q]];
}

template <int LA>
__global__ void __launch_bounds__(kThreads) fit_charges_kernel(int nShells, const PairItem *__restrict__ items,
                                                               const QShell *__restrict__ shells,
                                                               const double *__restrict__ exps,
                                                               const double *__restrict__ coefs, int spherical,
                                                               double *__restrict__ charges) {
    const int k = blockIdx.x * kThreads + threadIdx.x;
    if (k >= nShells) return;
    const QShell A = shells[items[k].a];
    overlap_kinetic<LA, 0>(A, shells[items[k].b], exps, coefs, spherical,
                           [&](int i, int, double s, double) { charges[A.f0 + i] = s; });
}

// ------------------------------------------------------------------------------------------------------------------------
// Per SCF iteration: b = sum_rows w_row P_row B_row (partial sums over row chunks, then a fixed-order reduction) and
// F_row += B_row . c (one wave per row).  w_row = 2 off the diagonal, 1 on it, 0 for a duplicate row.
// ------------------------------------------------------------------------------------------------------------------------
constexpr int kRowChunk = 1024;

// Partial sums of b over kRowChunk rows: 16 waves per work-group, each 64 rows and the same 64 fit functions, their sums
// added in order.  The rows' weights w_row P_row are gathered once into LDS, so that the rows' loads are independent of
// each other.  Bound by reading the integrals: 1.7 GB on (H2O)48 in 0.29 ms, against 0.61 with a thread for 1,024 rows,
// whose every load waited for the row's index and density, and on (H2O)16, whose chunks then were too few to
// fill the chip, 0.02 ms against 0.37.
__global__ void __launch_bounds__(1024) fit_b_partial_kernel(long long rows, int nFit, const double *__restrict__ B,
                                                            const long long *__restrict__ rowPacked,
                                                            const unsigned char *__restrict__ rowDiag,
                                                            const double *__restrict__ P, double *__restrict__ partial) {
    __shared__ double sw[kRowChunk];
    __shared__ double sums[16][64];
    const long long r0 = static_cast<long long>(blockIdx.y) * kRowChunk;
    const int n = static_cast<int>(rows - r0 < kRowChunk ? rows - r0 : kRowChunk);
    for (int k = threadIdx.x; k < n; k += 1024) {
        const long long o = rowPacked[r0 + k];
        sw[k] = o < 0 ? 0.0 : (rowDiag[r0 + k] ? 1.0 : 2.0) * P[o];
    }
    __syncthreads();
    const int c = threadIdx.x & 63, wv = threadIdx.x >> 6, col = blockIdx.x * 64 + c;
    const int k0 = wv * (kRowChunk / 16), k1 = k0 + kRowChunk / 16 < n ? k0 + kRowChunk / 16 : n;
    double acc = 0.0;
    if (col < nFit) {
        const double *row = B + r0 * nFit + col;
#pragma unroll 8
        for (int k = k0; k < k1; k++) acc = fma(sw[k], row[static_cast<size_t>(k) * nFit], acc);
    }
    sums[wv][c] = acc;
    __syncthreads();
    if (wv != 0 || col >= nFit) return;
    for (int k = 1; k < 16; k++) acc += sums[k][c];
    partial[static_cast<size_t>(blockIdx.y) * nFit + col] = acc;
}

// b from the partial sums: 64 fit functions per work-group, 16 threads each (chunks j, j + 16, ...), then their 16 sums in
// order.
__global__ void __launch_bounds__(1024) fit_b_reduce_kernel(int nChunks, int nFit, const double *__restrict__ partial,
                                                            double *__restrict__ b) {
    __shared__ double s[16][64];
    const int c = threadIdx.x & 63, j = threadIdx.x >> 6, col = blockIdx.x * 64 + c;
    double acc = 0.0;
    if (col < nFit) {
#pragma unroll 4
        for (int k = j; k < nChunks; k += 16) acc += partial[static_cast<size_t>(k) * nFit + col];
    }
    s[j][c] = acc;
    __syncthreads();
    if (j == 0 && col < nFit) {
        for (int k = 1; k < 16; k++) acc += s[k][c];
        b[col] = acc;
    }
}

__global__ void __launch_bounds__(256) zero_packed_kernel(size_t n, double *__restrict__ F) {
    for (size_t k = blockIdx.x * 256ull + threadIdx.x; k < n; k += gridDim.x * 256ull) F[k] = 0.0;
}

// F_row = B_row . c, four rows per wave: each value of c serves four loads.  Bound by reading the integrals ((H2O)48: one row
// per wave 0.37 ms, this 0.29 ms).
constexpr int kFockRows = 4;

__global__ void __launch_bounds__(256) fit_fock_kernel(long long rows, int nFit, const double *__restrict__ B,
                                                      const long long *__restrict__ rowPacked,
                                                      const double *__restrict__ c, double *__restrict__ F) {
    const long long r0 = (blockIdx.x * 256LL + threadIdx.x) / 64 * kFockRows;
    const int lane = threadIdx.x & 63;
    if (r0 >= rows) return;
    const int n = static_cast<int>(rows - r0 < kFockRows ? rows - r0 : kFockRows);
    const double *row[kFockRows];
    double acc[kFockRows];
#pragma unroll
    for (int i = 0; i < kFockRows; i++) {
        row[i] = B + (r0 + (i < n ? i : 0)) * nFit;     // the last rows' waves repeat a row
        acc[i] = 0.0;
    }
#pragma unroll 2
    for (int k = lane; k < nFit; k += 64) {
        const double x = c[k];
#pragma unroll
        for (int i = 0; i < kFockRows; i++) acc[i] = fma(row[i][k], x, acc[i]);
    }
#pragma unroll
    for (int i = 0; i < kFockRows; i++) {
#pragma unroll
        for (int s = 32; s > 0; s >>= 1) acc[i] += __shfl_xor(acc[i], s, 64);
        const long long o = i < n ? rowPacked[r0 + i] : -1;
        if (lane == 0 && o >= 0) F[o] = acc[i];
    }
}

}  // namespace

}  // namespace qs

// ------------------------------------------------------------------------------------------------------------------------
// Handles.
// ------------------------------------------------------------------------------------------------------------------------
struct qs_basis : qs::QBasis {
    qs::QShell *d_shells = nullptr;
    double *d_exps = nullptr, *d_coefs = nullptr;
    hipStream_t stream = nullptr;      // the one-electron kernel's stream
};

struct qs_fit {
    int nFit = 0, nOrbital = 0;
    long long rows = 0, nPairs = 0;
    qs::FitLaunch launch = {};         // the fit shells and functions in the order of the columns
    qs::QShell *d_fitSorted = nullptr;
    std::vector<int> column;           // stored column of each fit function
    double *staging = nullptr;         // pinned: b or c in the order of the columns (nFit), then packed P or F
    std::mutex step;                   // held while a call's matrices are in the staging and the device arrays
    const qs_basis *orbital = nullptr, *fit = nullptr;
    double *d_B = nullptr;
    long long *d_rowPacked = nullptr;
    unsigned char *d_rowDiag = nullptr;
    double *d_P = nullptr, *d_F = nullptr, *d_b = nullptr, *d_c = nullptr, *d_partial = nullptr;
    hipStream_t stream = nullptr;
};

namespace qs {
namespace {

// Device arrays come from the quadrature library's caching allocator: a request loop sets up and releases molecules
// while other jobs compute, and hipFree would synchronise the whole device.
template <typename T>
int qs_alloc(T **p, size_t n) {
    *p = nullptr;
    if (xq::cache_alloc(reinterpret_cast<void **>(p), (n > 0 ? n : 1) * sizeof(T)) != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
        set_error("hipMalloc failed (" + std::to_string((n > 0 ? n : 1) * sizeof(T)) + " bytes)");
        return kOutOfMemory;
    }
    return kOK;
}

template <typename T>
void qs_release(T **p) {
    if (*p != nullptr) { (void)xq::cache_free(*p); *p = nullptr; }
}

// An array with at least `count` elements; one that is too small is replaced (the work on it must be done).
template <typename T>
int qs_room(T **p, size_t *room, size_t count) {
    if (*p != nullptr && count <= *room) return kOK;
    qs_release(p);
    *room = count;
    return qs_alloc(p, count);
}

// Shell pairs sorted by class, and where each class starts; doubles of all their records.
struct PairSet {
    std::vector<PairItem> items;
    int start[7] = {0, 0, 0, 0, 0, 0, 0};
    long long doubles = 0;
};

int pair_class(const QShell &a, const QShell &b) {
    const int la = std::max(a.l, b.l), lb = std::min(a.l, b.l);
    return la * (la + 1) / 2 + lb;
}

// Doubles of the dense rows of the fit matrix that are held at once (256 MB; all of them up to about 150 waters' fit
// functions): as a whole they would take twice the packed result's memory beside it.
constexpr long long kSlabDoubles = 1LL << 25;

// Doubles of the records a set may hold where its pairs may be fewer (256 MB): the records have room for every primitive
// pair, 50 KB for each pair of 6-31G* waters, and those of all pairs would grow with the square of the molecule
// (6 GB for 500 waters).  One set covers up to about 100 waters.
constexpr long long kSliceDoubles = 1LL << 25;

// The pairs first .. last - 1 by class, in their order within a class, last the number of pairs or the first whose records
// would pass `limit` doubles (at least one is taken); row: the first row of each pair's electron-fit integrals, or empty.
PairSet pair_set(const QBasis *b, const std::vector<QPair> &pairs, const std::vector<long long> &row, size_t first = 0,
                 size_t *last = nullptr, long long limit = LLONG_MAX) {
    PairSet set;
    // A pair's records have six doubles or more.
    std::vector<unsigned char> cls(std::min<size_t>(pairs.size() - first, static_cast<size_t>(limit / 6) + 1));
    size_t end = first;
    for (long long doubles = 0; end < pairs.size(); end++) {
        const QShell &A = b->shells[pairs[end].x], &B = b->shells[pairs[end].y];
        doubles += record_room(A, B);
        if (doubles > limit && end > first) break;
        cls[end - first] = static_cast<unsigned char>(pair_class(A, B));
        set.start[cls[end - first] + 1]++;
    }
    if (last != nullptr) *last = end;
    set.items.resize(end - first);
    for (int c = 0; c < 6; c++) set.start[c + 1] += set.start[c];
    int at[6];
    for (int c = 0; c < 6; c++) at[c] = set.start[c];
    for (size_t k = first; k < end; k++) {
        const QShell &A = b->shells[pairs[k].x], &B = b->shells[pairs[k].y];
        set.items[at[cls[k - first]]++] =
            pair_item(b->shells.data(), pairs[k].x, pairs[k].y, row.empty() ? 0 : row[k], set.doubles);
        set.doubles += record_room(A, B);
    }
    return set;
}

// launch(la, lb, items of the class, their number) for every class of the set that has pairs.
template <class Launch>
int for_classes(const PairSet &set, PairItem *d_items, const char *what, Launch launch) {
    for (int la = 0, c = 0; la <= kMaxL; la++)
        for (int lb = 0; lb <= la; lb++, c++) {
            const int n = set.start[c + 1] - set.start[c];
            if (n == 0) continue;
            with_pair_class(la, lb, [&](auto A, auto B) { launch(A, B, d_items + set.start[c], n); });
            XQ_TRY(check(hipGetLastError(), what));
        }
    return kOK;
}

inline dim3 groups(long long items, int perGroup) { return dim3(static_cast<unsigned>((items + perGroup - 1) / perGroup)); }

int launch_records(const qs_basis *b, const PairSet &set, PairItem *d_items, double *d_records, hipStream_t s) {
    return for_classes(set, d_items, "pair_records_kernel", [&](auto la, auto lb, PairItem *items, int n) {
        hipLaunchKernelGGL((pair_records_kernel<la, lb>), groups(n, kThreads), dim3(kThreads), 0, s, n, items, b->d_shells,
                           b->d_exps, b->d_coefs, d_records);
    });
}

}  // namespace
}  // namespace qs

using namespace qs;

extern "C" {

int qs_basis_create(int nAtoms, const int *Z, const double *xyzBohr, int nSpec, const double *spec, int spherical,
                    qs_basis **basis) {
    if (basis == nullptr || nAtoms <= 0 || Z == nullptr || xyzBohr == nullptr || spec == nullptr || nSpec <= 0) {
        set_error("invalid basis arguments");
        return kInvalidArgument;
    }
    *basis = nullptr;
    XQ_TRY(ensure_boys());
    qs_basis *b = new qs_basis();
    b->nAtoms = nAtoms;
    b->spherical = spherical ? 1 : 0;
    b->Z.assign(Z, Z + nAtoms);
    b->xyz.assign(xyzBohr, xyzBohr + 3 * nAtoms);
    const std::string err = build_shells(b, nSpec, spec);
    int status = kOK;
    if (!err.empty()) { set_error(err); status = kInvalidArgument; }
    if (status == kOK) status = check(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking), "hipStreamCreate");
    // On the device the unit shell and its primitive follow the basis's own.
    std::vector<QShell> shells(b->shells);
    std::vector<double> exps(b->exps), coefs(b->coefs);
    shells.push_back(unit_shell(static_cast<int>(exps.size())));
    exps.push_back(0.0);
    coefs.push_back(1.0);
    if (status == kOK) status = qs_alloc(&b->d_shells, shells.size());
    if (status == kOK) status = qs_alloc(&b->d_exps, exps.size());
    if (status == kOK) status = qs_alloc(&b->d_coefs, coefs.size());
    if (status == kOK) status = check(hipMemcpyAsync(b->d_shells, shells.data(), shells.size() * sizeof(QShell),
                                                     hipMemcpyHostToDevice, b->stream), "copy shells");
    if (status == kOK) status = check(hipMemcpyAsync(b->d_exps, exps.data(), exps.size() * sizeof(double),
                                                     hipMemcpyHostToDevice, b->stream), "copy exponents");
    if (status == kOK) status = check(hipMemcpyAsync(b->d_coefs, coefs.data(), coefs.size() * sizeof(double),
                                                     hipMemcpyHostToDevice, b->stream), "copy coefficients");
    if (status == kOK) status = check(hipStreamSynchronize(b->stream), "copy basis");
    if (status != kOK) { qs_basis_free(b); return status; }
    *basis = b;
    return kOK;
}

int qs_basis_size(const qs_basis *basis, int *nFunctions) {
    if (basis == nullptr || nFunctions == nullptr) { set_error("invalid arguments"); return kInvalidArgument; }
    *nFunctions = basis->nFunctions;
    return kOK;
}

void qs_basis_free(qs_basis *basis) {
    if (basis == nullptr) return;
    qs_release(&basis->d_shells);
    qs_release(&basis->d_exps);
    qs_release(&basis->d_coefs);
    if (basis->stream) (void)hipStreamDestroy(basis->stream);
    delete basis;
}

int qs_one_electron(qs_basis *basis, double *S, double *T, double *V) {
    if (basis == nullptr || S == nullptr || T == nullptr || V == nullptr) {
        set_error("invalid one-electron arguments");
        return kInvalidArgument;
    }
    const size_t n = static_cast<size_t>(basis->nFunctions), size = n * (n + 1) / 2;
    const std::vector<QPair> pairs = shell_pairs(basis, false);
    std::vector<double> atoms(4 * static_cast<size_t>(basis->nAtoms));
    for (int a = 0; a < basis->nAtoms; a++) {
        for (int c = 0; c < 3; c++) atoms[4 * a + c] = basis->xyz[3 * a + c];
        atoms[4 * a + 3] = static_cast<double>(basis->Z[a]);
    }
    PairItem *d_items = nullptr;
    double *d_records = nullptr, *d_atoms = nullptr, *d_S = nullptr, *d_T = nullptr, *d_V = nullptr;
    int status = qs_alloc(&d_atoms, atoms.size());
    if (status == kOK) status = qs_alloc(&d_S, size);
    if (status == kOK) status = qs_alloc(&d_T, size);
    if (status == kOK) status = qs_alloc(&d_V, size);
    if (status == kOK && !pairs.empty()) status = xq::make_runtime_room("one-electron integrals");
    hipStream_t s = basis->stream;
    if (status == kOK) status = check(hipMemcpyAsync(d_atoms, atoms.data(), atoms.size() * sizeof(double),
                                                     hipMemcpyHostToDevice, s), "copy atoms");
    PairSet set;        // one slice after another, each done before the next takes its place
    size_t room[2] = {0, 0};
    for (size_t first = 0, last = 0; status == kOK && first < pairs.size(); first = last) {
        if (first > 0) status = check(hipStreamSynchronize(s), "one-electron integrals");
        if (status != kOK) break;
        set = pair_set(basis, pairs, {}, first, &last, kSliceDoubles);
        status = qs_room(&d_items, &room[0], set.items.size());
        if (status == kOK) status = qs_room(&d_records, &room[1], static_cast<size_t>(set.doubles));
        if (status == kOK) status = check(hipMemcpyAsync(d_items, set.items.data(), set.items.size() * sizeof(PairItem),
                                                         hipMemcpyHostToDevice, s), "copy pairs");
        if (status == kOK) status = launch_records(basis, set, d_items, d_records, s);
        if (status != kOK) break;
        status = for_classes(set, d_items, "one-electron kernels", [&](auto la, auto lb, PairItem *items, int n) {
            hipLaunchKernelGGL((overlap_kinetic_kernel<la, lb>), groups(n, kThreads), dim3(kThreads), 0, s, n, items,
                               basis->d_shells, basis->d_exps, basis->d_coefs, basis->spherical, d_S, d_T);
            hipLaunchKernelGGL((nuclear_kernel<la, lb>), groups(n, 4), dim3(256), 0, s, n, items, basis->d_shells,
                               d_records, basis->nAtoms, d_atoms, basis->spherical, d_V);
        });
    }
    if (status == kOK) status = check(hipMemcpyAsync(S, d_S, size * sizeof(double), hipMemcpyDeviceToHost, s), "copy S");
    if (status == kOK) status = check(hipMemcpyAsync(T, d_T, size * sizeof(double), hipMemcpyDeviceToHost, s), "copy T");
    if (status == kOK) status = check(hipMemcpyAsync(V, d_V, size * sizeof(double), hipMemcpyDeviceToHost, s), "copy V");
    const int drained = check(hipStreamSynchronize(s), "one-electron integrals");
    if (status == kOK) status = drained;
    qs_release(&d_items);
    qs_release(&d_records);
    qs_release(&d_atoms);
    qs_release(&d_S);
    qs_release(&d_T);
    qs_release(&d_V);
    return status;
}

void qs_fit_free(qs_fit *fit) {
    if (fit == nullptr) return;
    if (fit->stream) (void)hipStreamSynchronize(fit->stream);
    qs_release(&fit->d_B);
    qs_release(&fit->d_rowPacked);
    qs_release(&fit->d_rowDiag);
    qs_release(&fit->d_P);
    qs_release(&fit->d_F);
    qs_release(&fit->d_b);
    qs_release(&fit->d_c);
    qs_release(&fit->d_partial);
    qs_release(&fit->d_fitSorted);
    if (fit->staging != nullptr) xq::cache_host_free(fit->staging);
    if (fit->stream) (void)hipStreamDestroy(fit->stream);
    delete fit;
}

int qs_fit_create(const qs_basis *orbital, const qs_basis *fitBasis, qs_fit **out) {
    if (orbital == nullptr || fitBasis == nullptr || out == nullptr) { set_error("invalid fit arguments"); return kInvalidArgument; }
    *out = nullptr;
    qs_fit *F = new qs_fit();
    F->orbital = orbital;
    F->fit = fitBasis;
    F->nFit = fitBasis->nFunctions;
    F->nOrbital = orbital->nFunctions;
    int status = check(hipStreamCreateWithFlags(&F->stream, hipStreamNonBlocking), "hipStreamCreate");
    // Significant shell pairs and their rows.
    std::vector<QPair> sp = status == kOK ? shell_pairs(orbital, true) : std::vector<QPair>();
    std::vector<long long> row(sp.size());
    std::vector<long long> rowPacked;
    std::vector<unsigned char> rowDiag;
    long long rows = 0;
    for (size_t k = 0; k < sp.size(); k++) {
        const QShell &A = orbital->shells[sp[k].x], &B = orbital->shells[sp[k].y];
        row[k] = rows;
        for (int i = 0; i < A.nf; i++)
            for (int j = 0; j < B.nf; j++) {
                const int mu = A.f0 + i, nu = B.f0 + j;
                rowPacked.push_back(mu >= nu ? packed_index(mu, nu) : -1);
                rowDiag.push_back(mu == nu ? 1 : 0);
            }
        rows += static_cast<long long>(A.nf) * B.nf;
    }
    F->rows = rows;
    F->nPairs = static_cast<long long>(sp.size());
    const size_t nOrbPacked = static_cast<size_t>(F->nOrbital) * (F->nOrbital + 1) / 2;
    const long long nChunks = (rows + kRowChunk - 1) / kRowChunk;
    const PairSet set = pair_set(orbital, sp, row);
    // The fit shells by angular momentum, and the stored column of every fit function: by angular momentum, then
    // by function of the shell, then by shell.
    std::vector<QShell> fitSorted(fitBasis->shells);
    std::stable_sort(fitSorted.begin(), fitSorted.end(), [](const QShell &u, const QShell &v) { return u.l < v.l; });
    FitLaunch &launch = F->launch;     // records and B differ between the set-up and the fit matrix
    launch.stream = F->stream;
    launch.cut = kUnderFlow;
    launch.oShells = orbital->d_shells;
    launch.oSpherical = orbital->spherical;
    launch.fSpherical = fitBasis->spherical;
    launch.fExps = fitBasis->d_exps;
    launch.fCoefs = fitBasis->d_coefs;
    launch.nFit = F->nFit;
    int *first = launch.first, *column = launch.column;
    F->column.resize(static_cast<size_t>(F->nFit));
    for (int l = 0; l <= kMaxL; l++) {
        int n = 0;
        while (first[l] + n < static_cast<int>(fitSorted.size()) && fitSorted[first[l] + n].l == l) n++;
        const int nf = n > 0 ? fitSorted[first[l]].nf : 0;
        for (int k = 0; k < n; k++)
            for (int m = 0; m < nf; m++) F->column[fitSorted[first[l] + k].f0 + m] = column[l] + m * n + k;
        first[l + 1] = first[l] + n;
        column[l + 1] = column[l] + n * nf;
    }
    PairItem *d_items = nullptr;
    double *d_records = nullptr;
    if (status == kOK) status = qs_alloc(&F->d_B, static_cast<size_t>(rows) * F->nFit);
    if (status == kOK) status = qs_alloc(&F->d_rowPacked, rowPacked.size());
    if (status == kOK) status = qs_alloc(&F->d_rowDiag, rowDiag.size());
    if (status == kOK) status = qs_alloc(&F->d_P, nOrbPacked);
    if (status == kOK) status = qs_alloc(&F->d_F, nOrbPacked);
    if (status == kOK) status = qs_alloc(&F->d_b, F->nFit);
    if (status == kOK) status = qs_alloc(&F->d_c, F->nFit);
    if (status == kOK) status = qs_alloc(&F->d_partial, static_cast<size_t>(nChunks > 0 ? nChunks : 1) * F->nFit);
    if (status == kOK) status = qs_alloc(&d_items, set.items.size());
    if (status == kOK) status = qs_alloc(&d_records, static_cast<size_t>(set.doubles));
    if (status == kOK) status = qs_alloc(&F->d_fitSorted, fitSorted.size());
    if (status == kOK)
        status = check(xq::cache_host_alloc(reinterpret_cast<void **>(&F->staging),
                                            (static_cast<size_t>(F->nFit) + nOrbPacked) * sizeof(double) + 8),
                       "hipHostMalloc");
    if (status == kOK && !fitSorted.empty())
        status = check(hipMemcpy(F->d_fitSorted, fitSorted.data(), fitSorted.size() * sizeof(QShell), hipMemcpyHostToDevice),
                       "copy fit shells");
    launch.fShells = F->d_fitSorted;
    if (status == kOK) status = boys_address(&launch.boys);
    if (status == kOK && rows > 0) {
        status = check(hipMemcpy(F->d_rowPacked, rowPacked.data(), rowPacked.size() * sizeof(long long),
                                 hipMemcpyHostToDevice), "copy rows");
        if (status == kOK) status = check(hipMemcpy(F->d_rowDiag, rowDiag.data(), rowDiag.size(), hipMemcpyHostToDevice),
                                          "copy rows");
        if (status == kOK) status = check(hipMemcpy(d_items, set.items.data(), set.items.size() * sizeof(PairItem),
                                                    hipMemcpyHostToDevice), "copy pairs");
        if (status == kOK && !fitSorted.empty()) status = xq::make_runtime_room("fit integrals");
        if (status == kOK) status = launch_records(orbital, set, d_items, d_records, F->stream);
        launch.records = d_records;
        launch.B = F->d_B;
        if (status == kOK)
            status = for_classes(set, d_items, "fit_integrals_kernel", [&](auto la, auto lb, PairItem *items, int n) {
                launch_fit<la, lb, 0>(launch, items, n);
                launch_fit<la, lb, 1>(launch, items, n);
                launch_fit<la, lb, 2>(launch, items, n);
            });
        const int drained = check(hipStreamSynchronize(F->stream), "fit integrals");
        if (status == kOK) status = drained;
    }
    qs_release(&d_items);
    qs_release(&d_records);
    if (status != kOK) { qs_fit_free(F); return status; }
    *out = F;
    return kOK;
}

int qs_fit_matrix(qs_fit *fit, double *M) {
    if (fit == nullptr || M == nullptr) { set_error("invalid fit matrix arguments"); return kInvalidArgument; }
    const size_t nFit = static_cast<size_t>(fit->nFit), size = (nFit + 1) * (nFit + 2) / 2;
    const qs_basis *basis = fit->fit;
    QBasis withUnit;
    withUnit.shells = basis->shells;
    withUnit.shells.push_back(unit_shell(static_cast<int>(basis->exps.size())));
    // Slabs of consecutive fit shells, whose functions are consecutive rows: the first shell of each, and the end.
    const int nShells = static_cast<int>(basis->shells.size());
    const long long slabRows = std::max<long long>(1, kSlabDoubles / std::max(1, fit->nFit));
    std::vector<int> slab(1, 0);
    long long rows = 0, mostRows = 0;
    for (int k = 0; k < nShells; k++) {
        if (rows > 0 && rows + basis->shells[k].nf > slabRows) {
            slab.push_back(k);
            rows = 0;
        }
        rows += basis->shells[k].nf;
        mostRows = std::max(mostRows, rows);
    }
    slab.push_back(nShells);
    PairItem *d_items = nullptr;
    double *d_records = nullptr, *d_dense = nullptr, *d_M = nullptr;
    int *d_column = nullptr;
    const hipStream_t s = fit->stream;
    int status = qs_alloc(&d_M, size);
    if (status == kOK) status = qs_alloc(&d_dense, static_cast<size_t>(mostRows) * nFit);
    if (status == kOK) status = qs_alloc(&d_column, nFit);
    if (status == kOK && nShells > 0) status = xq::make_runtime_room("fit matrix");
    if (status == kOK) status = check(hipMemcpyAsync(d_column, fit->column.data(), nFit * sizeof(int),
                                                     hipMemcpyHostToDevice, s), "copy columns");
    FitLaunch launch = fit->launch;
    launch.oShells = basis->d_shells;
    launch.oSpherical = basis->spherical;
    launch.cut = -1.0;
    launch.B = d_dense;
    PairSet set;        // one slab after another, each done before the next takes its place
    size_t room[2] = {0, 0};
    for (size_t b = 0; status == kOK && nShells > 0 && b + 1 < slab.size(); b++) {
        if (b > 0) status = check(hipStreamSynchronize(s), "fit matrix");
        if (status != kOK) break;
        // One pair of every fit shell of the slab with the unit shell; a shell's rows are its functions.
        const int k0 = slab[b], k1 = slab[b + 1], p0 = basis->shells[k0].f0,
                  p1 = basis->shells[k1 - 1].f0 + basis->shells[k1 - 1].nf;
        std::vector<QPair> pairs;
        std::vector<long long> row;
        for (int k = k0; k < k1; k++) {
            pairs.push_back(QPair{k, nShells});
            row.push_back(basis->shells[k].f0 - p0);
        }
        set = pair_set(&withUnit, pairs, row);
        status = qs_room(&d_items, &room[0], set.items.size());
        if (status == kOK) status = qs_room(&d_records, &room[1], static_cast<size_t>(set.doubles));
        if (status == kOK) status = check(hipMemcpyAsync(d_items, set.items.data(), set.items.size() * sizeof(PairItem),
                                                         hipMemcpyHostToDevice, s), "copy fit shells");
        if (status == kOK) status = launch_records(basis, set, d_items, d_records, s);
        if (status != kOK) break;
        launch.records = d_records;
        status = for_classes(set, d_items, "fit matrix kernels", [&](auto la, auto lb, PairItem *items, int n) {
            if constexpr (lb == 0) {     // the unit shell is the second of every pair
                launch_fit<la, 0, 0>(launch, items, n);
                launch_fit<la, 0, 1>(launch, items, n);
                launch_fit<la, 0, 2>(launch, items, n);
                hipLaunchKernelGGL(fit_charges_kernel<la>, groups(n, kThreads), dim3(kThreads), 0, s, n, items,
                                   basis->d_shells, basis->d_exps, basis->d_coefs, basis->spherical,
                                   d_M + nFit * (nFit + 1) / 2);
            }
        });
        if (status != kOK) break;
        hipLaunchKernelGGL(fit_matrix_pack_kernel, dim3(static_cast<unsigned>((nFit + 255) / 256),
                                                        static_cast<unsigned>(std::min(p1 - p0, 65535))),
                           dim3(256), 0, s, fit->nFit, p0, p1, d_dense, d_column, d_M);
        status = check(hipGetLastError(), "fit_matrix_pack_kernel");
    }
    const int drained = check(hipStreamSynchronize(s), "fit matrix");
    if (status == kOK) status = drained;
    if (status == kOK) status = check(hipMemcpy(M, d_M, size * sizeof(double), hipMemcpyDeviceToHost), "copy M");
    if (status == kOK) M[size - 1] = 0.0;      // the constraint's own entry
    qs_release(&d_M);
    qs_release(&d_dense);
    qs_release(&d_column);
    qs_release(&d_items);
    qs_release(&d_records);
    return status;
}

int qs_fit_b(qs_fit *fit, const double *P, double *b) {
    if (fit == nullptr || P == nullptr || b == nullptr) { set_error("invalid fit arguments"); return kInvalidArgument; }
    const size_t nPacked = static_cast<size_t>(fit->nOrbital) * (fit->nOrbital + 1) / 2;
    const int nChunks = static_cast<int>((fit->rows + kRowChunk - 1) / kRowChunk);
    if (nChunks == 0) {
        for (int k = 0; k < fit->nFit; k++) b[k] = 0.0;
        return kOK;
    }
    std::lock_guard<std::mutex> lock(fit->step);
    hipStream_t s = fit->stream;
    double *packed = fit->staging + fit->nFit;
    xq::host_copy(packed, P, nPacked);
    auto queue = [&]() -> int {
        XQ_CHECK(hipMemcpyAsync(fit->d_P, packed, nPacked * sizeof(double), hipMemcpyHostToDevice, s));
        hipLaunchKernelGGL(fit_b_partial_kernel, dim3((fit->nFit + 63) / 64, nChunks), dim3(1024), 0, s, fit->rows,
                           fit->nFit, fit->d_B, fit->d_rowPacked, fit->d_rowDiag, fit->d_P, fit->d_partial);
        hipLaunchKernelGGL(fit_b_reduce_kernel, dim3((fit->nFit + 63) / 64), dim3(1024), 0, s, nChunks, fit->nFit,
                           fit->d_partial, fit->d_b);
        XQ_CHECK(hipGetLastError());
        XQ_CHECK(hipMemcpyAsync(fit->staging, fit->d_b, fit->nFit * sizeof(double), hipMemcpyDeviceToHost, s));
        return kOK;
    };
    const int status = queue(), drained = check(hipStreamSynchronize(s), "fit b");
    if (status != kOK) return status;
    if (drained != kOK) return drained;
    for (int k = 0; k < fit->nFit; k++) b[k] = fit->staging[fit->column[k]];
    return kOK;
}

int qs_fit_fock(qs_fit *fit, const double *c, double *Fock) {
    if (fit == nullptr || c == nullptr || Fock == nullptr) { set_error("invalid fit arguments"); return kInvalidArgument; }
    const size_t nPacked = static_cast<size_t>(fit->nOrbital) * (fit->nOrbital + 1) / 2;
    if (fit->rows == 0) return kOK;
    std::lock_guard<std::mutex> lock(fit->step);
    hipStream_t s = fit->stream;
    double *packed = fit->staging + fit->nFit;
    for (int k = 0; k < fit->nFit; k++) fit->staging[fit->column[k]] = c[k];
    // The term is formed from zero and added on the host: F itself does not cross to the GPU.
    auto queue = [&]() -> int {
        XQ_CHECK(hipMemcpyAsync(fit->d_c, fit->staging, fit->nFit * sizeof(double), hipMemcpyHostToDevice, s));
        hipLaunchKernelGGL(zero_packed_kernel, dim3(static_cast<unsigned>(std::min<size_t>((nPacked + 255) / 256, 4096))),
                           dim3(256), 0, s, nPacked, fit->d_F);
        const long long waves = (fit->rows + kFockRows - 1) / kFockRows;
        hipLaunchKernelGGL(fit_fock_kernel, dim3(static_cast<unsigned>((waves * 64 + 255) / 256)), dim3(256), 0, s,
                           fit->rows, fit->nFit, fit->d_B, fit->d_rowPacked, fit->d_c, fit->d_F);
        XQ_CHECK(hipGetLastError());
        XQ_CHECK(hipMemcpyAsync(packed, fit->d_F, nPacked * sizeof(double), hipMemcpyDeviceToHost, s));
        return kOK;
    };
    const int status = queue(), drained = check(hipStreamSynchronize(s), "fit Fock");
    if (status != kOK) return status;
    if (drained != kOK) return drained;
    xq::host_add(Fock, packed, nPacked);
    return kOK;
}

int qs_fit_estimate_bytes(int nAtoms, const int *Z, const double *xyzBohr, int nSpec, const double *spec, int spherical,
                          int nFitSpec, const double *fitSpec, int fitSpherical, long long *bytes) {
    if (bytes == nullptr || nAtoms <= 0 || Z == nullptr || xyzBohr == nullptr || spec == nullptr || nSpec <= 0 ||
        fitSpec == nullptr || nFitSpec <= 0) {
        set_error("invalid fit estimate arguments");
        return kInvalidArgument;
    }
    *bytes = 0;
    QBasis orb, fit;
    for (QBasis *b : {&orb, &fit}) {
        b->nAtoms = nAtoms;
        b->Z.assign(Z, Z + nAtoms);
        b->xyz.assign(xyzBohr, xyzBohr + 3 * nAtoms);
    }
    orb.spherical = spherical ? 1 : 0;
    fit.spherical = fitSpherical ? 1 : 0;
    std::string err = build_shells(&orb, nSpec, spec);
    if (err.empty()) err = build_shells(&fit, nFitSpec, fitSpec);
    if (!err.empty()) { set_error(err); return kInvalidArgument; }
    // The arrays that stay: the integrals (rows x nFit), the row maps, P, F, b, c and the partial sums of b.
    long long rows = 0;
    for (const QPair &pq : shell_pairs(&orb, true))
        rows += static_cast<long long>(orb.shells[pq.x].nf) * orb.shells[pq.y].nf;
    const long long nFit = fit.nFunctions, n = orb.nFunctions, nPacked = n * (n + 1) / 2;
    const long long nChunks = (rows + kRowChunk - 1) / kRowChunk;
    *bytes = 8 * rows * nFit + 9 * rows + 16 * nPacked + 16 * nFit + 8 * (nChunks > 0 ? nChunks : 1) * nFit;
    return kOK;
}

int qs_fit_stats(const qs_fit *fit, long long *rows, long long *pairs, long long *deviceBytes) {
    if (fit == nullptr) { set_error("invalid arguments"); return kInvalidArgument; }
    if (rows) *rows = fit->rows;
    if (pairs) *pairs = fit->nPairs;
    if (deviceBytes) *deviceBytes = fit->rows * static_cast<long long>(fit->nFit) * 8;
    return kOK;
}

}  // extern "C"
