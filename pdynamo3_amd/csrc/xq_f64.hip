// FP64 quadrature on FP64 matrix cores (v_mfma_f64_16x16x4f64), same mathematics as the reference
// (DFTIntegrator.c:159-509, 517-618, 814-901):
//   X = P_red Phi, rho = sum Phi X, grad rho = 2 sum grad Phi X, functional, W = (w vrho / 2) Phi + 2 w vsigma
//   (grad rho . grad Phi), V += Phi W^T + W Phi^T (lower triangle).
// The basis values are stored once per geometry in the lane order the products consume, so every operand load is one
// coalesced 512-byte row per wave.  The kernels follow the mixed path's structure (xq_mixed.hip): a density kernel per row
// chunk of a block with P_red staged in LDS, the functional per block, a per-chunk W kernel, and a Fock kernel over a flat
// list of lower-triangle tiles with FP64 atomics; all read the same job table, so one launch serves one job or a batch.
//
// MFMA lane layout (16 x 16 x 4, FP64): lane l supplies A[l % 16][l / 16] and B[l / 16][l % 16] and receives
// D[4 v + l / 16][l % 16] for v = 0..3.
//
// Layouts (4096 doubles per chunk of 32 kept functions x 128 points; chunk C is chunk rc of block b):
//   FPB, GPB [C][g (4)][s (8)][h (2)][lane (64)]   Phi and grad Phi (GPB: 3 planes) in the density's B operand order:
//                                                  lane l holds row 4 s + l / 16 at point 32 g + 16 h + l % 16.  The
//                                                  density result register v of row half hm and point half hn is row
//                                                  16 hm + 4 v + l / 16, which is the operand entry (s = 4 hm + v, hn).
//   FPA, WPA [C][s (32)][h (2)][lane (64)]         Phi and W (per step) in the Fock product's A/B order: lane l holds
//                                                  row 16 h + l % 16 at point 4 s + l / 16.
#include <hip/hip_runtime.h>

#include <climits>
#include <type_traits>
#include <vector>

#include "xq_functional.h"
#include "xq_internal.h"

namespace xq {

typedef double v4d __attribute__((ext_vector_type(4)));

namespace {

constexpr int kC = 32;                   // chunk rows
constexpr int kChunk = 4096;             // doubles per chunk plane
// LDS row pitch of a staged P_red chunk in doubles: odd, so that the operands' 16 rows lie in different banks (39: two rows
// being written as well).  With 36, whose rows met in four banks, the density rows took 3.62 ms on (H2O)64, now 3.51.
constexpr int kRowPitch = kC + 7;
constexpr int kIdxCache = 1024;          // kept-function indices of a block cached in LDS by the density kernel

__device__ __forceinline__ v4d mfma_f64(double a, double b, const v4d &c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

template <typename F>
__device__ __forceinline__ int job_of(const MixedJob *jobs, int nJobs, int g, F base) {
    int lo = 0, hi = nJobs - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (base(jobs[mid]) <= g) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Set-up, once per geometry: one chunk per work-group (256 threads) from the FP64 rows of f, fx, fy, fz.
__global__ void __launch_bounds__(256) f64_prepare_kernel(
    const DevBlock *__restrict__ blocks, const int *__restrict__ chunkOffset, const int *__restrict__ chunkBlock,
    const double *__restrict__ f, const double *__restrict__ fx, const double *__restrict__ fy,
    const double *__restrict__ fz, double *__restrict__ FPB, double *__restrict__ GPB, double *__restrict__ FPA) {
    const size_t C = blockIdx.x;
    const int b = chunkBlock[C];
    const DevBlock blk = blocks[b];
    const int nb = blk.nKept, rc = static_cast<int>(C) - chunkOffset[b];
    const size_t R = static_cast<size_t>(blk.vOffset);
    auto value = [&](const double *a, int r, int p) -> double {
        const int row = kC * rc + r;
        return row < nb ? a[(R + row) * kBlockSize + p] : 0.0;
    };
    for (int e = threadIdx.x; e < kChunk; e += 256) {
        const int lane = e & 63, h = (e >> 6) & 1, s = (e >> 7) & 7, g = e >> 10;
        const int r = 4 * s + (lane >> 4), p = 32 * g + 16 * h + (lane & 15);
        FPB[C * kChunk + e] = value(f, r, p);
        GPB[(3 * C) * kChunk + e] = value(fx, r, p);
        GPB[(3 * C + 1) * kChunk + e] = value(fy, r, p);
        GPB[(3 * C + 2) * kChunk + e] = value(fz, r, p);
        const int lane2 = e & 63, h2 = (e >> 6) & 1, s2 = e >> 7;
        FPA[C * kChunk + e] = value(f, 16 * h2 + (lane2 & 15), 4 * s2 + (lane2 >> 4));
    }
}

// Density rows (one row chunk I of one block per work-group, 256 threads = 4 waves; wave wv owns points 32 wv .. + 31):
// X = P_red Phi for the chunk's 32 rows on FP64 MFMA (2 x 2 MFMA tiles per wave), then the chunk's share of rho and grad rho
// at the block's points, stored in part[chunk][4][point]; density_functional_kernel (xq_mixed.hip) sums the shares.  Each
// step multiplies one 32 x 32 chunk of P_red, gathered by all threads and staged in one of two LDS buffers (one barrier per
// step), with the matching Phi chunk, whose operands go straight to registers; the words of P_red are fetched one step
// ahead, and each Phi operand for the next step as soon as its products of this step are issued, into the same registers:
// four work-groups per CU instead of three with a second set of operand registers (3.62 ms against 4.13 then).  The row
// chunks of a block are consecutive items of one XCD, so that Phi comes from HBM about once per block.
// Bound by HBM (Phi and grad Phi once, 10.7 GB on (H2O)64, and the gathers of P_red) and the FP64 matrix cores (busy for
// half of the time).  One work-group per block, which read Phi once per row chunk from HBM and waited for each panel of
// gathers, took 8.26 ms on (H2O)64 (1.3e11 operations); this takes 3.51 ms and the functional 0.21 ms.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
density_rows_kernel_f64(const MixedJob *__restrict__ jobs, int nJobs, int interleaved) {
    __shared__ double sP[2][kC][kRowPitch];
    __shared__ int sIdx[kIdxCache];
    // Work-group g runs on XCD x = g % 8 and takes slot g / 8 of that XCD's item list, as the mixed density rows.
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const MixedJob &J = interleaved ? jobs[slot & 1]
                                    : jobs[job_of(jobs, nJobs, slot, [xcd](const MixedJob &j) { return j.itemBase[xcd]; })];
    const int local = interleaved ? slot >> 1 : slot - J.itemBase[xcd];
    if (local >= J.itemStart[xcd + 1] - J.itemStart[xcd]) return;
    // {chunk, kept functions x 1024 + row chunk, first kept index, block}.
    const int4 ent = J.items[J.itemStart[xcd] + local];
    const size_t CI = static_cast<size_t>(ent.x);
    const int nb = ent.y >> 10, I = ent.y & 1023, n = J.n;
    const size_t C = CI - I;
    const int nChunks = (nb + kC - 1) / kC;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, l16 = lane & 15, l4 = lane >> 4;
    // The block's kept-function indices, cached in LDS for the P_red gathers (blocks with more kept functions than the
    // cache read them from memory).
    const int *idxG = J.idx + ent.z;
    for (int k = t; k < nb && k < kIdxCache; k += 256) sIdx[k] = idxG[k];
    __syncthreads();
    const int *idx = nb <= kIdxCache ? sIdx : idxG;
    const double *__restrict__ P = J.P;
    const double *__restrict__ FPB = J.FPB;
    const double *__restrict__ GPB = J.GPB;
    // Operand entry (s, h) of this lane within a chunk plane of FPB / GPB.
    auto op = [&](int s, int h) { return ((wv * 8 + s) * 2 + h) * 64 + lane; };
    // Staging: row sr, columns 8 j + s8 (eight lanes read eight consecutive kept functions).
    const int sr = t >> 3, s8 = t & 7, r = kC * I + sr;
    const size_t rowOff = r < nb ? static_cast<size_t>(idx[r]) * n : 0;
    double pv[4], bq[8][2];
    auto fetch_p = [&](int c) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int k = kC * c + 8 * j + s8;
            pv[j] = r < nb && k < nb ? P[rowOff + idx[k]] : 0.0;
        }
    };
    const double *__restrict__ bp = FPB + C * kChunk + op(0, 0);    // operands of the chunk to fetch
    auto fetch_b = [&](int s) {
#pragma unroll
        for (int h = 0; h < 2; h++) bq[s][h] = bp[(2 * s + h) * 64];
    };
    v4d acc[2][2];
#pragma unroll
    for (int hm = 0; hm < 2; hm++)
#pragma unroll
        for (int hn = 0; hn < 2; hn++) acc[hm][hn] = v4d{0.0, 0.0, 0.0, 0.0};
    auto step = [&](int c, auto more) {
        double (&buf)[kC][kRowPitch] = sP[c & 1];
#pragma unroll
        for (int j = 0; j < 4; j++) buf[sr][8 * j + s8] = pv[j];
        // A wave writes this buffer again two steps on, after the next barrier, which every wave reaches done with it.
        __syncthreads();
        if constexpr (more) {
            fetch_p(c + 1);
            bp += kChunk;
        }
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const double a0 = buf[l16][4 * s + l4], a1 = buf[16 + l16][4 * s + l4];
            acc[0][0] = mfma_f64(a0, bq[s][0], acc[0][0]);
            acc[0][1] = mfma_f64(a0, bq[s][1], acc[0][1]);
            acc[1][0] = mfma_f64(a1, bq[s][0], acc[1][0]);
            acc[1][1] = mfma_f64(a1, bq[s][1], acc[1][1]);
            if constexpr (more) fetch_b(s);
        }
    };
    fetch_p(0);
#pragma unroll
    for (int s = 0; s < 8; s++) fetch_b(s);
#pragma unroll 1
    for (int c = 0; c + 1 < nChunks; c++) step(c, std::true_type{});
    step(nChunks - 1, std::false_type{});
    // Epilogue: register v of (hm, hn) is row 16 hm + 4 v + l / 16 of chunk I at point 32 wv + 16 hn + l % 16.
    double *q = J.part + CI * 4 * kBlockSize;
#pragma unroll 1
    for (int x = 0; x < 4; x++) {
        const double *__restrict__ plane = (x == 0 ? FPB + CI * kChunk : GPB + (3 * CI + (x - 1)) * kChunk) + op(0, 0);
        double pr[2] = {};
#pragma unroll
        for (int hm = 0; hm < 2; hm++)
#pragma unroll
            for (int v = 0; v < 4; v++)
#pragma unroll
                for (int hn = 0; hn < 2; hn++) pr[hn] += plane[(2 * (4 * hm + v) + hn) * 64] * acc[hm][hn][v];
        // Sum over the four lanes that share a point (l / 16 = 0..3).
#pragma unroll
        for (int hn = 0; hn < 2; hn++) {
            double e = pr[hn];
            e += __shfl_xor(e, 16, 64);
            e += __shfl_xor(e, 32, 64);
            if (l4 == 0) q[x * kBlockSize + kC * wv + 16 * hn + l16] = e;
        }
    }
}

// W (one chunk per work-group, 256 threads): W_rp = c0_p Phi_rp + c_p . grad Phi_rp from the density-order planes,
// transposed through LDS into the Fock order (WPA).
__global__ void __launch_bounds__(256) w_kernel_f64(const MixedJob *__restrict__ jobs, int nJobs) {
    __shared__ double sc[4][kBlockSize];
    __shared__ double sW[kC][kBlockSize + 1];
    const MixedJob &J = jobs[job_of(jobs, nJobs, blockIdx.x, [](const MixedJob &j) { return j.chunkBase; })];
    const size_t C = blockIdx.x - J.chunkBase;
    const int b = J.chunkBlock[C];
    if (J.skip[b]) return;
    const DevBlock blk = J.blocks[b];
    const int t = threadIdx.x;
    if (t < kBlockSize) {
#pragma unroll
        for (int k = 0; k < 4; k++) sc[k][t] = t < blk.nPoints ? J.wcoef[4 * (static_cast<size_t>(blk.pStart) + t) + k] : 0.0;
    }
    __syncthreads();
    for (int e = t; e < kChunk; e += 256) {
        const int lane = e & 63, h = (e >> 6) & 1, s = (e >> 7) & 7, g = e >> 10;
        const int r = 4 * s + (lane >> 4), p = 32 * g + 16 * h + (lane & 15);
        sW[r][p] = sc[0][p] * J.FPB[C * kChunk + e] + sc[1][p] * J.GPB[3 * C * kChunk + e] +
                   sc[2][p] * J.GPB[(3 * C + 1) * kChunk + e] + sc[3][p] * J.GPB[(3 * C + 2) * kChunk + e];
    }
    __syncthreads();
    for (int e = t; e < kChunk; e += 256) {
        const int lane = e & 63, h = (e >> 6) & 1, s = e >> 7;
        J.WPA[C * kChunk + e] = sW[16 * h + (lane & 15)][4 * s + (lane >> 4)];
    }
}

// The sums over a block's 128 points of one 32 x 32 tile, 32 steps of 4 points: Phi_I W_J^T, and, off the diagonal,
// W_I Phi_J^T as well (on it that is the transpose).  Operands are fetched four steps ahead, each into the registers of the
// one whose products have just been issued.
template <bool kDiagonal>
__device__ __forceinline__ void fock_tile_f64(const double *__restrict__ fI, const double *__restrict__ wI,
                                              const double *__restrict__ fJ, const double *__restrict__ wJ,
                                              v4d (&acc)[2][2]) {
    constexpr int kAhead = 4;
    double xf[kAhead][2], xw[kAhead][2], yf[kAhead][2], yw[kAhead][2];
    auto load = [&](int k) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int o = (2 * k + h) * 64;
            xf[k][h] = fI[o];
            yw[k][h] = wJ[o];
            if constexpr (!kDiagonal) {
                xw[k][h] = wI[o];
                yf[k][h] = fJ[o];
            }
        }
    };
    auto products = [&](int k) {
#pragma unroll
        for (int hm = 0; hm < 2; hm++)
#pragma unroll
            for (int hn = 0; hn < 2; hn++) {
                acc[hm][hn] = mfma_f64(xf[k][hm], yw[k][hn], acc[hm][hn]);
                if constexpr (!kDiagonal) acc[hm][hn] = mfma_f64(xw[k][hm], yf[k][hn], acc[hm][hn]);
            }
    };
#pragma unroll
    for (int k = 0; k < kAhead; k++) load(k);
#pragma unroll 1
    for (int s = kAhead; s < kBlockSize / 4; s += kAhead) {
        fI += 2 * 64 * kAhead;
        wI += 2 * 64 * kAhead;
        fJ += 2 * 64 * kAhead;
        wJ += 2 * 64 * kAhead;
#pragma unroll
        for (int k = 0; k < kAhead; k++) {
            products(k);
            load(k);
        }
    }
#pragma unroll
    for (int k = 0; k < kAhead; k++) products(k);
}

// Fock kernel: one wave per lower-triangle tile (I, J <= I), four tiles per work-group, no barriers.
// V += Phi_I W_J^T + W_I Phi_J^T with FP64 atomics; on a diagonal tile the second term is the first one's transpose, taken
// through LDS.  Work-group g runs on XCD g % 8; tiles are dealt so that each XCD takes a contiguous range of the tile list.
// Bound by the FP64 matrix cores and the atomics, which go to memory.  Groups of four steps whose loads were each waited
// for, and both products on the diagonal, took 3.99 and 4.03 ms in two runs on (H2O)64 and 27 us on one water; this takes
// 3.87 and 3.72 ms on the same box and 19 us (four waves per SIMD; three took 3% more).
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) fock_kernel_f64(const MixedJob *__restrict__ jobs, int nJobs, int groupsPerXcd,
                                                       int nGroups) {
    __shared__ double sT[4][kC][kC + 1];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6, l16 = lane & 15, l4 = lane >> 4;
    const int group = (blockIdx.x & 7) * groupsPerXcd + (blockIdx.x >> 3);
    if (group >= nGroups) return;
    const MixedJob &job = jobs[job_of(jobs, nJobs, group, [](const MixedJob &j) { return j.groupBase; })];
    const int tileIndex = 4 * (group - job.groupBase) + wv;
    if (tileIndex >= job.nTiles) return;
    const int4 tl = job.tiles[tileIndex];
    const int b = tl.x, I = tl.y, J = tl.z;
    if (job.skip[b]) return;
    const DevBlock blk = job.blocks[b];
    const int nb = blk.nKept;
    const int *idx = job.idx + blk.iOffset;
    const size_t CI = static_cast<size_t>(job.chunkOffset[b] + I), CJ = static_cast<size_t>(job.chunkOffset[b] + J);
    const double *fI = job.FPA + CI * kChunk + lane, *wI = job.WPA + CI * kChunk + lane;
    const double *fJ = job.FPA + CJ * kChunk + lane, *wJ = job.WPA + CJ * kChunk + lane;
    v4d acc[2][2];
#pragma unroll
    for (int hm = 0; hm < 2; hm++)
#pragma unroll
        for (int hn = 0; hn < 2; hn++) acc[hm][hn] = v4d{0.0, 0.0, 0.0, 0.0};
    if (I != J) {
        fock_tile_f64<false>(fI, wI, fJ, wJ, acc);
    } else {
        fock_tile_f64<true>(fI, wI, fJ, wJ, acc);
        double (&T)[kC][kC + 1] = sT[wv];
#pragma unroll
        for (int hm = 0; hm < 2; hm++)
#pragma unroll
            for (int hn = 0; hn < 2; hn++)
#pragma unroll
                for (int v = 0; v < 4; v++) T[16 * hm + 4 * v + l4][16 * hn + l16] = acc[hm][hn][v];
        // The wave's LDS accesses are in order; this keeps the compiler from moving them.
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int hm = 0; hm < 2; hm++)
#pragma unroll
            for (int hn = 0; hn < 2; hn++)
#pragma unroll
                for (int v = 0; v < 4; v++) acc[hm][hn][v] += T[16 * hn + l16][16 * hm + 4 * v + l4];
    }
    const int n = job.n;
#pragma unroll
    for (int hn = 0; hn < 2; hn++) {
        const int gj = kC * J + 16 * hn + l16;
        if (gj >= nb) continue;
        const size_t col = static_cast<size_t>(idx[gj]);
#pragma unroll
        for (int hm = 0; hm < 2; hm++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int gi = kC * I + 16 * hm + 4 * v + l4;
                if (gi < nb && gj <= gi) atomicAdd(&job.V[static_cast<size_t>(idx[gi]) * n + col], acc[hm][hn][v]);
            }
    }
}

}  // namespace

int prepare_f64(xq_grid *g, const double *f, const double *fx, const double *fy, const double *fz) {
    XQ_TRY(chunk_tables(g));
    const size_t nc = static_cast<size_t>(g->nChunks > 0 ? g->nChunks : 1);
    XQ_TRY(dev_alloc(g, &g->d_FPB, nc * kChunk));
    XQ_TRY(dev_alloc(g, &g->d_GPB, 3 * nc * kChunk));
    XQ_TRY(dev_alloc(g, &g->d_FPA, nc * kChunk));
    XQ_TRY(dev_alloc(g, &g->d_WPA, nc * kChunk));
    XQ_TRY(dev_alloc(g, &g->d_wcoef, 4 * static_cast<size_t>(g->nPoints > 0 ? g->nPoints : 1)));
    XQ_TRY(dev_alloc(g, &g->d_part, nc * 4 * kBlockSize));
    hipStream_t s = g->stream;
    if (g->nChunks > 0)
        hipLaunchKernelGGL(f64_prepare_kernel, dim3(static_cast<unsigned>(g->nChunks)), dim3(256), 0, s, g->d_blocks,
                           g->d_chunkOffset, g->d_chunkBlock, f, fx, fy, fz, g->d_FPB, g->d_GPB, g->d_FPA);
    XQ_CHECK(hipGetLastError());
    XQ_CHECK(hipStreamSynchronize(s));
    return kOK;
}

// Per-step arrays of a second job on the handle (the beta spin of an unrestricted quadrature): W planes and the density's
// row-chunk shares.  Complete or released.
int alloc_step_f64(xq_grid *g, StepArrays *a) {
    const size_t nc = static_cast<size_t>(g->nChunks > 0 ? g->nChunks : 1);
    int status = dev_alloc(g, &a->WPA, nc * kChunk);
    if (status == kOK) status = dev_alloc(g, &a->part, nc * 4 * kBlockSize);
    if (status != kOK) free_step_f64(g, a);
    return status;
}

void free_step_f64(xq_grid *g, StepArrays *a) {
    dev_free(g, &a->WPA);
    dev_free(g, &a->part);
}

void free_f64(xq_grid *g) {
    dev_free(g, &g->d_FPB);
    dev_free(g, &g->d_GPB);
    dev_free(g, &g->d_FPA);
    dev_free(g, &g->d_WPA);
}

int launch_f64(hipStream_t s, const StageEvents &ev, int nJobs, xq_grid *const *grids, const FunctionalSet *fs,
               MixedJob *h_table, MixedJob *d_table, int stages, const StepArrays *over) {
    long long rows, blocks, chunks, groups, itemSlots;
    fill_jobs(nJobs, grids, fs, h_table, &rows, &blocks, &chunks, &groups, over, &itemSlots);
    if (blocks > INT32_MAX / 2 || chunks > INT32_MAX / 2 || groups > INT32_MAX / 16 || itemSlots > INT32_MAX / 16) {
        set_error("batch too large for one launch");
        return kInvalidArgument;
    }
    XQ_CHECK(hipMemcpyAsync(d_table, h_table, nJobs * sizeof(MixedJob), hipMemcpyHostToDevice, s));
    XQ_CHECK(hipEventRecord(ev.evRho0, s));
    if ((stages & kStageDensity) && blocks > 0) {
        // The two spins of one handle (an unrestricted quadrature) run interleaved item by item.
        const int interleaved = nJobs == 2 && grids[0] == grids[1] ? 1 : 0;
        if (itemSlots > 0)
            hipLaunchKernelGGL(density_rows_kernel_f64, dim3(static_cast<unsigned>(8 * itemSlots)), dim3(256), 0, s, d_table,
                               nJobs, interleaved);
        launch_density_functional(s, nJobs, blocks, h_table[0].rhoOut != nullptr, d_table);
    }
    XQ_CHECK(hipEventRecord(ev.evDens1, s));
    XQ_CHECK(hipEventRecord(ev.evRho1, s));
    if ((stages & kStageFock) && chunks > 0) {
        hipLaunchKernelGGL(w_kernel_f64, dim3(static_cast<unsigned>(chunks)), dim3(256), 0, s, d_table, nJobs);
        const int perXcd = static_cast<int>((groups + 7) / 8);
        hipLaunchKernelGGL(fock_kernel_f64, dim3(static_cast<unsigned>(8 * perXcd)), dim3(256), 0, s, d_table, nJobs,
                           perXcd, static_cast<int>(groups));
    }
    XQ_CHECK(hipEventRecord(ev.evFock1, s));
    XQ_CHECK(hipGetLastError());
    return kOK;
}

}  // namespace xq
