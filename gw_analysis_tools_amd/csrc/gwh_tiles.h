/*
 * gwh_tiles.h -- the per-bin network log-likelihood kernels: one (instance, tile) work item per block, a tile of
 * TPB lanes x BPL bins per lane (TPB in 64..1024, BPL in 1..8, chosen per event: fixed default or autotuned).
 * Included by the engine (declarations, the block reduction and the work map) and by the three translation units that
 * instantiate the kernels of one (model, precision) each (IMRPhenomPv2 runs in FP64 in both modes), so the 75 kernels
 * compile in parallel.
 */
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

#include "gwh_engine.h"

/* ------------------------------------------------------------------------- */
/* reductions                                                                 */
/* ------------------------------------------------------------------------- */

/* Block-reduce NV values per thread of a TPB-lane block (fixed order) and write them to out[0..nv); a one-wave
 * block writes its wave sums directly.  The block's LDS is not reused afterwards (no closing barrier). */
template <int NV, int TPB = GWH_TPB>
__device__ __forceinline__ void block_reduce_store(double (&acc)[NV], double *__restrict__ out, double (*lds)[NV],
                                                   int nv = NV)
{
    int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int j = 0; j < NV; j++)
        if (j < nv) acc[j] = wave_sum(acc[j]); /* nv is uniform: unused slots are skipped, not masked */
    if (TPB == 64) {
        if (lane == 0) {
#pragma unroll
            for (int j = 0; j < NV; j++)
                if (j < nv) out[j] = acc[j];
        }
        return;
    }
    if (lane == 0) {
#pragma unroll
        for (int j = 0; j < NV; j++) lds[wv][j] = acc[j];
    }
    __syncthreads();
    if ((int)threadIdx.x < nv) {
        int j = threadIdx.x;
        double s = lds[0][j];
        for (int w = 1; w < TPB / 64; w++) s += lds[w][j];
        out[j] = s;
    }
}


/* ------------------------------------------------------------------------- */
/* the batched likelihood kernels                                             */
/* ------------------------------------------------------------------------- */

/* One (instance, tile) work item: TPB lanes x BPL bins of one instance's network log-likelihood, reduced
 * to the instance's partial sums for that tile.  Every early return is uniform over the block.
 * ANY: an item of a work list, whose event has TPB lanes and any number of bins per lane up to BPL = 8 (the unrolled
 * steps past it are skipped). */
template <int MODEL, int PREC, int BPL, int TPB, bool ANY = false>
__device__ __forceinline__ void gwh_loglike_tile(const WorkMap &W, const EventDesc *__restrict__ events,
                                                 const InstCoef *__restrict__ coefs, double *__restrict__ partial,
                                                 const int *__restrict__ active, const int ev, const int inst, const int tile,
                                                 double (*lds)[GWH_PARTIAL_STRIDE], double2 *__restrict__ tab,
                                                 double *__restrict__ etab)
{
    {
        const EventDesc &E = events[ev];
        if (!ANY && (E.bpl != BPL || E.lanes != TPB)) return; /* the instance's event is tiled by another launch */
        if (!ANY && tile >= active[inst]) return; /* above 0.2/M on an ascending grid: h = 0, nothing to add */
        const int bpl = ANY ? E.bpl : BPL;
        const int w = inst * W.tiles0 + tile;
        const InstCoef &C = coefs[inst];
        const int N = E.N, D = E.D;
        double acc[GWH_PARTIAL_STRIDE];
#pragma unroll
        for (int j = 0; j < GWH_PARTIAL_STRIDE; j++) acc[j] = 0;
        /* skip tiles entirely above the 0.2/M cutoff (h = 0 there, IMRPhenomD.cpp:475) */
        const int level = ANY ? gwh_tile_level(TPB) + (__ffs(bpl) - 1) : gwh_tile_level(TPB * BPL);
        const double fmin_tile = gwh_g(E.tile_fmin)[E.fmin_off[level] + tile];
        if (!(fmin_tile > C.fcut)) {
            /* the sin/cos and exponential tables in LDS: the detector phases (one gather per detector and bin), the
               merger-ringdown arctangent's correction and exponential and the IMRPhenomPv2 Euler angle read them
               there instead of through the vector memory path */
            for (int q = threadIdx.x; q < 256; q += TPB) tab[q] = gwh_turn_table[q];
            if (threadIdx.x < 64) etab[threadIdx.x] = gwh_exp2_table[threadIdx.x];
            __syncthreads();
#pragma unroll
            for (int j = 0; j < BPL; j++) {
                if (ANY && j >= bpl) break;
                /* Lanes past the end of the grid or above 0.2/M evaluate the last grid bin with a zero amplitude
                 * (and phase), so the accumulators never sit under divergent control flow; a wave without any
                 * bin at or below the cutoff skips the step on a uniform branch. */
                const int k0 = tile * TPB * bpl + j * TPB + threadIdx.x;
                const bool in = k0 < N;
                const int k = in ? k0 : N - 1;
                const double f = gwh_g(E.f)[k];
                const bool live = in && f <= C.fcut;
                if (!__ballot(live)) continue;
                const BinPow bp = gwh_load_bin(E, k);
                if (MODEL == GWH_IMRPHENOMD) {
                    double a, phi, u;
                    /* mixed: the merger-ringdown exponential in FP32, everything else as FP64 */
                    gwh_phenomd_fp64<PREC == GWH_MIXED>(C, f, bp, a, phi, u, tab, etab);
                    a = live ? a : 0.0;
                    phi = live ? phi : 0.0;
#pragma unroll
                    for (int d = 0; d < GWH_MAXDET; d++) {
                        if (d >= D) break;
                        double s, c;
                        gwh_sincos_tab(phi + C.det[d][3] * f, s, c, tab);
                        const double ws = gwh_g(E.wS)[(size_t)d * N + k];
                        const double2 dw = gwh_ld2(E.dwS, (size_t)d * N + k);
                        acc[3 * d] += a * a * ws;
                        acc[3 * d + 1] += a * (c * dw.x - s * dw.y);
                        acc[3 * d + 2] += a * (c * dw.y + s * dw.x);
                    }
                } else {
                    double A, Phi, hpr, hpi, hcr, hci;
                    gwh_pv2_fp64(C, f, bp, A, Phi, hpr, hpi, hcr, hci, tab, etab);
                    A = live ? A : 0.0;
                    Phi = live ? Phi : 0.0;
#pragma unroll
                    for (int d = 0; d < GWH_MAXDET; d++) {
                        if (d >= D) break;
                        const double P = C.det[d][0], Q = C.det[d][1];
                        const double Gr = P * hpr + Q * hcr, Gi = P * hpi + Q * hci;
                        double s, c;
                        gwh_sincos_tab(Phi + C.det[d][3] * f, s, c, tab);
                        const double ws = gwh_g(E.wS)[(size_t)d * N + k];
                        const double2 dw = gwh_ld2(E.dwS, (size_t)d * N + k);
                        acc[3 * d] += A * A * (Gr * Gr + Gi * Gi) * ws;
                        acc[3 * d + 1] += A * (dw.x * (Gr * c + Gi * s) - dw.y * (Gr * s - Gi * c));
                    }
                }
            }
        }
        block_reduce_store<GWH_PARTIAL_STRIDE, TPB>(acc, partial + (size_t)w * GWH_PARTIAL_STRIDE, lds, 3 * D);
    }
}

/* the flattened (instance, tile) work list of one number of lanes per tile (gwh_worklist_kernel): one block per live
 * work item, so batches mixing 10^3- and 10^5-bin events launch no empty blocks; entries fold over y beyond 2^20
 * blocks */
template <int MODEL, int PREC, int TPB>
__global__ __launch_bounds__(TPB) void gwh_loglike_wl_kernel(WorkMap W, const EventDesc *__restrict__ events,
                                                             const InstCoef *__restrict__ coefs,
                                                             double *__restrict__ partial,
                                                             const int2 *__restrict__ work,
                                                             const int *__restrict__ count)
{
    __shared__ double lds[TPB / 64][GWH_PARTIAL_STRIDE];
    __shared__ double2 tab[256];
    __shared__ double etab[64];
    const int w = blockIdx.y * gridDim.x + blockIdx.x;
    if (w >= *count) return;
    const int2 wi = work[w];
    if (wi.x < 0) return; /* a hole at the end of a column */
    gwh_loglike_tile<MODEL, PREC, 8, TPB, true>(W, events, coefs, partial, nullptr, wi.x >> 16, wi.x & 0xffff, wi.y, lds,
                                                tab, etab);
}

/* One block per (instance, tile) item, in tile-major order (item w = tile * n + instance).  Consecutive blocks go
 * to different XCDs, so the instances of every tile spread over all XCDs; in instance-major order tile t of every
 * instance would land on the same XCD, and the tiles below an instance's 0.2/M cutoff -- the only ones with work --
 * on a few XCDs.  Items above the cutoff cost one load.  count (optional, device): only instances i < *count are
 * visited, so a launch sized for the largest possible count costs little when the count is small.
 * One item per block rather than a resident grid striding over the items: with a loop around the item the compiler
 * keeps loop-invariant values (constants of the polynomial chains, lane offsets) in registers across iterations,
 * which doubles the kernel's VGPRs (IMRPhenomD 66 -> 134, IMRPhenomPv2 90 -> 165) and halves the waves a SIMD
 * holds (7 -> 3 or 4); the results are bit-identical either way (512 instances on 16225 bins: FP64 IMRPhenomD
 * 36.4 -> 30.4 us, IMRPhenomPv2 60.6 -> 52.8 / mixed 58.2 -> 49.7 us). */
template <int MODEL, int PREC, int BPL, int TPB>
__global__ __launch_bounds__(TPB) void gwh_loglike_grid_kernel(WorkMap W, const EventDesc *__restrict__ events,
                                                               const InstCoef *__restrict__ coefs,
                                                               double *__restrict__ partial,
                                                               const int *__restrict__ active,
                                                               const int *__restrict__ count)
{
    __shared__ double lds[TPB / 64][GWH_PARTIAL_STRIDE];
    __shared__ double2 tab[256];
    __shared__ double etab[64];
    const int nn = count ? min(*count, W.n) : W.n;
    const int w = blockIdx.y * gridDim.x + blockIdx.x; /* items fold over y beyond 2^20 blocks */
    if (nn <= 0 || w >= nn * W.tiles0) return;
    const int inst = w % nn;
    gwh_loglike_tile<MODEL, PREC, BPL, TPB>(W, events, coefs, partial, active, W.inst_event ? W.inst_event[inst] : W.event0,
                                            inst, w / nn, lds, tab, etab);
}

/* ------------------------------------------------------------------------- */
/* launch of one tiling class                                                 */
/* ------------------------------------------------------------------------- */

/* a dispatch counts work-items in 32 bits per dimension: at most 2^20 blocks along x */
static inline dim3 gwh_tile_grid(long long items)
{
    const long long gx = std::max(1LL, std::min(items, 1LL << 20)), gy = std::max(1LL, (items + gx - 1) / gx);
    return dim3((unsigned)gx, (unsigned)gy);
}

template <int MODEL, int PREC, int TPB>
static void gwh_launch_tiles_lanes(int bpl, long long items, hipStream_t st, const WorkMap &W, const EventDesc *ev,
                                   const InstCoef *c, double *part, const int *act, const int *count)
{
    const dim3 g = gwh_tile_grid(items), b(TPB);
#define GWH_GRID(BPL) hipLaunchKernelGGL((gwh_loglike_grid_kernel<MODEL, PREC, BPL, TPB>), g, b, 0, st, W, ev, c, part, act, count)
    switch (bpl) {
    case 1: GWH_GRID(1); break;
    case 2: GWH_GRID(2); break;
    case 4: GWH_GRID(4); break;
    default: GWH_GRID(8); break;
    }
#undef GWH_GRID
}

/* The per-bin kernel of one tiling class (bpl bins per lane x lanes per tile) over a batch on one event tiling: one
 * block per (instance, tile) item (items = n x tiles; count = the optional device instance count).  Each (MODEL, PREC)
 * is instantiated in its own translation unit (gwh_tiles_*.hip). */
template <int MODEL, int PREC>
void gwh_launch_tiles(int bpl, int lanes, long long items, hipStream_t st, const WorkMap &W, const EventDesc *ev,
                      const InstCoef *c, double *part, const int *act, const int *count)
{
    switch (lanes) {
    case 64: gwh_launch_tiles_lanes<MODEL, PREC, 64>(bpl, items, st, W, ev, c, part, act, count); break;
    case 128: gwh_launch_tiles_lanes<MODEL, PREC, 128>(bpl, items, st, W, ev, c, part, act, count); break;
    case 512: gwh_launch_tiles_lanes<MODEL, PREC, 512>(bpl, items, st, W, ev, c, part, act, count); break;
    case 1024: gwh_launch_tiles_lanes<MODEL, PREC, 1024>(bpl, items, st, W, ev, c, part, act, count); break;
    default: gwh_launch_tiles_lanes<MODEL, PREC, 256>(bpl, items, st, W, ev, c, part, act, count); break;
    }
}

/* The per-bin kernel over a work list of one number of lanes per tile: one block per entry (items = the list's upper
 * bound; count = its device length). */
template <int MODEL, int PREC>
void gwh_launch_worklist(int lanes, long long items, const int2 *work, hipStream_t st, const WorkMap &W,
                         const EventDesc *ev, const InstCoef *c, double *part, const int *count)
{
    const dim3 g = gwh_tile_grid(items);
#define GWH_WL(TPB) hipLaunchKernelGGL((gwh_loglike_wl_kernel<MODEL, PREC, TPB>), g, dim3(TPB), 0, st, W, ev, c, part, work, count)
    switch (lanes) {
    case 64: GWH_WL(64); break;
    case 128: GWH_WL(128); break;
    case 512: GWH_WL(512); break;
    case 1024: GWH_WL(1024); break;
    default: GWH_WL(256); break;
    }
#undef GWH_WL
}
/* Load the code object holding the kernels of one (MODEL, PREC) on the current device: the runtime loads a
 * translation unit's kernels at the first use of any of them, a few milliseconds that would otherwise fall on the
 * first likelihood launch (and on a serving loop's first request). */
template <int MODEL, int PREC> int gwh_tiles_load()
{
    hipFuncAttributes a;
    return hipFuncGetAttributes(&a, reinterpret_cast<const void *>(&gwh_loglike_grid_kernel<MODEL, PREC, 8, 256>)) ==
                   hipSuccess
               ? 0
               : -1;
}
#define GWH_TILES_DECLARE(M, P)                                                                                    \
    extern template void gwh_launch_tiles<M, P>(int, int, long long, hipStream_t, const WorkMap &,                  \
                                                const EventDesc *, const InstCoef *, double *, const int *,         \
                                                const int *);                                                       \
    extern template void gwh_launch_worklist<M, P>(int, long long, const int2 *, hipStream_t, const WorkMap &,      \
                                                   const EventDesc *, const InstCoef *, double *, const int *);     \
    extern template int gwh_tiles_load<M, P>();
GWH_TILES_DECLARE(GWH_IMRPHENOMD, GWH_FP64)
GWH_TILES_DECLARE(GWH_IMRPHENOMD, GWH_MIXED)
GWH_TILES_DECLARE(GWH_IMRPHENOMPV2, GWH_FP64)
