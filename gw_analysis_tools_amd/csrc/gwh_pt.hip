/*
 * gwh_pt.hip -- sampler steps as replayable HIP graphs.
 *
 *   likelihood step   the batched likelihood (setup, per-bin tiles, finalize) on fixed device buffers,
 *                     captured once; every replay reads the caller's parameter buffer and writes its
 *                     log-likelihood buffer (for samplers that make their own proposals)
 *   tempering step    a whole parallel-tempering step of n_temps x n_chains chains on the device:
 *                     Gaussian proposal, prior box, likelihood of every proposal, Metropolis-Hastings
 *                     decision, adjacent-temperature swaps along every ladder; the step counter lives in
 *                     device memory, so one captured graph serves every step with no host round trip
 *
 * Reference: src/mcmc_sampler_internals.cpp:35-145 (mcmc_step), :364-409 (gaussian_step),
 * :1086-1115 (chain_swap), :1121-1180 (single_chain_swap).
 *
 * Random numbers: Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11), key = the seed's two 32-bit halves,
 * counter = (instance or ladder pair, step low word, step high word, stream tag).  Per instance and step:
 * block A = tag 0, block B = tag 1; the proposal dimension is (A0 * dim) >> 32, the normal deviate is
 * Box-Muller sqrt(-2 ln(1 - u53(A1, A2))) cos(2 pi u53(A3, B0)), log U = ln u53(B1, B2); the swap uniform of
 * pair (k, chain c) is u53(C0, C1) of block (k * n_chains + c, step, tag 2).  u53(a, b) = ((a >> 5) 2^26 +
 * (b >> 6)) 2^-53.
 *
 * Mixed precision with the guard band: a Metropolis-Hastings decision whose margin (ll' - ll) / T - log U lies
 * within 2 tol / T of zero, and a swap whose margin lies within 2 tol |1/T2 - 1/T1|, is re-decided with FP64
 * likelihoods evaluated inside the same graph (a count-limited FP64 launch over the compacted states), so the
 * decision sequence equals the all-FP64 run's whenever the mixed likelihood error stays within tol.
 * A ladder with a swap inside the band is re-run with FP64 values for all of its states (the ladder's later
 * decisions depend on the earlier ones).
 */
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "gwh_basis.h"
#include "gwh_engine.h"

#define GWH_PT_MAXDIM 15
#define GWH_PT_MAXTEMPS 64
#define GWH_PT_MAXCHAINS 1024

/* ------------------------------------------------------------------------- */
/* Philox4x32-10                                                              */
/* ------------------------------------------------------------------------- */

struct U4 {
    uint32_t x, y, z, w;
};

__device__ __forceinline__ U4 philox4x32_10(U4 c, uint32_t k0, uint32_t k1)
{
#pragma unroll
    for (int r = 0; r < 10; r++) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c.x, p1 = (uint64_t)0xCD9E8D57u * c.z;
        U4 o;
        o.x = (uint32_t)(p1 >> 32) ^ c.y ^ k0;
        o.y = (uint32_t)p1;
        o.z = (uint32_t)(p0 >> 32) ^ c.w ^ k1;
        o.w = (uint32_t)p0;
        c = o;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    return c;
}

__device__ __forceinline__ double u53(uint32_t a, uint32_t b)
{
    return ((double)(a >> 5) * 67108864.0 + (double)(b >> 6)) * (1.0 / 9007199254740992.0);
}

/* ------------------------------------------------------------------------- */
/* device state of one tempering run                                          */
/* ------------------------------------------------------------------------- */

struct PtArgs {
    int n, nt, nc, dim, basis, swap_every, guard;
    double tol;
    uint32_t key0, key1;
    const double *temps;   /* nt */
    const double *width;   /* n x dim: Gaussian step width of every chain and dimension */
    const double *lower, *upper; /* dim: prior box */
    const gwh_params *tmpl; /* non-sampled fields */
    double *theta, *ll;    /* current states */
    double *prop, *llp;    /* this step's proposals and their log-likelihoods */
    double *logu;          /* n: this step's log U */
    gwh_params *params;    /* n: records of the proposals */
    int *mask;             /* n: proposal inside the prior box */
    int *acc;              /* n: 1 accepted, 0 rejected, 2 pending FP64 re-decision */
    int *swp;              /* (nt-1) x nc: pair swapped this step */
    long long *acc_count, *swap_count; /* n, (nt-1) x nc */
    unsigned long long *guard_evals;
    long long *step;
    /* guard band */
    int *gcount;           /* [0]: MH states, [1]: ladder states */
    int *gslot;            /* n: slot of instance i's pair in gparams */
    int *lslot;            /* nc: slot of ladder c's states in lparams, -1 none */
    gwh_params *gparams;   /* 2n */
    gwh_params *lparams;   /* n */
    double *gll, *lll;     /* FP64 log-likelihoods of gparams, lparams */
};

__device__ __forceinline__ gwh_params pt_record(const PtArgs &a, const double *v)
{
    gwh_params p = *a.tmpl;
    repack(v, a.basis, p);
    return p;
}

__device__ __forceinline__ double pt_T(const PtArgs &a, int i) { return a.temps[i / a.nc]; }

/* records of the initial states (for their likelihoods) */
__global__ void gwh_pt_init_kernel(PtArgs a)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    a.params[i] = pt_record(a, a.theta + (size_t)i * a.dim);
    a.mask[i] = 1;
}

/* gaussian_step (mcmc_sampler_internals.cpp:364-409): one dimension chosen uniformly, moved by
 * width * N(0, 1); the prior box decides whether the likelihood is needed at all (mcmc_step :83-92).
 * 64 chains per block, four waves with one lane of each per chain: all draw the proposal, then wave 0 writes it with
 * log U and the mask, waves 1 to 3 a part of its record each (repack_part), so the logarithms, powers and arctangents
 * run side by side: with one lane per chain the step's chain of them took 11.2 us, now 5.6. */
__global__ __launch_bounds__(256) void gwh_pt_propose_kernel(PtArgs a)
{
    const int role = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = blockIdx.x * 64 + (threadIdx.x & 63);
    if (i == 0 && role == 0) {
        a.gcount[0] = 0;
        a.gcount[1] = 0;
    }
    if (i >= a.n) return;
    const long long s = *a.step;
    const uint32_t slo = (uint32_t)s, shi = (uint32_t)((unsigned long long)s >> 32);
    const U4 A = philox4x32_10(U4{(uint32_t)i, slo, shi, 0u}, a.key0, a.key1);
    const U4 B = philox4x32_10(U4{(uint32_t)i, slo, shi, 1u}, a.key0, a.key1);
    const int beta = (int)(((uint64_t)A.x * (uint64_t)a.dim) >> 32);
    const double u1 = u53(A.y, A.z), u2 = u53(A.w, B.x);
    const double z = sqrt(-2.0 * log(1.0 - u1)) * cospi(2.0 * u2);
    const double *th = a.theta + (size_t)i * a.dim;
    const double t_beta = th[beta], x_beta = __dadd_rn(__dmul_rn(a.width[(size_t)i * a.dim + beta], z), t_beta);
    /* fixed trip count: every index of v is a compile-time constant, so v lives in registers */
    double v[GWH_PT_MAXDIM];
    int ok = 1;
#pragma unroll
    for (int d = 0; d < GWH_PT_MAXDIM; d++) v[d] = d < a.dim ? th[d] : 0.0;
#pragma unroll
    for (int d = 0; d < GWH_PT_MAXDIM; d++) {
        if (d >= a.dim) break;
        v[d] = (d == beta) ? x_beta : v[d];
        if (role == 0) a.prop[(size_t)i * a.dim + d] = v[d];
        ok &= (v[d] >= a.lower[d]) & (v[d] <= a.upper[d]);
    }
    if (role == 0) {
        a.mask[i] = ok;
        a.logu[i] = log(u53(B.y, B.z));
        return;
    }
    /* outside the prior box: the record of the current state (its likelihood is not used) */
#pragma unroll
    for (int d = 0; d < GWH_PT_MAXDIM; d++) v[d] = (!ok && d == beta) ? t_beta : v[d];
    /* a.params[i] holds the template's other fields since the init kernel: only the sampled ones change (the
     * sampling bases' repack reads no field of the record) */
    if (role == 1)
        repack_part(v, a.basis, 0, a.params[i]);
    else if (role == 2)
        repack_part(v, a.basis, 1, a.params[i]);
    else
        repack_part(v, a.basis, 2, a.params[i]);
}

/* Metropolis-Hastings (mcmc_sampler_internals.cpp:96-142): reject iff (ll' - ll) / T < log U; a proposal
 * outside the prior box or with a NaN likelihood is rejected */
__device__ __forceinline__ void pt_apply(const PtArgs &a, int i, bool accept)
{
    a.acc[i] = accept;
    if (!accept) return;
    for (int d = 0; d < a.dim; d++) a.theta[(size_t)i * a.dim + d] = a.prop[(size_t)i * a.dim + d];
    a.ll[i] = a.llp[i];
    a.acc_count[i]++;
}

__device__ __forceinline__ bool mh_accept(double ratio, double logu)
{
    return ratio > -INFINITY && !(ratio < logu);
}

/* The proposals' log-likelihoods from their tiles' partial sums (gwh_finalize_instance, one wave per chain), each followed
 * by its decision in lane 0 -- one launch instead of two -- and the step counter's advance: nothing in this kernel reads
 * it, the swaps that follow take it less one. */
__global__ __launch_bounds__(256) void gwh_pt_accept_kernel(PtArgs a, FinalizeArgs F)
{
    const int i = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (blockIdx.x == 0 && threadIdx.x == 0) ++*a.step;
    if (i >= a.n) return;
    double lp = gwh_finalize_instance(F, i);
    if ((threadIdx.x & 63) != 0) return;
    if (i < (a.nt - 1) * a.nc) a.swp[i] = 0; /* no swap so far in this step */
    const double T = pt_T(a, i), lu = a.logu[i];
    if (!a.mask[i]) lp = __longlong_as_double(0x7ff8000000000000ll);
    a.llp[i] = lp;
    const double ratio = (lp == lp) ? (-a.ll[i] + lp) / T : -INFINITY;
    const double margin = ratio - lu;
    if (a.guard && ratio > -INFINITY && isfinite(margin) && fabs(margin) < 2.0 * a.tol / T) {
        const int slot = atomicAdd(&a.gcount[0], 2);
        a.gslot[i] = slot;
        a.gparams[slot] = a.params[i];
        a.gparams[slot + 1] = pt_record(a, a.theta + (size_t)i * a.dim);
        a.acc[i] = 2;
        return;
    }
    pt_apply(a, i, mh_accept(ratio, lu));
}

__global__ void gwh_pt_accept_guard_kernel(PtArgs a)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n || a.acc[i] != 2) return;
    const int slot = a.gslot[i];
    const double T = pt_T(a, i);
    const double l1 = a.gll[slot], l0 = a.gll[slot + 1];
    const double ratio = (l1 == l1 && l0 == l0) ? (-l0 + l1) / T : -INFINITY;
    atomicAdd(a.guard_evals, 2ull);
    pt_apply(a, i, mh_accept(ratio, a.logu[i]));
}

/* chain_swap / single_chain_swap (mcmc_sampler_internals.cpp:1086-1180): pairs (k, k+1) of one ladder in
 * increasing k; reject iff exp((ll1 - ll2) / T2 - (ll1 - ll2) / T1) < U.
 *
 * One wave per ladder.  At pair k the state at temperature k + 1 is the one it started with and the state at k one of
 * those of temperatures 0..k, so the lanes decide every (pair, state) combination side by side (120 for 16 temperatures,
 * at most 2016), and lane 0 walks the ladder through the table of decisions; then all lanes move the states.  With one
 * lane per ladder, each walking its pairs' divisions and exponentials and moving its rows alone, a swap took 100 us for
 * 32 ladders of 16 temperatures, now 7.3.
 *
 * ll64: FP64 log-likelihoods of the ladder's states by temperature; without them a decision inside the guard band on the
 * walk ends it (-> the states are queued for FP64 evaluation). */
struct LadderShared {
    double ll[GWH_PT_MAXTEMPS], T[GWH_PT_MAXTEMPS], theta[GWH_PT_MAXTEMPS * GWH_PT_MAXDIM];
    unsigned char how[GWH_PT_MAXTEMPS][GWH_PT_MAXTEMPS]; /* pair k, state j: 1 swap, 2 undecided in this precision */
    int perm[GWH_PT_MAXTEMPS], flag[GWH_PT_MAXTEMPS], slot;
};

__device__ void pt_ladder(const PtArgs &a, int c, long long s, const double *ll64, LadderShared &sh)
{
    const int lane = threadIdx.x, nt = a.nt;
    if (lane < nt) {
        sh.ll[lane] = a.ll[lane * a.nc + c];
        sh.T[lane] = a.temps[lane];
    }
    for (int e = lane; e < nt * a.dim; e += 64) sh.theta[e] = a.theta[(size_t)((e / a.dim) * a.nc + c) * a.dim + e % a.dim];
    __syncthreads();
    const uint32_t slo = (uint32_t)s, shi = (uint32_t)((unsigned long long)s >> 32);
    for (int p = lane; p < nt * (nt - 1) / 2; p += 64) {
        int k = (int)((sqrtf(8.0f * p + 1.0f) - 1.0f) * 0.5f); /* p = k (k + 1) / 2 + j, 0 <= j <= k < nt - 1 */
        while (k * (k + 1) / 2 > p) k--;
        while ((k + 1) * (k + 2) / 2 <= p) k++;
        const int j = p - k * (k + 1) / 2;
        const U4 C = philox4x32_10(U4{(uint32_t)(k * a.nc + c), slo, shi, 2u}, a.key0, a.key1);
        const double alpha = u53(C.x, C.y);
        const double T1 = sh.T[k], T2 = sh.T[k + 1], l1 = sh.ll[j], l2 = sh.ll[k + 1];
        double pw = (l1 - l2) / T2 - (l1 - l2) / T1;
        bool near = a.guard && alpha > 0 && fabs(pw - log(alpha)) < 2.0 * a.tol * fabs(1.0 / T2 - 1.0 / T1);
        if (near && ll64) {
            const double m1 = ll64[j], m2 = ll64[k + 1];
            pw = (m1 - m2) / T2 - (m1 - m2) / T1;
            near = false;
        }
        sh.how[k][j] = near ? 2 : !(exp(pw) < alpha);
    }
    __syncthreads();
    if (lane == 0) {
        int cur = 0; /* the temperature whose state has come to temperature k */
        sh.slot = -1;
        for (int k = 0; k + 1 < nt; k++) {
            const int how = (sh.T[k] == sh.T[k + 1]) ? 0 : sh.how[k][cur];
            if (how == 2) { /* FP64 values of this ladder's states are needed */
                sh.slot = atomicAdd(&a.gcount[1], nt);
                break;
            }
            sh.flag[k] = how;
            sh.perm[k] = how ? k + 1 : cur;
            if (!how) cur = k + 1;
        }
        sh.perm[nt - 1] = cur;
    }
    __syncthreads();
    if (sh.slot >= 0) {
        if (lane == 0) a.lslot[c] = sh.slot;
        if (lane < nt) a.lparams[sh.slot + lane] = pt_record(a, a.theta + (size_t)(lane * a.nc + c) * a.dim);
        return;
    }
    if (lane < nt) a.ll[lane * a.nc + c] = sh.ll[sh.perm[lane]];
    for (int e = lane; e < nt * a.dim; e += 64)
        a.theta[(size_t)((e / a.dim) * a.nc + c) * a.dim + e % a.dim] = sh.theta[sh.perm[e / a.dim] * a.dim + e % a.dim];
    if (lane + 1 < nt) {
        a.swp[lane * a.nc + c] = sh.flag[lane];
        a.swap_count[lane * a.nc + c] += sh.flag[lane];
    }
}

/* one block of one wave per ladder; the accept kernel has advanced the step counter */
__global__ __launch_bounds__(64) void gwh_pt_swap_kernel(PtArgs a)
{
    __shared__ LadderShared sh;
    const int c = blockIdx.x, lane = threadIdx.x;
    const long long s = *a.step - 1;
    if (lane == 0) a.lslot[c] = -1;
    if (a.swap_every > 0 && (s + 1) % a.swap_every == 0) pt_ladder(a, c, s, nullptr, sh);
}

__global__ __launch_bounds__(64) void gwh_pt_swap_guard_kernel(PtArgs a)
{
    __shared__ LadderShared sh;
    const int c = blockIdx.x;
    const int slot = a.lslot[c];
    if (slot < 0) return; /* the whole block */
    pt_ladder(a, c, *a.step - 1, a.lll + slot, sh);
    if (threadIdx.x == 0) atomicAdd(a.guard_evals, (unsigned long long)a.nt);
}

/* ------------------------------------------------------------------------- */
/* host side                                                                  */
/* ------------------------------------------------------------------------- */

namespace {

struct StepGraph {
    std::mutex mu;
    bool dead = false;
    int kind = 0; /* 0 likelihood step, 1 tempering run */
    std::vector<int> pinned;
    hipStream_t stream = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    Scratch scr;
    /* tempering run */
    int steps_per_graph = 1;
    PtArgs a;
    DevBuf state;
    int event = -1, model = 0, precision = 0;
};

std::mutex g_mu;
std::map<int, std::shared_ptr<StepGraph>> g_graphs;
int g_next = 1;

std::shared_ptr<StepGraph> find_graph(int id, int kind)
{
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = g_graphs.find(id);
    if (it == g_graphs.end() || it->second->kind != kind) return nullptr;
    return it->second;
}

int register_graph(std::shared_ptr<StepGraph> g)
{
    std::lock_guard<std::mutex> lk(g_mu);
    int id = g_next++;
    g_graphs[id] = g;
    return id;
}

/* release device resources (engine lock held by the caller) */
void free_graph(StepGraph &g)
{
    Engine &E = gwh_engine();
    if (g.stream) (void)hipStreamSynchronize(g.stream);
    if (g.exec) (void)hipGraphExecDestroy(g.exec);
    if (g.graph) (void)hipGraphDestroy(g.graph);
    if (g.stream) (void)hipStreamDestroy(g.stream);
    g.exec = nullptr;
    g.graph = nullptr;
    g.stream = nullptr;
    g.scr.release();
    g.state.release();
    for (int e : g.pinned)
        if (e >= 0 && e < GWH_MAX_EVENTS && E.events[e].pins > 0) E.events[e].pins--;
    g.pinned.clear();
}

int pin_events(StepGraph &g, const int *events, int n, int event0)
{
    Engine &E = gwh_engine();
    std::vector<char> seen(GWH_MAX_EVENTS, 0);
    auto add = [&](int e) -> int {
        if (e < 0 || e >= GWH_MAX_EVENTS || !E.events[e].live)
            return gwh_set_error(GWH_ERR_INVALID, "unknown event " + std::to_string(e));
        if (!seen[e]) {
            seen[e] = 1;
            E.events[e].pins++;
            g.pinned.push_back(e);
        }
        return GWH_OK;
    };
    if (events) {
        for (int i = 0; i < n; i++) {
            int rc = add(events[i]);
            if (rc != GWH_OK) return rc;
        }
        return GWH_OK;
    }
    return add(event0);
}

/* capture what `body` enqueues on g.stream into g.graph / g.exec */
template <class F> int capture(StepGraph &g, F body)
{
    GWH_HIP(hipStreamBeginCapture(g.stream, hipStreamCaptureModeRelaxed));
    int rc = body();
    hipGraph_t graph = nullptr;
    hipError_t e = hipStreamEndCapture(g.stream, &graph);
    if (rc != GWH_OK) {
        if (graph) (void)hipGraphDestroy(graph);
        return rc;
    }
    if (e != hipSuccess) return gwh_set_error(GWH_ERR_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    g.graph = graph;
    GWH_HIP(hipGraphInstantiate(&g.exec, g.graph, nullptr, nullptr, 0));
    return GWH_OK;
}

inline dim3 blocks_of(int n) { return dim3((n + 255) / 256); }

} // namespace

/* ---- likelihood step ---- */

int gwh_loglike_graph_create(const int *events, const int *d_events, int events0, int model, int precision,
                             const void *d_params, int n, double *d_logl, int *graph)
{
    Engine &E = gwh_engine();
    std::lock_guard<std::recursive_mutex> lk(E.mu);
    int st = gwh_ensure_init();
    if (st != GWH_OK) return st;
    if (!graph || !d_params || !d_logl || n <= 0) return gwh_set_error(GWH_ERR_INVALID, "bad argument");
    if ((events == nullptr) != (d_events == nullptr))
        return gwh_set_error(GWH_ERR_INVALID, "events and d_events are given together or not at all");
    auto g = std::make_shared<StepGraph>();
    g->kind = 0;
    int rc = pin_events(*g, events, n, events0);
    if (rc == GWH_OK && hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking) != hipSuccess)
        rc = gwh_set_error(GWH_ERR_HIP, "hipStreamCreateWithFlags failed");
    LaunchExtra x;
    x.reserve_only = true;
    if (rc == GWH_OK)
        rc = gwh_loglike_launch(d_events, events ? events[0] : events0, model, precision, (const gwh_params *)d_params,
                                n, d_logl, g->stream, false, nullptr, events, 0, &g->scr, &x);
    if (rc == GWH_OK) {
        x.reserve_only = false;
        x.capturing = true;
        rc = capture(*g, [&]() {
            return gwh_loglike_launch(d_events, events ? events[0] : events0, model, precision,
                                      (const gwh_params *)d_params, n, d_logl, g->stream, false, nullptr, events, 0,
                                      &g->scr, &x);
        });
    }
    if (rc != GWH_OK) {
        free_graph(*g);
        return rc;
    }
    *graph = register_graph(g);
    return GWH_OK;
}

int gwh_graph_launch(int graph, void *stream)
{
    auto g = find_graph(graph, 0);
    if (!g) return gwh_set_error(GWH_ERR_INVALID, "unknown graph");
    std::lock_guard<std::mutex> lk(g->mu);
    if (g->dead) return gwh_set_error(GWH_ERR_INVALID, "unknown graph");
    GWH_HIP(hipGraphLaunch(g->exec, stream ? (hipStream_t)stream : g->stream));
    return GWH_OK;
}

int gwh_graph_synchronize(int graph)
{
    auto g = find_graph(graph, 0);
    if (!g) g = find_graph(graph, 1);
    if (!g) return gwh_set_error(GWH_ERR_INVALID, "unknown graph");
    std::lock_guard<std::mutex> lk(g->mu);
    if (g->dead) return gwh_set_error(GWH_ERR_INVALID, "unknown graph");
    GWH_HIP(hipStreamSynchronize(g->stream));
    return GWH_OK;
}

static int destroy_graph(int id, int kind)
{
    std::shared_ptr<StepGraph> g;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        auto it = g_graphs.find(id);
        if (it == g_graphs.end() || it->second->kind != kind) return gwh_set_error(GWH_ERR_INVALID, "unknown graph");
        g = it->second;
        g_graphs.erase(it);
    }
    Engine &E = gwh_engine();
    std::lock_guard<std::recursive_mutex> lk(E.mu);
    std::lock_guard<std::mutex> lk2(g->mu);
    g->dead = true;
    free_graph(*g);
    return GWH_OK;
}

int gwh_graph_destroy(int graph) { return destroy_graph(graph, 0); }

/* ---- tempering run ---- */

int gwh_pt_create(int event, const gwh_pt_config *cfg, const double *temps, const double *widths,
                  const double *lower, const double *upper, const gwh_params *tmpl, const double *theta0, int *pt)
{
    Engine &E = gwh_engine();
    std::lock_guard<std::recursive_mutex> lk(E.mu);
    int st = gwh_ensure_init();
    if (st != GWH_OK) return st;
    if (!cfg || !temps || !widths || !lower || !upper || !tmpl || !theta0 || !pt)
        return gwh_set_error(GWH_ERR_INVALID, "null argument");
    const int nt = cfg->n_temps, nc = cfg->n_chains;
    if (nt < 1 || nt > GWH_PT_MAXTEMPS) return gwh_set_error(GWH_ERR_INVALID, "n_temps must be 1..64");
    if (nc < 1 || nc > GWH_PT_MAXCHAINS) return gwh_set_error(GWH_ERR_INVALID, "n_chains must be 1..1024");
    const int n = nt * nc;
    if (2 * n > 65535) return gwh_set_error(GWH_ERR_INVALID, "at most 32767 chains in all");
    if (cfg->basis != GWH_BASIS_PHENOMD_MCMC && cfg->basis != GWH_BASIS_PV2_MCMC)
        return gwh_set_error(GWH_ERR_UNSUPPORTED, "sampling basis must be GWH_BASIS_PHENOMD_MCMC or GWH_BASIS_PV2_MCMC");
    if (cfg->model != GWH_IMRPHENOMD && cfg->model != GWH_IMRPHENOMPV2)
        return gwh_set_error(GWH_ERR_UNSUPPORTED, "model must be GWH_IMRPHENOMD or GWH_IMRPHENOMPV2");
    if (cfg->precision != GWH_FP64 && cfg->precision != GWH_MIXED)
        return gwh_set_error(GWH_ERR_INVALID, "bad precision");
    if (cfg->swap_every < 0 || cfg->steps_per_graph < 1 || cfg->steps_per_graph > 1000)
        return gwh_set_error(GWH_ERR_INVALID, "swap_every >= 0 and 1 <= steps_per_graph <= 1000");
    for (int k = 0; k < nt; k++)
        if (!(temps[k] > 0) || !std::isfinite(temps[k]))
            return gwh_set_error(GWH_ERR_INVALID, "temperatures must be positive and finite");
    const int dim = basis_dim(cfg->basis);
    const bool guard = cfg->guard && cfg->precision == GWH_MIXED;
    if (guard && !(cfg->tol > 0)) return gwh_set_error(GWH_ERR_INVALID, "guard band needs tol > 0");

    auto g = std::make_shared<StepGraph>();
    g->kind = 1;
    g->steps_per_graph = cfg->steps_per_graph;
    g->event = event;
    g->model = cfg->model;
    g->precision = cfg->precision;
    int rc = pin_events(*g, nullptr, 0, event);
    if (rc != GWH_OK) return rc;
    auto fail = [&](int code) {
        free_graph(*g);
        return code;
    };
    if (hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking) != hipSuccess)
        return fail(gwh_set_error(GWH_ERR_HIP, "hipStreamCreateWithFlags failed"));

    /* one allocation: doubles, then records, then 8-byte counters, then ints */
    const size_t nd = (size_t)nt + (size_t)n * dim + 2 * dim + 1 /* tmpl slot (aligned) */ + 2 * (size_t)n * dim +
                      3 * (size_t)n + 2 * (size_t)n + (size_t)n;
    const size_t nrec = (size_t)n + 2 * (size_t)n + (size_t)n + 1;
    const size_t ncnt = (size_t)n + (size_t)(nt - 1) * nc + 2;
    const size_t nint = (size_t)n * 3 + (size_t)(nt - 1) * nc + 2 + (size_t)n + (size_t)nc;
    const size_t bytes = nd * 8 + nrec * sizeof(gwh_params) + ncnt * 8 + nint * 4 + 256;
    if ((rc = g->state.ensure(bytes)) != GWH_OK) return fail(rc);
    char *base = (char *)g->state.p;
    size_t off = 0;
    auto take = [&](size_t b) {
        char *p = base + off;
        off += (b + 15) & ~(size_t)15;
        return p;
    };
    PtArgs &a = g->a;
    a.n = n;
    a.nt = nt;
    a.nc = nc;
    a.dim = dim;
    a.basis = cfg->basis;
    a.swap_every = cfg->swap_every;
    a.guard = guard;
    a.tol = cfg->tol;
    a.key0 = (uint32_t)cfg->seed;
    a.key1 = (uint32_t)(cfg->seed >> 32);
    double *d_temps = (double *)take(nt * 8);
    double *d_width = (double *)take((size_t)n * dim * 8);
    double *d_lower = (double *)take(dim * 8), *d_upper = (double *)take(dim * 8);
    a.temps = d_temps;
    a.width = d_width;
    a.lower = d_lower;
    a.upper = d_upper;
    a.theta = (double *)take((size_t)n * dim * 8);
    a.prop = (double *)take((size_t)n * dim * 8);
    a.ll = (double *)take(n * 8);
    a.llp = (double *)take(n * 8);
    a.logu = (double *)take(n * 8);
    a.gll = (double *)take(2 * (size_t)n * 8);
    a.lll = (double *)take((size_t)n * 8);
    gwh_params *d_tmpl = (gwh_params *)take(sizeof(gwh_params));
    a.tmpl = d_tmpl;
    a.params = (gwh_params *)take((size_t)n * sizeof(gwh_params));
    a.gparams = (gwh_params *)take(2 * (size_t)n * sizeof(gwh_params));
    a.lparams = (gwh_params *)take((size_t)n * sizeof(gwh_params));
    a.acc_count = (long long *)take((size_t)n * 8);
    a.swap_count = (long long *)take((size_t)std::max(nt - 1, 1) * nc * 8);
    a.guard_evals = (unsigned long long *)take(8);
    a.step = (long long *)take(8);
    a.mask = (int *)take((size_t)n * 4);
    a.acc = (int *)take((size_t)n * 4);
    a.gslot = (int *)take((size_t)n * 4);
    a.swp = (int *)take((size_t)std::max(nt - 1, 1) * nc * 4);
    a.gcount = (int *)take(2 * 4);
    a.lslot = (int *)take((size_t)nc * 4);
    if (off > g->state.cap) return fail(gwh_set_error(GWH_ERR_INVALID, "internal: state layout overflow"));

    hipStream_t s = g->stream;
    auto up = [&](void *dst, const void *src, size_t b) {
        return hipMemcpyAsync(dst, src, b, hipMemcpyHostToDevice, s) == hipSuccess;
    };
    bool ok = up(d_temps, temps, nt * 8) && up(d_width, widths, (size_t)n * dim * 8) &&
              up(d_lower, lower, dim * 8) && up(d_upper, upper, dim * 8) &&
              up(a.theta, theta0, (size_t)n * dim * 8) && up(d_tmpl, tmpl, sizeof(gwh_params));
    ok = ok && hipMemsetAsync(a.acc_count, 0, (size_t)n * 8, s) == hipSuccess &&
         hipMemsetAsync(a.swap_count, 0, (size_t)std::max(nt - 1, 1) * nc * 8, s) == hipSuccess &&
         hipMemsetAsync(a.guard_evals, 0, 8, s) == hipSuccess && hipMemsetAsync(a.step, 0, 8, s) == hipSuccess &&
         hipMemsetAsync(a.acc, 0, (size_t)n * 4, s) == hipSuccess &&
         hipMemsetAsync(a.swp, 0, (size_t)std::max(nt - 1, 1) * nc * 4, s) == hipSuccess &&
         hipMemsetAsync(a.lslot, 0xff, (size_t)nc * 4, s) == hipSuccess &&
         hipMemsetAsync(a.prop, 0, (size_t)n * dim * 8, s) == hipSuccess &&
         hipMemsetAsync(a.llp, 0, (size_t)n * 8, s) == hipSuccess;
    if (!ok) return fail(gwh_set_error(GWH_ERR_HIP, "initial copies failed"));

    /* scratch sized for the largest launch before anything is captured */
    LaunchExtra x;
    x.reserve_only = true;
    const int P = cfg->precision, M = cfg->model;
    if ((rc = gwh_loglike_launch(nullptr, event, M, P, a.params, n, a.llp, s, false, nullptr, nullptr, 0, &g->scr,
                                 &x)) != GWH_OK)
        return fail(rc);
    if (guard && (rc = gwh_loglike_launch(nullptr, event, M, GWH_FP64, a.gparams, 2 * n, a.gll, s, false, nullptr,
                                          nullptr, 0, &g->scr, &x)) != GWH_OK)
        return fail(rc);

    /* likelihoods of the initial states (eager) */
    x.reserve_only = false;
    hipLaunchKernelGGL(gwh_pt_init_kernel, blocks_of(n), dim3(256), 0, s, a);
    if ((rc = gwh_loglike_launch(nullptr, event, M, P, a.params, n, a.ll, s, false, nullptr, nullptr, 0, &g->scr,
                                 &x)) != GWH_OK)
        return fail(rc);
    if (hipStreamSynchronize(s) != hipSuccess) return fail(gwh_set_error(GWH_ERR_HIP, "initial likelihoods failed"));

    x.capturing = true;
    rc = capture(*g, [&]() -> int {
        int r;
        for (int k = 0; k < g->steps_per_graph; k++) {
            hipLaunchKernelGGL(gwh_pt_propose_kernel, dim3((n + 63) / 64), dim3(256), 0, s, a);
            LaunchExtra m = x;
            FinalizeArgs fin;
            m.d_mask = a.mask;
            m.finalize_later = &fin;
            if ((r = gwh_loglike_launch(nullptr, event, M, P, a.params, n, a.llp, s, false, nullptr, nullptr, 0,
                                        &g->scr, &m)) != GWH_OK)
                return r;
            hipLaunchKernelGGL(gwh_pt_accept_kernel, dim3((n + 3) / 4), dim3(256), 0, s, a, fin);
            if (guard) {
                LaunchExtra c0 = x;
                c0.d_count = a.gcount;
                if ((r = gwh_loglike_launch(nullptr, event, M, GWH_FP64, a.gparams, 2 * n, a.gll, s, false, nullptr,
                                            nullptr, 0, &g->scr, &c0)) != GWH_OK)
                    return r;
                hipLaunchKernelGGL(gwh_pt_accept_guard_kernel, blocks_of(n), dim3(256), 0, s, a);
            }
            /* runs advance by whole graphs from step 0, so with a swap interval that divides the graph's steps the place
               in the graph tells whether a step swaps; otherwise the kernel asks the step counter */
            const bool swaps = cfg->swap_every > 0 && nt > 1 &&
                               (g->steps_per_graph % cfg->swap_every != 0 || (k + 1) % cfg->swap_every == 0);
            if (swaps) hipLaunchKernelGGL(gwh_pt_swap_kernel, dim3(nc), dim3(64), 0, s, a);
            if (swaps && guard) {
                LaunchExtra c1 = x;
                c1.d_count = a.gcount + 1;
                if ((r = gwh_loglike_launch(nullptr, event, M, GWH_FP64, a.lparams, n, a.lll, s, false, nullptr,
                                            nullptr, 0, &g->scr, &c1)) != GWH_OK)
                    return r;
                hipLaunchKernelGGL(gwh_pt_swap_guard_kernel, dim3(nc), dim3(64), 0, s, a);
            }
            GWH_HIP(hipGetLastError());
        }
        return GWH_OK;
    });
    if (rc != GWH_OK) return fail(rc);
    *pt = register_graph(g);
    return GWH_OK;
}

int gwh_pt_run(int pt, int steps)
{
    auto g = find_graph(pt, 1);
    if (!g) return gwh_set_error(GWH_ERR_INVALID, "unknown tempering run");
    std::lock_guard<std::mutex> lk(g->mu);
    if (g->dead) return gwh_set_error(GWH_ERR_INVALID, "unknown tempering run");
    if (steps < 0 || steps % g->steps_per_graph != 0)
        return gwh_set_error(GWH_ERR_INVALID, "steps must be a non-negative multiple of steps_per_graph");
    for (int k = 0; k < steps / g->steps_per_graph; k++) GWH_HIP(hipGraphLaunch(g->exec, g->stream));
    return GWH_OK;
}

int gwh_pt_synchronize(int pt)
{
    auto g = find_graph(pt, 1);
    if (!g) return gwh_set_error(GWH_ERR_INVALID, "unknown tempering run");
    std::lock_guard<std::mutex> lk(g->mu);
    if (g->dead) return gwh_set_error(GWH_ERR_INVALID, "unknown tempering run");
    GWH_HIP(hipStreamSynchronize(g->stream));
    return GWH_OK;
}

static int pt_read(int pt, const std::vector<std::pair<void *, std::pair<const void *, size_t>>> &items)
{
    auto g = find_graph(pt, 1);
    if (!g) return gwh_set_error(GWH_ERR_INVALID, "unknown tempering run");
    std::lock_guard<std::mutex> lk(g->mu);
    if (g->dead) return gwh_set_error(GWH_ERR_INVALID, "unknown tempering run");
    GWH_HIP(hipStreamSynchronize(g->stream));
    for (auto &it : items)
        if (it.first) GWH_HIP(hipMemcpy(it.first, it.second.first, it.second.second, hipMemcpyDeviceToHost));
    return GWH_OK;
}

int gwh_pt_state(int pt, double *theta, double *ll, long long *step)
{
    auto g = find_graph(pt, 1);
    if (!g) return gwh_set_error(GWH_ERR_INVALID, "unknown tempering run");
    const PtArgs &a = g->a;
    return pt_read(pt, {{theta, {a.theta, (size_t)a.n * a.dim * 8}}, {ll, {a.ll, (size_t)a.n * 8}},
                        {step, {a.step, 8}}});
}

int gwh_pt_last_step(int pt, double *prop, double *llp, int *accept, int *swapped)
{
    auto g = find_graph(pt, 1);
    if (!g) return gwh_set_error(GWH_ERR_INVALID, "unknown tempering run");
    const PtArgs &a = g->a;
    return pt_read(pt, {{prop, {a.prop, (size_t)a.n * a.dim * 8}}, {llp, {a.llp, (size_t)a.n * 8}},
                        {accept, {a.acc, (size_t)a.n * 4}},
                        {swapped, {a.swp, (size_t)std::max(a.nt - 1, 0) * a.nc * 4}}});
}

int gwh_pt_counters(int pt, long long *accepts, long long *swaps, long long *guard_evals)
{
    auto g = find_graph(pt, 1);
    if (!g) return gwh_set_error(GWH_ERR_INVALID, "unknown tempering run");
    const PtArgs &a = g->a;
    return pt_read(pt, {{accepts, {a.acc_count, (size_t)a.n * 8}},
                        {swaps, {a.swap_count, (size_t)std::max(a.nt - 1, 0) * a.nc * 8}},
                        {guard_evals, {a.guard_evals, 8}}});
}

int gwh_pt_destroy(int pt) { return destroy_graph(pt, 1); }
