/*
 * gwh_fisher.hip -- numerical Fisher matrices on MI355X.
 *
 *   host      unpack the point into the basis of the generation method, build the central-difference
 *             stencil (the perturbed parameter sets, fisher.cpp:148-557), run the FP64 setup for all of
 *             them in one launch
 *   fused     one block per (point, 64 bins): the stencil evaluations of every parameter projected on every detector,
 *             the FP64 difference quotients scaled by sqrt(w/S) as operand rows (parameters padded to 16) in LDS, and
 *             F = sum_rows a a^T of the block with v_mfma_f64_16x16x4
 *   reduce    the blocks' partial matrices of every point, FP64, in a fixed order
 *   FP32 Gram and bare derivatives: a stencil kernel (one lane per bin, point and row) writes the rows to memory,
 *             v_mfma_f32_16x16x4 contracts them with FP64 sums across waves and row chunks
 *   invert    FP64 LU inverse per point (util.cpp:828-855) -> marginal sigmas
 *
 * Reference: src/fisher.cpp:81-145 (fisher_numerical), :148-557 (calculate_derivatives),
 * :1754-2572 (basis maps), :2704-2781 (calculate_fisher_elements).
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "gwh_engine.h"
#include "gwh_tables.h"

typedef double gwh_d4 __attribute__((ext_vector_type(4)));
typedef float gwh_f4 __attribute__((ext_vector_type(4)));

#define GWH_FROWS 16      /* parameters padded to the MFMA tile */
#define GWH_MAXSTEN 4     /* order 4 uses 4 evaluations per parameter */
#define GWH_GRAM_ROWS 4096 /* operand rows per Gram block */
#define GWH_FUSED_BINS 64  /* bins per block of the fused stencil + Gram kernel: one per lane of each wave */
#define GWH_FUSED_MAX_POINTS 128 /* points per pass of the fused path (passes pipeline with the host staging) */
#define GWH_FUSED_MIN_POINTS 16  /* fewer than these are not left for a last pass of their own */
#ifndef GWH_FUSED_WAVES
#define GWH_FUSED_WAVES 8 /* waves per block of the fused kernel: GWH_FROWS / GWH_FUSED_WAVES operand rows each */
#endif

#define GWH_FUSED_SLOTS 3 /* operand rows a wave of the fused kernel can take */

#include "gwh_basis.h"

static gwh_params non_parameter_options(const gwh_params &in)
{
    gwh_params w;
    memset(&w, 0, sizeof(w));
    w.chip = -1;
    w.phip = -1;
    w.sky_average = in.sky_average;
    w.f_ref = in.f_ref;
    w.gmst = in.gmst;
    w.shift_time = 0; /* fisher.cpp:2527 */
    w.shift_phase = in.shift_phase;
    w.dep_postmerger = in.dep_postmerger;
    /* fisher.cpp:2541-2570: the ppE terms and the gIMR lists travel with the parameters */
    w.ppe_nmod = in.ppe_nmod;
    w.ppe_theory = in.ppe_theory; /* a theory's map and redshift travel with its parameters (:2541-2545) */
    w.cosmology = in.cosmology;
    for (int i = 0; i < GWH_PPE_MAX; i++) {
        w.ppe_b[i] = in.ppe_b[i];
        w.ppe_beta[i] = in.ppe_beta[i];
    }
    memcpy(w.gimr_dphi, in.gimr_dphi, sizeof(w.gimr_dphi));
    memcpy(w.gimr_dsigma, in.gimr_dsigma, sizeof(w.gimr_dsigma));
    memcpy(w.gimr_dbeta, in.gimr_dbeta, sizeof(w.gimr_dbeta));
    memcpy(w.gimr_dalpha, in.gimr_dalpha, sizeof(w.gimr_dalpha));
    w.gimr_nlist = in.gimr_nlist;
    memcpy(w.gimr_list, in.gimr_list, sizeof(w.gimr_list));
    return w;
}

/* the table entry of a gIMR Fisher-basis code (GWH_GIMR_CODE_*), null for a parameter the waveform does not read */
static const double *gimr_slot(const gwh_params &p, int code)
{
    if (code < 0 || code >= GWH_GIMR_NCODES) return nullptr;
    if (code < GWH_GIMR_CODE_SIGMA(2)) return &p.gimr_dphi[code];
    if (code < GWH_GIMR_CODE_BETA(2)) return &p.gimr_dsigma[code - GWH_GIMR_CODE_SIGMA(2)];
    if (code < GWH_GIMR_CODE_ALPHA(2)) return &p.gimr_dbeta[code - GWH_GIMR_CODE_BETA(2)];
    return &p.gimr_dalpha[code - GWH_GIMR_CODE_ALPHA(2)];
}

/* Fisher basis of a model: the GR basis, with betappe[0..nmod) appended for the ppE methods
 * (fisher.cpp:2083-2088 unpack, :2424-2429 repack) or the listed gIMR deltas for the gIMR methods
 * (:2128-2158, :2473-2505; a repeated entry repacks into the table only through its first occurrence, the one
 * the waveform reads) */
static void unpack_mod(const gwh_params &p, int basis, int var, int nmod, double *v, int *lf)
{
    unpack(p, basis, v, lf);
    const int base = basis_dim(basis);
    for (int i = 0; i < nmod; i++) {
        const double *s = (var == 3) ? gimr_slot(p, p.gimr_list[i]) : &p.ppe_beta[i];
        v[base + i] = s ? *s : 0.0;
        lf[base + i] = 0;
    }
}
/* the fields of a record that depend on its vector's element i (-1: on any).  q may hold only the bytes of a record that
 * its model reads (gwh_record_bytes). */
static void repack_mod(const double *v, int basis, int var, int nmod, int element, gwh_params &q)
{
    const int base = basis_dim(basis);
    if (element < 0)
        repack(v, basis, q);
    else if (element < base)
        repack_element(v, basis, element, q);
    if (element >= 0 && element < base) return;
    for (int i = 0; i < nmod; i++) {
        if (var != 3) {
            q.ppe_beta[i] = v[base + i];
            continue;
        }
        bool first = true;
        for (int j = 0; j < i; j++) first &= (q.gimr_list[j] != q.gimr_list[i]);
        double *s = const_cast<double *>(gimr_slot(q, q.gimr_list[i]));
        if (first && s) *s = v[base + i];
    }
}

/* appended parameters of a model's Fisher basis: the ppE betas or the listed gIMR deltas (every point of a
 * batch with the same count) */
static int fisher_mods(int model, const gwh_params *params, int n, int *nmod)
{
    *nmod = 0;
    if (!gwh_model_valid(model)) return gwh_set_error(GWH_ERR_UNSUPPORTED, "unknown model");
    const int var = gwh_ppe_variant(model);
    if (var == 0 || n <= 0) return GWH_OK;
    const int m = (var == 3) ? params[0].gimr_nlist : params[0].ppe_nmod;
    if (var != 3 && (m < 0 || m > GWH_PPE_MAX))
        return gwh_set_error(GWH_ERR_UNSUPPORTED, "ppE term count outside 0..4");
    if (var == 3 && (m < 0 || m > GWH_GIMR_LIST_MAX))
        return gwh_set_error(GWH_ERR_UNSUPPORTED, "at most 16 gIMR deltas in a Fisher basis");
    for (int i = 0; i < n; i++) {
        if (((var == 3) ? params[i].gimr_nlist : params[i].ppe_nmod) != m)
            return gwh_set_error(GWH_ERR_INVALID, "every point of a modified-gravity Fisher batch needs the same "
                                                  "number of ppE terms / gIMR deltas");
        if (var == 3)
            for (int k = 0; k < m; k++)
                if (params[i].gimr_list[k] < -1 || params[i].gimr_list[k] >= GWH_GIMR_NCODES)
                    return gwh_set_error(GWH_ERR_INVALID, "bad gIMR Fisher-basis code");
    }
    *nmod = m;
    return GWH_OK;
}

static double host_dtoa(double ra, double dec, double gmst, int d1, int d2)
{
    const double *l1 = gwh_det_location[d1], *l2 = gwh_det_location[d2];
    double ha = gmst - ra;
    double e0 = cos(dec) * cos(ha), e1 = cos(dec) * -sin(ha), e2 = sin(dec);
    return ((l1[0] - l2[0]) * e0 + (l1[1] - l2[1]) * e1 + (l1[2] - l2[2]) * e2) / GWH_C_SI;
}

/* Bits of one stencil evaluation.  The GWH_EV_SAME_* ones compare it with the evaluation that its wave of the fused
 * kernel does just before it (of the previous row of the wave for the first evaluation of a row): the records are
 * functions of the parameter sets, so parts that depend on fields with equal bits only are equal bit for bit. */
#define GWH_EV_NO_TOF 1     /* order 4, +-2 eps: no time-of-flight phase (tc is shifted instead) */
#define GWH_EV_SAME_CORE 2  /* masses and spins: amplitude without prefactor, phase without shifts, Euler angles */
#define GWH_EV_SAME_TWIST 4 /* core and frame: the IMRPhenomPv2 twist-up factors */
#define GWH_EV_SAME_PHASE 8 /* core, time and phase shift: the phase at the first detector */

/* Stencil of one point: for every parameter i, S evaluations with weights c[i][s] (the difference
 * quotient including 1/eps and the log factor theta_i); the dim * S parameter sets go to `inst`, record_bytes apart,
 * their GWH_EV_* bits to `flags`: GWH_EV_NO_TOF marks the order-4 +-2 eps evaluations that shift tc instead
 * of using the time-of-flight phase (fisher.cpp:433-453). */
struct PointStencil {
    int S;
    double c[GWH_FROWS][GWH_MAXSTEN];
};

/* Step of one basis coordinate v: step > 0 is the absolute epsilon of fisher.cpp:158; step < 0 is a
 * step relative to the coordinate, |step| * |v| (|step| where v is exactly 0). */
static double coordinate_step(double step, double v)
{
    if (step > 0) return step;
    return v != 0 ? -step * fabs(v) : -step;
}

static int build_stencil(const gwh_params &p, int basis, int var, int nmod, int order, double step, int det,
                         int ref_det, char *inst, int record_bytes, int *flags, PointStencil &ps)
{
    int dim = basis_dim(basis) + nmod;
    double v[GWH_FROWS];
    int lf[GWH_FROWS];
    unpack_mod(p, basis, var, nmod, v, lf);
    gwh_params base = non_parameter_options(p);
    repack_mod(v, basis, var, nmod, -1, base); /* a stencil record differs from it where its one element enters */
    ps.S = (order >= 4) ? 4 : 2;
    for (int i = 0; i < GWH_FROWS; i++)
        for (int s = 0; s < GWH_MAXSTEN; s++) ps.c[i][s] = 0;
    for (int i = 0; i < dim; i++) {
        double eps = coordinate_step(step, v[i]);
        bool edge = (i == 8 && v[i] > .25 - eps); /* eta at the equal-mass boundary: one-sided */
        double fac = lf[i] ? v[i] : 1.0;
        double off[4];
        int S = ps.S;
        if (S == 2) {
            off[0] = edge ? 0 : eps;
            off[1] = -eps;
            double den = edge ? eps : 2 * eps;
            ps.c[i][0] = fac / den;
            ps.c[i][1] = -fac / den;
        } else {
            off[0] = edge ? 0 : 2 * eps;
            off[1] = eps;
            off[2] = -eps;
            off[3] = -2 * eps;
            double den = edge ? 6. * eps : 12. * eps;
            ps.c[i][0] = -fac / den;
            ps.c[i][1] = 8. * fac / den;
            ps.c[i][2] = -8. * fac / den;
            ps.c[i][3] = fac / den;
        }
        for (int s = 0; s < S; s++) {
            double w[GWH_FROWS];
            for (int j = 0; j < dim; j++) w[j] = v[j];
            w[i] = v[i] + off[s];
            gwh_params &q = *(gwh_params *)inst;
            memcpy(inst, &base, record_bytes);
            repack_mod(w, basis, var, nmod, i, q);
            bool two = (S == 4) && (s == 0 || s == 3);
            if (two && det != ref_det) q.tc -= host_dtoa(q.RA, q.DEC, q.gmst, ref_det, det);
            *flags++ = two ? GWH_EV_NO_TOF : 0;
            inst += record_bytes;
        }
    }
    return dim;
}

/* The GWH_EV_SAME_* bits of parameter set b evaluated right after a: which parts of its record (gwh_setup_kernel)
 * follow from fields with equal bits.  Core: masses, spins, the chi_p given, the ringdown option, the ppE / gIMR terms
 * (and for a theory's terms the distance, through its redshift).  IMRPhenomPv2 frame: core, phi_p, f_ref, inclination
 * and phase.  Phase: core, t_c and the reference: for IMRPhenomD the phase and f_ref, for IMRPhenomPv2 phi_p and f_ref
 * (its phase offset is the azimuth of J, in which inclination and phase do not enter).  mod: the model has ppE / gIMR
 * terms (the records of the others end before them). */
static int shared_parts(const gwh_params &a, const gwh_params &b, bool pv2, bool mod)
{
    auto eq = [](const void *x, const void *y, size_t n) { return memcmp(x, y, n) == 0; };
#define GWH_SAME(F) eq(&a.F, &b.F, sizeof(a.F))
    if (!(GWH_SAME(mass1) && GWH_SAME(mass2) && GWH_SAME(spin1) && GWH_SAME(spin2) && GWH_SAME(chip) &&
          GWH_SAME(dep_postmerger)))
        return 0;
    if (mod && !(GWH_SAME(ppe_nmod) && GWH_SAME(ppe_theory) && GWH_SAME(cosmology) && GWH_SAME(ppe_b) &&
                 GWH_SAME(ppe_beta) && GWH_SAME(gimr_dphi) && GWH_SAME(gimr_dsigma) && GWH_SAME(gimr_dbeta) &&
                 GWH_SAME(gimr_dalpha) && (!a.ppe_theory || GWH_SAME(DL))))
        return 0;
    int bits = GWH_EV_SAME_CORE;
    const bool ref = GWH_SAME(f_ref) && GWH_SAME(phip);
    if (ref && GWH_SAME(incl) && GWH_SAME(phiRef)) bits |= GWH_EV_SAME_TWIST;
    if (ref && GWH_SAME(tc) && GWH_SAME(shift_time) && GWH_SAME(shift_phase) && (pv2 || GWH_SAME(phiRef)))
        bits |= GWH_EV_SAME_PHASE;
    return bits;
}

/* vector operations of one evaluation after another (the fused kernel's code, counted by hand; only the proportions
 * matter): the projections always, the rest where it is not shared */
static int evaluation_cost(const gwh_params *prev, const gwh_params &p, bool pv2, bool mod, int ndet)
{
    const int same = prev ? shared_parts(*prev, p, pv2, mod) : 0;
    int c = 20 + 14 * ndet;
    if (!(same & GWH_EV_SAME_CORE)) c += pv2 ? 330 : 150;
    if (pv2 && !(same & GWH_EV_SAME_TWIST)) c += 130;
    if (!(same & GWH_EV_SAME_PHASE))
        c += 10 + 28 * ndet;
    else if (memcmp(&prev->RA, &p.RA, sizeof(p.RA)) || memcmp(&prev->DEC, &p.DEC, sizeof(p.DEC)))
        c += 28 * (ndet - 1); /* the arrival times; the first detector is their reference */
    return c;
}

/* Rows of the waves of the fused kernel: rows in decreasing order of their cost alone, each to the wave that ends
 * earliest with it, where what it shares with the wave's last row costs nothing.  inst: the dim * S parameter sets of
 * one point.  The choice changes only the time: an operand's value does not depend on its wave. */
static void assign_rows(const char *inst, int record_bytes, int dim, int S, bool pv2, bool mod, int ndet, int slots,
                        int (*row)[GWH_FUSED_SLOTS])
{
    int load[GWH_FUSED_WAVES] = {0}, used[GWH_FUSED_WAVES] = {0}, order[GWH_FROWS], alone[GWH_FROWS];
    auto cost = [&](int last, int i) { /* row i after row `last` (-1: first of its wave) */
        int c = 0;
        for (int s = 0; s < S; s++) {
            const int e = i * S + s, b = s ? e - 1 : (last >= 0 ? last * S + S - 1 : -1);
            const gwh_params *prev = b >= 0 ? (const gwh_params *)(inst + (size_t)b * record_bytes) : nullptr;
            c += evaluation_cost(prev, *(const gwh_params *)(inst + (size_t)e * record_bytes), pv2, mod, ndet);
        }
        return c;
    };
    for (int i = 0; i < dim; i++) {
        order[i] = i;
        alone[i] = cost(-1, i);
    }
    std::stable_sort(order, order + dim, [&](int x, int y) { return alone[x] > alone[y]; });
    for (int w = 0; w < GWH_FUSED_WAVES; w++)
        for (int h = 0; h < GWH_FUSED_SLOTS; h++) row[w][h] = -1;
    for (int n = 0; n < dim; n++) {
        int best = -1, end = 0;
        for (int w = 0; w < GWH_FUSED_WAVES; w++) {
            if (used[w] >= slots) continue;
            const int e = load[w] + cost(used[w] ? row[w][used[w] - 1] : -1, order[n]);
            if (best < 0 || e < end) {
                best = w;
                end = e;
            }
        }
        row[best][used[best]++] = order[n];
        load[best] = end;
    }
}

/* ------------------------------------------------------------------------- */
/* device: stencil                                                            */
/* ------------------------------------------------------------------------- */

/* One stencil evaluation's share in the difference quotient of a detector, dr + i di += c h, with the fused
 * multiply-adds written out: the operand rows and the bare derivatives round it alike wherever they are inlined (at
 * the reference's step of 1e-8 the quotient magnifies a last-bit difference a millionfold). */
#pragma clang fp contract(off)
/* IMRPhenomD: h = A K e^{-i x} from cos x and sin x */
__device__ __forceinline__ void add_response_d(double c, double A, double cs, double sn, const double *K, double &dr,
                                               double &di)
{
    const double er = A * cs, ei = A * sn;
    dr = fma(c, fma(er, K[0], ei * K[1]), dr);
    di = fma(c, fma(er, K[1], -(ei * K[0])), di);
}
/* IMRPhenomPv2: h = A (P h+ + Q hx) e^{-i x} */
__device__ __forceinline__ void add_response_pv2(double c, double A, double cs, double sn, const double *K, double hpr,
                                                 double hpi, double hcr, double hci, double &dr, double &di)
{
    const double Gr = fma(K[0], hpr, K[1] * hcr), Gi = fma(K[0], hpi, K[1] * hci), cA = c * A;
    dr = fma(cA, fma(Gr, cs, Gi * sn), dr);
    di = fma(cA, fma(Gi, cs, -(Gr * sn)), di);
}
#pragma clang fp contract(fast)

struct StencilArgs {
    const InstCoef *coef;        /* points x (dim*S [+1 central]) records */
    const int *flags;            /* points x records: GWH_EV_* bits of every stencil evaluation */
    const double *cw;            /* points x 16 x 4 stencil weights */
    int dim, S, per_point;       /* records per point */
    int d_first, d_count;        /* detectors of the event accumulated */
    int skyavg;                  /* sky-averaged IMRPhenomD: amplitude / phase derivatives */
    double sa_sign;              /* +1 (order 2) or -1 (order 4): i d(phase) A sign of fisher.cpp:299-315 */
    double *raw;                 /* non-null: write the bare derivatives dim x N complex (one point, one
                                    detector) instead of weighted Gram operand rows */
    int row[GWH_FUSED_WAVES][GWH_FUSED_SLOTS]; /* fused kernel: the operand rows of every wave, -1 none */
};

/* One lane per (bin, point, operand row): blockIdx.z is the row, and the S = 2 or 4 stencil evaluations of that
 * component are unrolled (S = a.S, a template parameter).  With the rows and stencil points as loops inside the
 * lane the compiler kept loop-invariant values live across them (IMRPhenomD 154, IMRPhenomPv2 190 VGPRs: 3 and
 * 2 waves per SIMD); now 115-127 VGPRs, 4 waves.  The arithmetic is unchanged. */
template <int MODEL, typename T, int S>
__global__ __launch_bounds__(GWH_TPB) void gwh_fisher_stencil_kernel(StencilArgs a, const EventDesc *__restrict__ events,
                                                                     int event0, T *__restrict__ rows)
{
    const int pt = blockIdx.y;
    const int i = blockIdx.z; /* operand row: component i < dim, zero padding up to GWH_FROWS */
    const int k = blockIdx.x * GWH_TPB + threadIdx.x;
    const EventDesc &E = events[event0];
    const int N = E.N;
    if (k >= N) return;
    const double f = E.f[k];
    const InstCoef *C = a.coef + (size_t)pt * a.per_point;
    const double *cw = a.cw + (size_t)pt * GWH_FROWS * GWH_MAXSTEN;
    const int *nt = a.flags + (size_t)pt * a.per_point;
    const size_t nrows = (size_t)a.d_count * N * 2;
    T *base = rows + (size_t)pt * nrows * GWH_FROWS;
    if (a.skyavg) {
        /* d h = dA + i sign d(phase) A_central (fisher.cpp:292-316); no detector projection */
        const InstCoef &Cc = C[a.dim * S];
        const BinPow bp = gwh_load_bin(E, k);
        double Ac = 0, u, ph;
        if (f <= Cc.fcut) gwh_phenomd_fp64(Cc, f, bp, Ac, ph, u);
        double sw = sqrt(E.wS[(size_t)a.d_first * N + k]);
        double dA = 0, dP = 0;
        if (i < a.dim) {
#pragma unroll
            for (int s = 0; s < S; s++) {
                const InstCoef &Ci = C[i * S + s];
                double A = 0, phi;
                gwh_phenomd_fp64(Ci, f, bp, A, phi, u);
                if (!(f <= Ci.fcut)) A = 0;
                dA += cw[i * GWH_MAXSTEN + s] * A;
                dP += cw[i * GWH_MAXSTEN + s] * (-phi); /* construct_phase returns -(Psi - tc (f-fref) - phic) */
            }
        }
        if (a.raw) {
            if (i < a.dim) {
                a.raw[((size_t)i * N + k) * 2] = dA;
                a.raw[((size_t)i * N + k) * 2 + 1] = a.sa_sign * dP * Ac;
            }
            return;
        }
        base[(size_t)i * N + k] = (T)(dA * sw);
        base[(size_t)(GWH_FROWS + i) * N + k] = (T)(a.sa_sign * dP * Ac * sw);
        return;
    }
    const BinPow bp = gwh_load_bin(E, k);
    double sw[GWH_MAXDET];
    for (int dd = 0; dd < GWH_MAXDET; dd++) sw[dd] = (dd < a.d_count) ? sqrt(E.wS[(size_t)(a.d_first + dd) * N + k]) : 0;
    double dr[GWH_MAXDET] = {0, 0, 0, 0}, di[GWH_MAXDET] = {0, 0, 0, 0};
    if (i < a.dim) {
#pragma unroll
        for (int s = 0; s < S; s++) {
            const InstCoef &Ci = C[i * S + s];
            if (!(f <= Ci.fcut)) continue; /* h = 0 above 0.2/M of this evaluation */
            const double c = cw[i * GWH_MAXSTEN + s];
            const bool tof = !(nt[i * S + s] & GWH_EV_NO_TOF);
            if (MODEL == GWH_IMRPHENOMD) {
                double A, phi, u;
                gwh_phenomd_fp64(Ci, f, bp, A, phi, u);
                for (int dd = 0; dd < GWH_MAXDET; dd++) {
                    if (dd >= a.d_count) break;
                    int d = a.d_first + dd;
                    double sn, cs;
                    gwh_sincos_table(phi + (tof ? Ci.det[d][3] : 0.0) * f, sn, cs);
                    add_response_d(c, A, cs, sn, Ci.det[d], dr[dd], di[dd]);
                }
            } else {
                double A, Phi, hpr, hpi, hcr, hci;
                gwh_pv2_fp64(Ci, f, bp, A, Phi, hpr, hpi, hcr, hci);
                for (int dd = 0; dd < GWH_MAXDET; dd++) {
                    if (dd >= a.d_count) break;
                    int d = a.d_first + dd;
                    double sn, cs;
                    gwh_sincos_table(Phi + (tof ? Ci.det[d][3] : 0.0) * f, sn, cs);
                    add_response_pv2(c, A, cs, sn, Ci.det[d], hpr, hpi, hcr, hci, dr[dd], di[dd]);
                }
            }
        }
    }
    if (a.raw) {
        if (i < a.dim) {
            a.raw[((size_t)i * N + k) * 2] = dr[0];
            a.raw[((size_t)i * N + k) * 2 + 1] = di[0];
        }
        return;
    }
    for (int dd = 0; dd < GWH_MAXDET; dd++) {
        if (dd >= a.d_count) break;
        T *pl = base + (size_t)dd * 2 * GWH_FROWS * N; /* planes (detector, re/im), component-major */
        pl[(size_t)i * N + k] = (T)(dr[dd] * sw[dd]);
        pl[(size_t)(GWH_FROWS + i) * N + k] = (T)(di[dd] * sw[dd]);
    }
}

/* the stencil kernel of a model, operand type and stencil size (a.S: 2 for order 2, 4 for order 4) */
template <typename T>
static void launch_stencil(bool pv2, dim3 g, hipStream_t st, const StencilArgs &a, const EventDesc *evp, int event,
                           T *rows)
{
    if (!pv2) {
        if (a.S == 4)
            hipLaunchKernelGGL((gwh_fisher_stencil_kernel<GWH_IMRPHENOMD, T, 4>), g, dim3(GWH_TPB), 0, st, a, evp,
                               event, rows);
        else
            hipLaunchKernelGGL((gwh_fisher_stencil_kernel<GWH_IMRPHENOMD, T, 2>), g, dim3(GWH_TPB), 0, st, a, evp,
                               event, rows);
    } else {
        if (a.S == 4)
            hipLaunchKernelGGL((gwh_fisher_stencil_kernel<GWH_IMRPHENOMPV2, T, 4>), g, dim3(GWH_TPB), 0, st, a, evp,
                               event, rows);
        else
            hipLaunchKernelGGL((gwh_fisher_stencil_kernel<GWH_IMRPHENOMPV2, T, 2>), g, dim3(GWH_TPB), 0, st, a, evp,
                               event, rows);
    }
}

/* ------------------------------------------------------------------------- */
/* device: Gram on the matrix cores                                           */
/* ------------------------------------------------------------------------- */

/* elements before row i of a packed lower triangle (and of a whole triangle of i rows): partial Gram matrices hold
 * only element (i, j <= i) of the parameters, 91 of the 256 for 13 parameters */
__host__ __device__ constexpr int gram_tri(int i) { return i * (i + 1) / 2; }

/* The operand rows of a point lie in planes (detector, real / imaginary part), component-major: component i of
 * bin k at plane[i * N + k], so the stencil kernels write whole waves of consecutive bins.  Each block: up to
 * GWH_GRAM_ROWS bins of one plane of one point, 4 waves; each wave accumulates a 16x16 tile of a a^T over its
 * bins, 4 bins per MFMA (lane l supplies component l%16 of bin k0 + l/16 as both A and B operand; eight
 * MFMAs' operands are loaded first, 32 consecutive bins of each component).  Output: per block the FP64 partial
 * sums of the lower triangle of the dim parameters (gram_tri). */
__global__ __launch_bounds__(GWH_TPB) void gwh_gram_kernel(const float *__restrict__ rows, int N, int nplanes,
                                                           int blk_per_plane, double *__restrict__ partial, int nblk,
                                                           int dim)
{
    __shared__ double lds[GWH_TPB / 64][256];
    const int pt = blockIdx.y, blk = blockIdx.x;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int plane = blk / blk_per_plane;
    const float *a = rows + ((size_t)pt * nplanes + plane) * GWH_FROWS * N + (size_t)(lane & 15) * N;
    int r0 = (blk % blk_per_plane) * GWH_GRAM_ROWS + wv * (GWH_GRAM_ROWS / 4);
    int r1 = r0 + GWH_GRAM_ROWS / 4;
    if (r1 > N) r1 = N;
    gwh_f4 acc = {0, 0, 0, 0};
    for (int r = r0; r < r1; r += 32) {
        float x[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int rr = r + 4 * u + (lane >> 4);
            x[u] = (rr < r1) ? a[rr] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[u], x[u], acc, 0, 0, 0);
    }
    /* result layout on gfx950 (checked on the device): column l % 16; row 4 (l / 16) + j for the FP32 instruction
     * (l / 16 + 4 j for the FP64 one of the fused kernel) */
    for (int j = 0; j < 4; j++) lds[wv][(4 * (lane >> 4) + j) * 16 + (lane & 15)] = acc[j];
    __syncthreads();
    const int ei = threadIdx.x >> 4, ej = threadIdx.x & 15;
    if (ei < dim && ej <= ei) {
        double s = lds[0][threadIdx.x];
        for (int w = 1; w < GWH_TPB / 64; w++) s += lds[w][threadIdx.x];
        partial[((size_t)pt * nblk + blk) * gram_tri(dim) + gram_tri(ei) + ej] = s;
    }
}

/* Column of the LDS plane that holds bin `col` of operand row `row` in the fused kernel: rows are rotated by two
 * bins each, so that the 32 lanes of a half wave, which read bins 4 q + {0, 1} or {2, 3} of all 16 rows, touch 32
 * different bank pairs.  Unrotated, the 16 rows (512 bytes apart) share their banks: SQ_LDS_BANK_CONFLICT was 9.4e7
 * of 1.2e8 LDS cycles of a 128-point pass of the 13-parameter IMRPhenomPv2 Fisher (846 -> 838 us: the
 * evaluations covered most of them). */
__device__ __forceinline__ int fused_col(int row, int col) { return (col + 2 * row) & (GWH_FUSED_BINS - 1); }

/* The stencil and the FP64 Gram in one kernel: one block of WAVES waves per (point, chunk of 64 bins).  Each wave
 * evaluates the operand rows the host gave it (a.row) -- the S stencil evaluations of a component, unrolled,
 * projected on every detector and weighted by sqrt(4 w / S_n) -- for the chunk's bins, one per lane, into LDS planes
 * (detector, re/im) x row x bin (zero for padding rows and bins past the grid); then the waves contract every plane
 * on the FP64 matrix cores (v_mfma_f64_16x16x4f64: 4 bins per instruction, lane l supplying component l % 16 of bin
 * l / 16 as both operands; wave w takes the (plane, 4-bin) slices w, w + WAVES, ...), and the block writes one
 * partial Gram, summed over its waves in a fixed order.  The operand rows never leave the CU.
 *
 * Most parameters of a basis leave most of the waveform as it is: sky position, polarisation, inclination, phase,
 * time and distance move neither the amplitude's shape nor the phase's, and polarisation and distance not even the
 * phase in a detector.  What an evaluation shares with the one its wave did before (GWH_EV_SAME_*, equal bits by
 * construction) is kept in registers instead of computed again, and rows that share are given to the same wave:
 * 12 instead of 22 evaluations of the waveform for the 11 IMRPhenomD parameters (4 rows change it, the other 7 lie
 * in 4 waves), 13 instead of 26 for the 13 of IMRPhenomPv2.  The arithmetic of an operand does not depend on which
 * wave does it or after what.  Per launch, every evaluation in full -> shared, over the live chunks only:
 * IMRPhenomPv2, 128 points x 16225 bins x 3 detectors 838 -> 307 us, IMRPhenomD, 12 points x 65539 bins x 3 418 -> 238
 * us; the 7-parameter sky-averaged matrix of one point on 4017 bins, which went through operand rows in HBM, 36 ->
 * 8.5 us.
 *
 * Two blocks share a CU by their LDS: 4 waves a SIMD, which issue 41 % (IMRPhenomPv2) and 46 % (IMRPhenomD) of the
 * vector rate and wait for 62 and 50 % of their cycles.
 *
 * SKY: the sky-averaged IMRPhenomD basis, d h = dA + i sign d(phase) A_central (fisher.cpp:292-316) in planes
 * (dA, d(phase) A) of one detector row. */
template <int MODEL, int S, int WAVES, int SLOTS, bool SKY>
__global__ __launch_bounds__(WAVES * 64) void gwh_fisher_fused_kernel(StencilArgs a,
                                                                     const EventDesc *__restrict__ events,
                                                                     int event0, double *__restrict__ partial, int nbc)
{
    __shared__ double lds[2 * GWH_MAXDET][GWH_FROWS][GWH_FUSED_BINS]; /* 64 KiB */
    const int pt = blockIdx.y, bc = blockIdx.x;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const EventDesc &E = events[event0];
    const int N = E.N;
    const int k0 = bc * GWH_FUSED_BINS + lane;
    const bool in = k0 < N;
    const int k = in ? k0 : N - 1;
    const InstCoef *C = a.coef + (size_t)pt * a.per_point;
    const double *cw = a.cw + (size_t)pt * GWH_FROWS * GWH_MAXSTEN;
    const int *fl = a.flags + (size_t)pt * a.per_point;
    const int nplanes = 2 * a.d_count;
    for (int e = threadIdx.x; e < nplanes * (GWH_FROWS - a.dim) * GWH_FUSED_BINS; e += WAVES * 64) {
        const int r = e / GWH_FUSED_BINS;
        lds[r % nplanes][a.dim + r / nplanes][e % GWH_FUSED_BINS] = 0.0; /* padding rows */
    }
    double f = 0, sw[GWH_MAXDET] = {0, 0, 0, 0}, Ac = 0;
    BinPow bp = {0, 0, 0, 0, 0};
    /* the previous evaluation of this wave */
    double a0 = 0, psi = 0, u = 0, Phi = 0, hpr = 0, hpi = 0, hcr = 0, hci = 0;
    Pv2Angles ang = {0, 0, 0, 0};
    double zc[GWH_MAXDET] = {0, 0, 0, 0}, zs[GWH_MAXDET] = {0, 0, 0, 0}, kz[GWH_MAXDET] = {0, 0, 0, 0};
    if (a.row[wv][0] >= 0) {
        f = gwh_g(E.f)[k];
        bp = gwh_load_bin(E, k);
#pragma unroll
        for (int dd = 0; dd < (SKY ? 1 : GWH_MAXDET); dd++)
            if (dd < a.d_count) sw[dd] = in ? sqrt(gwh_g(E.wS)[(size_t)(a.d_first + dd) * N + k]) : 0.0;
        /* a lane above the cutoff evaluates its bin with a zero amplitude, so the phase has to be finite: a bin of
           infinite frequency, or none, is taken at 1e15 Hz, above every cutoff (a branch that no other wave enters, behind the
           loads: selects in every wave took 2 % of the kernel, the branch in front of the weights' loads 1.5 %) */
        if (!SKY && __ballot(!(f < HUGE_VAL))) {
            const bool none = !(f < HUGE_VAL);
            f = none ? 1e15 : f;
            bp = none ? BinPow{34.538776394910684, 1e5, 1e-5, 3.1622776601683795e-18, 1.7782794100389228e11} : bp;
        }
        if (SKY) {
            const InstCoef &Cc = C[a.dim * S];
            double ph;
            if (f <= Cc.fcut) gwh_phenomd_fp64(Cc, f, bp, Ac, ph, u);
        }
    }
    /* unrolled: no loop for the compiler to hoist values across */
#pragma unroll
    for (int h = 0; h < SLOTS; h++) {
        const int i = a.row[wv][h]; /* uniform over the wave */
        if (i < 0) break;
        double dr[GWH_MAXDET] = {0, 0, 0, 0}, di[GWH_MAXDET] = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < S; s++) {
            const InstCoef &Ci = C[i * S + s];
            const int same = fl[i * S + s];
            const double c = cw[i * GWH_MAXSTEN + s];
            const bool live = f <= Ci.fcut; /* h = 0 above 0.2/M of this evaluation */
            if (SKY) {
                /* the phase counts up to the cutoff of the central amplitude */
                if (!__ballot(!(f > Ci.fcut) || !(f > C[a.dim * S].fcut))) continue;
                if (!(same & GWH_EV_SAME_CORE)) gwh_phenomd_core(Ci, f, bp, a0, psi, u);
                dr[0] += c * (live ? Ci.amp_pref * a0 : 0.0);
                di[0] += c * -gwh_phase_shift(Ci, f, psi); /* construct_phase returns -(Psi - tc (f-fref) - phic) */
                continue;
            }
            if (!__ballot(live)) continue;
            if (!(same & GWH_EV_SAME_CORE)) {
                gwh_phenomd_core<false, MODEL == GWH_IMRPHENOMPV2>(Ci, f, bp, a0, psi, u);
                if (MODEL == GWH_IMRPHENOMPV2) ang = gwh_pv2_angles(Ci, u, bp);
            }
            if (MODEL == GWH_IMRPHENOMPV2 && !(same & GWH_EV_SAME_TWIST)) gwh_pv2_twist(Ci, ang, hpr, hpi, hcr, hci);
            if (!(same & GWH_EV_SAME_PHASE)) {
                Phi = gwh_phase_shift(Ci, f, psi);
                if (MODEL == GWH_IMRPHENOMPV2) Phi = gwh_pv2_phase(Ci, f, Phi, ang);
            }
            const double A = live ? Ci.amp_pref * a0 : 0.0;
#pragma unroll
            for (int dd = 0; dd < GWH_MAXDET; dd++) {
                if (dd >= a.d_count) break;
                const int d = a.d_first + dd;
                const double kd = (same & GWH_EV_NO_TOF) ? 0.0 : Ci.det[d][3];
                if (!(same & GWH_EV_SAME_PHASE) || __double_as_longlong(kd) != __double_as_longlong(kz[dd])) {
                    gwh_sincos_table(Phi + kd * f, zs[dd], zc[dd]);
                    kz[dd] = kd;
                }
                if (MODEL == GWH_IMRPHENOMD)
                    add_response_d(c, A, zc[dd], zs[dd], Ci.det[d], dr[dd], di[dd]);
                else
                    add_response_pv2(c, A, zc[dd], zs[dd], Ci.det[d], hpr, hpi, hcr, hci, dr[dd], di[dd]);
            }
        }
        if (SKY) {
            lds[0][i][fused_col(i, lane)] = dr[0] * sw[0];
            lds[1][i][fused_col(i, lane)] = a.sa_sign * di[0] * Ac * sw[0];
        } else {
#pragma unroll
            for (int dd = 0; dd < GWH_MAXDET; dd++) {
                if (dd >= a.d_count) break;
                lds[2 * dd][i][fused_col(i, lane)] = dr[dd] * sw[dd];
                lds[2 * dd + 1][i][fused_col(i, lane)] = di[dd] * sw[dd];
            }
        }
    }
    __syncthreads();
    gwh_d4 acc = {0, 0, 0, 0};
    const int nslice = nplanes * (GWH_FUSED_BINS / 4);
    for (int t = wv; t < nslice; t += WAVES) {
        const int pl = t / (GWH_FUSED_BINS / 4), q = t % (GWH_FUSED_BINS / 4);
        const int row = lane & 15;
        const double x = lds[pl][row][fused_col(row, 4 * q + (lane >> 4))];
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x, x, acc, 0, 0, 0);
    }
    __syncthreads(); /* the planes are read: the LDS now holds the waves' partial matrices */
    double(*part)[256] = reinterpret_cast<double(*)[256]>(&lds[0][0][0]);
    for (int j = 0; j < 4; j++) part[wv][((lane >> 4) + 4 * j) * 16 + (lane & 15)] = acc[j];
    __syncthreads();
    /* the product of the operand with itself is symmetric bit for bit: the lower triangle of the parameters */
    const int ei = threadIdx.x >> 4, ej = threadIdx.x & 15;
    if (ei < a.dim && ej <= ei) {
        double sum = part[0][threadIdx.x];
        for (int w = 1; w < WAVES; w++) sum += part[w][threadIdx.x];
        partial[((size_t)pt * nbc + bc) * gram_tri(a.dim) + gram_tri(ei) + ej] = sum;
    }
}

/* the fused kernel of a model, stencil size and basis; grid: chunks of 64 bins x points.  Order 2 gives a wave up to
 * three rows; order 4 (single points only) two, which keeps its unrolled code within the instruction cache. */
static void launch_fused(bool pv2, bool sky, dim3 g, hipStream_t st, const StencilArgs &a, const EventDesc *evp,
                         int event, double *partial)
{
    constexpr int W = GWH_FUSED_WAVES;
    const dim3 b(W * 64);
    const int nbc = (int)g.x;
#define GWH_FUSED(M, S, SLOTS, SKY)                                                                                 \
    hipLaunchKernelGGL((gwh_fisher_fused_kernel<M, S, W, SLOTS, SKY>), g, b, 0, st, a, evp, event, partial, nbc)
    if (sky && a.S == 4)
        GWH_FUSED(GWH_IMRPHENOMD, 4, 2, true);
    else if (sky)
        GWH_FUSED(GWH_IMRPHENOMD, 2, 2, true);
    else if (!pv2 && a.S == 4)
        GWH_FUSED(GWH_IMRPHENOMD, 4, 2, false);
    else if (!pv2)
        GWH_FUSED(GWH_IMRPHENOMD, 2, GWH_FUSED_SLOTS, false);
    else if (a.S == 4)
        GWH_FUSED(GWH_IMRPHENOMPV2, 4, 2, false);
    else
        GWH_FUSED(GWH_IMRPHENOMPV2, 2, GWH_FUSED_SLOTS, false);
#undef GWH_FUSED
}

/* Fixed-order FP64 sum of the Gram partials: one block of 1024 threads per (point, 16 elements of the packed lower
 * triangle).  Thread (q, e) sums its element over blocks q, q + 64, ... in increasing order (16 consecutive elements
 * per load, 128 bytes), the 64 sums are added pairwise in LDS, and each element is written to both halves of the
 * matrix, as calculate_fisher_elements assigns out[k][j] = out[j][k].  The loads of a thread are a serial chain, so
 * the blocks are spread over 64 threads per element and not over four: 12 points of 1025 blocks 68 -> 8.5 us, 128
 * points of 254 blocks 18.7 -> 7.3 us. */
__global__ __launch_bounds__(1024) void gwh_gram_reduce_kernel(const double *__restrict__ partial, int nblk, int dim,
                                                               double scale, double *__restrict__ out,
                                                               double *__restrict__ host)
{
    __shared__ double red[64][17];
    const int pt = blockIdx.x, tri = gram_tri(dim);
    const int e = blockIdx.y * 16 + (threadIdx.x & 15), q = threadIdx.x >> 4;
    const double *pp = partial + (size_t)pt * nblk * tri + e;
    double acc = 0;
    if (e < tri)
        for (int b = q; b < nblk; b += 64) acc += pp[(size_t)b * tri];
    red[q][threadIdx.x & 15] = acc;
    __syncthreads();
    for (int w = 32; w > 0; w >>= 1) {
        if (q < w) red[q][threadIdx.x & 15] += red[q + w][threadIdx.x & 15];
        __syncthreads();
    }
    if (q == 0 && e < tri) {
        int i = 0;
        while (gram_tri(i + 1) <= e) i++;
        const int j = e - gram_tri(i);
        const double v = red[0][threadIdx.x] * scale;
        double *o = out + (size_t)pt * dim * dim;
        o[i * dim + j] = v;
        o[j * dim + i] = v;
        o = host + (size_t)pt * dim * dim;
        o[i * dim + j] = v;
        o[j * dim + i] = v;
    }
}

/* FP64 LU inverse with partial pivoting per point -> marginal sigmas sqrt(Sigma_ii): one wave per point.  The
 * elimination of step k updates every element (i, j > k) once, spread over the lanes, in the same order of steps
 * as a serial elimination; the pivot is the first row of largest |a_ik| (a NaN diagonal keeps its row); lane c then
 * solves L U x = P e_c by forward and back substitution (loops of fixed length, so x stays in registers). */
__global__ __launch_bounds__(64) void gwh_fisher_invert_kernel(const double *__restrict__ F, int n, int dim,
                                                               double *__restrict__ sigma)
{
    __shared__ double a[GWH_FROWS][GWH_FROWS + 1];
    __shared__ int perm[GWH_FROWS];
    __shared__ int piv_s;
    const int pt = blockIdx.x, lane = threadIdx.x;
    if (pt >= n) return; /* the whole block */
    const double *M = F + (size_t)pt * dim * dim;
    for (int e = lane; e < dim * dim; e += 64) a[e / dim][e % dim] = M[e];
    if (lane < dim) perm[lane] = lane;
    __syncthreads();
    bool sing = false;
    for (int k = 0; k < dim; k++) {
        /* pivot: the first row i >= k of largest |a_ik| */
        if (lane == 0) {
            int piv = k;
            double mx = fabs(a[k][k]);
            for (int i = k + 1; i < dim; i++)
                if (fabs(a[i][k]) > mx) {
                    mx = fabs(a[i][k]);
                    piv = i;
                }
            piv_s = (mx == 0) ? -1 : piv;
        }
        __syncthreads();
        const int piv = piv_s;
        if (piv < 0) {
            sing = true;
            break;
        }
        if (piv != k) {
            if (lane < dim) {
                const double t = a[k][lane];
                a[k][lane] = a[piv][lane];
                a[piv][lane] = t;
            }
            if (lane == 0) {
                const int t = perm[k];
                perm[k] = perm[piv];
                perm[piv] = t;
            }
            __syncthreads();
        }
        if (lane > k && lane < dim) a[lane][k] /= a[k][k];
        __syncthreads();
        const int m = dim - k - 1;
        for (int e = lane; e < m * m; e += 64) {
            const int i = k + 1 + e / m, j = k + 1 + e % m;
            a[i][j] -= a[i][k] * a[k][j];
        }
        __syncthreads();
    }
    const int c = lane;
    if (c >= dim) return;
    if (sing) {
        sigma[(size_t)pt * dim + c] = __longlong_as_double(0x7ff8000000000000LL);
        return;
    }
    double x[GWH_FROWS];
#pragma unroll
    for (int i = 0; i < GWH_FROWS; i++) {
        x[i] = 0;
        if (i < dim) {
            double s = (perm[i] == c) ? 1.0 : 0.0;
#pragma unroll
            for (int j = 0; j < i; j++) s -= a[i][j] * x[j];
            x[i] = s;
        }
    }
#pragma unroll
    for (int i = GWH_FROWS - 1; i >= 0; i--) {
        if (i < dim) {
            double s = x[i];
#pragma unroll
            for (int j = i + 1; j < GWH_FROWS; j++)
                if (j < dim) s -= a[i][j] * x[j];
            x[i] = s / a[i][i];
        }
    }
    double xc = 0;
#pragma unroll
    for (int i = 0; i < GWH_FROWS; i++)
        if (i == c) xc = x[i];
    sigma[(size_t)pt * dim + c] = sqrt(xc);
}

/* ------------------------------------------------------------------------- */
/* host driver                                                                */
/* ------------------------------------------------------------------------- */

/* Fisher matrices of `n` points on a resident event.  d_first/d_count select the detectors whose
 * responses enter (network sum = all); ref_det is the arrival-time reference. */
static int fisher_run(int event, int model, int basis, int precision, const gwh_params *params, int n, int order,
                      double eps, int d_first, int d_count, int det_for_tof, int ref_det, double scale, double *out,
                      double *sigma, FisherScratch &F, double *raw = nullptr)
{
    Engine &E = gwh_engine();
    if (!(eps != 0) || !std::isfinite(eps))
        return gwh_set_error(GWH_ERR_INVALID, "the Fisher step must be finite and nonzero");
    Event ev;
    {
        /* copy of the descriptor; the device block stays valid because broker requests pin the
           event (gwh_event_destroy then refuses) and direct callers hold it for the call */
        std::lock_guard<std::recursive_mutex> lk(E.mu);
        ev = E.events[event];
    }
    int nmod, rc0;
    if ((rc0 = fisher_mods(model, params, n, &nmod)) != GWH_OK) return rc0;
    const bool pv2 = gwh_is_pv2(model);
    int dim = basis_dim(basis) + nmod;
    if (dim > GWH_FROWS) return gwh_set_error(GWH_ERR_UNSUPPORTED, "at most 16 Fisher parameters");
    bool sky = (basis == GWH_BASIS_PHENOMD_SKYAVG);
    if (sky && pv2)
        return gwh_set_error(GWH_ERR_UNSUPPORTED, "Sky averaged IMRPhenomP is not supported for regular fishers.");
    int S = (order >= 4) ? 4 : 2;
    int per_point = dim * S + (sky ? 1 : 0);
    const int N = ev.N;
    const size_t nrows = (size_t)(sky ? 1 : d_count) * N * 2;
    const size_t row_bytes = GWH_FROWS * (raw ? 8 : 4); /* operand rows: FP32 Gram, bare derivatives */
    /* the FP64 Gram runs fused with the stencil (no operand rows in HBM); the FP32 Gram and the bare derivatives go
       through operand rows */
    const bool fused = !raw && precision != GWH_FISHER_GRAM_FP32;
    /* points per pass: bounded operand buffer (F.max_operand, 1 GiB unless a caller's budget says less); fused,
       the partial Gram matrices take its place */
    size_t per_pt_bytes = nrows * row_bytes;
    const int nplanes = (int)(nrows / N); /* (detector, re/im) planes of a point's operand rows */
    const int blk_per_plane = (N + GWH_GRAM_ROWS - 1) / GWH_GRAM_ROWS;
    int nblk = fused ? (N + GWH_FUSED_BINS - 1) / GWH_FUSED_BINS : nplanes * blk_per_plane;
    const size_t part_bytes = (size_t)nblk * gram_tri(dim) * 8; /* partial Gram matrices of a point */
    if (fused) per_pt_bytes = part_bytes;
    int chunk = (int)std::max<size_t>(1, F.max_operand / per_pt_bytes);
    if (chunk > n) chunk = n;
    if (chunk > 65535) chunk = 65535;
    if (fused && chunk > GWH_FUSED_MAX_POINTS) chunk = GWH_FUSED_MAX_POINTS;
    int rc;
    if (!fused && (rc = F.deriv.ensure((size_t)chunk * per_pt_bytes)) != GWH_OK) return rc;
    if ((rc = F.gram.ensure((size_t)chunk * part_bytes)) != GWH_OK) return rc;
    if ((rc = F.out.ensure((size_t)n * dim * dim * 8)) != GWH_OK) return rc;
    const bool mod = gwh_ppe_variant(model) != 0;
    const int record_bytes = gwh_record_bytes(model);
    StencilArgs a;
    const int slots = (S == 4 || sky) ? 2 : GWH_FUSED_SLOTS; /* as launch_fused */
    const size_t out_bytes = (size_t)dim * dim * 8; /* a point's matrix */
    /* the pass that each staging holds, whose matrices the caller does not have yet */
    struct Pending {
        int p0, np;
        const char *m;
    } pending[2] = {{0, 0, nullptr}, {0, 0, nullptr}};
    auto collect = [&](int sl) {
        if (!pending[sl].np) return GWH_OK;
        GWH_HIP(hipEventSynchronize(F.stage_done[sl]));
        memcpy(out + (size_t)pending[sl].p0 * dim * dim, pending[sl].m, pending[sl].np * out_bytes);
        pending[sl].np = 0;
        return GWH_OK;
    };
    /* buffers of the largest pass */
    const size_t ni_max = (size_t)chunk * per_point,
                 misc_max = (size_t)chunk * GWH_FROWS * GWH_MAXSTEN * 8 + (ni_max * 4 + 7) / 8 * 8,
                 stage_max = ni_max * record_bytes + misc_max + chunk * out_bytes;
    if ((rc = F.coef.ensure(ni_max * sizeof(InstCoef))) != GWH_OK) return rc;
    if ((rc = F.misc.ensure(misc_max + 256)) != GWH_OK) return rc;
    /* the device waits for the host to build the first pass: of several, the first two are a quarter and a half of the
       others */
    SettleStream settle(F.stream);
    int slot = 0, pass = (fused && n > chunk) ? std::max(1, chunk / 4) : chunk;
    for (int p0 = 0, np; p0 < n; p0 += np, slot ^= 1, pass = std::min(2 * pass, chunk)) {
        np = std::min(pass, n - p0);
        if (fused && n - p0 - np < GWH_FUSED_MIN_POINTS && n - p0 <= chunk) np = n - p0;
        const int ni = np * per_point;
        const size_t ncw = (size_t)np * GWH_FROWS * GWH_MAXSTEN;
        /* a pass in pinned memory, which the kernels read and write: records, weights and flags (these two copied by the
           setup's launch), then the matrices.  As copies on the stream these took 50 us between two passes (384 points:
           1241 -> 1065 us; building whole records anew for every stencil point, and the first pass no shorter than the
           others: 1348 us). */
        const size_t rec_bytes = (size_t)ni * record_bytes, flag_bytes = ((size_t)ni * 4 + 7) / 8 * 8,
                     misc_bytes = ncw * 8 + flag_bytes;
        if (F.stage_done[slot]) GWH_HIP(hipEventSynchronize(F.stage_done[slot])); /* its last pass has ended */
        else GWH_HIP(hipEventCreateWithFlags(&F.stage_done[slot], hipEventDisableTiming));
        if ((rc = collect(slot)) != GWH_OK) return rc;
        if (F.stage_cap[slot] < stage_max) {
            if (F.stage[slot]) GWH_HIP(hipHostFree(F.stage[slot]));
            F.stage[slot] = nullptr;
            F.stage_cap[slot] = 0;
            if ((rc = gwh_pinned_alloc(&F.stage[slot], &F.stage_dev[slot], stage_max + stage_max / 4)) != GWH_OK) return rc;
            F.stage_cap[slot] = stage_max + stage_max / 4;
        }
        char *st = (char *)F.stage[slot];
        double *cw = (double *)(st + rec_bytes);
        int *flags = (int *)(cw + ncw); /* GWH_EV_* bits of every record */
        double fcut = 0;                /* highest cutoff of a record */
        for (int q = 0; q < np; q++) {
            PointStencil ps;
            char *rec = st + (size_t)q * per_point * record_bytes;
            int *fl = flags + (size_t)q * per_point;
            build_stencil(params[p0 + q], basis, gwh_ppe_variant(model), nmod, order, eps, det_for_tof, ref_det, rec,
                          record_bytes, fl, ps);
            if (sky) { /* central amplitude: the caller's parameters */
                memcpy(rec + (size_t)(per_point - 1) * record_bytes, &params[p0 + q], record_bytes);
                fl[per_point - 1] = 0;
            }
            auto at = [&](int e) -> const gwh_params & { return *(const gwh_params *)(rec + (size_t)e * record_bytes); };
            if (fused) {
                if (p0 == 0 && q == 0)
                    assign_rows(rec, record_bytes, dim, S, pv2, mod, sky ? 1 : d_count, slots, a.row);
                for (int w = 0; w < GWH_FUSED_WAVES; w++) {
                    int prev = -1;
                    for (int h = 0; h < slots && a.row[w][h] >= 0; h++)
                        for (int e = a.row[w][h] * S; e < (a.row[w][h] + 1) * S; prev = e++)
                            if (prev >= 0) fl[e] |= shared_parts(at(prev), at(e), pv2, mod);
                }
            }
            for (int e = 0; e < per_point; e++) {
                const double c = .2 / (at(e).mass1 * GWH_MSOL_SEC + at(e).mass2 * GWH_MSOL_SEC);
                if (!(c <= fcut || fcut != fcut)) fcut = c; /* NaN stays: every chunk */
            }
            memcpy(cw + (size_t)q * GWH_FROWS * GWH_MAXSTEN, ps.c, sizeof(ps.c));
        }
        char *misc = (char *)F.misc.p, *dev = (char *)F.stage_dev[slot];
        if ((rc = gwh_setup_launch(nullptr, event, model, (const gwh_params *)dev, ni, F.coef.as<InstCoef>(), F.stream,
                                   record_bytes, {(const double *)(dev + rec_bytes), (double *)misc,
                                                  (int)(misc_bytes / 8)})) != GWH_OK)
            return rc;
        a.coef = F.coef.as<const InstCoef>();
        a.cw = (const double *)misc;
        a.flags = (const int *)(misc + ncw * 8);
        a.dim = dim;
        a.S = S;
        a.per_point = per_point;
        a.d_first = d_first;
        a.d_count = sky ? 1 : d_count;
        a.skyavg = sky;
        a.sa_sign = (S == 4) ? -1.0 : 1.0;
        a.raw = nullptr;
        dim3 g((N + GWH_TPB - 1) / GWH_TPB, np, GWH_FROWS); /* z: operand row */
        const EventDesc *evp = (const EventDesc *)E.d_events;
        if (raw) {
            /* bare derivatives of one point on one detector (calculate_derivatives) */
            if ((rc = F.raw.ensure((size_t)dim * N * 16)) != GWH_OK) return rc;
            a.raw = F.raw.as<double>();
            a.d_count = 1;
            dim3 g1((N + GWH_TPB - 1) / GWH_TPB, 1, dim);
            launch_stencil<double>(pv2, g1, F.stream, a, evp, event, F.deriv.as<double>());
            GWH_HIP(hipGetLastError());
            GWH_HIP(hipMemcpyAsync(raw, F.raw.p, (size_t)dim * N * 16, hipMemcpyDeviceToHost, F.stream));
            GWH_HIP(hipStreamSynchronize(F.stream));
            return settle.done();
        }
        int nb = nblk; /* partial Gram matrices of a point */
        if (fused) {
            /* only the 64-bin chunks that begin at or below some record's cutoff 0.2/M hold anything (a margin covers
               the rounding of the device's own cutoff, which decides bin by bin): 77 of 254 chunks for 65 solar masses
               on 20-2048 Hz */
            const std::vector<double> &cf = *ev.chunk_fmin;
            while (nb > 1 && cf[nb - 1] > fcut * (1 + 1e-9)) nb--;
            launch_fused(pv2, sky, dim3(nb, np), F.stream, a, evp, event, F.gram.as<double>());
        } else {
            launch_stencil<float>(pv2, g, F.stream, a, evp, event, F.deriv.as<float>());
            GWH_HIP(hipGetLastError());
            hipLaunchKernelGGL(gwh_gram_kernel, dim3(nblk, np), dim3(GWH_TPB), 0, F.stream, F.deriv.as<const float>(), N,
                               nplanes, blk_per_plane, F.gram.as<double>(), nblk, dim);
        }
        GWH_HIP(hipGetLastError());
        hipLaunchKernelGGL(gwh_gram_reduce_kernel, dim3(np, (gram_tri(dim) + 15) / 16), dim3(1024), 0, F.stream, F.gram.as<const double>(),
                           nb, dim, scale, F.out.as<double>() + (size_t)p0 * dim * dim,
                           (double *)(dev + rec_bytes + misc_bytes));
        GWH_HIP(hipGetLastError());
        GWH_HIP(hipEventRecord(F.stage_done[slot], F.stream));
        pending[slot] = {p0, np, st + rec_bytes + misc_bytes};
    }
    if (sigma) {
        if ((rc = F.sig.ensure((size_t)n * dim * 8)) != GWH_OK) return rc;
        hipLaunchKernelGGL(gwh_fisher_invert_kernel, dim3(n), dim3(64), 0, F.stream,
                           F.out.as<const double>(), n, dim, F.sig.as<double>());
        GWH_HIP(hipGetLastError());
        GWH_HIP(hipMemcpyAsync(sigma, F.sig.p, (size_t)n * dim * 8, hipMemcpyDeviceToHost, F.stream));
    }
    for (int k = 0; k < 2; k++, slot ^= 1)
        if ((rc = collect(slot)) != GWH_OK) return rc;
    if (sigma) GWH_HIP(hipStreamSynchronize(F.stream));
    return settle.done();
}

int gwh_fisher_batch_with(int event, int model, int basis, int precision, const gwh_params *params, int n, int dim,
                          double epsilon, double *out, double *sigma, FisherScratch &F)
{
    Engine &E = gwh_engine();
    int rc = gwh_ensure_init();
    if (rc != GWH_OK) return rc;
    if (n <= 0) return GWH_OK;
    if (!params || !out) return gwh_set_error(GWH_ERR_INVALID, "null argument");
    Event ev;
    {
        std::lock_guard<std::recursive_mutex> lk(E.mu);
        if (event < 0 || event >= GWH_MAX_EVENTS || !E.events[event].live)
            return gwh_set_error(GWH_ERR_INVALID, "unknown event");
        ev = E.events[event];
    }
    int nmod;
    if ((rc = fisher_mods(model, params, n, &nmod)) != GWH_OK) return rc;
    if (basis_dim(basis) < 0 || basis_dim(basis) + nmod != dim)
        return gwh_set_error(GWH_ERR_INVALID, "dimension does not match the parameter basis (and ppE terms)");
    if (precision != GWH_FP64 && precision != GWH_MIXED && precision != GWH_FISHER_GRAM_FP32)
        return gwh_set_error(GWH_ERR_INVALID, "bad precision");
    if ((basis == GWH_BASIS_PV2_FULL || basis == GWH_BASIS_PV2_MCMC) != gwh_is_pv2(model))
        return gwh_set_error(GWH_ERR_INVALID, "basis does not belong to the model");
    /* the event's weights use the likelihood's df = f[N/2]-f[N/2-1]; the Fisher uses f[1]-f[0] */
    double scale = ev.df_fisher / ev.df_like;
    return fisher_run(event, model, basis, precision, params, n, 2, epsilon, 0, ev.D, ev.det[0], ev.det[0], scale, out,
                      sigma, F);
}

size_t gwh_fisher_batch_bytes(int event, int model, int basis, int precision, const gwh_params *params, int n,
                              size_t max_operand, const FisherScratch &F, bool want_sigma)
{
    Engine &E = gwh_engine();
    Event ev;
    {
        std::lock_guard<std::recursive_mutex> lk(E.mu);
        if (event < 0 || event >= GWH_MAX_EVENTS || !E.events[event].live) return 0;
        ev = E.events[event];
    }
    int nmod;
    if (n <= 0 || !params || fisher_mods(model, params, n, &nmod) != GWH_OK || basis_dim(basis) < 0) return 0;
    /* the buffers fisher_run ensures (order 2) */
    const int dim = basis_dim(basis) + nmod;
    const bool sky = (basis == GWH_BASIS_PHENOMD_SKYAVG);
    const size_t per_point = (size_t)dim * 2 + (sky ? 1 : 0);
    const size_t nrows = (size_t)(sky ? 1 : ev.D) * ev.N * 2;
    const bool fused = precision != GWH_FISHER_GRAM_FP32;
    const size_t nblk = fused ? (ev.N + GWH_FUSED_BINS - 1) / GWH_FUSED_BINS
                              : (nrows / ev.N) * ((ev.N + GWH_GRAM_ROWS - 1) / GWH_GRAM_ROWS);
    const size_t part_bytes = nblk * gram_tri(dim) * 8;
    const size_t per_pt_bytes = fused ? part_bytes : nrows * GWH_FROWS * ((precision == GWH_FISHER_GRAM_FP32) ? 4 : 8);
    size_t chunk = std::max<size_t>(1, max_operand / per_pt_bytes);
    chunk = std::min<size_t>(chunk, std::min(n, 65535));
    if (fused) chunk = std::min<size_t>(chunk, GWH_FUSED_MAX_POINTS);
    const size_t ni = chunk * per_point;
    return (fused ? F.deriv.cap : gwh_grown_capacity(chunk * per_pt_bytes, F.deriv.cap)) +
           gwh_grown_capacity(chunk * part_bytes, F.gram.cap) +
           gwh_grown_capacity((size_t)n * dim * dim * 8, F.out.cap) +
           (want_sigma ? gwh_grown_capacity((size_t)n * dim * 8, F.sig.cap) : F.sig.cap) +
           gwh_grown_capacity(ni * sizeof(InstCoef), F.coef.cap) +
           gwh_grown_capacity(chunk * GWH_FROWS * GWH_MAXSTEN * 8 + (ni * 4 + 7) / 8 * 8 + 256, F.misc.cap) + F.raw.cap;
}

extern "C" {

/* detector_util.cpp:573-636 name matching (exact strings only; anything else is unsupported) */
int gwh_detector_id(const char *name)
{
    if (!name) return -1;
    static const struct {
        const char *s;
        int id;
    } names[] = {{"Hanford", GWH_HANFORD},
                 {"hanford", GWH_HANFORD},
                 {"Livingston", GWH_LIVINGSTON},
                 {"livingston", GWH_LIVINGSTON},
                 {"Virgo", GWH_VIRGO},
                 {"virgo", GWH_VIRGO},
                 {"Kagra", GWH_KAGRA},
                 {"kagra", GWH_KAGRA},
                 {"Indigo", GWH_INDIGO},
                 {"indigo", GWH_INDIGO},
                 {"Cosmic Explorer", GWH_CE},
                 {"cosmic explorer", GWH_CE},
                 {"CE", GWH_CE},
                 {"Einstein Telescope 1", GWH_ET1},
                 {"einstein telescope 1", GWH_ET1},
                 {"ET1", GWH_ET1},
                 {"Einstein Telescope 2", GWH_ET2},
                 {"einstein telescope 2", GWH_ET2},
                 {"ET2", GWH_ET2},
                 {"Einstein Telescope 3", GWH_ET3},
                 {"einstein telescope 3", GWH_ET3},
                 {"ET3", GWH_ET3}};
    for (auto &n : names)
        if (!strcmp(n.s, name)) return n.id;
    return -1;
}

double gwh_dtoa(double RA, double DEC, double gmst, int detector1, int detector2)
{
    if (detector1 < 0 || detector1 >= GWH_NDET_TABLE || detector2 < 0 || detector2 >= GWH_NDET_TABLE) {
        gwh_set_error(GWH_ERR_UNSUPPORTED, "unsupported detector");
        return __builtin_nan("");
    }
    return host_dtoa(RA, DEC, gmst, detector1, detector2);
}

/* util.cpp:1797-1846: GPS seconds -> Greenwich mean sidereal time in radians (the reference's
 * low-order series in Julian days from J2000, hours wrapped to [0, 24)) */
double gwh_gps_to_gmst_radian(double gps)
{
    const double jd_j2000 = 2451545.0, gps_at_j2000 = 630763213.0;
    double jd = jd_j2000 + (gps - gps_at_j2000) / 86400.0;
    double jd0 = floor(jd) + 0.5;
    double hours_ut = (jd - jd0) * 24.0;
    double d0 = jd0 - jd_j2000, centuries = (jd - jd_j2000) / 36525.0;
    double g = 6.697374558 + 0.06570982441908 * d0 + 1.00273790935 * hours_ut + 0.000026 * centuries * centuries;
    double whole = (double)((long long)floor(g) % 24);
    return (whole + (g - floor(g))) * M_PI / 12.0;
}

int gwh_unpack_parameters(const gwh_params *params, int basis, double *v, int *log_factors)
{
    if (!params || !v) return gwh_set_error(GWH_ERR_INVALID, "null argument");
    int dim = basis_dim(basis);
    if (dim < 0) return gwh_set_error(GWH_ERR_INVALID, "unknown basis");
    int lf[GWH_FROWS];
    unpack(*params, basis, v, lf);
    if (log_factors)
        for (int i = 0; i < dim; i++) log_factors[i] = lf[i];
    return GWH_OK;
}

int gwh_repack_parameters(const double *v, int basis, gwh_params *params)
{
    if (!params || !v) return gwh_set_error(GWH_ERR_INVALID, "null argument");
    if (basis_dim(basis) < 0) return gwh_set_error(GWH_ERR_INVALID, "unknown basis");
    repack(v, basis, *params);
    return GWH_OK;
}

/* one-point Fisher on a temporary event holding the PSD for (reference detector, detector): the
 * time-of-flight phase of the second is relative to the first; the weights use df = f[1]-f[0]
 * (fisher.cpp:2746).  deriv != null: return the bare derivatives instead (calculate_derivatives). */
static int single_point(const double *frequencies, int length, int model, int basis, int detector,
                        int reference_detector, double *out, int dim, const gwh_params *params, int order,
                        const double *psd, double epsilon, double *deriv)
{
    Engine &E = gwh_engine();
    int rc = gwh_ensure_init();
    if (rc != GWH_OK) return rc;
    if (!frequencies || !(out || deriv) || !params || length < 2 || (!psd && !deriv))
        return gwh_set_error(GWH_ERR_INVALID, "null argument or length < 2");
    int nmod;
    if ((rc = fisher_mods(model, params, 1, &nmod)) != GWH_OK) return rc;
    if (basis_dim(basis) < 0 || basis_dim(basis) + nmod != dim)
        return gwh_set_error(GWH_ERR_INVALID, "dimension does not match the parameter basis (and ppE terms)");
    if ((basis == GWH_BASIS_PV2_FULL || basis == GWH_BASIS_PV2_MCMC) != gwh_is_pv2(model))
        return gwh_set_error(GWH_ERR_INVALID, "basis does not belong to the model");
    if (order != 2 && order != 4) return gwh_set_error(GWH_ERR_INVALID, "order must be 2 or 4");
    if (detector < 0 || detector >= GWH_NDET_TABLE || reference_detector < 0 || reference_detector >= GWH_NDET_TABLE)
        return gwh_set_error(GWH_ERR_UNSUPPORTED, "unsupported detector");
    if (basis == GWH_BASIS_PHENOMD_SKYAVG && !params->sky_average)
        return gwh_set_error(GWH_ERR_INVALID, "the sky-averaged basis needs params->sky_average");
    if (basis != GWH_BASIS_PHENOMD_SKYAVG && params->sky_average)
        return gwh_set_error(GWH_ERR_UNSUPPORTED, "sky_average selects the sky-averaged IMRPhenomD basis only");
    int dets[2] = {reference_detector, detector};
    int nd = (detector != reference_detector) ? 2 : 1;
    if (nd == 1) dets[0] = detector;
    /* the PSD of the Fisher detector on both rows (the reference detector's row only carries the arrival-time
     * reference); derivatives alone need no PSD: a unit one */
    std::vector<double> unit;
    const double *ps = psd;
    if (!ps) {
        unit.assign((size_t)length, 1.0);
        ps = unit.data();
    }
    const double *fp[2] = {frequencies, frequencies}, *pp[2] = {ps, ps};
    int ev;
    /* a cached event (no allocation after the first call on these arrays) */
    if ((rc = gwh_single_call_event(fp, length, nd, dets, nullptr, pp, GWH_SIMPSONS, nullptr, 0, &ev, 1)) != GWH_OK)
        return rc;
    E.events[ev].pins++;
    rc = fisher_run(ev, model, basis, GWH_FP64, params, 1, order, epsilon, nd - 1, 1, detector, reference_detector,
                    1.0, out, nullptr, E.fisher, deriv);
    E.events[ev].pins--;
    return rc;
}

static int gr_model_of(int basis)
{
    return (basis == GWH_BASIS_PV2_FULL || basis == GWH_BASIS_PV2_MCMC) ? GWH_IMRPHENOMPV2 : GWH_IMRPHENOMD;
}

int gwh_fisher_derivatives_model(const double *frequencies, int length, int model, int basis, int detector,
                                 int reference_detector, int dim, const gwh_params *params, int order, double epsilon,
                                 double *deriv)
{
    Engine &E = gwh_engine();
    std::lock_guard<std::recursive_mutex> lk(E.mu);
    if (!deriv) return gwh_set_error(GWH_ERR_INVALID, "null argument");
    return single_point(frequencies, length, model, basis, detector, reference_detector, nullptr, dim, params, order,
                        nullptr, epsilon, deriv);
}

int gwh_fisher_numerical_model(const double *frequencies, int length, int model, int basis, int detector,
                               int reference_detector, double *out, int dim, const gwh_params *params, int order,
                               const double *psd, double epsilon)
{
    Engine &E = gwh_engine();
    std::lock_guard<std::recursive_mutex> lk(E.mu);
    if (!out || !psd) return gwh_set_error(GWH_ERR_INVALID, "null argument");
    return single_point(frequencies, length, model, basis, detector, reference_detector, out, dim, params, order, psd,
                        epsilon, nullptr);
}

int gwh_fisher_derivatives(const double *frequencies, int length, int basis, int detector, int reference_detector,
                           int dim, const gwh_params *params, int order, double epsilon, double *deriv)
{
    return gwh_fisher_derivatives_model(frequencies, length, gr_model_of(basis), basis, detector, reference_detector,
                                        dim, params, order, epsilon, deriv);
}

int gwh_fisher_numerical(const double *frequencies, int length, int basis, int detector, int reference_detector,
                         double *out, int dim, const gwh_params *params, int order, const double *psd, double epsilon)
{
    return gwh_fisher_numerical_model(frequencies, length, gr_model_of(basis), basis, detector, reference_detector,
                                      out, dim, params, order, psd, epsilon);
}

int gwh_fisher_batch(int event, int model, int basis, int precision, const gwh_params *params, int n, int dim,
                     double epsilon, double *out, double *sigma)
{
    Engine &E = gwh_engine();
    std::lock_guard<std::recursive_mutex> lk(E.mu);
    int rc = gwh_ensure_init();
    if (rc != GWH_OK) return rc;
    return gwh_fisher_batch_with(event, model, basis, precision, params, n, dim, epsilon, out, sigma, E.fisher);
}

} /* extern "C" */
