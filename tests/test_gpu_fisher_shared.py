"""The fused Fisher kernel against the engine's own bare derivatives (the stencil kernel, which evaluates every
stencil point in full): what the fused kernel keeps from one evaluation to the next, the rows it gives to each wave
and the chunks of bins it leaves out may not show in the matrix.

Bound: both round an operand alike, so only the order of the sums over n bins and two quadratures differs, at most
2 n eps / 2 relative to sqrt(F_ii F_jj) (1e-12 for n < 4500, where the rounding errors average far below it) -- at the
reference's step of 1e-8 a last-bit difference of one operand would show at 1e-10."""
import numpy as np
import pytest

import gw_analysis_tools_amd as G
from gw_analysis_tools_amd import workloads as W

pytestmark = pytest.mark.gpu

TOL = 1e-12
SRC = dict(mass1=36., mass2=29., spin1=[0, 0, 0.3], spin2=[0, 0, -0.1], DL=410., tc=0.01, phiRef=0.3, f_ref=20.,
           RA=1.37, DEC=-1.26, psi=2.66, incl=2.9, gmst=W.GMST)
PREC = dict(SRC, spin1=[0.3, 0.1, 0.3], spin2=[-0.1, 0.2, -0.1])
PPE = dict(ppe_nmod=2, ppe_b=[-7., -3.], ppe_beta=[3e-5, -3e-3])
GIMR = dict(gimr_nlist=2, gimr_list=[6, 17], gimr_dphi=[0] * 6 + [0.05] + [0] * 7)
CASES = [  # (model, basis, dimension, parameters)
    (G.IMRPHENOMD, G.BASIS_PHENOMD_SKYAVG, 7, dict(SRC, sky_average=1)),
    (G.IMRPHENOMD, G.BASIS_PHENOMD_FULL, 11, SRC),
    (G.IMRPHENOMD, G.BASIS_PHENOMD_MCMC, 11, SRC),
    (G.IMRPHENOMPV2, G.BASIS_PV2_FULL, 13, dict(PREC, chip=0.35, phip=0.8)),
    (G.IMRPHENOMPV2, G.BASIS_PV2_MCMC, 15, PREC),
    (G.PPE_IMRPHENOMD_IMR, G.BASIS_PHENOMD_MCMC, 13, dict(SRC, **PPE)),
    (G.GIMRPHENOMPV2, G.BASIS_PV2_FULL, 15, dict(PREC, chip=0.35, phip=0.8, **GIMR)),
    # a theory's term depends on the distance through its redshift: DL shares nothing here
    (G.PPE_IMRPHENOMD_INSPIRAL, G.BASIS_PHENOMD_FULL, 12,
     dict(SRC, ppe_theory=G.THEORY_EDGB, ppe_nmod=1, ppe_beta=[1e-12])),
]


def _gram(f, psd, d):
    n = len(f)
    w = np.ones(n)
    w[1:n - 1:2] = 4
    w[2:n - 1:2] = 2
    w = w * (f[1] - f[0]) / 3 * 4 / psd
    return np.real((d * w) @ np.conj(d).T)


def _norm_err(a, b):
    s = np.sqrt(np.abs(np.diag(b)))
    s[s == 0] = 1
    return np.max(np.abs(a - b) / np.outer(s, s))


def _params(kw):
    return G.make_params(**{k: (list(v) if isinstance(v, (list, tuple)) else v) for k, v in kw.items()})


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("model,basis,dim,kw", CASES)
def test_fused_gram_is_the_gram_of_the_derivatives(model, basis, dim, kw, order):
    f = W.uniform_grid(20., 1024., 0.25)
    psd = W.analytic_psd(f)
    p, det = _params(kw), 0 if kw.get("sky_average") else 1
    d = G.fisher_derivatives(f, basis, det, 0, dim, p, order=order, model=model)
    F = G.fisher_numerical(f, psd, basis, det, 0, dim, p, order=order, model=model)
    assert _norm_err(F, _gram(f, psd, d)) <= TOL
    assert np.array_equal(F, F.T)


# lengths around the 64-bin chunks, and a grid whose chunks do not ascend (the cutoff 0.2/M of 65 solar masses, 625
# Hz, lies inside its first half): every chunk holding a live bin is visited
@pytest.mark.parametrize("n", [3, 64, 65, 127, 129, 2001])
@pytest.mark.parametrize("folded", [False, True])
def test_fused_gram_lengths_and_orders_of_the_grid(n, folded):
    f = np.linspace(20., 1500., n)
    if folded:
        f = np.concatenate([f[n // 2:], f[:n // 2]])
    psd = W.analytic_psd(f)
    for model, basis, dim, kw in (CASES[0], CASES[2], CASES[3]):
        p, det = _params(kw), 0 if kw.get("sky_average") else 2
        d = G.fisher_derivatives(f, basis, det, 0, dim, p, model=model)
        F = G.fisher_numerical(f, psd, basis, det, 0, dim, p, model=model)
        assert _norm_err(F, _gram(f, psd, d)) <= TOL


def test_points_of_very_different_mass_share_a_pass():
    """the chunks of a pass follow its lightest point, the bins of a point its own cutoff; a point in a pass with
    others equals the point alone, bit for bit, and the sum of the one-detector matrices"""
    f = W.uniform_grid(20., 1800., 0.5)
    psd = W.analytic_psd(f)
    ev = G.Event(f, [np.zeros(len(f), complex)] * 3, [psd] * 3, [0, 1, 2])
    P = np.concatenate([W.injection_params(1, mass1=m, mass2=0.6 * m) for m in (90., 20., 8., 60.)])
    F = G.fisher_batch(ev, P, G.IMRPHENOMD, G.BASIS_PHENOMD_MCMC, 11, epsilon=-1e-7)
    for i in range(len(P)):
        one = G.fisher_batch(ev, P[i:i + 1], G.IMRPHENOMD, G.BASIS_PHENOMD_MCMC, 11, epsilon=-1e-7)
        assert np.array_equal(F[i], one[0])
        p = _params({k: (P[i][k].tolist() if P[i][k].shape else P[i][k].item()) for k in P.dtype.names})
        s = sum(G.fisher_numerical(f, psd, G.BASIS_PHENOMD_MCMC, d, 0, 11, p, epsilon=-1e-7) for d in range(3))
        assert _norm_err(F[i], s) <= TOL
    ev.close()


def test_a_point_without_masses_leaves_the_others_alone():
    """the batch's chunks end at the highest cutoff 0.2 / M of its points; one without a cutoff does not hide the
    light point before it behind the heavy point after it"""
    f = W.uniform_grid(20., 2048., 0.5)
    psd = W.analytic_psd(f)
    ev = G.Event(f, [np.zeros(len(f), complex)], [psd], [0])
    P = W.perturbed_params(W.injection_params(1)[0], 3, step=1)
    P["mass1"], P["mass2"] = [8., np.nan, 90.], [6., 20., 70.]
    a = G.fisher_batch(ev, P, G.IMRPHENOMD, G.BASIS_PHENOMD_FULL, 11, epsilon=1e-6)
    for i in (0, 2):
        alone = G.fisher_batch(ev, P[i:i + 1], G.IMRPHENOMD, G.BASIS_PHENOMD_FULL, 11, epsilon=1e-6)[0]
        assert np.linalg.norm(a[i] - alone) <= 1e-12 * np.linalg.norm(alone)
    ev.close()


@pytest.mark.parametrize("psd_bin", [0., -1e-46, np.nan])
@pytest.mark.parametrize("at", [0.6, 0.95])
def test_a_weight_without_a_value_does_not_depend_on_the_neighbours(psd_bin, at):
    """a bin whose noise is zero, negative or not a number leaves no matrix of the event a value, above a point's cutoff
    too (0 times such a weight), whether or not a lighter point in the pass reaches the bin's chunk"""
    f = W.uniform_grid(20., 2000., 0.5)
    psd = W.analytic_psd(f)
    psd[int(at * len(f))] = psd_bin
    ev = G.Event(f, [np.zeros(len(f), complex)] * 2, [W.analytic_psd(f), psd], [0, 1])
    P = np.concatenate([W.injection_params(1, mass1=m, mass2=0.6 * m) for m in (90., 4., 60.)])
    for model, basis, dim in ((G.IMRPHENOMD, G.BASIS_PHENOMD_MCMC, 11), (G.IMRPHENOMPV2, G.BASIS_PV2_FULL, 13)):
        P["chip"], P["phip"] = 0.3, 0.7
        F = G.fisher_batch(ev, P, model, basis, dim, epsilon=-1e-7)
        for i in range(len(P)):
            one = G.fisher_batch(ev, P[i:i + 1], model, basis, dim, epsilon=-1e-7)
            assert not np.any(np.isfinite(F[i])) and np.array_equal(F[i], one[0], equal_nan=True)
    ev.close()


@pytest.mark.parametrize("tail", [np.inf, np.nan])
def test_bins_without_a_frequency_count_nothing(tail):
    """a grid padded with infinities or NaN, below and above the cutoff inside one chunk of 64: such bins are above every cutoff"""
    f = np.linspace(20., 800., 100)
    psd = W.analytic_psd(f)
    f[-3:] = tail
    for model, basis, dim, kw in CASES[1:5]:
        p = _params(kw)
        d = G.fisher_derivatives(f, basis, 1, 0, dim, p, model=model)
        assert np.all(d[:, -3:] == 0)
        F = G.fisher_numerical(f, psd, basis, 1, 0, dim, p, model=model)
        assert _norm_err(F, _gram(f, psd, d)) <= TOL
