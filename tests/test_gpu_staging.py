"""Calls whose inputs and results go through pinned memory, against the same calls beyond its 4 MiB, which do not; and
Fisher batches on either side of their pass sizes.  The kernels are the same, so the results are too."""
import numpy as np
import pytest

import gw_analysis_tools_amd as G
from gw_analysis_tools_amd import workloads as W

pytestmark = pytest.mark.gpu


def _event(n=101):
    f = 20. + np.arange(n) * 2.
    psd = W.analytic_psd(f)
    return G.Event(f, [np.full(n, 1e-23 + 2e-23j)] * 2, [psd] * 2, [0, 1])


@pytest.mark.parametrize("model,n", [(G.IMRPHENOMD, 30000), (G.IMRPHENOMPV2, 30000), (G.PPE_IMRPHENOMD_IMR, 12000)])
def test_likelihoods_beyond_the_staging(model, n):
    a, b = _event(), _event(77)
    base = W.precessing_params(1) if model == G.IMRPHENOMPV2 else W.injection_params(1)
    P = np.repeat(base, n)
    P["DL"] *= np.linspace(0.5, 2.0, n)
    P["ppe_nmod"], P["ppe_b"][:, 0], P["ppe_beta"][:, 0] = 1, -7., 1e-5  # the GR models do not read them
    ids = np.where(np.arange(n) % 3 == 0, a.id, b.id).astype(np.int32)
    for events in (None, ids):
        full = G.loglike_batch(a, P, model, events=events)
        for lo, hi in ((0, 1), (5, 12), (n - 3, n)):
            part = G.loglike_batch(a, P[lo:hi], model, events=None if events is None else ids[lo:hi])
            assert np.array_equal(full[lo:hi], part)
    assert len(set(full[:50])) == 50
    snr = G.snr_batch(a, P, model)
    assert np.array_equal(snr[-3:], G.snr_batch(a, P[-3:], model))
    a.close()
    b.close()


@pytest.mark.parametrize("model", [G.IMRPHENOMD, G.IMRPHENOMPV2])
def test_single_waveforms_beyond_the_staging(model):
    n = 280000  # 4.5 MiB an output
    f = 20. + np.arange(n) / 512.
    P = W.precessing_params(1) if model == G.IMRPHENOMPV2 else W.injection_params(1)
    p = G.Params.from_buffer_copy(P[0].tobytes())
    hp, hc = G.fourier_waveform(f, p, model)
    r = G.fourier_detector_response(f, p, 1, model)
    c = G.create_coherent_GW_detection(f, p, [0, 1, 2], model)
    for lo, hi in ((0, 1), (3, 1000), (n - 77, n)):
        sp, sc = G.fourier_waveform(f[lo:hi], p, model)
        assert np.array_equal(hp[lo:hi], sp) and np.array_equal(hc[lo:hi], sc)
        assert np.array_equal(r[lo:hi], G.fourier_detector_response(f[lo:hi], p, 1, model))
        s = G.create_coherent_GW_detection(f[lo:hi], p, [0, 1, 2], model)
        assert all(np.array_equal(x[lo:hi], y) for x, y in zip(c, s))
    assert np.any(hp != 0)


@pytest.mark.parametrize("model,basis,dim", [(G.IMRPHENOMD, G.BASIS_PHENOMD_FULL, 11),
                                             (G.IMRPHENOMPV2, G.BASIS_PV2_MCMC, 15),
                                             (G.PPE_IMRPHENOMD_IMR, G.BASIS_PHENOMD_MCMC, 12)])
def test_fisher_passes(model, basis, dim):
    ev = _event()
    P = W.precessing_params(300) if model == G.IMRPHENOMPV2 else W.perturbed_params(W.injection_params(1)[0], 300, step=1)
    P["mass1"] = np.linspace(30., 40., 300)
    if dim == 12:
        P["ppe_nmod"], P["ppe_b"][:, 0], P["ppe_beta"][:, 0] = 1, -7., 1e-5
    full, sig = G.fisher_batch(ev, P, model, basis, dim, epsilon=1e-6, with_sigma=True)
    for n in (1, 31, 33, 127, 128, 129, 143, 145, 225):
        assert np.array_equal(G.fisher_batch(ev, P[:n], model, basis, dim, epsilon=1e-6), full[:n])
    assert np.all(np.isfinite(full)) and len({m[0, 0] for m in full}) == 300
    ev.close()
