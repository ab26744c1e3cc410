"""The batched maximised likelihood over lengths where its reductions and transforms change shape -- a few bins, one bin
around a block of 256 and around 1024 threads, primes, powers of two -- and over batch sizes, against the CPU
restatement (oracle/gwo_maxll.py) to 1e-9 relative, the FP64 likelihood bar."""
import numpy as np
import pytest

import gw_analysis_tools_amd as G
import oracle as O
from gw_analysis_tools_amd import workloads as W
from oracle import gwo_maxll as M

pytestmark = pytest.mark.gpu

TOL = 1e-9


def _op(rec):
    return O.make_params(**{k: (rec[k].tolist() if rec[k].shape else rec[k].item()) for k in rec.dtype.names})


@pytest.mark.parametrize("n", [5, 64, 251, 256, 257, 1023, 1024, 1025, 2048, 4099, 8191])
@pytest.mark.parametrize("model", [G.IMRPHENOMD, G.IMRPHENOMPV2])
def test_lengths(n, model):
    f = 20. + np.arange(n) * (480. / (n - 1))
    psd = W.analytic_psd(f)
    g = W.rng(3, 40 + n)
    nd = 1 + n % 3
    data = [O.detector_response(f, _op(W.injection_params(1)[0]), d) + W.noise(f, psd, g) for d in range(nd)]
    P = W.precessing_params(3) if model == G.IMRPHENOMPV2 else W.perturbed_params(W.injection_params(1)[0], 3, step=n)
    ev = G.Event(f, data, [psd] * nd, list(range(nd)))
    got = G.maximized_loglike_batch(ev, P, model)
    for i in range(3):
        ref = M.intrinsic_network(f, data, [psd] * nd, _op(P[i]), model)
        assert abs(got[i] - ref) <= TOL * abs(ref), (n, model, i, got[i], ref)
        one = G.maximized_loglike_batch(ev, P[i:i + 1], model)
        assert abs(one[0] - got[i]) <= 1e-13 * abs(ref) * np.log2(n + 2)
    ev.close()


def test_no_finite_maximum():
    """NaN data give a statistic without a maximum, as the serial rule: the comparison never picks a NaN"""
    f = 20. + np.arange(300) * 1.5
    psd = W.analytic_psd(f)
    ev = G.Event(f, [np.full(300, np.nan + 0j)], [psd], [0])
    assert not np.isfinite(G.maximized_loglike_batch(ev, W.injection_params(2), G.IMRPHENOMD)).any()
    ev.close()
