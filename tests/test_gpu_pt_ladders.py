"""The tempering step on the device over ladder shapes: one temperature (no pair), two, more than a wave's worth of pairs
per lane (64 temperatures, 2016 pairs), equal temperatures next to each other, one ladder and chain counts that fill no
block, swap intervals that divide a graph's steps (a graph without swap launches on the other steps) and ones that do
not.  Every decision equals the CPU restatement's (oracle/pt_oracle.py) fed with the engine's own likelihoods."""
import numpy as np
import pytest

import gw_analysis_tools_amd as G
from gw_analysis_tools_amd import pt
from gw_analysis_tools_amd import workloads as W
from oracle import pt_oracle as PO

pytestmark = pytest.mark.gpu

WIDTHS = np.array([0.02, 0.02, 0.05, 0.03, 0.05, 2e-4, 0.03, 2e-4, 2e-3, 0.05, 0.05])


@pytest.fixture(scope="module")
def event():
    f = W.uniform_grid(20., 300., 0.5)
    psd = W.analytic_psd(f)
    inj = W.injection_params(1)[0]
    p = G.make_params(**{k: (inj[k].tolist() if inj[k].shape else inj[k].item()) for k in inj.dtype.names})
    data = [r + W.noise(f, psd, W.rng(1, 9)) for r in G.create_coherent_GW_detection(f, p, [0, 1])]
    ev = G.Event(f, data, [psd] * 2, [0, 1])
    yield ev, inj
    ev.close()


@pytest.mark.parametrize("nt,nc,swap_every,per_graph", [(1, 5, 1, 1), (2, 3, 1, 2), (3, 70, 2, 4), (4, 1, 3, 2),
                                                        (16, 4, 2, 2), (64, 2, 1, 1), (5, 3, 0, 3)])
def test_ladder_shapes(event, nt, nc, swap_every, per_graph):
    ev, inj = event
    temps = 1.08 ** np.arange(nt)
    if nt >= 5:
        temps[3] = temps[2]  # equal temperatures never swap
    th0 = pt.theta_from_params(inj)

    def like(th):
        return G.loglike_batch(ev, pt.params_from_theta(th, inj), G.IMRPHENOMD, G.FP64)

    dev = G.DevicePT(ev, inj, th0, WIDTHS, temps, nc, pt.LOWER, pt.UPPER, precision=G.FP64, seed=77 + nt,
                     swap_every=swap_every, steps_per_graph=per_graph)
    ref = PO.PTOracle(like, th0, WIDTHS, temps, nc, pt.LOWER, pt.UPPER, 77 + nt, swap_every)
    swaps = np.zeros((max(nt - 1, 0), nc), dtype=int)
    for _ in range(12 // per_graph):
        dev.run(per_graph)
        for _ in range(per_graph):
            ref.step()
            swaps += ref.history[-1]["swapped"]
        _, _, acc, sw = dev.last_step()
        assert np.array_equal(acc, ref.history[-1]["accept"])
        assert np.array_equal(sw, ref.history[-1]["swapped"])
    th, ll, steps = dev.state()
    assert steps == 12 and np.allclose(th, ref.theta, rtol=1e-13, atol=1e-15)
    assert np.all(np.abs(ll - ref.ll) <= 1e-9 * np.abs(ref.ll))
    assert np.array_equal(dev.counters()[1], swaps)
    if nt > 2 and swap_every:
        assert swaps.sum() > 0
    dev.close()
