"""Multi-event batches (the flattened work list) against the same instances on their event alone (the tile-major grid):
bit-identical, whatever the number of instances, their order, and the number of lanes per tile of their events.  The
list takes instances in groups of 8, writes its items in 8 columns of equal length and fills the last places with
holes, so counts around multiples of 8 and lists shorter than 8 items are where it can go wrong."""
import numpy as np
import pytest

import gw_analysis_tools_amd as G
from gw_analysis_tools_amd import workloads as W

pytestmark = pytest.mark.gpu


def _event(f, step):
    psd = W.analytic_psd(f)
    g = W.rng(2, 100 + step)
    return G.Event(f, [W.noise(f, psd, g) for _ in range(3)], [psd] * 3, [0, 1, 2])


def _params(n, step):
    """total masses from 9 to 130 solar masses: some instances keep every tile, others only the first"""
    P = W.perturbed_params(W.injection_params(1)[0], n, step=step)
    s = np.exp(np.linspace(np.log(0.15), np.log(2.0), n)) if n > 1 else np.array([0.3])
    P["mass1"], P["mass2"] = P["mass1"] * s, P["mass2"] * s
    return P


@pytest.fixture(scope="module")
def events():
    """three tilings: 2003 bins (256 lanes x 2), 40001 bins (256 x 8), and 9001 bins of 64 lanes, held by a step graph
    while the others are tiled"""
    G.set_tile_lanes(64)
    a = _event(W.uniform_grid(20., 20. + 9000 * 0.125, 0.125), 0)
    d = G.DeviceArray(448), G.DeviceArray(8)
    graph = G.LoglikeGraph(a, d[0].ptr, 1, d[1].ptr)
    G.set_tile_lanes(0)
    ev = [a, _event(W.uniform_grid(20., 20. + 2002 * 0.5, 0.5), 1), _event(W.uniform_grid(20., 20. + 40000 / 32, 1 / 32), 2)]
    yield ev
    graph.close()
    for e in ev:
        e.close()


@pytest.mark.parametrize("model", [G.IMRPHENOMD, G.IMRPHENOMPV2])
@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 17, 64, 300])
@pytest.mark.parametrize("order", ["blocks", "interleaved", "one"])
def test_work_list_equals_single_event_batches(events, model, n, order):
    P = _params(n, n)
    if model == G.IMRPHENOMPV2:
        P["spin1"][:, 0], P["spin2"][:, 1] = 0.3, -0.2
    i = np.arange(n)
    which = {"blocks": i * 3 // n, "interleaved": i % 3, "one": np.full(n, 1)}[order]
    got = G.loglike_batch(events[0], P, model, G.FP64, events=[events[k] for k in which])
    for k in range(3):
        sel = which == k
        if sel.any():
            assert np.array_equal(got[sel], G.loglike_batch(events[k], P[sel], model, G.FP64)), (n, order, k)
    assert np.all(np.isfinite(got))
