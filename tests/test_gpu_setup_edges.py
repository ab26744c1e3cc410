"""The per-instance setup where its geometry degenerates or its angles leave the ordinary range: spins along and
against the orbital axis and in its plane, line of sight on the axis and within an underflowing square of it, equal and
inverted masses, angles of 2^40 rad and beyond, reference frequencies in every phase region; and instance counts around
the 32 lanes of a setup block.  1e-9 against the oracle is the FP64 likelihood bar of the other tests here."""
import numpy as np
import pytest

import gw_analysis_tools_amd as G
import oracle as O
from gw_analysis_tools_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def net():
    f = W.uniform_grid(20., 512., 0.5)
    psd = W.analytic_psd(f)
    g = W.rng(7, 1)
    data = [O.detector_response(f, O.make_params(**W.INJECTION), d) + W.noise(f, psd, g) for d in (0, 1)]
    ev = G.Event(f, data, [psd] * 2, [0, 1])
    yield f, psd, data, ev
    ev.close()


def _edges(kind, model):
    base = W.precessing_params(1) if model == G.IMRPHENOMPV2 else W.injection_params(1)
    out = []

    def add(**kw):
        r = base.copy()
        for k, v in kw.items():
            r[k] = v
        out.append(r[0])

    if kind == "geometry":
        for s in ([0, 0, 0], [0, 0, .9], [0, 0, -.9], [.3, 0, 0], [-.3, 0, 0], [0, .3, 0], [0, -.3, .2]):
            for inc in (0., np.pi, 1e-300, .7, -2.):
                add(spin1=s, spin2=[0, 0, 0], incl=inc)
            add(spin1=s, spin2=s, mass1=29., mass2=36.)
        for m in ((30., 30.), (1.4, 1.4), (29., 36.), (100., 5.)):
            add(mass1=m[0], mass2=m[1])
        for c in (0., .3, 1.):
            add(chip=c, phip=2.)
    elif kind == "cancelling":
        # J along the orbital axis with chi_p > 0: exactly, to rounding, within a tilt that acos(J_z / J) cannot resolve,
        # with zeros of either sign, and against the axis; the line of sight in all four quadrants
        for phi in (0.2, 1.9, 3.5, 5.5):
            for s in (.5, .25, .3, .7):
                for a in (s, -s):
                    add(mass1=30., mass2=30., spin1=[a, 0, .2], spin2=[-a, 0, .2], incl=1.2, phiRef=phi)
                    add(mass1=30., mass2=30., spin1=[0, a, .2], spin2=[0, -a, -.1], incl=2.3, phiRef=phi)
                    add(mass1=30., mass2=30., spin1=[a, -.1, .2], spin2=[-a, .1, .2], incl=1.2, phiRef=phi)
                    add(mass1=30., mass2=15., spin1=[a / 4, 0, .2], spin2=[-a, 0, .2], incl=.8, phiRef=phi)
                    add(mass1=80., mass2=10., spin1=[a / 64, 0, -.95], spin2=[-a, 0, 0], incl=1.2, phiRef=phi)
            for x in (1e-12, -1e-12):
                add(mass1=30., mass2=30., spin1=[.5, x, .2], spin2=[-.5, 0, .2], incl=1.2, phiRef=phi)
                add(mass1=30., mass2=30., spin1=[x, .5, .2], spin2=[0, -.5, .2], incl=1.2, phiRef=phi)
            add(mass1=30., mass2=30., spin1=[-0., .5, .2], spin2=[-0., -.5, .2], incl=1.2, phiRef=phi)
        # the line of sight in a coordinate plane, where its azimuth is a rounding error away from a quadrant
        for phi in (0., -0., np.pi / 2, np.pi, -np.pi / 2, 2 * np.pi):
            for inc in (1.2, -1.2, 2.5, -2.5):
                for a in (.5, -.3):
                    add(mass1=30., mass2=30., spin1=[a, -.1, .2], spin2=[-a, .1, .2], incl=inc, phiRef=phi)
                    add(mass1=30., mass2=30., spin1=[0, a, -.7], spin2=[0, -a, .7], incl=inc, phiRef=phi)
    elif kind == "reference":
        for fr in (5., 20., 60., 100., 200., 300., 500., 1000.):
            for st in (0, 1):
                add(f_ref=fr, shift_time=st, shift_phase=1)
                add(f_ref=fr, shift_time=st, shift_phase=0)
    else:
        for k in ("incl", "psi", "RA", "DEC", "gmst"):
            for v in (-1e5, 2. ** 40, -2. ** 40 * (1 - 2. ** -53), 1e17, 1e300):
                add(**{k: v})
        if model == G.IMRPHENOMPV2:  # phiRef only places the line of sight there, as pi/2 - phiRef
            for v in (1e5, -1e7, 1e10, 1e17, -1e300):
                add(phiRef=v)
    return np.array(out, dtype=base.dtype)


@pytest.mark.parametrize("kind,model", [("geometry", G.IMRPHENOMPV2), ("cancelling", G.IMRPHENOMPV2),
                                        ("reference", G.IMRPHENOMD),
                                        ("reference", G.IMRPHENOMPV2), ("angles", G.IMRPHENOMD),
                                        ("angles", G.IMRPHENOMPV2)])
def test_degenerate_setups_match_oracle(net, kind, model):
    f, psd, data, ev = net
    P = _edges(kind, model)
    a = G.loglike_batch(ev, P, model)
    for i, r in enumerate(P):
        p = O.make_params(**{k: (r[k].tolist() if r[k].shape else r[k].item()) for k in r.dtype.names})
        ref = O.network_loglike(f, data, [psd] * 2, [0, 1], p, model)
        assert abs(a[i] - ref) <= 1e-9 * max(1.0, abs(ref)), (i, r, a[i], ref)


@pytest.mark.parametrize("n", [1, 31, 32, 33, 64, 65])
def test_instances_around_a_setup_block(net, n):
    ev = net[3]
    P = W.precessing_params(n)
    a = G.loglike_batch(ev, P, G.IMRPHENOMPV2)
    for i in {0, n // 2, n - 1}:
        assert a[i] == G.loglike_batch(ev, P[i:i + 1], G.IMRPHENOMPV2)[0]


def test_angles_without_a_value_give_none(net):
    ev = net[3]
    for k in ("incl", "psi", "RA", "DEC", "gmst"):
        P = W.precessing_params(2)
        P[k] = [np.inf, np.nan]
        for m in (G.IMRPHENOMD, G.IMRPHENOMPV2):
            assert np.all(np.isnan(G.loglike_batch(ev, P, m)))
