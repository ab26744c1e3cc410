"""The kernel's IMRPhenomPv2 twist-up (gwh_pv2_twist with the setup's constants of the line of sight), bin by bin, against
the sum over m = -2..2 of the rotation elements and spherical harmonics that it stands for (IMRPhenomP.cpp:290-361),
written out from the oracle's pieces.  The ratio of the polarisations is free of amplitude and phase, so only the angles count:
Euler angles of up to 1e2 rad, 1e2 x 2^-52 x a few roundings of their terms, 4e-13; and the tilt of the orbital axis,
which the oracle takes as acos(Jz / J) as the reference does: that ratio's few 2^-53 are as much over the tilt, in each of
the angles that follow from it: 16 x 2^-53 / tilt."""
import numpy as np
import pytest

import gw_analysis_tools_amd as G
import oracle as O
from gw_analysis_tools_amd import workloads as W

F = np.array([20., 31., 55., 90., 140., 210., 330., 480., 600.])
BASE = dict(DL=410., RA=1.37, DEC=-1.26, psi=2.66, f_ref=20., gmst=W.GMST, tc=0.01, phiRef=0.3, phip=1.1)
# (masses, aligned spins, chi_p): opening angles from 3e-7 rad to 90 degrees
SOURCES = [((36., 29.), (0.3, -0.1), 1e-6), ((36., 29.), (0.3, -0.1), 0.02), ((30., 12.), (-0.5, 0.2), 0.5),
           ((50., 7.), (-0.6, 0.), 0.75), ((9., 1.5), (0., 0.), 0.99)]
INCLINATIONS = [0.05, 0.7, 1.57, 2.4, 3.1]


def _kw(src, incl):
    return dict(BASE, mass1=src[0][0], mass2=src[0][1], spin1=[0, 0, src[1][0]], spin2=[0, 0, src[1][1]], chip=src[2],
                incl=incl)


def _bound(p):
    q = O.pv2_setup_summary(p)
    return 4e-13 + 16 * 2.0 ** -53 * abs((O.pv2_pieces(p, BASE["f_ref"])["L2PN"] + q["SL"]) / q["SP"])


def _factors(p, f, wrong=None):
    """h+ and hx factors at f with the polarisation turned by zeta; wrong: m whose rotation element changes sign"""
    q, z = O.pv2_pieces(p, f), O.pv2_setup_summary(p)["zeta"]
    hp = hc = 0
    for m in range(-2, 3):
        d2 = -q["d2"][m + 2] if m == wrong else q["d2"][m + 2]
        t2 = np.exp(-1j * m * q["alpha"]) * q["dm2"][m + 2] * q["ylm"][m + 2]
        tm = np.exp(1j * m * q["alpha"]) * d2 * q["ylm"][m + 2]
        hp, hc = hp + t2 + tm, hc + 1j * (t2 - tm)
    c, s = np.cos(2 * z), np.sin(2 * z)
    return c * hp + s * hc, c * hc - s * hp


def _apart(hp, hc, p, wrong=None):
    """how far hp : hc is from the ratio of the sum's factors, over the size of the vector"""
    worst = 0.0
    for k, f in enumerate(F):
        if hp[k] == 0 and hc[k] == 0:
            continue
        a, b = _factors(p, f, wrong)
        worst = max(worst, abs(hp[k] * b - hc[k] * a) / (np.hypot(abs(hp[k]), abs(hc[k])) * np.hypot(abs(a), abs(b))))
    return worst


@pytest.mark.gpu
@pytest.mark.parametrize("src", SOURCES)
@pytest.mark.parametrize("incl", INCLINATIONS)
def test_the_kernel_twists_up_as_the_sum_over_m(src, incl):
    kw = _kw(src, incl)
    hp, hc = G.fourier_waveform(F, G.make_params(**kw), G.IMRPHENOMPV2)
    p = O.make_params(**kw)
    assert np.any(hp != 0)
    assert _apart(hp, hc, p) <= _bound(p)


def test_the_comparison_sees_every_term():
    """on the oracle's own waveform: within the bound as it is, beyond it with any one rotation element changed"""
    for m in range(-2, 3):
        seen = 0.0
        for src in SOURCES:
            for incl in INCLINATIONS:
                p = O.make_params(**_kw(src, incl))
                hp, hc = O.fourier_waveform(F, p, O.IMRPHENOMPV2)
                assert _apart(hp, hc, p) <= _bound(p)
                seen = max(seen, _apart(hp, hc, p, m))
        assert seen > 1e-3, (m, seen)
