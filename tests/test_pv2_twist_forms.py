"""The identity behind gwh_pv2_twist: the IMRPhenomPv2 twist-up collected by powers of e^{i alpha}, restated here, against
the sum over m of the rotation elements d^2_{m,+-2}(beta) and the -2Y_2m it stands for (IMRPhenomP.cpp:290-361), over
small and large opening angles.  The kernel itself is compared with that sum in test_gpu_pv2_twist.py.  Every
coefficient is a polynomial in cos beta and sin beta, so 8 ulp of the largest term covers its ~10 roundings."""
import numpy as np
import pytest


def _sum_over_m(beta, alpha, th):
    """the reference's sum: h+ = sum t2 + tm, hx = i sum (t2 - tm)"""
    c, s = np.cos(beta / 2), np.sin(beta / 2)
    d2 = [s ** 4, 2 * c * s ** 3, np.sqrt(6) * s * s * c * c, 2 * c ** 3 * s, c ** 4]  # m = -2..2 to +2
    dm = [d2[4], -d2[3], d2[2], -d2[1], d2[0]]
    ct, st = np.cos(th), np.sin(th)
    y = [np.sqrt(5 / (64 * np.pi)) * (1 - ct) ** 2, np.sqrt(5 / (16 * np.pi)) * st * (1 - ct),
         np.sqrt(15 / (32 * np.pi)) * st * st, np.sqrt(5 / (16 * np.pi)) * st * (1 + ct),
         np.sqrt(5 / (64 * np.pi)) * (1 + ct) ** 2]
    hp = hc = 0
    for m in range(-2, 3):
        t2 = np.exp(-1j * m * alpha) * dm[m + 2] * y[m + 2]
        tm = np.exp(1j * m * alpha) * d2[m + 2] * y[m + 2]
        hp, hc = hp + t2 + tm, hc + 1j * (t2 - tm)
    return hp, hc


def _closed(beta, alpha, th, sign=1.0):
    cb, sb = np.cos(beta), np.sin(beta)
    ct, st = np.cos(th), np.sin(th)
    tw = [np.sqrt(5 / (64 * np.pi)) * 2 * (1 + ct * ct), np.sqrt(5 / (64 * np.pi)) * 4 * ct,
          np.sqrt(5 / (16 * np.pi)) * 2 * st, np.sqrt(5 / (16 * np.pi)) * 2 * st * ct,
          np.sqrt(15 / (32 * np.pi)) * (np.sqrt(6) / 2) * st * st]
    sa, ca = np.sin(alpha), np.cos(alpha)
    c2, s2 = ca * ca - sa * sa, 2 * sa * ca
    e, g = 0.5 + 0.5 * cb * cb, sb * cb
    hp = tw[0] * (e * c2) + tw[3] * (g * ca) + tw[4] * (sb * sb) + 1j * (tw[0] * (cb * s2) + tw[3] * (sb * sa))
    hc = tw[1] * (e * s2) + tw[2] * (g * sa) - 1j * sign * (tw[1] * (cb * c2) + tw[2] * (sb * ca))
    return hp, hc


@pytest.mark.parametrize("lo,hi", [(1e-9, 1e-3), (1e-3, 1.5), (1.5, np.pi / 2)])
def test_closed_forms_equal_the_sum_over_m(lo, hi):
    g = np.random.default_rng(3)
    worst = planted = 0.0
    for _ in range(400):
        beta = np.exp(g.uniform(np.log(lo), np.log(hi)))
        alpha, th = g.uniform(-30, 30), g.uniform(0, np.pi)
        a, b, p = _sum_over_m(beta, alpha, th), _closed(beta, alpha, th), _closed(beta, alpha, th, -1.0)
        worst = max(worst, abs(a[0] - b[0]), abs(a[1] - b[1]))
        planted = max(planted, abs(a[1] - p[1]))
    assert worst <= 8 * 2.0 ** -52 * 1.3, worst  # |h| is at most 2 (5 / (4 pi))^(1/2) = 1.26
    assert planted > 0.1
