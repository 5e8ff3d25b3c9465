"""The FP64 shifted-force Coulomb pair by itself: two charges on the x axis, from
1e-6 apart to the last number below the cutoff, force and energy against long
double, through the Coulomb call alone and through the walk it shares with a pair
call.

With u = 2^-53, r exact (one atom at x = 0), A = 1/r^2, B = 1/rc^2, and every
operation of qq (1/r2 - 1/rc2) / r and qq (1/r + (r - rc)/rc2 - 1/rc) at its own
rounding, reciprocals within an ulp:
  r2 and 1/r2 leave 3 u A, 1/rc2 leaves 2 u B, and the difference, the charge, the
  division by r and the product with dx 5.5 u |A - B|:  |dF| <= 9 u |qq| (A + B);
  1/r leaves 2.5 u/r, r and rc2 in the middle term u B (1.5 r + 4 (rc - r)), the sums
  and the charge the rest:  |dE| <= u |qq| (6/r + 11/rc).
"""
import numpy as np
import pytest

from seplib_amd import sep as S
from seplib_amd.sim import SepSystem

pytestmark = pytest.mark.gpu

RC = 2.5
Q = (0.7, -1.3)


def _distances():
    below = RC * (1.0 - np.array([2.0 ** -52, 1e-15, 1e-13, 1e-10, 1e-7, 1e-4]))
    r = np.concatenate([np.geomspace(1e-6, 0.3, 120), np.linspace(0.3, RC, 400, endpoint=False),
                        below])
    return r[r < RC]


def _system(product, update):
    w = dict(x=np.full((2, 3), 4.0), v=np.zeros((2, 3)), m=np.ones(2), q=np.array(Q),
             type=np.full(2, b"A"), L=np.full(3, 14.0), mol=np.full(2, -1))
    w["x"][0, 0] = 0.0
    return SepSystem.from_workload(product, w, cf=RC, dt=0.001, skin=0.25, update=update,
                                   nsubbox=(5, 5, 5))


def _call(s, r):
    s.view["x"][1, 0] = r
    s.reset_retval()
    s.reset_force()
    s.coulomb_sf(RC)


def _walk(s, r):
    s.view["x"][1, 0] = r
    s.sys.neighb_flag = 1
    s.check(s._lib().sep_gpu_upload(s.atoms, s.sysp))
    s.gpu_run([s.op_pairs("BB", RC), s.op_coulomb(RC)], 1)
    s.gpu_sync()


@pytest.mark.parametrize("way", ["call", "walk"])
def test_pair_within_rounding(product, way):
    s = _system(product, S.SEP_BRUTE if way == "call" else S.SEP_LLIST_NEIGHBLIST)
    try:
        if way == "walk":
            s.gpu_resident(True)
        ld, u = np.longdouble, 2.0 ** -53
        qq = ld(Q[0] * Q[1])
        worst = [0.0, 0.0]
        for r in _distances():
            (_call if way == "call" else _walk)(s, r)
            f, e = np.array(s.view["f"]), s.ret.ecoul
            assert np.array_equal(f[0], -f[1]) and not f[:, 1:].any()
            A, B = 1 / ld(r) ** 2, 1 / ld(RC) ** 2
            F = qq * (A - B)
            E = qq * (1 / ld(r) + (ld(r) - ld(RC)) * B - 1 / ld(RC))
            dF = abs(ld(f[1, 0]) - F) / (u * abs(qq) * (A + B))
            dE = abs(ld(e) - E) / (u * abs(qq) * (6 / ld(r) + 11 / ld(RC)))
            assert dF <= 9.0, (r, dF)
            assert dE <= 1.0, (r, dE)
            worst = [max(worst[0], float(dF)), max(worst[1], float(dE))]
        print("largest: force %.2f of 9, energy %.2f of 1" % tuple(worst), flush=True)
    finally:
        s.close()


@pytest.mark.parametrize("way", ["call", "walk"])
def test_charges_in_one_place(product, way):
    """The division's infinities: the energy is infinite, the force undefined."""
    s = _system(product, S.SEP_BRUTE if way == "call" else S.SEP_LLIST_NEIGHBLIST)
    try:
        if way == "walk":
            s.gpu_resident(True)
        (_call if way == "call" else _walk)(s, 0.0)
        assert s.ret.ecoul == -np.inf
        assert np.isnan(s.view["f"]).all()
    finally:
        s.close()
