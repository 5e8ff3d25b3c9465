"""The near build of a batch against the general one, which serves lists of more
than 256 entries: the same forces, energies and stress to the bit, for systems
of three to six cells an axis, for cells of few atoms and of more candidates than
the near build stages, with atoms on the faces of the box and outside it, pairs
at the rounding of the list cutoff, and any number of lanes an atom.
"""
import numpy as np
import pytest

from seplib_amd import batch as B
from seplib_amd import sep as S
from seplib_amd import workloads as W

pytestmark = pytest.mark.gpu

RL = B.RC + B.SKIN


def _lattice(n, L, seed):
    k = int(np.ceil(n ** (1.0 / 3.0)))
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n] + 0.5
    return np.mod(g * (L / k) + 0.05 * (W.uniform(seed, 3 * n).reshape(n, 3) - 0.5), L)


def _edge(x, L):
    """Atoms 30.. at the list cutoff from atoms 0.., a few ulps up to 1e-5 either way."""
    u = W.normal(3, 48).reshape(16, 3)
    u /= np.linalg.norm(u, axis=1)[:, None]
    eps = np.array([0, 1e-16, 4e-16, 1e-12, 1e-9, 1e-7, 1e-6, 1e-5])
    x[30:46] = np.mod(x[:16] + (RL * (1.0 + np.concatenate([eps, -eps])))[:, None] * u, L)
    return x


def _systems():
    out = []
    for k, (cells, per) in enumerate([(3.01, 4), (3.4, 23), (3.9, 45), (4.5, 12), (5.2, 30), (6.0, 22)]):
        L = RL * cells
        n = max(60, int(per * int(cells) ** 3))
        out.append((_lattice(n, L, 5 + k), L))
    x, L = _lattice(900, RL * 3.6, 21), RL * 3.6
    out.append((_edge(x.copy(), L), L))
    x = x.copy()
    x[0] = [0.0, 0.0, 0.0]
    x[1] = [np.nextafter(L, 0.0)] * 3
    out.append((x, L))
    x = x.copy()
    x[2] = [L, 0.4 * L, 0.6 * L]
    out.append((x, L))
    reps = []
    for k, (x, L) in enumerate(out):
        n = len(x)
        w = dict(x=x, v=W.normal(40 + k, 3 * n).reshape(n, 3), m=np.ones(n), q=np.zeros(n),
                 type=np.full(n, b"A"), L=np.full(3, L), mol=np.full(n, -1))
        reps.append(dict(n=n, rho=n / L ** 3, T=1.0, w=w))
    return reps


def _forces(product, reps, cap, lanes, precision):
    systems = B.make_systems(product, reps)
    b = B.Batch(product, systems, [1.0] * len(reps), precision=precision, cap=cap)
    try:
        if lanes:
            b.set_shape([lanes] * len(reps))
        b.eval(precision)
        rets, _ = b.sync()
        return [(np.array(s.view["f"]), r.epot, S.mat(r.pot_P).copy())
                for s, r in zip(systems, rets)]
    finally:
        b.close()


@pytest.mark.parametrize("lanes", [0, 1, 2, 8, 16])
@pytest.mark.parametrize("precision", [S.SEP_GPU_FP64, S.SEP_GPU_MIXED], ids=["fp64", "mixed"])
def test_near_build_same_bits(product, lanes, precision):
    reps = _systems()
    near = _forces(product, reps, 256, lanes, precision)
    far = _forces(product, reps, 320, lanes, precision)
    # (atoms 0 and 1 at the corners of the box meet across it: what is not finite
    # in the mixed form has to be so in both)
    for k, (a, c) in enumerate(zip(near, far)):
        assert np.nanmax(np.abs(c[0])) > 0.0, k
        assert np.array_equal(a[0], c[0], equal_nan=True), (k, "f")
        assert np.array_equal(a[1], c[1], equal_nan=True), (k, "epot")
        assert np.array_equal(a[2], c[2], equal_nan=True), (k, "pot_P")


@pytest.mark.parametrize("n", [8192, 8193])
def test_binning_same_bits(product, n):
    """A system beside one that decides which binning serves the batch."""
    small = W.random_packed(700, 0.8, 1.0, seed=9)
    alone = _forces(product, [dict(n=700, rho=0.8, T=1.0, w=small)], 0, 0, S.SEP_GPU_FP64)
    reps = [dict(n=700, rho=0.8, T=1.0, w=small),
            dict(n=n, rho=0.7, T=1.0, w=W.random_packed(n, 0.7, 1.0, seed=10))]
    both = _forces(product, reps, 0, 0, S.SEP_GPU_FP64)
    assert np.array_equal(alone[0][0], both[0][0])
    assert alone[0][1] == both[0][1]


def test_build_choice_same_bits(product):
    """A system of 1000 cells alone, built by the general path, and beside small
    ones, with which the batch takes the near one."""
    big = dict(n=20000, rho=0.9, T=1.0, w=W.random_packed(20000, 0.9, 1.0, seed=12))
    small = dict(n=200, rho=0.8, T=1.0, w=W.random_packed(200, 0.8, 1.0, seed=13))
    alone = _forces(product, [big], 0, 0, S.SEP_GPU_FP64)
    both = _forces(product, [big, small, small], 0, 0, S.SEP_GPU_FP64)
    for a, b in zip(alone[0], both[0]):
        assert np.array_equal(np.asarray(a), np.asarray(b))
