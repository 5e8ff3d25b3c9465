"""The walk of LJ and Coulomb together by 16 lanes an atom gives the bits of the
two calls made one after the other, which walk by four: at sizes on either side
of its workgroups, of a wave, and of the largest system it serves; with lists of
no, few and many batches; with and without a type filter, into a cleared and a
used force; in boxes where few and most pairs cross a face; with atoms that
carry no charge or neither type.
"""
import numpy as np
import pytest

from seplib_amd import sep as S
from seplib_amd import workloads as W
from seplib_amd.sim import SepSystem

pytestmark = pytest.mark.gpu

STEPS = 3


def _system(n, rho, seed):
    L = max(6.6, (n / rho) ** (1.0 / 3.0))
    k = int(np.ceil(n ** (1.0 / 3.0)))
    g = (np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n] + 0.5)
    x = np.mod(g * (L / k) + 0.1 * (W.uniform(seed, 3 * n).reshape(n, 3) - 0.5), L)
    q = np.where(np.arange(n) % 3 == 0, 0.0, np.where(np.arange(n) % 2 == 0, 0.4, -0.4))
    t = np.where(np.arange(n) % 5 == 0, b"B", np.where(np.arange(n) % 7 == 0, b"C", b"A"))
    return dict(x=x, v=0.1 * W.normal(seed + 1, 3 * n).reshape(n, 3), m=np.ones(n), q=q,
                type=t, L=np.full(3, L), mol=np.full(n, -1))


def _run(product, w, types, precision, used, together, room=0):
    s = SepSystem.from_workload(product, w, cf=2.5, dt=0.001, skin=0.25)
    try:
        s.gpu_precision(precision)
        if room:  # the list's allocation, without a bound on it
            for entries in (room, 0):
                s.check(s._lib().sep_gpu_list_limit(s.atoms, s.sysp, entries))
        s.gpu_resident(True)
        if together:
            ops = [s.op_pairs(types, 2.5, "sep_lj_shift"), s.op_coulomb(2.4), s.op_leapfrog()]
            if used:
                ops.insert(0, s.op_pairs("BB", 2.0, "sep_lj_shift"))
            s.gpu_run(ops, STEPS, graph=True)
        else:
            for _ in range(STEPS):
                s.reset_retval()
                s.reset_force()
                if used:
                    s.force_pairs("BB", 2.0, "sep_lj_shift")
                s.force_pairs(types, 2.5, "sep_lj_shift")
                s.coulomb_sf(2.4)
                s.leapfrog()
        s.gpu_sync()
        out = {k: np.array(s.view[k]) for k in ("x", "v", "f")}
        out.update(epot=s.ret.epot, ecoul=s.ret.ecoul, potP=S.mat(s.ret.pot_P).copy())
        return out
    finally:
        s.close()


@pytest.mark.parametrize("precision", [S.SEP_GPU_FP64, S.SEP_GPU_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("n,rho", [(1, 0.001), (15, 0.05), (17, 0.05), (64, 0.2), (257, 0.9),
                                   (1000, 0.9), (3001, 0.5), (8192, 0.7), (8193, 0.7)])
@pytest.mark.parametrize("types,used", [("AB", False), ("AA", True)])
def test_wide_walk_same_bits(product, n, rho, types, used, precision):
    w = _system(n, rho, 11 + n)
    a = _run(product, w, types, precision, used, True)
    b = _run(product, w, types, precision, used, False)
    for k in a:
        assert np.array_equal(np.asarray(a[k]), np.asarray(b[k])), k


@pytest.mark.parametrize("room", [128, 512])
@pytest.mark.parametrize("n,rho", [(1, 0.001), (15, 0.05), (17, 0.05), (64, 0.2), (4096, 0.1),
                                   (4097, 0.1), (8192, 0.1), (8193, 0.1)])
def test_walks_of_short_lists(product, n, rho, room):
    """Short lists, whose allocation decides how many lanes walk them."""
    w = _system(n, rho, 11 + n)
    a = _run(product, w, "AB", S.SEP_GPU_FP64, False, True, room)
    b = _run(product, w, "AB", S.SEP_GPU_FP64, False, False)
    for k in a:
        assert np.array_equal(np.asarray(a[k]), np.asarray(b[k])), k
