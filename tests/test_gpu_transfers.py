"""The atoms' way to the device and back: every field survives bit for bit, in
original order, at sizes on either side of a workgroup of a transfer, of a
chunk of a download, of the host threads and of the most chunks there are, and
again once the device has sorted the atoms.  The same for batches whose
systems share chunks, fill one, or exceed one.
"""
import ctypes as C

import numpy as np
import pytest

from seplib_amd import batch as B
from seplib_amd import sep as S
from seplib_amd import workloads as W
from seplib_amd.sim import SepSystem

pytestmark = pytest.mark.gpu

DOUBLES = ("x", "v", "f", "a", "xn")
INTS = ("cross_neighb", "crossings")


def _fill(view, seed):
    n = len(view["x"])
    for k, name in enumerate(DOUBLES[1:]):
        view[name] = W.normal(seed + k, 3 * n).reshape(n, 3)
    for k, name in enumerate(INTS):
        view[name] = np.arange(3 * n).reshape(n, 3) * (k + 1) % 1013 - 500


def _clear(view):
    for name in DOUBLES + INTS:
        view[name] = 0


@pytest.mark.parametrize("n", [1, 63, 64, 65, 16384, 16385, 32767, 32768, 32769, 262145])
def test_fields_survive(product, n):
    L = max(12.0, (n / 0.2) ** (1.0 / 3.0))
    w = dict(x=W.uniform(n, 3 * n).reshape(n, 3) * L, v=np.zeros((n, 3)),
             m=1.0 + W.uniform(n + 1, n), q=W.normal(n + 2, n), type=np.full(n, b"A"),
             L=np.full(3, L), mol=np.full(n, -1))
    s = SepSystem.from_workload(product, w, cf=2.5, dt=0.005, skin=0.3, nneighb=8)
    try:
        _fill(s.view, 7)
        s.view["xn"] = w["x"]
        want = {k: np.array(s.view[k]) for k in DOUBLES + INTS}
        s.gpu_resident(True)
        _clear(s.view)
        s.gpu_sync()
        for k in want:
            assert np.array_equal(s.view[k], want[k]), (k, "as uploaded")
        # a pair call sorts the atoms and replaces f alone
        s.gpu_run([s.op_pairs("AA", 2.5, "sep_lj_shift")], 1)
        _clear(s.view)
        s.gpu_sync()
        for k in want:
            if k != "f":
                assert np.array_equal(s.view[k], want[k]), (k, "sorted")
    finally:
        s.close()


@pytest.mark.parametrize("n", [16384, 49151, 49152])
def test_synchronised_step(product, n):
    """A synchronised leapfrog without forces, packed and unpacked by the caller
    alone and by several threads: x moves by v dt, and nothing else does."""
    L, dt = 50.0, 0.004
    x = W.uniform(n, 3 * n).reshape(n, 3) * (L - 2.0) + 1.0
    v = W.normal(n + 1, 3 * n).reshape(n, 3)
    w = dict(x=x, v=v, m=1.0 + W.uniform(n + 2, n), q=np.zeros(n), type=np.full(n, b"A"),
             L=np.full(3, L), mol=np.full(n, -1))
    s = SepSystem.from_workload(product, w, cf=2.5, dt=dt, skin=0.3, nneighb=8)
    try:
        s.view["crossings"] = np.arange(3 * n).reshape(n, 3)
        s.view["xn"] = x
        s.leapfrog()
        assert np.array_equal(s.view["x"], x + v * dt)
        assert np.array_equal(s.view["v"], v) and not np.array(s.view["a"]).any()
        assert np.array_equal(s.view["crossings"], np.arange(3 * n).reshape(n, 3))
        assert np.array_equal(s.view["xn"], x)
    finally:
        s.close()


@pytest.mark.parametrize("sizes", [[33], [64, 65, 200], [300] * 70, [17000, 40, 20000, 900, 50]])
def test_batch_survives(product, sizes):
    reps = [dict(n=n, rho=0.3, T=1.0, w=W.random_packed(n, 0.1, 1.0, seed=5 + k))
            for k, n in enumerate(sizes)]
    systems = B.make_systems(product, reps)
    b = B.Batch(product, systems, [1.0] * len(reps), precision=S.SEP_GPU_FP64)
    try:
        want = [(np.array(s.view["x"]), np.array(s.view["v"])) for s in systems]
        b.eval(S.SEP_GPU_FP64)
        for s in systems:
            s.view["x"] = 0
            s.view["v"] = 0
        b.sync()
        for k, s in enumerate(systems):
            assert np.array_equal(s.view["x"], want[k][0]), (k, "x")
            assert np.array_equal(s.view["v"], want[k][1]), (k, "v")
    finally:
        b.close()


@pytest.mark.parametrize("n,clump", [(2, 0), (64, 64), (65, 65), (500, 400), (3000, 700)])
def test_half_rows(product, oracle, n, clump):
    """The rows written to neighb, in atom order and within their own arrays,
    from few atoms up to clumps whose rows take more room than the buffer has
    (several passes)."""
    L = 14.0
    x = W.uniform(n, 3 * n).reshape(n, 3) * L
    x[:clump] = 4.0 + W.uniform(n + 1, 3 * clump).reshape(clump, 3) * 1.5
    w = dict(x=x, v=np.zeros((n, 3)), m=np.ones(n), q=np.zeros(n), type=np.full(n, b"A"),
             L=np.full(3, L), mol=np.full(n, -1))

    pairs = []
    for api in (product, oracle):
        s = SepSystem.from_workload(api, w, cf=2.5, dt=0.005, skin=0.3, nneighb=n + 2,
                                    nsubbox=(5, 5, 5))
        try:
            s.reset_retval()
            s.reset_force()
            s.force_pairs("AA", 2.5, "sep_lj_shift")
            pairs.append(s.half_pairs())
            if api is product:
                pairs.append(s.gpu_pairs())
        finally:
            s.close()
    assert np.array_equal(pairs[0], pairs[2])
    assert np.array_equal(pairs[1], pairs[2])


def test_batch_in_several_passes(product):
    """More records than the pinned buffer holds (64 MiB: 9362 systems of one to
    three atoms, each with 64 slots), a larger system among each pass's."""
    reps = []
    for k in range(9500):
        n = 300 if k in (4000, 9450) else 1 + k % 3
        x = (W.uniform(k, 3 * n).reshape(n, 3) + 0.01) * 5.8
        reps.append(dict(n=n, rho=n / 216.0, T=1.0, w=dict(
            x=x, v=W.normal(k, 3 * n).reshape(n, 3), m=np.ones(n), q=np.zeros(n),
            type=np.full(n, b"A"), L=np.full(3, 6.0), mol=np.full(n, -1))))
    systems = B.make_systems(product, reps, nneighb=4)
    b = B.Batch(product, systems, [1.0] * len(reps), precision=S.SEP_GPU_FP64)
    try:
        b.eval(S.SEP_GPU_FP64)
        for s in systems:
            for k in ("x", "v"):
                s.view[k] = 0
            for k in ("f", "a", "crossings"):
                s.view[k] = 7
        b.sync()
        for s, r in zip(systems, reps):
            assert np.array_equal(s.view["x"], r["w"]["x"])
            assert np.array_equal(s.view["v"], r["w"]["v"])
            assert not (np.array(s.view["f"]) == 7).any()
            assert not np.array(s.view["a"]).any() and not np.array(s.view["crossings"]).any()
    finally:
        b.close()
        for s in systems:
            s.close()


def test_half_rows_in_several_passes(product):
    """Rows that fill more than the largest buffer (256 MiB), against the count
    of the full lists."""
    n, L, cf = 38000, 15.0, 4.9
    x = W.uniform(91, 3 * n).reshape(n, 3) * L
    w = dict(x=x, v=np.zeros((n, 3)), m=np.ones(n), q=np.zeros(n), type=np.full(n, b"A"),
             L=np.full(3, L), mol=np.full(n, -1))
    s = SepSystem.from_workload(product, w, cf=cf, dt=0.005, skin=0.0, nneighb=4,
                                nsubbox=(3, 3, 3))
    lib = product.lib
    try:
        s.gpu_resident(True)
        s.gpu_run([s.op_pairs("BB", cf)], 1)
        mean, mx = C.c_double(0.0), C.c_int(0)
        assert lib.sep_gpu_list_stats(s.atoms, C.byref(mean), C.byref(mx)) == 0
        total = int(round(mean.value * n)) // 2
        assert total > 64 * 1024 * 1024 * 1.5
        got = np.empty(2 * total, dtype=np.int32)
        cnt = C.c_long(0)
        assert lib.sep_gpu_neighbour_pairs(s.atoms, s.sysp, got.ctypes.data_as(C.POINTER(C.c_int)),
                                           total, C.byref(cnt)) == 0
        assert cnt.value == total
        # rows in atom order, their entries above the atom
        i, j = got[0::2], got[1::2]
        assert (np.diff(i) >= 0).all() and (j > i).all() and j.max() < n
        # the counts of a few atoms, from the positions
        deg = np.bincount(i, minlength=n) + np.bincount(j, minlength=n)
        for a in (0, 1, 777, 20000, 31000, n - 1):
            d = x - x[a]
            d -= L * np.rint(d / L)
            r2 = (d * d).sum(1)
            lo, hi = (r2 < (cf * cf) * (1 - 1e-12)).sum() - 1, (r2 < (cf * cf) * (1 + 1e-12)).sum() - 1
            assert lo <= deg[a] <= hi, a
            row = j[slice(*np.searchsorted(i, [a, a + 1]))]
            assert len(np.unique(row)) == len(row)
    finally:
        s.close()
