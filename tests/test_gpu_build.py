"""The list build where its path changes: the quantized build's grids from 3
cells an axis up, cells fuller than a wave, home atoms whose candidates take
several passes, atoms on and outside the faces of the box, pairs within the
rounding of the list cutoff, the exclusion rules, and the FP64 build of a
box that is not cubic.  The pair set is the oracle's, pair for pair.
"""
import numpy as np
import pytest

from seplib_amd import sep as S
from seplib_amd import workloads as W
from seplib_amd.sim import SepSystem

pytestmark = pytest.mark.gpu

CF, SKIN = 2.5, 0.3
RL = CF + SKIN


def _points(n, L, seed, clump=0):
    """n random points in the box, `clump` of them inside one cell's size."""
    x = W.uniform(seed, 3 * n).reshape(n, 3) * L
    x[:clump] = 0.3 * L + W.uniform(seed + 1, 3 * clump).reshape(clump, 3) * 2.0
    return x


def _edge_pairs(x, L, seed):
    """Moves the second half of 40 of the points to the list cutoff from the
    first half, inside and outside it by a few ulps up to 1e-4."""
    u = W.normal(seed, 60).reshape(20, 3)
    u /= np.linalg.norm(u, axis=1)[:, None]
    eps = np.array([0, 1e-16, 4e-16, 1e-12, 1e-9, 1e-7, 1e-6, 1e-5, 3e-5, 1e-4])
    r = RL * (1.0 + np.concatenate([eps, -eps]))
    x[20:40] = np.mod(x[:20] + r[:, None] * u, L)
    return x


def _workload(x, L, mol=None, **more):
    n = len(x)
    return dict(x=x, v=np.zeros((n, 3)), m=np.ones(n), q=np.zeros(n), type=np.full(n, b"A"),
                L=np.asarray(L, dtype=np.float64), mol=np.full(n, -1) if mol is None else mol, **more)


def _chains(n, k):
    """Bonds and angles of chains of k consecutive atoms, molecule by molecule."""
    mol = np.arange(n) // k
    a = np.arange(n - 1)
    a = a[mol[a] == mol[a + 1]]
    bonds = np.stack([mol[a], a, a + 1, 0 * a], axis=1)
    b = np.arange(n - 2)
    b = b[mol[b] == mol[b + 2]]
    return mol, bonds, np.stack([mol[b], b, b + 1, b + 2, 0 * b], axis=1)


def _pairs(api, w, opt, nneighb):
    s = SepSystem.from_workload(api, w, cf=CF, dt=0.005, skin=SKIN, nneighb=nneighb,
                                nsubbox=[int(l / RL) for l in w["L"]])
    try:
        s.reset_retval()
        s.reset_force()
        s.force_pairs("AA", CF, "sep_lj", opt)
        return s.half_pairs()
    finally:
        s.close()


def _check(product, oracle, w, opt=S.SEP_ALL, nneighb=800):
    a, b = _pairs(product, w, opt, nneighb), _pairs(oracle, w, opt, nneighb)
    assert len(b) > 0
    assert np.array_equal(a, b)


@pytest.mark.parametrize("cells", [2, 3, 4, 5, 7])
@pytest.mark.parametrize("per_cell", [0.3, 12, 40])
def test_grids(product, oracle, cells, per_cell):
    L = RL * cells * 1.0001
    n = max(41, int(per_cell * cells ** 3))
    _check(product, oracle, _workload(_edge_pairs(_points(n, L, 3), L, 5), [L] * 3))


@pytest.mark.parametrize("cells,per_cell", [(5, 64), (5, 65), (6, 130)])
def test_slices(product, oracle, cells, per_cell):
    """Cells of more atoms than a wave, cut into more slices."""
    L = RL * cells * 1.0001
    n = per_cell * cells ** 3
    _check(product, oracle, _workload(_edge_pairs(_points(n, L, 15), L, 17), [L] * 3), nneighb=1200)


@pytest.mark.parametrize("clump", [60, 65, 200, 700])
@pytest.mark.parametrize("opt", [S.SEP_ALL, S.SEP_EXCL_SAME_MOL, S.SEP_EXCL_BONDED])
def test_full_cells(product, oracle, clump, opt):
    """Cells of more than 64 atoms and more candidates than a wave holds."""
    L = RL * 3.3
    n = 900
    mol, bonds, angles = _chains(n, 5)
    w = _workload(_points(n, L, 7, clump), [L] * 3, mol, bonds=bonds, angles=angles)
    _check(product, oracle, w, opt)


@pytest.mark.parametrize("opt", [S.SEP_ALL, S.SEP_EXCL_SAME_MOL, S.SEP_EXCL_BONDED])
@pytest.mark.parametrize("where", ["inside", "face", "outside"])
def test_faces(product, oracle, opt, where):
    """Atoms on the faces; at x == L, and below 0, the FP64 test of every
    candidate decides."""
    L = RL * 5.2
    n = 1200
    mol, bonds, angles = _chains(n, 4)
    x = _points(n, L, 11)
    x[0] = [0.0, 0.0, 0.0]
    x[1] = [np.nextafter(L, 0.0), 0.5 * L, 0.25 * L]
    x[2] = [0.5 * L, np.nextafter(L, 0.0), np.nextafter(L, 0.0)]
    if where == "face":
        x[3] = [L, 0.5 * L, 0.5 * L]
    if where == "outside":
        x[3] = [-1e-3, 0.5 * L, 0.5 * L]
    _check(product, oracle, _workload(x, [L] * 3, mol, bonds=bonds, angles=angles), opt)


@pytest.mark.parametrize("shape", [(3, 4, 5), (5, 6, 7)])
def test_box_not_cubic(product, oracle, shape):
    L = np.array([RL * k * 1.01 for k in shape])
    _check(product, oracle, _workload(_points(1500, L, 13), L))


@pytest.mark.parametrize("n,clump", [(4096, 0), (4097, 2500), (9000, 2100), (32768, 0), (32769, 0)])
def test_wide_cells(product, oracle, n, clump):
    """Cells much wider than the list cutoff: more members in one than the
    one-launch ordering ranks in LDS, and its largest and the next system."""
    L = 30.0
    x = W.uniform(17, 3 * n).reshape(n, 3) * L
    x[:clump] = 10.1 + W.uniform(18, 3 * clump).reshape(clump, 3) * 9.8
    w = _workload(x, [L] * 3)
    pairs = []
    for api in (product, oracle):
        s = SepSystem.from_workload(api, w, cf=1.0, dt=0.005, skin=0.2, nneighb=100,
                                    nsubbox=(3, 3, 3))
        try:
            s.reset_retval()
            s.reset_force()
            s.force_pairs("AA", 1.0, "sep_lj", S.SEP_ALL)
            pairs.append(s.half_pairs())
        finally:
            s.close()
    assert len(pairs[1]) > 0
    assert np.array_equal(*pairs)


@pytest.mark.parametrize("resident", [False, True])
@pytest.mark.parametrize("n", [4097, 16384, 16385, 32768])
def test_orderings(product, oracle, n, resident):
    """A call that is sure to rebuild and a step that rebuilds when flagged order
    the atoms in one launch up to different sizes."""
    w = W.random_packed(n, 0.5, 1.0, seed=33)
    grid = [int(l / RL) for l in w["L"]]
    s = SepSystem.from_workload(product, w, cf=CF, dt=0.005, skin=SKIN, nneighb=200, nsubbox=grid)
    o = SepSystem.from_workload(oracle, w, cf=CF, dt=0.005, skin=SKIN, nneighb=200, nsubbox=grid)
    try:
        if resident:
            s.gpu_resident(True)
            s.gpu_run([s.op_pairs("AA", CF, "sep_lj")], 1)
        else:
            s.force_pairs("AA", CF, "sep_lj")
        o.force_pairs("AA", CF, "sep_lj")
        assert np.array_equal(s.gpu_pairs(), o.half_pairs())
    finally:
        s.close()
        o.close()


@pytest.mark.parametrize("n", [1024, 1025, 2047, 2049, 4097])
def test_one_cell(product, oracle, n):
    """A box of fewer than three list cutoffs an edge: all atoms in one cell,
    ranked by several rounds of threads against several rounds of keys."""
    L = 6.0
    w = _workload(W.uniform(29, 3 * n).reshape(n, 3) * L, [L] * 3)
    pairs = []
    for api in (product, oracle):
        s = SepSystem.from_workload(api, w, cf=1.9, dt=0.005, skin=0.15, nneighb=n + 1,
                                    update=S.SEP_NEIGHBLIST)
        try:
            s.reset_retval()
            s.reset_force()
            s.force_pairs("AA", 1.9, "sep_lj", S.SEP_ALL)
            pairs.append(s.half_pairs())
        finally:
            s.close()
    assert len(pairs[1]) > 0
    assert np.array_equal(*pairs)


@pytest.mark.parametrize("n", [2, 63, 65, 4096, 4097, 32767, 32768, 32769])
def test_sums_over_blocks(product, oracle, n):
    """Energies and stress where the number of partial rows crosses the
    finisher's limits: sums of n terms in another order than the oracle's,
    each within n roundings, so 1e-12 relative holds with room to spare."""
    w = W.random_packed(n, 0.8442, 1.0, seed=23)
    if n < 1000:  # the box holds three cells an axis
        w["L"] = np.maximum(w["L"], 3.1 * RL)
    out = []
    for api in (product, oracle):
        s = SepSystem.from_workload(api, w, cf=CF, dt=0.005, skin=SKIN, nneighb=128,
                                    nsubbox=[int(l / RL) for l in w["L"]])
        try:
            s.reset_retval()
            s.reset_force()
            s.force_pairs("AA", CF, "sep_lj_shift", S.SEP_ALL)
            s.leapfrog()
            out.append((s.ret.epot, s.ret.ekin, S.mat(s.ret.pot_P), S.mat(s.ret.kin_P),
                        s.sys.max_dist2))
        finally:
            s.close()
    for a, b in zip(*out):
        scale = np.abs(b).max()
        assert np.abs(np.asarray(a) - b).max() <= 1e-12 * scale, (a, b)
