"""A device failure inside a resident run: a neighbour-list overflow, forced
from the host with sep_gpu_list_limit (the build truncates each list at the
bound and raises SEP_GPU_ENEIGHB; every access stays inside the allocated
list).

  * the failing graph-replayed run returns SEP_GPU_ENEIGHB, and the system
    stays at the step before the rebuild that overflowed: x, v, f, a, xn,
    crossings, sepret, alpha, tnow and the rebuild counters equal those of
    an unbounded run stopped there, bit for bit (for an odd and an even
    count of frozen steps, which end on either position buffer);
  * with the bound lifted, the next run continues from there and ends bit
    for bit where an uninterrupted run ends.

No kernel faults or waits here: the overflow only sets the device error
word, and every later kernel of the run reads it and leaves the state
alone.
"""
import ctypes as C
import re

import numpy as np
import pytest

from seplib_amd import sep as S
from seplib_amd import workloads as W
from seplib_amd.sim import SepSystem

pytestmark = pytest.mark.gpu

KW = dict(cf=2.5, dt=0.005, skin=0.3)


def _ops(s):
    return [s.op_pairs("AA", 2.5), s.op_nosehoover(1.0, 10.0), s.op_leapfrog()]


def _run(s, nsteps, graph=True):
    ops = _ops(s)
    arr = (S.sep_gpu_op * len(ops))(*ops)
    return s._lib().sep_gpu_run(s.atoms, s.sysp, s.retp, arr, len(ops), nsteps,
                                S.SEP_GPU_RUN_GRAPH if graph else 0)


def _snap(s):
    s.gpu_sync()
    st = s.state()
    r = s.ret
    st.update(epot=r.epot, ekin=r.ekin, potP=S.mat(r.pot_P), kinP=S.mat(r.kin_P))
    return st


def _same(a, b):
    for k in ("x", "v", "f", "a", "xn", "cross_neighb", "crossings", "potP", "kinP"):
        assert np.array_equal(a[k], b[k]), k
    for k in ("epot", "ekin", "alpha", "max_dist2", "nupdate_neighb", "neighb_flag", "tnow"):
        assert a[k] == b[k], k


@pytest.mark.parametrize("precision", [S.SEP_GPU_FP64, S.SEP_GPU_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("extra", [10, 11])
def test_list_overflow_freezes_a_graph_run(product, precision, extra):
    w = W.lj_fcc(10, 0.8442, 1.0, seed=4)  # 4000 atoms
    lib = product.lib
    a = SepSystem.from_workload(product, w, **KW)
    b = SepSystem.from_workload(product, w, **KW)
    try:
        for s in (a, b):
            s.gpu_precision(precision)
            s.gpu_resident(True)
            # the first build (checked on the host) and the second, which the
            # reference's zero xn triggers after step 1
            assert _run(s, 2, graph=False) == 0
        mean, mx = C.c_double(0.0), C.c_int(0)
        assert lib.sep_gpu_list_stats(b.atoms, C.byref(mean), C.byref(mx)) == 0
        assert mean.value > 60.0
        # reference: one step at a time until the next step rebuilds
        steps = 0
        while True:
            a.gpu_sync()
            if a.sys.neighb_flag == 1:
                break
            assert _run(a, 1, graph=False) == 0
            steps += 1
            assert steps < 200
        assert steps > 2
        ref = _snap(a)
        assert ref["nupdate_neighb"] >= 1
        # bounded well below the mean list: the next rebuild overflows
        assert lib.sep_gpu_list_limit(b.atoms, b.sysp, 48) == 0
        print("case: precision %d, rebuild after %d steps, %d frozen steps" %
              (precision, steps, extra), flush=True)
        rc = _run(b, steps + extra)
        assert rc == S.SEP_GPU_ENEIGHB, rc
        assert b"overflow" in lib.sep_gpu_last_error_message() or \
            b"neighbours" in lib.sep_gpu_last_error_message()
        _same(_snap(b), ref)
        # lifted: both continue and agree
        assert lib.sep_gpu_list_limit(b.atoms, b.sysp, 0) == 0
        assert _run(b, 30) == 0
        assert _run(a, 30) == 0
        end_a, end_b = _snap(a), _snap(b)
        assert end_a["nupdate_neighb"] > ref["nupdate_neighb"]
        _same(end_b, end_a)
    finally:
        a.close()
        b.close()


def test_list_limit_in_synchronised_mode(product):
    """The synchronised API with a bound below the lists it needs reports
    SEP_GPU_ENEIGHB (the reference's "Too many neighbours") instead of
    growing the list; lifting the bound lets the same call succeed."""
    w = W.lj_fcc(8, 0.8442, 1.0, seed=5)
    lib = product.lib
    s = SepSystem.from_workload(product, w, **KW)
    try:
        assert lib.sep_gpu_list_limit(s.atoms, s.sysp, 32) == 0
        lib.sep_gpu_clear_error()
        s.reset_retval()
        s.reset_force()
        s.force_pairs("AA", 2.5)
        assert lib.sep_gpu_last_error() == S.SEP_GPU_ENEIGHB
        assert lib.sep_gpu_list_limit(s.atoms, s.sysp, 0) == 0
        lib.sep_gpu_clear_error()
        s.sys.neighb_flag = 1
        s.reset_retval()
        s.reset_force()
        s.force_pairs("AA", 2.5)
        assert lib.sep_gpu_last_error() == 0
        assert np.abs(np.array(s.view["f"])).max() > 0
    finally:
        s.close()


@pytest.mark.parametrize("graph", [False, True], ids=["eager", "graph"])
@pytest.mark.parametrize("k,extra", [(10, 1), (10, 40), (21, 5)])
def test_overflow_of_a_bound_names_it(product, k, extra, graph):
    """However many steps follow the one that overflowed, the report holds the
    length that build found and the bound (4000 and 37044 atoms: the two ways
    the atoms are ordered)."""
    w = W.lj_fcc(k, 0.8442, 1.0, seed=4)
    lib = product.lib
    s = SepSystem.from_workload(product, w, **KW)
    try:
        s.gpu_resident(True)
        assert _run(s, 2, graph=False) == 0
        mean, mx = C.c_double(0.0), C.c_int(0)
        assert lib.sep_gpu_list_stats(s.atoms, C.byref(mean), C.byref(mx)) == 0
        assert lib.sep_gpu_list_limit(s.atoms, s.sysp, 48) == 0
        s.sys.neighb_flag = 1  # the next step rebuilds
        assert lib.sep_gpu_upload(s.atoms, s.sysp) == 0
        assert _run(s, 1 + extra, graph) == S.SEP_GPU_ENEIGHB
        said = lib.sep_gpu_last_error_message().decode()
        found = re.search(r"a list of (\d+) entries exceeds the limit of 48", said)
        assert found, said
        # the lists of a liquid two steps apart: nearly the same
        assert 0.8 * mx.value <= int(found.group(1)) <= 1.25 * mx.value, (said, mx.value)
    finally:
        s.close()


def _implosion(n, seed):
    """Atoms of type B (no pair call of "AA" moves them) on their way to the
    centre, which they would reach after 200 steps, and a few of type A at
    rest, whose forces the run computes."""
    L = (n / 0.25) ** (1.0 / 3.0)
    x = W.uniform(seed, 3 * n).reshape(n, 3) * L
    v = (0.5 * L - x) / (200 * 0.005)
    t = np.full(n, b"B")
    t[::50], v[::50] = b"A", 0.0
    na = len(t[::50])
    k = int(np.ceil(na ** (1.0 / 3.0)))
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:na]
    x[::50] = (g + 0.5) * (L / k)
    return dict(x=x, v=v, m=np.ones(n), q=np.zeros(n), type=t, L=np.full(3, L),
                mol=np.full(n, -1))


@pytest.mark.parametrize("graph", [False, True], ids=["eager", "graph"])
@pytest.mark.parametrize("n", [2000, 20000, 33000])
def test_run_continues_after_its_list_outgrew_the_allocation(product, n, graph):
    """Lists that grow several times beyond what the first build was given: each
    run that overflows says how long its longest list was and grows the list,
    the next one goes on, and the end is bit for bit that of a system whose
    list had room for all of it."""
    w = _implosion(n, 31)
    lib = product.lib
    a = SepSystem.from_workload(product, w, **KW)
    b = SepSystem.from_workload(product, w, **KW)
    steps = 110
    try:
        for s in (a, b):
            s.gpu_resident(True)
        assert lib.sep_gpu_list_limit(a.atoms, a.sysp, 1024) == 0
        ops = [b.op_pairs("AA", 2.5), b.op_leapfrog()]
        arr = (S.sep_gpu_op * len(ops))(*ops)
        flags = S.SEP_GPU_RUN_GRAPH if graph else 0

        def go(s, k):
            return lib.sep_gpu_run(s.atoms, s.sysp, s.retp, arr, len(ops), k, flags)

        assert go(a, steps) == 0
        done, grown, longest = 0, 0, 0
        while done < steps:
            t0 = b.sys.tnow
            rc = go(b, steps - done)
            if rc:
                assert rc == S.SEP_GPU_ENEIGHB
                found = re.search(r"longest list (\d+)", lib.sep_gpu_last_error_message().decode())
                assert int(found.group(1)) > max(longest, 64)
                longest = int(found.group(1))
                grown += 1
                assert grown < 12
            b.gpu_sync()
            new = int(round((b.sys.tnow - t0) / KW["dt"]))
            assert (new > 0 or grown > 0) and (rc or new == steps - done)
            done += new
        assert grown >= 2
        _same(_snap(b), _snap(a))
    finally:
        a.close()
        b.close()
