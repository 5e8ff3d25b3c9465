"""The library's host sources (seplib_amd/csrc/host/*.c) with the device calls
replaced by the test program's own (CPU), one program a promise:

  * tests/host/adjoint_noalloc.c: sep_gpu_lj_adjoint_noalloc neither allocates
    nor starts a thread;
  * tests/host/thread_signals.c: the threads that calls on many atoms start
    take none of the program's signals, and the caller's mask is as it was.
"""
import glob
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIBDIR = os.path.join(ROOT, "seplib_amd")


def _run(tmp_path, name, wrap):
    if shutil.which("gcc") is None:
        pytest.skip("gcc not available")
    if not os.path.exists(os.path.join(LIBDIR, "libsep.so")):
        pytest.skip("libsep.so not built")
    exe = os.path.join(str(tmp_path), name)
    host = sorted(glob.glob(os.path.join(LIBDIR, "csrc", "host", "*.c")))
    # the device calls a program does not define come from the library, and
    # are not reached
    p = subprocess.run(["gcc", "-std=c99", "-g", "-O1", "-D_GNU_SOURCE",
                        "-I", os.path.join(ROOT, "include"), "-I", os.path.join(LIBDIR, "csrc"),
                        "-I", os.path.join(LIBDIR, "csrc", "host"),
                        os.path.join(ROOT, "tests", "host", name + ".c")] + host +
                       ["-Wl,--wrap=" + f for f in wrap] +
                       ["-o", exe, "-L", LIBDIR, "-lsep", "-Wl,-rpath," + LIBDIR, "-lm",
                        "-lpthread"], capture_output=True, text=True)
    assert p.returncode == 0, p.stderr[-3000:]
    p = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, (p.returncode, p.stdout[-2000:], p.stderr[-2000:])


def test_noalloc_adjoint_allocates_nothing(tmp_path):
    _run(tmp_path, "adjoint_noalloc", ["malloc", "calloc", "realloc", "pthread_create"])


def test_helper_threads_take_no_signals(tmp_path):
    _run(tmp_path, "thread_signals", [])
