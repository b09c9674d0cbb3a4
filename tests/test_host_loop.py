"""What a trip-scheduled call leaves behind: its kernels have all finished when it returns.

The workspace, lists and counts belong to the reactor, and the next call may come on
another stream, which nothing orders behind the first: a kernel of the first call still
running then would read the second call's cells and append to its lists, beyond their
ends.  emu_host.cpp counts the launches that the host has waited for, on every way out of
the loop: trips issued in batches and one by one, the evaluation issued before the wait
and after it, plain and compacted lists, all cells done and the cap on trips reached.
"""
import ctypes as C
import glob
import os
import subprocess

import numpy as np
import pytest

from oracle import oracle as O
from pelelm_amd import cells

HERE = os.path.dirname(os.path.abspath(__file__))
EMU = os.path.join(HERE, "cpu_emulation")
CSRC = os.path.join(os.path.dirname(HERE), "pelelm_amd", "csrc")
SRC = [os.path.join(EMU, "emu_host.cpp"), os.path.join(EMU, "hip", "hip_runtime.h")]
SRC += [os.path.join(CSRC, f) for f in ("reactor_bdf.hip", "reactor_internal.h", "mlp_internal.h")]
SRC += sorted(glob.glob(os.path.join(CSRC, "mech", "*.inc")))
CLANG = "/opt/rocm/llvm/bin/clang++"
MECH, N = "LiDryer", 1000


@pytest.fixture(scope="module")
def lib():
    out = os.path.join(EMU, "_build", "libhost.so")
    if not os.path.exists(out) or any(os.path.getmtime(s) > os.path.getmtime(out) for s in SRC):
        os.makedirs(os.path.dirname(out), exist_ok=True)
        subprocess.run([CLANG, "-O2", "-std=c++17", "-fPIC", "-shared", "-DPELE_TU_MECH",
                        f'-DPELE_TU_MECH_INC="mech/{MECH}.inc"', f"-DPELE_TU_MECH_TYPE=mech_{MECH}",
                        f"-DPELE_TU_MECH_FN=mech_table_{MECH}", "-I" + EMU, "-I" + CSRC, "-o", out, SRC[0]], check=True)
    return C.CDLL(out)


def _react(lib, d, n, compact, gmres, ahead, cap, profile=0):
    p = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
    rY, T, rE = (d[k][..., :n].copy() for k in ("rY", "T", "rE"))
    FC, cnt, out = np.zeros(n), np.zeros(16, dtype=np.uint64), (C.c_long * 4)()
    rc = lib.host_react(C.c_long(n), p(rY), p(T), p(rE), p(FC), C.c_double(d["dt"]), C.c_double(1e-6),
                        C.c_double(1e-10), compact, gmres, ahead, profile, C.c_long(cap), p(cnt), out)
    assert rc == 0
    return rY, T, FC, cnt, {"launched": out[0], "left": out[1], "looks": out[2], "trips": out[3]}


@pytest.fixture(scope="module")
def box():
    return cells.generate_workload("lidryer_16", ncell=N)


@pytest.mark.parametrize("n", [130, N])
@pytest.mark.parametrize("compact,gmres", [(0, 0), (1, 0), (0, 1)])
@pytest.mark.parametrize("ahead,profile", [(0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("cap", [60100, 19])
def test_no_kernel_outlives_the_call(lib, box, n, compact, gmres, ahead, profile, cap):
    FC, cnt, out = _react(lib, box, n, compact, gmres, ahead, cap, profile)[2:]
    assert out["launched"] > 0
    assert out["left"] == 0
    if cap == 19:   # no multiple of a batch: exactly 19 trips, and every unfinished cell failed
        assert out["trips"] == 19
        assert cnt[8] == np.count_nonzero(FC < 0) > 0
        assert np.abs(FC).max() <= 19


@pytest.mark.parametrize("compact,gmres", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("cap", [60100, 19])
def test_batches_and_early_evaluations_change_nothing(lib, box, compact, gmres, cap):
    """The same cells with their trips as the call issues them (in batches of eight for
    compacted lists and GMRES, else each evaluation before the wait), without the early
    evaluation, and one by one: the same states, counts and number of trips."""
    usual, late, single = [_react(lib, box, N, compact, gmres, ahead, cap, profile)
                           for ahead, profile in ((1, 0), (0, 0), (1, 1))]
    for other in (late, single):
        for a, b in zip(usual[:4], other[:4]):
            np.testing.assert_array_equal(a, b)
        assert usual[4]["trips"] == other[4]["trips"]
    trips = usual[4]["trips"]
    assert single[4]["looks"] == trips + (cap != 19)
    assert usual[4]["looks"] == (-(-trips // 8) if compact or gmres else trips + (cap != 19))
