"""CPU: the slab pass's tables, walked the way its kernel walks them
(tests/slab_emu.cpp): bounds of every read, the split of the terms between the
pass and the fast-block sweep, and the result against the step lists."""
import ctypes
import os
import shutil
import subprocess

import pytest

from nadvibs_amd.engine import problem_struct
from nadvibs_amd.synth import make_problem, workload

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "nadvibs_amd", "csrc")

# ns, nfunc, offdiag_even, quirks (ordr 3): one to three L modes, none to four G modes, basis sizes of one
# and two (monomials whose steps shrink), one to four states, 33 to 64 fast rows
CASES = [
    (4, [3, 4, 4, 4], 0.0, 3),
    (4, [3, 5, 4, 4, 4, 4], 0.0, 3),
    (3, [2, 3, 4, 6, 6], 30.0, 3),
    (2, [3, 2, 1, 3, 5, 8], 0.0, 0),
    (1, [5, 6, 7, 7], 0.0, 0),
    (3, [3, 1, 4, 4, 4], 5.0, 3),
    (4, [5, 2, 2, 3, 6, 6], 10.0, 3),
    (4, [2, 2, 3, 2, 3, 4, 4, 4], 0.0, 3),
    (2, [12, 11, 13, 7, 7], 0.0, 3),
    (3, [40, 3, 60], 0.0, 3),
    (4, [3, 3, 3, 3, 3, 3, 2, 37], 0.0, 0),
]


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    out = str(tmp_path_factory.mktemp("slabemu") / "libslabemu.so")
    subprocess.check_call([gxx, "-O2", "-std=c++17", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "include"),
                           "-I" + CSRC, os.path.join(ROOT, "tests", "slab_emu.cpp"),
                           os.path.join(CSRC, "nv_operator.cpp"), "-o", out])
    lib = ctypes.CDLL(out)
    lib.slab_emulate.restype = ctypes.c_double
    lib.slab_emulate.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_long] + [ctypes.POINTER(ctypes.c_int)] * 3
    return lib


def _run(lib, prob, el, maxgroups):
    desc, keep = problem_struct(prob)
    on, bad, shape = ctypes.c_int(), ctypes.c_int(), (ctypes.c_int * 6)()
    err = lib.slab_emulate(ctypes.byref(desc), el, maxgroups, ctypes.byref(on), ctypes.byref(bad), shape)
    del keep
    return err, on.value, bad.value, list(shape)


@pytest.mark.parametrize("el", [4, 8])
@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}x{'-'.join(map(str, c[1]))}" for c in CASES])
def test_slab_tables(emu, case, el):
    ns, nf, offe, quirks = case
    p = make_problem(ns, nf, 3, (400, 2500), 200.0, 60.0, 40.0, cubic=10.0, seed=len(nf), quirks=quirks,
                     offdiag_even=offe)
    err, on, bad, shape = _run(emu, p, el, 60)
    assert on == 1, shape
    assert bad == 0, (bad, shape)
    assert err < 1e-13, (err, shape)


def test_slab_tables_of_the_ten_mode_operator(emu):
    for el in (4, 8):
        err, on, bad, shape = _run(emu, workload("cfg3"), el, 12)
        assert on == 1 and bad == 0 and err < 1e-13, (err, bad, shape)
        assert shape[0] == 3 and shape[1] == 4  # modes 4..6 in LDS, 0..3 gathered


def test_no_slab_without_cubic_slow_terms_or_above_four_states(emu):
    for p in (make_problem(3, [4, 4, 6, 6], 2, (400, 2500), 200.0, 60.0, 40.0, seed=1),
              make_problem(5, [4, 4, 6, 6], 3, (400, 2500), 200.0, 60.0, 40.0, cubic=10.0, seed=1)):
        assert _run(emu, p, 4, 10)[1] == 0
