"""How a staged device-to-host copy is cut (nimblesm_amd/csrc/nsm_copy_plan.h):
the pinned memory that a copy may use first costs its first touch, 370 us per
MB, so it stays a small share of what a plain copy of that size takes."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("plan") / "libplan.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-o", out,
                    os.path.join(ROOT, "tests", "copy_plan_shim.cpp")], check=True)
    lib = C.CDLL(out)
    lib.copy_plan.argtypes = [C.c_size_t, C.c_void_p]
    lib.copy_plan.restype = None

    def of(size):
        p = np.zeros(4, np.uint64)
        lib.copy_plan(size, p.ctypes.data)
        return [int(v) for v in p]

    return of


@pytest.mark.parametrize("mb", [2, 2.1, 6.6, 15.9, 16, 21.9, 31.9, 32, 51.5, 800])
def test_pinned_memory_is_in_proportion(plan, mb):
    size = int(mb * (1 << 20))
    chunk, own, helpers, pinned = plan(size)
    assert chunk % 8 == 0 and chunk * 2 <= size  # whole values, something to overlap
    assert own >= 2 and pinned == chunk * (own + 2 * helpers)
    assert pinned <= 0.5625 * size  # 370 us per MB of it, 70 to 100 us per MB of a plain copy, several copies
    assert pinned <= (1 << 20) or helpers > 0
    assert pinned <= 18 << 20
