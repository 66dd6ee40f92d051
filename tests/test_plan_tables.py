"""Pass tables are cached and shared by plans of every thread: what one plan
holds, and a running call reads, planning elsewhere leaves alone."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SO = os.path.join(HERE, "_build", "libplan_tables_host.so")
CSRC = os.path.join(HERE, "..", "eithot_amd", "csrc")


@pytest.fixture(scope="module")
def pt():
    src = os.path.join(HERE, "plan_tables_harness.cpp")
    deps = [src] + [os.path.join(CSRC, f) for f in ("plan.cpp", "plan.hpp", "maps.hpp")]
    if not os.path.exists(SO) or os.path.getmtime(SO) < max(map(os.path.getmtime, deps)):
        os.makedirs(os.path.dirname(SO), exist_ok=True)
        tmp = f"{SO}.{os.getpid()}.tmp"
        subprocess.check_call(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "-O1",
                               "-std=c++17", "-fPIC", "-shared", "-pthread", "-o", tmp, src])
        os.replace(tmp, SO)
    L = ctypes.CDLL(SO)
    shape = [ctypes.POINTER(ctypes.c_int64), ctypes.POINTER(ctypes.c_int), ctypes.c_int,
             ctypes.c_int64]
    L.pt_replan.argtypes = shape + [ctypes.c_int64, ctypes.POINTER(ctypes.c_int)]
    L.pt_plan_ms.argtypes = shape + [ctypes.c_int, ctypes.c_int]
    L.pt_plan_ms.restype = ctypes.c_double
    return L


# short cycles (grouped by length), long ones, cells of 128 bytes to beyond 1 KiB
@pytest.mark.parametrize("dims,perm,elem,other", [
    ([32, 15, 15, 16, 15, 15], [1, 4, 3, 6, 2, 5], 4, 8), ([32, 15, 15, 32, 15, 15], [4, 3, 6, 2, 1, 5], 4, 2),
    ([32, 48, 64, 40], [4, 2, 3, 1], 4, 2), ([7248, 724], [2, 1], 4, 2), ([40, 30, 30, 30], [1, 4, 3, 2], 8, 4)])
def test_tables_of_a_plan_stay(pt, dims, perm, elem, other):
    n = ctypes.c_int()
    r = pt.pt_replan((ctypes.c_int64 * len(dims))(*dims), (ctypes.c_int * len(perm))(*perm),
                     len(dims), elem, other, ctypes.byref(n))
    assert r == 0, f"pass {r - 1}'s table changed"
    assert n.value > 0


# plans that cost less than any with a pass of small cells could
@pytest.mark.parametrize("dims,perm,elem", [([150, 300, 300], [3, 2, 1], 8),
                                            ([32, 15, 15, 32, 15, 15], [4, 3, 6, 2, 1, 5], 4)])
def test_plans_that_small_cells_cannot_beat_are_searched_once(pt, dims, perm, elem):
    a = ((ctypes.c_int64 * len(dims))(*dims), (ctypes.c_int * len(perm))(*perm), len(dims), elem)
    without, both = pt.pt_plan_ms(*a, 0, 9), pt.pt_plan_ms(*a, 1, 9)
    assert 0 < both < 1.5 * without, (without, both)
