"""Composed cycle maps as digit permutations: the host's digit form and the
kernel's arithmetic on it against the maps, position by position."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import eithot_amd as E

HERE = os.path.dirname(os.path.abspath(__file__))
SO = os.path.join(HERE, "_build", "libcycle16_host.so")
CSRC = os.path.join(HERE, "..", "eithot_amd", "csrc")


@pytest.fixture(scope="module")
def ch():
    src = os.path.join(HERE, "cycle16_harness.cpp")
    deps = [src] + [os.path.join(CSRC, f) for f in ("plan.cpp", "plan.hpp", "maps.hpp")]
    if not os.path.exists(SO) or os.path.getmtime(SO) < max(map(os.path.getmtime, deps)):
        os.makedirs(os.path.dirname(SO), exist_ok=True)
        tmp = f"{SO}.{os.getpid()}.tmp"
        subprocess.check_call(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "-O1",
                               "-std=c++17", "-fPIC", "-shared", "-o", tmp, src])
        os.replace(tmp, SO)
    L = ctypes.CDLL(SO)
    L.c16_digits.restype = ctypes.c_int64
    L.c16_digits.argtypes = [ctypes.c_int, ctypes.POINTER(ctypes.c_int64), ctypes.c_int64,
                             ctypes.c_int64]
    L.c16_div.restype = ctypes.c_int64
    L.c16_div.argtypes = [ctypes.c_uint32, ctypes.c_int, ctypes.POINTER(ctypes.c_uint32)]
    L.c16_groups.restype = ctypes.c_int64
    L.c16_groups.argtypes = [ctypes.c_uint32]
    return L


def cycle_maps(dims, perm, elem):
    ops, _ = E.plan_describe(dims, perm, elem)
    return [(o["maps"], o["R"] * o["C"]) for o in ops if o["kind"] == 4]


PLANS = [([32, 15, 15, 32, 15, 15], [4, 3, 6, 2, 1, 5], 4), ([80, 96, 75, 96], [1, 4, 3, 2], 4),
         ([352, 4, 28, 48, 28], [4, 3, 2, 5, 1], 4), ([48, 151, 2, 19, 2, 7], [4, 6, 5, 2, 1, 3], 4),
         ([43, 280, 37, 3], [3, 4, 2, 1], 1), ([128, 200, 300], [1, 3, 2], 4)]


@pytest.mark.parametrize("dims,perm,elem", PLANS)
def test_digit_form_of_plans(ch, dims, perm, elem):
    passes = cycle_maps(dims, perm, elem)
    assert passes
    for maps, n in passes:
        flat = (ctypes.c_int64 * (4 * len(maps)))(*[v for m in maps for v in m])
        got = ch.c16_digits(len(maps), flat, n, 1)
        assert 1 <= got <= len(maps), (maps, n, got)


def test_digit_form_of_random_compositions(ch):
    # maps over random factorizations of N: one digit permutation where their
    # factors divide each other's digits, several where they do not
    rng = np.random.default_rng(6)
    forms = {True: 0, False: 0}
    for _ in range(400):
        f = [int(x) for x in rng.choice([1, 2, 3, 4, 5, 7, 8], size=5)]
        n = int(np.prod(f))
        if n < 2:
            continue
        maps = []
        for _ in range(int(rng.integers(1, 6))):
            g = [f[i] for i in rng.permutation(5)] if rng.random() < 0.8 else f
            m, r, c = g[0], g[1] * g[2], g[3]
            maps.append((m * r * c, r, c, m))
        flat = (ctypes.c_int64 * (4 * len(maps)))(*[v for m in maps for v in m])
        got = ch.c16_digits(len(maps), flat, n, 1)
        assert 1 <= got <= len(maps), (maps, n, got)
        forms[got > 1] += 1
    assert min(forms.values()) > 20, forms


def test_two_instruction_division(ch):
    rng = np.random.default_rng(7)
    x = (ctypes.c_uint32 * 200)(*[int(v) for v in rng.integers(0, 1 << 31, size=200)])
    edge = [2 ** k + e for k in range(1, 31) for e in (-1, 0, 1) if 2 <= 2 ** k + e < 2 ** 31]
    for d in edge + [int(v) for v in rng.integers(2, 1 << 31, size=500)]:
        assert ch.c16_div(d, 200, x) == -1, d


def test_cell_groups(ch):
    assert ch.c16_groups(1 << 20) == -1
