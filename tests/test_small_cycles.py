"""Cycle passes over cells of 16 bytes to a line: the planner's rule against
the plans without it, and on the device from unaligned tensors."""
import numpy as np
import pytest

import eithot_amd as E
from oracle import pyoracle as O
from plan_sim import simulate

# cells of 16, 20, 33, 50, 64, 76, 100 and 124 bytes: replacing column and row
# passes in LDS, staged and in narrow slices, tiles, and two passes by one
CASES = [([4, 500, 1213], [1, 3, 2], 4), ([20, 30259, 2], [3, 1, 2], 4),
         ([33, 1427, 24], [1, 3, 2], 1), ([25, 1193, 43], [1, 3, 2], 2),
         ([16, 541, 113], [1, 3, 2], 4), ([50, 2593, 14], [1, 3, 2], 2),
         ([31, 279, 61], [1, 3, 2], 4), ([9110, 78], [2, 1], 4),
         ([14, 7, 1138], [2, 3, 1], 8), ([719, 7, 1724], [3, 2, 1], 1)]
# these take the rule (16 bytes in LDS, and the last two, keep their passes)
SMALL = CASES[1:8]


def small_cells(ops):
    return [o["U"] for o in ops if o["kind"] == 4 and o["U"] < 128]


@pytest.mark.parametrize("dims,perm,elem", CASES)
def test_plan(dims, perm, elem):
    rng = np.random.default_rng(3)
    a = rng.integers(0, 256, int(np.prod(dims)) * elem, dtype=np.uint8)
    want = O.permute(a, dims, [p - 1 for p in perm], elem=elem)
    ops, scratch = E.plan_describe(dims, perm, elem)
    got = a.copy()
    simulate(got, ops)
    assert np.array_equal(got, want.view(np.uint8).reshape(-1))
    if (dims, perm, elem) in SMALL:
        assert small_cells(ops)
    # less extra memory than its tables need: the plan without small cells
    alpha = 1e-3
    try:
        tight, _ = E.plan_describe(dims, perm, elem, alpha=alpha)
    except E.EithotError:
        tight = []
    old = E.set_tuning("lower_mask", 15)
    try:
        assert not small_cells(E.plan_describe(dims, perm, elem)[0])
        if not tight:
            with pytest.raises(E.EithotError):
                E.plan_describe(dims, perm, elem, alpha=alpha)
    finally:
        E.set_tuning("lower_mask", old)
    got = a.copy()
    if tight:
        simulate(got, tight)
        assert np.array_equal(got, want.view(np.uint8).reshape(-1))


@pytest.mark.gpu
@pytest.mark.parametrize("dims,perm,elem", CASES)
def test_device(torch_cuda, dims, perm, elem):
    torch = torch_cuda
    rng = np.random.default_rng(4)
    n = int(np.prod(dims)) * elem
    a = rng.integers(0, 256, n, dtype=np.uint8)
    want = O.permute(a, dims, [p - 1 for p in perm], elem=elem).view(np.uint8).reshape(-1)
    whole = E.set_tuning("whole", 0)
    try:
        for lead in (0, elem):
            buf = torch.zeros(n + 64, dtype=torch.uint8, device="cuda")
            buf[lead:lead + n] = torch.from_numpy(a).cuda()
            torch.cuda.synchronize()
            print(f"small cycles dims={dims} perm={perm} lead={lead}", flush=True)
            E.transpose_ptr(buf.data_ptr() + lead, dims, perm, elem)
            torch.cuda.synchronize()
            out = buf.cpu().numpy()
            assert np.array_equal(out[lead:lead + n], want), (dims, lead)
            assert not out[:lead].any() and not out[lead + n:].any()
    finally:
        E.set_tuning("whole", whole)
