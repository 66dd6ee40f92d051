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


# a plan without tables or scratch before; with small cells it has both
LIMITED = ([31, 279, 1213], [1, 3, 2], 4)


@pytest.mark.gpu
def test_captured_first_and_pool_too_small(torch_cuda):
    # what needed neither a table nor scratch before still runs where neither
    # has a place: captured on its first call, and served without a pool
    torch = torch_cuda
    dims, perm, elem = LIMITED
    rng = np.random.default_rng(5)
    n = int(np.prod(dims)) * elem
    a = rng.integers(0, 256, n, dtype=np.uint8)
    want = O.permute(a, dims, [p - 1 for p in perm], elem=elem).view(np.uint8).reshape(-1)
    src = torch.from_numpy(a).cuda()
    buf = src.clone()
    ops, scratch = E.plan_describe(dims, perm, elem)
    assert small_cells(ops) and scratch > 256
    old = E.set_tuning("whole", 0)
    try:
        E.transpose_ptr(src.clone().data_ptr(), [64, 64], [2, 1], 4)  # the library is set up
        side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        print("small cells: first call captured", flush=True)
        with torch.cuda.stream(side):
            graph.capture_begin(capture_error_mode="thread_local")
            try:
                E.transpose_ptr(buf.data_ptr(), dims, perm, elem, stream=side.cuda_stream)
            finally:
                graph.capture_end()
        for _ in range(3):
            buf.copy_(src)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(buf.cpu().numpy(), want)
        buf.copy_(src)
        torch.cuda.synchronize()
        print("small cells: served without a pool", flush=True)
        server = E.Server(0)
        server.submit(buf.data_ptr(), dims, perm, elem)
        server.drain()
        torch.cuda.synchronize()
        assert np.array_equal(buf.cpu().numpy(), want)
        # and with a call before, captured on the passes of that call
        E.transpose_ptr(src.clone().data_ptr(), dims, perm, elem)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(side):
            graph.capture_begin(capture_error_mode="thread_local")
            try:
                E.transpose_ptr(buf.data_ptr(), dims, perm, elem, stream=side.cuda_stream)
            finally:
                graph.capture_end()
        for _ in range(3):
            buf.copy_(src)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(buf.cpu().numpy(), want)
    finally:
        E.set_tuning("whole", old)
