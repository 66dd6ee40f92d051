"""The whole-permutation passes (one kernel instead of a plan's passes):
emulated on the host against the oracle over random shapes of every form, and
on the GPU at the sizes where tiles, runs and regions end raggedly."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle import pyoracle as O

HERE = os.path.dirname(os.path.abspath(__file__))
SO = os.path.join(HERE, "_build", "libwhole_host.so")
CSRC = os.path.join(HERE, "..", "eithot_amd", "csrc")
ORBIT, RESIDENT = 1, 2


@pytest.fixture(scope="module")
def wh():
    src = os.path.join(HERE, "whole_harness.cpp")
    deps = [src] + [os.path.join(CSRC, f) for f in ("whole.hpp", "whole_plan.cpp", "maps.hpp")]
    if not os.path.exists(SO) or os.path.getmtime(SO) < max(map(os.path.getmtime, deps)):
        os.makedirs(os.path.dirname(SO), exist_ok=True)
        tmp = f"{SO}.{os.getpid()}.tmp"
        subprocess.check_call(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "-O1",
                               "-std=c++17", "-fPIC", "-shared", "-o", tmp, src])
        os.replace(tmp, SO)
    L = ctypes.CDLL(SO)
    i64p = ctypes.POINTER(ctypes.c_int64)
    L.wh_run.argtypes = [i64p, ctypes.POINTER(ctypes.c_int), ctypes.c_int, ctypes.c_int64,
                         ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, i64p, i64p]
    return L


def emulate(wh, dims, perm, elem, cus=256, passes=2, weak=0):
    vol = int(np.prod(dims))
    host = O.fill(vol, elem, 7, 1)
    buf = host.copy()
    tiles, lds = ctypes.c_int64(), ctypes.c_int64()
    mode = wh.wh_run((ctypes.c_int64 * len(dims))(*dims), (ctypes.c_int * len(dims))(*perm),
                     len(dims), elem, cus, passes, weak, buf.ctypes.data, tiles, lds)
    assert mode >= 0, (dims, perm, elem, "access out of bounds")
    if mode:
        want = O.permute(host, dims, [p - 1 for p in perm], elem)
        assert np.array_equal(buf, want), (dims, perm, elem, mode, tiles.value)
    return mode, tiles.value


def test_emulated_random_shapes(wh):
    # every order, element size and permutation; few CUs make large tiles and
    # regions that do not fit, many make small tiles
    rng = np.random.default_rng(5)
    seen = {0: 0, ORBIT: 0, RESIDENT: 0}
    for k in range(600):
        r = int(rng.integers(2, 8))
        vol = int(np.exp(rng.uniform(np.log(1 << 6), np.log(1 << 18))))
        w = rng.dirichlet(np.ones(r))
        dims = [max(1, int(round(vol ** x))) for x in w]
        if k % 3 == 0:  # lengths that recur, as the orbit form wants
            a = max(2, int(vol ** (1 / r)))
            dims = [a if rng.random() < 0.6 else max(2, a // 2 + 1) for _ in range(r)]
        if k % 6 == 0:  # squares, and palindromes reversed
            r = int(rng.integers(2, 5))
            a, b = int(rng.integers(33, 400)), int(rng.integers(2, 6))
            dims = {2: [a, a], 3: [a, b, a], 4: [a, b, b, a]}[r]
            perm = list(range(r, 0, -1))
        else:
            perm = [int(p) + 1 for p in rng.permutation(r)]
        elem = int(rng.choice([1, 2, 4, 8]))
        cus = int(rng.choice([4, 32, 256]))
        mode, _ = emulate(wh, dims, perm, elem, cus, passes=int(rng.integers(1, 4)),
                          weak=int(rng.integers(2)))
        seen[mode] += 1
    assert min(seen.values()) > 30, seen


EDGES = [
    # (dims, perm, elem, mode): square of whole tiles, one short of and one past them
    ([256, 256], [2, 1], 4, ORBIT),
    ([255, 255], [2, 1], 4, ORBIT),
    ([257, 257, 3], [2, 1, 3], 4, ORBIT),
    ([1021, 1021], [2, 1], 1, ORBIT),
    ([515, 515, 2], [2, 1, 3], 2, ORBIT),
    ([130, 130, 5], [2, 1, 3], 8, ORBIT),
    # four dims, runs of a whole dim each
    ([96, 5, 5, 96], [4, 3, 2, 1], 4, ORBIT),
    # pairs of elements kept together, odd lengths, the last region too
    ([2, 333, 501, 3], [1, 3, 2, 4], 4, RESIDENT),
    ([61, 7, 45], [3, 1, 2], 4, RESIDENT),
    ([129, 33, 65, 2], [4, 2, 3, 1], 8, RESIDENT),
    ([3, 641, 481, 5], [2, 3, 1, 4], 1, RESIDENT),
    ([128, 2049, 3], [2, 1, 3], 2, RESIDENT),
    ([3, 1000, 1001], [1, 3, 2], 1, RESIDENT),
    ([5, 77, 3, 19, 41], [4, 1, 5, 3, 2], 2, RESIDENT),
    # the most tiles a region may have of the smaller and the larger kind
    ([1999, 2003], [2, 1], 4, RESIDENT),
    ([2047, 2039], [2, 1], 4, RESIDENT),
]


@pytest.mark.parametrize("dims,perm,elem,mode", EDGES)
def test_emulated_edges(wh, dims, perm, elem, mode):
    got, tiles = emulate(wh, dims, perm, elem)
    assert got == mode and tiles > 1, (got, tiles)


@pytest.mark.gpu
@pytest.mark.parametrize("dims,perm,elem,mode", EDGES)
def test_gpu_edges(torch_cuda, dims, perm, elem, mode):
    # bit for bit against the oracle, at the tensor's own address and one
    # element past an allocation's start, and with the passes it replaces
    import eithot_amd as E
    from gpu_util import assert_bitexact
    torch = torch_cuda
    vol = int(np.prod(dims))
    host = O.fill(vol, elem, 11, 1)
    want = O.permute(host, dims, [p - 1 for p in perm], elem)
    for shift in (0, elem):
        buf = torch.zeros(vol * elem + 64, dtype=torch.uint8, device="cuda:0")
        buf[shift:shift + vol * elem] = torch.from_numpy(host.copy()).to("cuda:0").view(torch.uint8)
        for whole in (1, 0):
            print(f"whole case dims={dims} perm={perm} elem={elem} shift={shift} whole={whole}",
                  flush=True)
            buf[shift:shift + vol * elem] = torch.from_numpy(host.copy()).to("cuda:0").view(torch.uint8)
            old = E.set_tuning("whole", whole)
            try:
                E.transpose_ptr(buf.data_ptr() + shift, dims, perm, elem)
            finally:
                E.set_tuning("whole", old)
            got = buf[shift:shift + vol * elem].cpu().numpy().view(want.dtype)
            assert_bitexact(got, want, f"{dims} {perm} shift {shift} whole {whole}")
            # nothing around the tensor is written
            assert int(buf[:shift].count_nonzero()) == 0
            assert int(buf[shift + vol * elem:].count_nonzero()) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dims,perm,elem", [([1000, 999], [2, 1], 1),
                                            ([500, 500], [2, 1], 4),
                                            ([1001, 997], [2, 1], 2)])
def test_gpu_captured_after_a_plain_call(torch_cuda, dims, perm, elem):
    # a call made before can be captured (its passes with scratch and tables,
    # without, one whole pass), and every replay equals the eager call, with
    # eager calls in between
    import eithot_amd as E
    from gpu_util import assert_bitexact
    torch = torch_cuda
    vol = int(np.prod(dims))
    host = O.fill(vol, elem, 13, 1)
    want = O.permute(host, dims, [p - 1 for p in perm], elem)
    buf = torch.from_numpy(host.copy()).to("cuda:0")
    src = buf.clone()
    print(f"capture dims={dims} perm={perm}", flush=True)
    E.transpose_ptr(buf.data_ptr(), dims, perm, elem)
    assert_bitexact(buf.cpu().numpy(), want, "eager")
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        graph.capture_begin(capture_error_mode="thread_local")
        try:
            E.transpose_ptr(buf.data_ptr(), dims, perm, elem, stream=side.cuda_stream)
        finally:
            graph.capture_end()
    for k in range(3):
        buf.copy_(src)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert_bitexact(buf.cpu().numpy(), want, f"replay {k}")
        buf.copy_(src)
        E.transpose_ptr(buf.data_ptr(), dims, perm, elem, stream=torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert_bitexact(buf.cpu().numpy(), want, f"eager {k}")
