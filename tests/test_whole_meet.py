"""Resident passes where a region's workgroups are kept from meeting: threads
on the host share too little room, workgroups on the GPU have no patience.
Also the passes of batches and the pairs of tiles, emulated."""
import ctypes
import os
import subprocess
import threading

import numpy as np
import pytest

from oracle import pyoracle as O
from test_whole import CSRC, EDGES, HERE, RESIDENT

SO = os.path.join(HERE, "_build", "libwhole_meet_host.so")


@pytest.fixture(scope="module")
def wm():
    src = os.path.join(HERE, "whole_meet_harness.cpp")
    deps = [src, os.path.join(HERE, "whole_harness.cpp")] + [
        os.path.join(CSRC, f) for f in ("whole.hpp", "whole_plan.cpp", "maps.hpp")]
    if not os.path.exists(SO) or os.path.getmtime(SO) < max(map(os.path.getmtime, deps)):
        os.makedirs(os.path.dirname(SO), exist_ok=True)
        tmp = f"{SO}.{os.getpid()}.tmp"
        subprocess.check_call(["/opt/rocm/bin/hipcc", "-x", "hip", "--offload-arch=gfx950", "-O1",
                               "-std=c++17", "-fPIC", "-shared", "-pthread", "-o", tmp, src])
        os.replace(tmp, SO)
    L = ctypes.CDLL(SO)
    i64p = ctypes.POINTER(ctypes.c_int64)
    shape = [i64p, ctypes.POINTER(ctypes.c_int), ctypes.c_int, ctypes.c_int64, ctypes.c_int,
             ctypes.c_int]
    L.wm_run.argtypes = shape + [ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_void_p,
                                 ctypes.c_void_p, i64p]
    L.wm_once.argtypes = shape + [ctypes.c_int64, ctypes.c_void_p, i64p]
    return L


def args(dims, perm, elem, cus, batched):
    return ((ctypes.c_int64 * len(dims))(*dims), (ctypes.c_int * len(perm))(*perm), len(dims), elem,
            cus, batched)


# room for one launch's region, for both, for one workgroup less than one
# region, and for half of one: the last two never meet, and the first may not
@pytest.mark.parametrize("room,always", [(1.0, False), (2.0, False), (-1, True), (0.5, True)])
@pytest.mark.parametrize("dims,perm,elem,batched", [([61, 7, 45], [3, 1, 2], 4, 0),
                                                    ([40, 37, 41, 5], [3, 2, 1, 4], 2, 0),
                                                    ([333, 121, 3], [2, 1, 3], 8, 1)])
def test_regions_that_cannot_meet(wm, dims, perm, elem, batched, room, always):
    vol, rounds = int(np.prod(dims)), 5
    want, bufs = [], []
    for seed in (1, 2):
        x = O.fill(vol, elem, seed, 1)
        bufs.append(x.copy())
        for _ in range(rounds):
            x = O.permute(x, dims, [p - 1 for p in perm], elem)
        want.append(x)
    wgs, probe = ctypes.c_int64(), bufs[0].copy()
    a = args(dims, perm, elem, 256, batched)
    per = ctypes.c_int64()
    n = wm.wm_once(*a, 160 * 1024, probe.ctypes.data, per)
    assert n > 2
    slots = n - 1 if room < 0 else max(1, int(n * room))
    # 1 ms of patience; 20 ms where it may do
    alone = wm.wm_run(*a, slots, 100000 if always else 2000000, rounds, bufs[0].ctypes.data,
                      bufs[1].ctypes.data, wgs)
    assert alone >= 0, alone
    regions = dims[-1] if perm[-1] == len(dims) else 1
    if always:
        assert alone == 2 * rounds * regions
    for got, w in zip(bufs, want):
        assert np.array_equal(got, w.view(got.dtype))


@pytest.mark.parametrize("batched", [0, 1])
def test_emulated_workgroups(wm, batched):
    # every order, element size and permutation; few CUs, or little LDS, make
    # large tiles and regions that do not fit, many make small tiles
    rng = np.random.default_rng(17 + batched)
    seen = {0: 0, 1: 0, 2: 0}
    for k in range(1000):
        r = int(rng.integers(2, 7))
        vol = int(np.exp(rng.uniform(np.log(1 << 9), np.log(1 << 20))))
        dims = [max(1, int(round(vol ** x))) for x in rng.dirichlet(np.ones(r))]
        if k % 5 == 0:
            dims = [int(rng.integers(300, 1100)), int(rng.integers(300, 1100))]
            r = 2
        perm = [int(p) + 1 for p in rng.permutation(r)]
        elem, cus = int(rng.choice([1, 2, 4, 8])), int(rng.choice([8, 32, 256]))
        lds = int(rng.choice([64, 160])) * 1024
        host = O.fill(int(np.prod(dims)), elem, 7, 1)
        buf, per = host.copy(), ctypes.c_int64()
        n = wm.wm_once(*args(dims, perm, elem, cus, batched), lds, buf.ctypes.data, per)
        assert n >= 0, (dims, perm, elem, cus, lds)
        seen[per.value if n else 0] += 1
        if n:
            want = O.permute(host, dims, [p - 1 for p in perm], elem)
            assert np.array_equal(buf, want), (dims, perm, elem, cus, lds)
    assert min(seen.values()) > 20, seen


@pytest.fixture
def impatient():
    import eithot_amd as E
    old = E.set_tuning("whole_patience", 0)
    yield E
    E.set_tuning("whole_patience", old)


@pytest.mark.gpu
@pytest.mark.parametrize("dims,perm,elem", [e[:3] for e in EDGES if e[3] == RESIDENT])
def test_gpu_without_patience(torch_cuda, impatient, dims, perm, elem):
    # most regions are called off and moved by one workgroup, others meet:
    # either way the whole tensor is, and nothing around it
    E = impatient
    from gpu_util import assert_bitexact
    torch = torch_cuda
    vol = int(np.prod(dims))
    host = O.fill(vol, elem, 21, 1)
    want = O.permute(host, dims, [p - 1 for p in perm], elem)
    back = np.argsort([p - 1 for p in perm])
    dims_t = [dims[p - 1] for p in perm]
    for shift in (0, elem):
        print(f"no patience dims={dims} perm={perm} elem={elem} shift={shift}", flush=True)
        buf = torch.zeros(vol * elem + 64, dtype=torch.uint8, device="cuda:0")
        view = buf[shift:shift + vol * elem]
        view.copy_(torch.from_numpy(host.copy()).to("cuda:0").view(torch.uint8))
        for k in range(4):
            E.transpose_ptr(view.data_ptr(), dims, perm, elem)
            assert_bitexact(view.cpu().numpy().view(want.dtype), want, f"{dims} shift {shift} there {k}")
            E.transpose_ptr(view.data_ptr(), dims_t, [int(p) + 1 for p in back], elem)
            assert_bitexact(view.cpu().numpy().view(host.dtype), host, f"{dims} shift {shift} back {k}")
        assert int(buf[:shift].count_nonzero()) == 0
        assert int(buf[shift + vol * elem:].count_nonzero()) == 0


def batch_shapes():
    rng = np.random.default_rng(8)
    out = [([333, 121, 3], [2, 1, 3], 8), ([40, 37, 41, 5], [3, 2, 1, 4], 2), ([1999, 501], [2, 1], 1)]
    for _ in range(20):
        dims = [int(x) for x in rng.integers(20, 90, 3)]
        out.append((dims, [3, 1, 2], int(rng.choice([1, 2, 4, 8]))))
    return out


class Tensors:
    def __init__(self, torch, shapes, seed):
        self.shapes, self.src, self.want, self.buf = shapes, [], [], []
        for k, (dims, perm, elem) in enumerate(shapes):
            host = O.fill(int(np.prod(dims)), elem, seed + k, 1)
            self.want.append(O.permute(host, dims, [p - 1 for p in perm], elem))
            self.src.append(torch.from_numpy(host.copy()).to("cuda:0"))
            self.buf.append(self.src[-1].clone())

    def reset(self):
        for b, s in zip(self.buf, self.src):
            b.copy_(s)

    def check(self, what):
        from gpu_util import assert_bitexact
        for b, w, s in zip(self.buf, self.want, self.shapes):
            assert_bitexact(b.cpu().numpy(), w, f"{s} {what}")


@pytest.mark.gpu
def test_gpu_batch_and_server_without_patience(torch_cuda, impatient):
    E, torch = impatient, torch_cuda
    t = Tensors(torch, batch_shapes(), 30)
    batch = E.Batch()
    for b, (dims, perm, elem) in zip(t.buf, t.shapes):
        batch.add(b.data_ptr(), dims, perm, elem)
    print("batch without patience", flush=True)
    batch.build()
    for k in range(4):
        t.reset()
        torch.cuda.synchronize()
        batch.run()
        t.check(f"batch {k}")
    print("server without patience", flush=True)
    server = E.Server(1 << 20, max_inflight=16, nstreams=4)
    for k in range(3):
        t.reset()
        torch.cuda.synchronize()
        ids = [server.submit(b.data_ptr(), *s) for b, s in zip(t.buf, t.shapes)]
        server.drain()
        assert all(server.status(i)[0] == 2 for i in ids)
        t.check(f"server {k}")


@pytest.mark.gpu
@pytest.mark.parametrize("patience", [100000, 0])
def test_gpu_streams_threads_and_a_batch(torch_cuda, patience):
    # resident passes of the null stream, two side streams, a batch and three
    # threads follow each other in every order
    import eithot_amd as E
    torch = torch_cuda
    old = E.set_tuning("whole_patience", patience)
    try:
        shapes = batch_shapes()[:8]
        single, batched = Tensors(torch, shapes, 60), Tensors(torch, shapes, 80)
        batch = E.Batch()
        for b, s in zip(batched.buf, batched.shapes):
            batch.add(b.data_ptr(), *s)
        batch.build()
        streams = [None, torch.cuda.Stream(), torch.cuda.Stream()]
        rng = np.random.default_rng(3)
        print(f"streams and a batch, patience {patience}", flush=True)
        for k in range(6):
            single.reset()
            batched.reset()
            torch.cuda.synchronize()
            when = int(rng.integers(8))
            for i, (b, s) in enumerate(zip(single.buf, single.shapes)):
                if i == when:
                    batch.run(stream=streams[1].cuda_stream if k % 2 else None, sync=False)
                st = streams[int(rng.integers(3))]
                E.transpose_ptr(b.data_ptr(), *s, stream=st.cuda_stream if st else None)
            torch.cuda.synchronize()
            single.check(f"streams {k}")
            batched.check(f"batch {k}")
        print(f"threads, patience {patience}", flush=True)
        single.reset()
        torch.cuda.synchronize()
        errors = []

        def work(j):
            try:
                st = streams[j]
                for b, s in list(zip(single.buf, single.shapes))[j::3]:
                    E.transpose_ptr(b.data_ptr(), *s, stream=st.cuda_stream if st else None)
                if st:
                    st.synchronize()
            except Exception as e:  # reported by the test's own thread
                errors.append(e)

        threads = [threading.Thread(target=work, args=(j,)) for j in range(3)]
        for th in threads:
            th.start()
        for th in threads:
            th.join()
        assert not errors, errors
        torch.cuda.synchronize()
        single.check("threads")
    finally:
        E.set_tuning("whole_patience", old)
