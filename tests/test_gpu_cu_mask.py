"""Streams that see part of the chip: a region's workgroups may not all fit
there, so calls on them run the plan's passes."""
import ctypes

import numpy as np
import pytest

import eithot_amd as E
from gpu_graph import VP, runtime
from gpu_util import assert_bitexact
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

# regions of 256 workgroups at two to a CU, and of a few
CASES = [([2, 4096, 1024, 2], [1, 3, 2, 4], 4), ([2047, 2039], [2, 1], 4), ([61, 7, 45], [3, 1, 2], 4)]


class MaskedStream:
    def __init__(self, torch, cus):
        self.hip, self.s = runtime(), VP()
        total = torch.cuda.get_device_properties(0).multi_processor_count
        n = (total + 31) // 32
        words = (ctypes.c_uint32 * n)(*[sum(1 << b for b in range(32) if 32 * k + b < cus)
                                        for k in range(n)])
        assert self.hip.hipExtStreamCreateWithCUMask(ctypes.byref(self.s), n, words) == 0

    def wait(self):
        assert self.hip.hipStreamSynchronize(self.s) == 0

    def close(self):
        assert self.hip.hipStreamDestroy(self.s) == 0


def transpose(dims, perm, elem, stream, buf):
    """The call's passes, by their times."""
    E.lib().eithot_set_pass_timing(1)
    try:
        E.transpose_ptr(buf.data_ptr(), dims, perm, elem, stream=stream)
    finally:
        E.lib().eithot_set_pass_timing(0)
    return E.lib().eithot_last_pass_times(None, 0)


@pytest.mark.parametrize("dims,perm,elem", CASES)
@pytest.mark.parametrize("cus", [32, 64, 255, 256])
def test_calls_on_part_of_the_chip(torch_cuda, dims, perm, elem, cus):
    torch = torch_cuda
    ops, _ = E.plan_describe(dims, perm, elem)
    host = O.fill(int(np.prod(dims)), elem, 5, 1)
    want = O.permute(host, dims, [p - 1 for p in perm], elem)
    st = MaskedStream(torch, cus)
    total = torch.cuda.get_device_properties(0).multi_processor_count
    print(f"{cus} of {total} CUs dims={dims}", flush=True)
    for _ in range(3):
        buf = torch.from_numpy(host.copy()).to("cuda:0")
        torch.cuda.synchronize()
        passes = transpose(dims, perm, elem, st.s.value, buf)
        st.wait()
        assert_bitexact(buf.cpu().numpy(), want, f"{dims} on {cus} CUs")
        if cus < total and len(ops) > 1:
            assert passes == len(ops)
        if cus >= total:
            assert passes == 1
    st.close()


def test_batch_on_part_of_the_chip(torch_cuda):
    # a batch keeps its launches: regions that find no room are called off
    torch = torch_cuda
    shapes = CASES[1:] + [([1021, 523, 2], [2, 1, 3], 4)] * 3
    old = E.set_tuning("whole_patience", 2000)
    try:
        hosts = [O.fill(int(np.prod(d)), e, 40 + k, 1) for k, (d, _, e) in enumerate(shapes)]
        bufs = [torch.from_numpy(h.copy()).to("cuda:0") for h in hosts]
        batch = E.Batch()
        for b, s in zip(bufs, shapes):
            batch.add(b.data_ptr(), *s)
        batch.build()
        st = MaskedStream(torch, 32)
        print("batch on 32 CUs", flush=True)
        for _ in range(3):
            for b, h in zip(bufs, hosts):
                b.copy_(torch.from_numpy(h.copy()))
            torch.cuda.synchronize()
            batch.run(stream=st.s.value, sync=False)
            st.wait()
            for b, h, (d, p, e) in zip(bufs, hosts, shapes):
                assert_bitexact(b.cpu().numpy(), O.permute(h, d, [q - 1 for q in p], e), f"{d}")
        st.close()
    finally:
        E.set_tuning("whole_patience", old)
