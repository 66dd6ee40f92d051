"""Fused block passes whose fastest output digits are shorter than a 16-byte
chunk: aligned and dense runs, short and long first digits."""
import numpy as np
import pytest

import eithot_amd as E
from oracle import pyoracle as O

# the first output digits: 2 x 3 x 57, 3 x 7, 2 x 2 x 2 x 17, 15 x 16, 3 x 5
CASES = [([3, 2, 181, 57, 37], [2, 1, 4, 3, 5], 1), ([601, 7, 3, 40], [3, 2, 1, 4], 1),
         ([17, 301, 2, 2, 2, 50], [3, 4, 5, 1, 2, 6], 1), ([16, 163, 15, 9], [3, 1, 2, 4], 1),
         ([1011, 5, 3, 31], [3, 2, 1, 4], 2), ([2048, 2, 2, 3, 20], [3, 2, 4, 1, 5], 2),
         ([1007, 3, 5, 20], [2, 3, 1, 4], 4), ([1024, 3, 5, 20], [3, 2, 1, 4], 4)]


@pytest.mark.gpu
@pytest.mark.parametrize("dims,perm,elem", CASES)
def test_short_digits(torch_cuda, dims, perm, elem):
    torch = torch_cuda
    rng = np.random.default_rng(8)
    n = int(np.prod(dims)) * elem
    a = rng.integers(0, 256, n, dtype=np.uint8)
    want = O.permute(a, dims, [p - 1 for p in perm], elem=elem).view(np.uint8).reshape(-1)
    whole = E.set_tuning("whole", 0)
    try:
        assert [o["kind"] for o in E.plan_describe(dims, perm, elem)[0]] == [5]
        for lead in (0, elem, 16 - elem):
            buf = torch.zeros(n + 64, dtype=torch.uint8, device="cuda")
            buf[lead:lead + n] = torch.from_numpy(a).cuda()
            torch.cuda.synchronize()
            print(f"block runs dims={dims} perm={perm} lead={lead}", flush=True)
            E.transpose_ptr(buf.data_ptr() + lead, dims, perm, elem)
            torch.cuda.synchronize()
            out = buf.cpu().numpy()
            assert np.array_equal(out[lead:lead + n], want), (dims, lead)
            assert not out[:lead].any() and not out[lead + n:].any()
    finally:
        E.set_tuning("whole", whole)
