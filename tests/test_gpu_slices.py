"""Staged row passes of unit slices of 16 bytes and more: slices of one whole
piece, a piece and a byte, two pieces that overlap, both row maps, at the
tensor's address and past it."""
import numpy as np
import pytest

import eithot_amd as E
from oracle import pyoracle as O

CASES = [([32, 170003, 3], [1, 3, 2], 1, 0.2), ([34, 170003, 3], [1, 3, 2], 1, 0.2),
         ([50, 3, 170003], [1, 3, 2], 1, 0.2), ([30, 170003, 3], [1, 3, 2], 4, 0.1),
         ([80, 170003, 3], [1, 3, 2], 1, 0.2)]


@pytest.mark.gpu
@pytest.mark.parametrize("dims,perm,elem,alpha", CASES)
def test_staged_slices(torch_cuda, dims, perm, elem, alpha):
    torch = torch_cuda
    rng = np.random.default_rng(6)
    n = int(np.prod(dims)) * elem
    a = rng.integers(0, 256, n, dtype=np.uint8)
    want = O.permute(a, dims, [p - 1 for p in perm], elem=elem).view(np.uint8).reshape(-1)
    old = {k: E.set_tuning(k, 0) for k in ("whole", "cycle_min_cell", "regroup")}
    try:
        ops, _ = E.plan_describe(dims, perm, elem, alpha=alpha)
        assert any(o["kind"] == 3 and o["staged"] and 16 <= o["us"] < o["U"] for o in ops)
        for lead in (0, elem):
            buf = torch.zeros(n + 64, dtype=torch.uint8, device="cuda")
            buf[lead:lead + n] = torch.from_numpy(a).cuda()
            torch.cuda.synchronize()
            print(f"staged slices dims={dims} perm={perm} lead={lead}", flush=True)
            E.transpose_ptr(buf.data_ptr() + lead, dims, perm, elem, 1, alpha)
            torch.cuda.synchronize()
            out = buf.cpu().numpy()
            assert np.array_equal(out[lead:lead + n], want), (dims, lead)
            assert not out[:lead].any() and not out[lead + n:].any()
    finally:
        for k, v in old.items():
            E.set_tuning(k, v)
