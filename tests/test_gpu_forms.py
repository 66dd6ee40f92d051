"""Which form a call ran in: the plan's passes or one whole pass."""
import numpy as np
import pytest

import eithot_amd as E
from gpu_util import run_case

pytestmark = pytest.mark.gpu

# (dims, perm, elem, form): a square, regions of a plan with two passes, a
# region in place of a plan's only pass, a tensor that no whole pass takes
CASES = [([500, 500], [2, 1], 4, 1), ([129, 33, 65, 2], [4, 2, 3, 1], 8, 2),
         ([61, 7, 45], [3, 1, 2], 4, 2), ([64, 64, 64], [1, 3, 2], 4, 0)]


@pytest.mark.parametrize("dims,perm,elem,form", CASES)
def test_form_is_told(torch_cuda, dims, perm, elem, form):
    # (one pass either way in the third: the number of pass times cannot tell)
    for whole in (1, 0):
        old = E.set_tuning("whole", whole)
        try:
            got, want, _ = run_case(torch_cuda, dims, perm, elem)
        finally:
            E.set_tuning("whole", old)
        assert np.array_equal(got, want)
        assert E.last_whole_pass() == (form if whole else 0)


def test_knob_without_effect_leaves_the_form(torch_cuda):
    for value in (6, 8):
        old = E.set_tuning("cycle_u_depth", value)
        try:
            run_case(torch_cuda, [500, 500], [2, 1], 4)
        finally:
            E.set_tuning("cycle_u_depth", old)
        assert E.last_whole_pass() == 1
