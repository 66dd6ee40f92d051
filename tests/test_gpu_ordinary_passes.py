"""The parity tests whose shapes a whole pass takes by default, with the
plans' own passes: whole passes are off here, in plain calls and in batches."""
import pytest

import eithot_amd as E
from test_gpu_batch_serve import test_batch_matches_oracle, test_server_alone_and_in_the_mix  # noqa: F401
from test_gpu_configs import test_decomposer_orders, test_partitioned_transposes  # noqa: F401
from test_gpu_parity import (test_all_perms_rank4_small, test_composite_cycle_passes,  # noqa: F401
                             test_cycle_following_passes, test_dense_block_passes,
                             test_fused_block_passes, test_known_answer_2x4096x1024x2,
                             test_narrow_slice_row_passes, test_narrow_unit_catanzaro_passes,
                             test_narrow_word_tiles, test_random_high_order, test_regroup_plans,
                             test_segtile_plans, test_shifted_cycle_passes, test_staged_passes,
                             test_staged_row_tiles)

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def ordinary_passes():
    old = E.set_tuning("whole", 0)
    yield
    assert E.set_tuning("whole", old) == 0
