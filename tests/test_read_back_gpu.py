"""GPU tests of the decode kernel where its merge reads the splits' rows at constant distances (split counts that are a multiple of
16 and fill a batch) and on both sides of that rule, and where a tile is a wavefront's first, ragged or the query group padded."""
import numpy as np
import pytest

from llminfer_amd import _binding as B
from llminfer_amd import synth

from helpers import assert_parity, assert_tap_parity, run_hip, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side", [0, "measure"])
@pytest.mark.parametrize("n_q,n_kv", [(32, 8), (16, 8), (24, 8), (64, 8), (40, 8)])  # (groups of 3 and 5: padded to 4 and 8)
@pytest.mark.parametrize("num_splits", [8, 15, 16, 17, 24, 31, 32, 33, 48, 63, 64])
def test_split_counts_either_side_of_the_rule(oracle, dev, n_q, n_kv, num_splits, side):
    ctx = 64 * 16 + 5 + num_splits  # a tile for every split, the last one ragged
    case = synth.make_case(100 + num_splits, n_q=n_q, n_kv=n_kv, ctx=ctx)
    kw = dict(workspace_side=side) if side else {}
    got16, got32, plan = run_hip(case, dev, kv_layout=B.KV_LAYOUT_HEAD_MAJOR, want_plan=True, workspace_bytes=64 << 20,
                                 force_path=B.PATH_SPLIT_FUSED, num_splits=num_splits, **kw)
    assert plan.num_splits == num_splits and plan.workspace_side == (1 if side else 0)
    ref = run_oracle(oracle, case)
    assert_parity(got16, ref, "splits %d" % num_splits)
    assert_tap_parity(got32, ref, "splits %d" % num_splits)


@pytest.mark.parametrize("n_q,n_kv", [(2, 2), (6, 2), (10, 2), (16, 2), (26, 2)])
@pytest.mark.parametrize("ctx", [1, 15, 16, 17, 63, 64, 65, 127, 129])
def test_first_and_ragged_tiles_of_a_single_pass(oracle, dev, n_q, n_kv, ctx):
    case = synth.make_case(200 + ctx, n_q=n_q, n_kv=n_kv, ctx=ctx)
    got16, got32 = run_hip(case, dev, kv_layout=B.KV_LAYOUT_POS_MAJOR, force_path=B.PATH_SINGLE_PASS)[:2]
    ref = run_oracle(oracle, case)
    assert_parity(got16, ref, "ctx %d" % ctx)
    # (a probability enters as a sum of two bf16 numbers, 2^-17 of it off at most, so an output is off by 2^-17 of the largest |V|, 4 here: 3e-5,
    # however near to zero the output itself is: no bound relative to it alone)
    assert np.all(np.abs(got32 - ref) <= 3e-5 + 2e-4 * np.abs(ref)), "ctx %d" % ctx
