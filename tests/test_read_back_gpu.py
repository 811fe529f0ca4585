"""GPU tests of the decode kernel where its merge reads the splits' rows at constant distances (split counts that are a multiple of
16 and fill a batch) and on both sides of that rule, and where a tile is a wavefront's first, ragged or the query group padded."""
import numpy as np
import pytest

from llminfer_amd import _binding as B
from llminfer_amd import synth

from helpers import assert_parity, assert_round_off, assert_tap_parity, run_hip, run_oracle

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


def _in_64_bits(case):
    """The case's output in 64 bits and how far off an fp32 evaluation of it with probabilities as sums of two bf16 numbers may be, u = 2^-24: a
    score is 128 exact products added in fp32 (128 u of the sum of their magnitudes) times a rounded factor and less a maximum; exp2 is good to
    2^-22, of a probability and of each tile's and wavefront's rescale; the sums over the positions lose 2 u a position (the matrix cores need not
    round to nearest), above and below the fraction bar; a probability is cut at 2^-17."""
    n_q, n_kv, ctx, u = case["head_num"], case["kv_dim"] // 128, case["pos"] + 1, 2.0 ** -24
    k, v = (synth.bf16_bits_to_f32(case[c][0, :ctx]).astype(np.float64).reshape(ctx, n_kv, 128).repeat(n_q // n_kv, axis=1) for c in "kv")
    q = synth.bf16_bits_to_f32(case["q"]).astype(np.float64).reshape(n_q, 128)
    factor = np.log2(np.e) / np.sqrt(128.0)
    s = np.einsum("hd,thd->th", q, k) * factor
    below = s.max(axis=0) - s
    p = np.exp2(-below)
    p /= p.sum(axis=0)
    off = np.log(2) * (128 * u * factor * np.einsum("hd,thd->th", abs(q), abs(k)) + 3 * u * abs(s) + u * below) + 2.0 ** -22
    out, mean_abs = np.einsum("th,thd->hd", p, v), np.einsum("th,thd->hd", p, abs(v))
    bound = np.einsum("th,thd->hd", p * off, abs(v)) + abs(out) * (p * off).sum(axis=0)[:, None]
    bound += mean_abs * (2.0 ** -17 + 4 * ctx * u + 2 * (-(-ctx // 16) + 8) * 2.0 ** -22)
    return out.reshape(-1), bound.reshape(-1)


@pytest.mark.parametrize("layout", [B.KV_LAYOUT_POS_MAJOR, B.KV_LAYOUT_HEAD_MAJOR])
@pytest.mark.parametrize("n_q,n_kv", [(2, 2), (6, 2), (10, 2), (16, 2), (26, 2)])
@pytest.mark.parametrize("ctx", [1, 15, 16, 17, 63, 64, 65, 127, 129])
def test_first_and_ragged_tiles_of_a_single_pass(oracle, dev, n_q, n_kv, ctx, layout):
    case = synth.make_case(200 + ctx, n_q=n_q, n_kv=n_kv, ctx=ctx)
    ref, (exact, bound) = run_oracle(oracle, case), _in_64_bits(case)
    for waves in (0, 1, 2, 4, 8):  # (which wavefront has the ragged tile, and whether it is its first)
        if waves * (1 << (n_q // n_kv - 1).bit_length()) > 64:
            continue
        got16, got32 = run_hip(case, dev, kv_layout=layout, force_path=B.PATH_SINGLE_PASS, waves_per_group=waves)[:2]
        what = "ctx %d, %d wavefronts" % (ctx, waves)
        assert_parity(got16, ref, what)
        assert_round_off(got32, exact, what)
        over = abs(got32 - exact) / bound
        assert over.max() <= 1.0, "%s: %.2f of the bound" % (what, over.max())
