"""GPU tests of how a query head's splits are merged at the edges of the rules that choose: more splits than one wavefront
merges, a head of a large group per workgroup, and the split counts a position read on the device asks for."""
import numpy as np
import pytest
import torch

from llminfer_amd import _binding as B
from llminfer_amd import ops, synth

from helpers import assert_parity, assert_tap_parity, from_dev_bf16, run_hip, run_oracle, to_dev
from test_resident_stack_gpu import timeouts

pytestmark = pytest.mark.gpu

HEAD, POS = B.KV_LAYOUT_HEAD_MAJOR, B.KV_LAYOUT_POS_MAJOR


@pytest.mark.parametrize("n_q,n_kv,ctx,layout,kw", [
    (8, 1, 4500, HEAD, {}),                                                # 256 splits, four wavefronts for a group of 8
    (8, 1, 4500, HEAD, dict(num_splits=256)),                              # ... eight
    (14, 2, 517, POS, {}),                                                 # four wavefronts, 7 heads in a group
    (8, 2, 2100, POS, {}),                                                 # 128 splits, four wavefronts
    (16, 2, 1040, HEAD, dict(num_splits=65)),                              # the last wavefronts' shares are short or empty
    (4, 1, 4200, HEAD, dict(num_splits=250, waves_per_group=4)),           # 63 splits for each wavefront
    (4, 1, 4200, HEAD, dict(num_splits=256, waves_per_group=2)),           # two wavefronts: one merges them all
    (2, 2, 1700, HEAD, dict(num_splits=100)),                              # one head per KV head
    (32, 8, 1700, HEAD, dict(num_splits=100, workspace_side="measure")),   # two homes per row
    (64, 8, 1700, HEAD, dict(num_splits=70, workspace_side=0x66666666)),
    (32, 2, 256, HEAD, {}),                                                # 16 splits for 16 heads: a head each
    (32, 2, 240, HEAD, dict(num_splits=15)),                               # one split too few: the last workgroup merges
    (26, 2, 209, POS, {}),                                                 # 13 heads in a group
    (9, 1, 3000, HEAD, dict(num_splits=9)),
    (16, 1, 20000, HEAD, {}),                                              # 256 splits, 16 heads, two columns a thread
    (8, 1, 200, HEAD, dict(num_splits=12, waves_per_group=4)),             # 8 heads, four wavefronts: a head each
    (16, 2, 250, POS, dict(num_splits=15, waves_per_group=4)),
    (14, 2, 130, HEAD, dict(num_splits=7, waves_per_group=4)),             # ... as many splits as heads
    (8, 1, 120, POS, dict(num_splits=7, waves_per_group=4)),               # ... one split too few
])
def test_merges_of_many_splits_and_large_groups(oracle, dev, n_q, n_kv, ctx, layout, kw):
    case = synth.make_case(7 + ctx, n_q=n_q, n_kv=n_kv, ctx=ctx)
    force = dict(force_path=B.PATH_SPLIT_FUSED) if "num_splits" in kw else {}
    got16, got32, plan = run_hip(case, dev, kv_layout=layout, want_plan=True, workspace_bytes=64 << 20, **force, **kw)
    ref = run_oracle(oracle, case)
    what = "splits %d waves %d side %d" % (plan.num_splits, plan.waves_per_group, plan.workspace_side)
    assert plan.num_splits == kw.get("num_splits", plan.num_splits) and plan.num_splits > 1, what
    assert plan.workspace_side == (1 if kw.get("workspace_side") else 0), what
    assert_parity(got16, ref, what)
    assert_tap_parity(got32, ref, what)


@pytest.mark.parametrize("n_q,n_kv,ctx,kw", [
    (512, 32, 3000, {}), (320, 20, 1000, {}), (288, 32, 700, {}), (144, 9, 250, {}),
    (288, 32, 700, dict(num_splits=16)),    # more splits than heads in the group
    (256, 32, 2100, dict(num_splits=32)),   # groups of 8
    (128, 8, 700, {}), (126, 9, 900, {}),   # the most heads that are merged a workgroup each
])
def test_many_heads_do_not_wait_for_each_other(oracle, dev, n_q, n_kv, ctx, kw):
    """More query heads than half the compute units: no workgroup per head waits (the launch would not fit the chip)."""
    case = synth.make_case(3 + n_q, n_q=n_q, n_kv=n_kv, ctx=ctx)
    force = dict(force_path=B.PATH_SPLIT_FUSED) if kw else {}
    before = timeouts()
    got16, got32, plan = run_hip(case, dev, kv_layout=HEAD, want_plan=True, workspace_bytes=64 << 20, **force, **kw)
    ref = run_oracle(oracle, case)
    assert plan.num_splits > 1 and timeouts() == before
    assert_parity(got16, ref, "splits %d" % plan.num_splits)
    assert_tap_parity(got32, ref, "splits %d" % plan.num_splits)


@pytest.mark.parametrize("n_q,n_kv,msl,layout,short_workspace", [
    (288, 18, 1024, HEAD, False),   # more heads than may wait for each other: the counts of the smaller groups
    (32, 8, 4096, HEAD, False), (64, 8, 4096, POS, False), (32, 2, 4096, HEAD, False),
    (8, 1, 4096, HEAD, False),      # 256 splits and a reciprocal for each count
    (16, 8, 4096, HEAD, True),      # a workspace for 11 splits: every count is capped by it
])
def test_device_position_takes_the_planned_split_counts(oracle, dev, n_q, n_kv, msl, layout, short_workspace):
    """One captured launch sized for the whole window; the position walks over the lengths at which the rule changes from a
    single pass to a quarter of the splits, half of them and all of them, and over odd ones between."""
    case = synth.make_case(60 + n_q + n_kv, n_q=n_q, n_kv=n_kv, ctx=msl)
    hm = layout == HEAD
    q = to_dev(case["q"], dev)
    k, v = (to_dev(synth.to_head_major(c, n_kv) if hm else c, dev) for c in (case["k"], case["v"]))
    out = torch.zeros(n_q * 128, dtype=torch.int16, device=dev)
    out32 = torch.zeros(n_q * 128, dtype=torch.float32, device=dev)
    nbytes = n_q * 11 * 528 + 16 if short_workspace else ops.workspace_bytes(n_q, 128, msl)
    ws = torch.full((nbytes // 4,), float("nan"), dtype=torch.float32, device=dev)
    pos = torch.zeros(1, dtype=torch.int32, device=dev)
    stream, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    kw = dict(layer_id=0, pos=msl - 1, kv_dim=n_kv * 128, kv_mul=n_q // n_kv, head_num=n_q, head_dim=128, max_seq_len=msl,
              kv_layout=layout, output_f32=out32, pos_device=pos)
    with torch.cuda.stream(stream):
        with torch.cuda.graph(g, stream=stream):
            ops.mha_decode(q, k, v, out, ws, stream=stream, **kw)
    half = max(128 // n_kv, n_q // n_kv if n_q // n_kv > 8 and n_q <= 128 else 2)
    edges = [11 * 16, 12 * 16, 15 * 16, 16 * 16, 16 * half, 16 * (4 * half), 16 * (256 // n_kv)]
    lengths = sorted({1, 2, 16, 17, 100, 777, msl - 1, msl} | {e + d for e in edges for d in (-16, -1, 0, 1, 16)})
    for n in [x for x in lengths if 0 < x <= msl]:
        pos.fill_(n - 1)
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        ref = oracle.mha_cpu(case["q"], case["k"], case["v"], 0, n - 1, n_kv * 128, n_q // n_kv, n_q, 128, msl)
        assert_parity(from_dev_bf16(out), ref, "%d positions" % n)
        if n > 4:  # (the tap's absolute bound is for averages, not for a single V row)
            assert np.all(np.abs(out32.cpu().numpy() - ref) <= 2e-5 + 2e-4 * np.abs(ref)), "%d positions" % n
