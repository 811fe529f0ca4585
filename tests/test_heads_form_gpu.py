"""GPU tests of the multi-layer launch that takes a KV head of a layer at a time (independent layers): bits of one
llmi_hip_mha_decode_append launch per layer, replays, the wait of heads that are cut between workgroups."""
import ctypes

import numpy as np
import pytest
import torch

from llminfer_amd import _binding as B
from llminfer_amd import ops

import test_independent_layers_gpu as independent
from helpers import from_dev_bf16
from test_resident_stack_gpu import Stack, timeouts

pytestmark = pytest.mark.gpu

HEAD, POS = B.KV_LAYOUT_HEAD_MAJOR, B.KV_LAYOUT_POS_MAJOR


def _form(st, **over):
    """What the planner says of the stack's layers: llmi_hip_heads_form."""
    t, s, form = st.fresh(), B.MhaStackArgs(), (ctypes.c_int32 * 6)()
    s.first.mha = ops.make_mha_args(t["q"], t["k"], t["v"], t["out"], st.ws, **dict(st.kw, **over))
    s.first.key_new, s.first.value_new, s.first.norm_weight = t["kn"].data_ptr(), t["vn"].data_ptr(), t["w"].data_ptr()
    s.first.sin_cache, s.first.cos_cache, s.first.eps = st.sin_d.data_ptr(), st.cos_d.data_ptr(), 1e-6
    s.layer_count, s.query_stride, s.output_stride = st.layers, st.dim, st.dim
    s.key_new_stride, s.value_new_stride, s.norm_weight_stride = st.kv_dim, st.kv_dim, 2 * 128
    B.check(B.lib().llmi_hip_heads_form(ctypes.byref(s), 0, form), "llmi_hip_heads_form")
    return list(form)


@pytest.mark.parametrize("layers,ctx,n_q,n_kv,layout", [
    (4, 1, 32, 8, HEAD),     # one cached position, one wavefront with a tile
    (5, 17, 32, 8, POS),     # two tiles, a row in the second
    (8, 100, 64, 8, HEAD),   # a single pass of eight wavefronts
    (8, 170, 24, 8, HEAD),   # ... with groups of three: more tiles than wavefronts
    (7, 300, 64, 8, POS),    # sixteen splits, wavefronts without a tile
    (9, 420, 40, 8, HEAD),   # groups of five
    (4, 500, 16, 16, HEAD),  # one query head per KV head, sixteen of them
    (64, 60, 16, 8, HEAD),   # two heads per workgroup
    (36, 300, 32, 8, HEAD),  # 32 heads over: cut
    (35, 270, 24, 8, POS),   # 24 heads over
    (33, 1000, 64, 8, HEAD),  # 8 heads over: a split per part
    (12, 2100, 64, 8, HEAD),  # fewer heads than workgroups: every head cut
])
def test_heads_one_by_one_give_the_bits_of_one_launch_per_layer(dev, layers, ctx, n_q, n_kv, layout):
    assert _form(Stack(dev, layers, ctx, n_q=n_q, n_kv=n_kv, layout=layout))[0] > 0
    independent.test_independent_layers_give_the_bits_of_one_launch_per_layer(dev, layers, ctx, n_q, n_kv, layout, None, None, {})


@pytest.mark.parametrize("layers,regions", [(16, 3), (16, 4), (14, 5), (16, 9)])
def test_layers_one_by_one_reuse_the_regions_of_a_small_workspace(dev, layers, regions):
    """Lengths at which the stream by layers stays the faster form."""
    independent.test_independent_layers_give_the_bits_of_one_launch_per_layer(dev, layers, 2000, 32, 8, HEAD, 32, regions, {})


def test_cut_heads_give_up_with_nan_instead_of_hanging(dev):
    """36 layers x 8 heads on 256 compute units: the last four layers' heads are cut. With the poll limit forced to zero they are NaN,
    the others do not notice; with it restored the same call is right."""
    st = Stack(dev, 36, 300, seed=7)
    a = st.fresh()
    st.run_per_layer(a)
    before, prev = timeouts(), B.lib().llmi_hip_set_poll_limit(0)
    try:
        b = st.fresh()
        assert st.run_stack(b) == 1
    finally:
        assert B.lib().llmi_hip_set_poll_limit(prev) == 0
    cut = 36 * 8 % torch.cuda.get_device_properties(dev).multi_processor_count // 8
    assert cut == 4 and timeouts() > before
    whole = (36 - cut) * st.dim
    assert torch.equal(b["out"][:whole], a["out"][:whole])
    assert np.all(np.isnan(from_dev_bf16(b["out"][whole:36 * st.dim])))
    after = timeouts()
    st.ws.fill_(float("nan"))
    c = st.fresh()
    assert st.run_stack(c) == 1
    assert torch.equal(c["out"], a["out"]) and timeouts() == after


@pytest.mark.parametrize("layers,ctx,n_q,n_kv,layout,forced,splits,at_once,parts", [
    (5, 250, 64, 8, HEAD, 0, 16, 8, 1),     # a tile each
    (5, 257, 64, 8, POS, 0, 16, 4, 1),      # one of them has two
    (33, 256, 40, 8, HEAD, 0, 16, 8, 1),    # groups of five, two heads for some workgroups
    (5, 300, 64, 8, POS, 19, 19, 8, 1),     # the last round has three splits
    (35, 432, 64, 8, HEAD, 27, 27, 8, 2),   # ... and heads are cut: 13 splits and 14
    (33, 304, 56, 8, HEAD, 19, 19, 8, 16),  # ... a part has one or two
    (4, 512, 64, 8, HEAD, 0, 16, 4, 8),     # two whole tiles each
    (33, 352, 64, 8, HEAD, 11, 11, 4, 8),   # ... eleven splits
    (40, 330, 64, 8, HEAD, 11, 11, 4, 1),   # ... uncut: four, four and three
    (4, 513, 64, 8, HEAD, 0, 16, 2, 8),     # three
    (6, 1023, 64, 8, POS, 0, 16, 2, 4),     # four, the last one ragged
    (33, 440, 64, 8, POS, 7, 7, 2, 4),      # seven splits of four
    (5, 1041, 64, 8, HEAD, 0, 32, 2, 4),    # two or three
    (36, 2048, 64, 8, HEAD, 0, 32, 2, 8),   # four
    (4, 2049, 64, 8, HEAD, 0, 32, 1, 8),    # five: one split at a time
    (9, 186, 32, 8, HEAD, 0, 8, 2, 1),      # four wavefronts stream: splits of one tile or two
    (9, 256, 24, 8, POS, 0, 16, 4, 1),      # a tile each, groups of three
    (33, 256, 16, 8, HEAD, 0, 16, 4, 16),   # ... a split per part
    (5, 300, 32, 8, HEAD, 19, 19, 4, 1),    # ... the last round has three
    (35, 368, 32, 8, POS, 23, 23, 4, 2),    # ... cut: eleven and twelve
    (5, 500, 32, 8, HEAD, 0, 16, 2, 4),     # two each
    (35, 512, 8, 8, HEAD, 0, 16, 2, 8),     # ... whole tiles
    (12, 300, 16, 4, HEAD, 0, 16, 2, 1),    # ... or one
    (12, 280, 16, 4, HEAD, 9, 9, 2, 1),     # ... nine splits
    (4, 513, 32, 8, HEAD, 0, 16, 1, 8),     # three: one split at a time
])
def test_splits_side_by_side_give_the_bits_of_one_launch_per_layer(dev, layers, ctx, n_q, n_kv, layout, forced, splits, at_once, parts):
    over = dict(num_splits=forced, force_path=B.PATH_SPLIT_FUSED) if forced else {}
    grid, *form = _form(Stack(dev, layers, ctx, n_q=n_q, n_kv=n_kv, layout=layout), **over)
    assert grid > 0 and form == [parts, layers * n_kv % 256 if parts > 1 else 0, 8 if n_q // n_kv > 4 else 4, splits, at_once]
    independent.test_independent_layers_give_the_bits_of_one_launch_per_layer(dev, layers, ctx, n_q, n_kv, layout, None, None, over)
