"""GPU tests of the multi-layer launch that takes a KV head of a layer at a time (independent layers): bits of one
llmi_hip_mha_decode_append launch per layer, replays, the wait of heads that are cut between workgroups."""
import numpy as np
import pytest
import torch

from llminfer_amd import _binding as B

import test_independent_layers_gpu as independent
from helpers import from_dev_bf16
from test_resident_stack_gpu import Stack, timeouts

pytestmark = pytest.mark.gpu

HEAD, POS = B.KV_LAYOUT_HEAD_MAJOR, B.KV_LAYOUT_POS_MAJOR


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


@pytest.mark.parametrize("layers,ctx,n_q,n_kv,layout", [
    (5, 250, 64, 8, HEAD),    # 16 splits of a tile each: eight at a time
    (5, 257, 64, 8, POS),     # one of them has two: four
    (33, 256, 40, 8, HEAD),   # ... cut heads, groups of five
    (4, 512, 64, 8, HEAD),    # two each, whole
    (4, 513, 64, 8, HEAD),    # three: two at a time
    (6, 1023, 64, 8, POS),    # four, the last one ragged
    (5, 1041, 64, 8, HEAD),   # 32 splits of two or three
    (36, 2048, 64, 8, HEAD),  # ... of four, cut heads
    (4, 2049, 64, 8, HEAD),   # five: one at a time
    (9, 186, 32, 8, HEAD),    # four wavefronts: 8 splits of one or two, two at a time
    (9, 256, 24, 8, POS),     # 16 of a tile each, four at a time, groups of three
    (33, 256, 16, 8, HEAD),   # ... cut heads
    (5, 500, 32, 8, HEAD),    # two each
    (35, 512, 8, 8, HEAD),    # ... whole, cut heads
    (5, 513, 32, 8, HEAD),    # three: one at a time
    (12, 300, 16, 4, HEAD),   # 19 splits, an odd number, of a tile each
])
def test_splits_side_by_side_give_the_bits_of_one_launch_per_layer(dev, layers, ctx, n_q, n_kv, layout):
    independent.test_independent_layers_give_the_bits_of_one_launch_per_layer(dev, layers, ctx, n_q, n_kv, layout, None, None, {})
