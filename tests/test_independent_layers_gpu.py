"""GPU tests of llmi_hip_mha_decode_append_stack on layers that cannot see each other's writes: they run as one stream whose
partial results go round in a few regions of the workspace. Reference: one llmi_hip_mha_decode_append launch per layer, same bits."""
import pytest
import torch

from llminfer_amd import _binding as B
from llminfer_amd import ops

from test_resident_stack_gpu import D, Stack, timeouts

pytestmark = pytest.mark.gpu

HEAD, POS = B.KV_LAYOUT_HEAD_MAJOR, B.KV_LAYOUT_POS_MAJOR


def _workspace_for(st, splits, regions):
    """A workspace with room for exactly `regions` layers' partial rows and records (None: as it is)."""
    if regions is None:
        return st.ws
    region = (st.n_q * splits * 528 + 16 + 255) // 256 * 256
    need = regions * region + 256 + 16 * 64 * 4  # ... and the done tags
    return torch.full((need // 4,), float("nan"), dtype=torch.float32, device=st.dev)


@pytest.mark.parametrize("layers,ctx,n_q,n_kv,layout,splits,regions,over", [
    (3, 300, 32, 8, HEAD, 8, None, {}),     # a region per layer: records are cleared for replays
    (11, 300, 32, 8, HEAD, 8, 3, {}),       # three regions: a merge takes its steps one after the other
    (11, 300, 32, 8, POS, 8, 4, {}),
    (14, 300, 32, 8, HEAD, 8, 5, {}),       # five: a step per layer, region reuse checked layer by layer
    (37, 300, 24, 8, HEAD, 8, 9, {}),       # ... and three layers at a time; groups of three heads
    (40, 200, 8, 8, POS, 8, None, {}),      # one head per KV head, more layers than tag lines
    (20, 1030, 32, 8, HEAD, 32, None, {}),  # two or three tiles per split: idle wavefronts, a one-row tile
    (9, 1100, 16, 4, HEAD, 64, None, {"num_splits": 64, "force_path": B.PATH_SPLIT_FUSED}),  # two batches of rows per merge
    (9, 700, 32, 8, HEAD, 4, 6, {"num_splits": 4, "force_path": B.PATH_SPLIT_FUSED}),  # every workgroup merges in every layer
])
def test_independent_layers_give_the_bits_of_one_launch_per_layer(dev, layers, ctx, n_q, n_kv, layout, splits, regions, over):
    st = Stack(dev, layers, ctx, n_q=n_q, n_kv=n_kv, layout=layout)
    a = st.fresh()
    tap_a = torch.zeros(layers * st.dim, dtype=torch.float32, device=dev)
    st.run_per_layer(a, **over)
    for l in range(layers):
        kw = dict(st.kw, layer_id=l, output_f32=tap_a[l * st.dim:], **over)
        ops.mha_decode_append(a["q"][l * st.dim:], a["kn"][l * st.kv_dim:], a["vn"][l * st.kv_dim:], a["w"][l * 2 * D:], st.sin_d,
                              st.cos_d, a["k"], a["v"], a["out"][l * st.dim:], st.ws, **kw)
    full, st.ws = st.ws, _workspace_for(st, splits, regions)
    before = timeouts()
    tap = torch.zeros_like(tap_a)
    b = st.fresh()
    assert st.run_stack(b, output_f32=tap, **over) == 1
    assert torch.equal(b["out"], a["out"]) and torch.equal(tap, tap_a)
    assert torch.equal(b["k"], a["k"]) and torch.equal(b["v"], a["v"])
    # replays carry the same tags: nothing the last one left behind may be taken for this one's
    stream, g, c = torch.cuda.Stream(), torch.cuda.CUDAGraph(), st.fresh()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(g, stream=stream):
            st.run_stack(c, stream=stream, **over)
    for rep in range(3):
        c["q"].copy_(torch.roll(b["q"], st.dim * rep))  # another query per layer: a stale record would show
        for l in range(layers):
            kw = dict(st.kw, layer_id=l, **over)
            ops.mha_decode_append(c["q"][l * st.dim:], b["kn"][l * st.kv_dim:], b["vn"][l * st.kv_dim:], b["w"][l * 2 * D:], st.sin_d,
                                  st.cos_d, b["k"], b["v"], b["out"][l * st.dim:], torch.empty_like(full), **kw)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(c["out"], b["out"]), "replay %d" % rep
    assert timeouts() == before


def test_interleaved_buffers_keep_the_order_between_layers(dev):
    """Queries and outputs row by row in one array: the ranges overlap, so the layers stay a chain."""
    st = Stack(dev, 6, 900)
    a, b = st.fresh(), st.fresh()
    st.run_per_layer(a)
    rows = torch.zeros((st.layers, 2, st.dim), dtype=torch.int16, device=dev)
    rows[:, 0] = b["q"].view(-1, st.dim)[:st.layers]
    n = ops.mha_decode_append_stack(rows.view(-1), b["kn"], b["vn"], b["w"], st.sin_d, st.cos_d, b["k"], b["v"], rows.view(-1)[st.dim:], st.ws,
                                    layer_count=st.layers, query_stride=2 * st.dim, key_new_stride=st.kv_dim, value_new_stride=st.kv_dim,
                                    norm_weight_stride=2 * D, output_stride=2 * st.dim, **st.kw)
    torch.cuda.synchronize()
    assert n == 1 and torch.equal(rows[:, 1].reshape(-1), a["out"])
    assert torch.equal(b["k"], a["k"]) and torch.equal(b["v"], a["v"])
