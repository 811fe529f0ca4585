"""A new token whose score overflows to minus infinity has no weight: the output is the softmax over the cached positions. The wavefront
that starts its running softmax from the new token holds that token's value row by then, and its first tile has to clear it. Key norm
weights of 1e37 and raw keys that are the negated raw queries: every appended row is finite, its score with each query head is below the least fp32
number. Against the CPU oracle, in every kernel that starts from the new token."""
import numpy as np
import pytest
import torch

from llminfer_amd import _binding as B
from llminfer_amd import ops, synth

from helpers import assert_parity, from_dev_bf16, to_dev
from test_resident_stack_gpu import D, Stack

pytestmark = pytest.mark.gpu

HEAD, POS = B.KV_LAYOUT_HEAD_MAJOR, B.KV_LAYOUT_POS_MAJOR


def _overflowing(oracle, dev, layers, ctx, group, n_kv, layout=HEAD, chained=False):
    """The stack and the oracle's output of each layer. A group's query heads are one row, so that no other head of it moves its maximum; in a chain
    that holds for every layer, whose query is the output of the one before."""
    st = Stack(dev, layers, ctx, n_q=group * n_kv, n_kv=n_kv, layout=layout, chained=chained)
    st.w[:, :D], st.w[:, D:] = 0x3F80, synth.f32_to_bf16_bits(np.float32([1e37]))[0]
    negated = lambda rows: (rows.reshape(n_kv, group, D)[:, 0] ^ 0x8000).reshape(-1)
    refs = []
    for l in range(layers):
        if chained and l:
            st.q_raw[l] = synth.f32_to_bf16_bits(refs[-1])
        st.q_raw[l] = st.q_raw[l].reshape(n_kv, group, D)[:, :1].repeat(group, axis=1).reshape(-1)
        st.k_new[l] = negated(st.q_raw[l])
        one = _one_layer(st, l)
        refs.append(one.oracle_outputs(oracle)[0])
        # (what the test is about: without the new position the oracle has the same output)
        shown = oracle.mha_cpu(oracle.qk_norm_rope(one.q_raw[0].reshape(-1, D), one.w[0, :D], *(t[ctx] for t in oracle.sincos_table(D, one.msl))).reshape(-1),
                               one.k_all, one.v_all, 0, ctx - 1, st.kv_dim, group, st.n_q, D, st.msl)
        assert np.array_equal(refs[-1], shown) and np.all(np.isfinite(shown))
    return st, refs


def _one_layer(st, l):
    one = object.__new__(Stack)
    one.__dict__.update(st.__dict__, layers=1)
    for name in ("k_all", "v_all", "q_raw", "k_new", "v_new", "w"):
        setattr(one, name, getattr(st, name)[l:l + 1])
    return one


def _check(st, out, refs, what):
    for l, ref in enumerate(refs):
        assert_parity(from_dev_bf16(out[l * st.dim:(l + 1) * st.dim]), ref, "%s, layer %d" % (what, l))


@pytest.mark.parametrize("group,n_kv", [(1, 8), (3, 8), (4, 8), (8, 8), (16, 2)])
@pytest.mark.parametrize("ctx", [1, 40, 700, 3001])
def test_one_launch_per_layer(oracle, dev, group, n_kv, ctx):
    st, refs = _overflowing(oracle, dev, 1, ctx, group, n_kv)
    for waves in (0, 1, 4):
        t = st.fresh()
        st.run_per_layer(t, waves_per_group=waves)
        _check(st, t["out"], refs, "%d wavefronts" % waves)
    t = st.fresh()
    st.run_per_layer(t, pos=st.msl - 1, pos_device=torch.tensor([ctx], dtype=torch.int32, device=dev))
    _check(st, t["out"], refs, "device position")


@pytest.mark.parametrize("layers,ctx,group,chained", [
    (3, 300, 4, False),    # a few independent layers: one stream of all tiles
    (8, 300, 4, False),    # more of them: a KV head at a time
    (8, 1100, 8, False),
    (8, 40, 1, False),     # single passes
    (4, 300, 4, True),     # a chain
    (4, 2000, 1, True),
])
def test_one_launch_for_the_layers(oracle, dev, layers, ctx, group, chained):
    st, refs = _overflowing(oracle, dev, layers, ctx, group, 8, chained=chained)
    t = st.fresh()
    assert st.run_stack(t) == 1
    _check(st, t["out"], refs, "one launch")


def test_with_the_output_projection_in_one_launch(oracle, dev):
    st, refs = _overflowing(oracle, dev, 1, 1100, 4, 8)
    t, hidden = st.fresh(), 256
    wo = to_dev(synth.f32_to_bf16_bits(np.random.RandomState(3).standard_normal((hidden, st.dim)).astype(np.float32)), dev)
    residual = torch.zeros(hidden, dtype=torch.int16, device=dev)
    assert ops.mha_decode_append(t["q"], t["kn"], t["vn"], t["w"], st.sin_d, st.cos_d, t["k"], t["v"], t["out"], st.ws, o_weight=wo,
                                 residual=residual, one_launch=True, **st.kw) == 1
    torch.cuda.synchronize()
    _check(st, t["out"], refs, "with the projection")
