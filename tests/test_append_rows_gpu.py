"""The append variant's rows: a workgroup's query rows, and in the last split's the new K and V rows, are dealt to its wavefronts
in pairs. Every group size and wavefront count the kernels are built for, where the deal changes (odd groups, more rows than
wavefronts have places for in one pass), against the CPU oracle."""
import numpy as np
import pytest
import torch

from llminfer_amd import _binding as B
from llminfer_amd import ops, synth

from helpers import assert_parity, from_dev_bf16, to_dev

pytestmark = pytest.mark.gpu

D = 128


def _append(oracle, dev, group, n_kv, ctx, *, waves=0, splits=0, on_device=False, scale=1.0, eps=1e-6, msl=None):
    """One call; its output, its appended rows, and what the oracle has for them."""
    n_q, pos, msl, kv_dim = group * n_kv, ctx, msl or ctx + 2, n_kv * D
    rng = np.random.RandomState(1000 * group + ctx)
    case = synth.make_case(ctx + group, n_q=n_q, n_kv=n_kv, ctx=max(ctx, 1), max_seq_len=msl)
    row = lambda *shape: rng.standard_normal(shape).astype(np.float32)
    q_raw, k_new = (synth.f32_to_bf16_bits(row(n, D) * np.float32(scale)) for n in (n_q, n_kv))
    v_new = synth.f32_to_bf16_bits(row(n_kv, D))
    w = synth.f32_to_bf16_bits(1 + 0.02 * row(2 * D))
    sin_o, cos_o = oracle.sincos_table(D, msl)
    k_n = oracle.qk_norm_rope(k_new, w[D:], sin_o[pos], cos_o[pos], eps)
    q_n = oracle.qk_norm_rope(q_raw, w[:D], sin_o[pos], cos_o[pos], eps)
    k_ref, v_ref = case["k"].copy(), case["v"].copy()
    k_ref[0, pos], v_ref[0, pos] = k_n.reshape(-1), v_new.reshape(-1)
    ref = oracle.mha_cpu(q_n.reshape(-1), k_ref, v_ref, 0, pos, kv_dim, group, n_q, D, msl)

    k_d, v_d = (to_dev(synth.to_head_major(case[c], n_kv), dev) for c in "kv")
    out = torch.zeros(n_q * D, dtype=torch.int16, device=dev)
    ws = torch.full((ops.workspace_bytes(n_q, D, msl) // 4,), float("nan"), dtype=torch.float32, device=dev)
    sin_d, cos_d = ops.sincos_table(D, msl, dev)
    kw = dict(layer_id=0, pos=pos, kv_dim=kv_dim, kv_mul=group, head_num=n_q, head_dim=D, max_seq_len=msl,
              kv_layout=B.KV_LAYOUT_HEAD_MAJOR, waves_per_group=waves, num_splits=splits, eps=eps)
    if on_device:
        kw.update(pos=msl - 1, pos_device=torch.tensor([pos], dtype=torch.int32, device=dev))
    up = lambda a: to_dev(a.reshape(-1), dev)
    ops.mha_decode_append(up(q_raw), up(k_new), up(v_new), up(w), sin_d, cos_d, k_d, v_d, out, ws, **kw)
    torch.cuda.synchronize()
    rows = [c.cpu().numpy().view(np.uint16)[0, :, pos] for c in (k_d, v_d)]
    return from_dev_bf16(out), ref, rows, k_n, v_new


def _check(got, ref, rows, k_n, v_new, what):
    assert_parity(got, ref, what)
    assert np.array_equal(rows[1], v_new), what
    k_got, k_want = (synth.bf16_bits_to_f32(x).astype(np.float64) for x in (rows[0], k_n))
    # (a bf16 step where a sum in another order rounds the other way)
    assert np.all(np.abs(k_got - k_want) <= np.abs(k_want) / 128 + 1e-6) and (rows[0] == k_n).mean() > 0.99, what


@pytest.mark.parametrize("waves", [0, 1, 2, 4, 8])
@pytest.mark.parametrize("group", [1, 2, 3, 4, 5, 7, 8, 9, 15, 16])
def test_every_deal_of_the_rows(oracle, dev, group, waves):
    if waves * (1 << (group - 1).bit_length()) > 64:
        pytest.skip("no kernel of this many wavefronts for the group")
    for ctx, splits in ((0, 0), (33, 1), (150, 3)):
        what = "group %d, %d waves, %d positions, %d splits" % (group, waves, ctx, splits)
        _check(*_append(oracle, dev, group, 2, ctx, waves=waves, splits=splits), what)


@pytest.mark.parametrize("group,n_kv", [(2, 8), (4, 8), (8, 8), (5, 3), (16, 1)])
def test_rows_at_a_device_position(oracle, dev, group, n_kv):
    for ctx in (1, 129, 700):
        _check(*_append(oracle, dev, group, n_kv, ctx, on_device=True, msl=1024), "group %d, %d positions" % (group, ctx))


@pytest.mark.parametrize("scale,eps", [(1e16, 1e-6), (1e-17, 0.0), (1e-3, 1e-6), (0.0, 1e-6)])
def test_rows_of_any_size(oracle, dev, scale, eps):
    """Mean squares in and out of the range of the reciprocal root."""
    got, ref, rows, k_n, v_new = _append(oracle, dev, 4, 8, 40, scale=scale, eps=eps)
    _check(got, ref, rows, k_n, v_new, "rows of size %g" % scale)
