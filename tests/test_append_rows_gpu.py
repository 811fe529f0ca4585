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


def _bf16(bits):
    return synth.bf16_bits_to_f32(bits)


def _fma(a, b, c):
    return (np.asarray(a, np.longdouble) * b + c).astype(np.float32)


def _chain(rows, w, sin, cos, eps):
    """Norm and rotation of raw bf16 rows [..., 128], operation by operation as the append kernels declare them: squares of four neighbouring
    pairs in a chain, folded neighbour by neighbour, root and division each rounded, bf16 once. sin, cos: [..., 64]."""
    x, w = _bf16(rows).reshape(rows.shape[:-1] + (2, 16, 4)), _bf16(w).reshape(2, 16, 4)
    a, b = x[..., 0, :, :], x[..., 1, :, :]
    ss = _fma(a[..., 0], a[..., 0], a[..., 1] * a[..., 1])
    for v in (a[..., 2], a[..., 3], b[..., 0], b[..., 1], b[..., 2], b[..., 3]):
        ss = _fma(v, v, ss)
    while ss.shape[-1] > 1:
        ss = ss[..., 0::2] + ss[..., 1::2]
    r = np.float32(1) / np.sqrt(_fma(ss, np.float32(1 / 128), np.float32(eps)))[..., None]
    sn, cs = (t.reshape(t.shape[:-1] + (16, 4)) for t in (sin, cos))
    av, bv = a * w[0] * r, b * w[1] * r
    lo, hi = _fma(av, cs, -(bv * sn)), _fma(av, sn, bv * cs)
    return synth.f32_to_bf16_bits(np.stack([lo, hi], axis=-3).reshape(rows.shape).astype(np.float32))


def _append_positions(dev, n_q, n_kv, count, k_new, v_new, w, eps=1e-6):
    """`count` positions appended one call after the other to an empty cache; the cached K rows and the tables' rows."""
    kv_dim = n_kv * D
    kc, vc = (torch.zeros(count, kv_dim, dtype=torch.int16, device=dev) for _ in "kv")
    ws = torch.zeros(ops.workspace_bytes(n_q, D, count) // 4, dtype=torch.float32, device=dev)
    sin, cos = ops.sincos_table(D, count, dev)
    k_d, v_d, w_d = to_dev(k_new, dev), to_dev(v_new, dev), to_dev(w, dev)
    q_d, out = torch.zeros(n_q * D, dtype=torch.int16, device=dev), torch.zeros(n_q * D, dtype=torch.int16, device=dev)
    for pos in range(count):
        ops.mha_decode_append(q_d, k_d[pos], v_d[pos], w_d, sin, cos, kc, vc, out, ws, layer_id=0, pos=pos, kv_dim=kv_dim, kv_mul=n_q // n_kv,
                              head_num=n_q, head_dim=D, max_seq_len=count, kv_layout=B.KV_LAYOUT_POS_MAJOR, eps=eps)
    torch.cuda.synchronize()
    assert np.array_equal(vc.cpu().numpy().view(np.uint16), v_new)
    tables = (t.cpu().numpy().reshape(count, 1, D // 2) for t in (sin, cos))
    return (kc.cpu().numpy().view(np.uint16).reshape(count, n_kv, D), *tables)


@pytest.mark.parametrize("group", [1, 3, 4, 8, 16])
def test_key_rows_have_the_bits_of_the_declared_chain(dev, group):
    """A last fp32 bit turns a bf16 rounding once in some ten thousand values: half a million of them, every one the chain's."""
    n_kv, count = 32, 128
    rng = np.random.RandomState(group)
    bits = lambda *shape: synth.f32_to_bf16_bits(rng.standard_normal(shape).astype(np.float32))
    k_new, v_new, w = bits(count, n_kv * D), bits(count, n_kv * D), synth.f32_to_bf16_bits(1 + 0.02 * rng.standard_normal(2 * D).astype(np.float32))
    got, sin, cos = _append_positions(dev, group * n_kv, n_kv, count, k_new, v_new, w)
    want = _chain(k_new.reshape(count, n_kv, D), w[D:], sin, cos, 1e-6)
    assert np.array_equal(got, want), "%d of %d values differ" % ((got != want).sum(), want.size)


# Value rows whose mean square, with eps, lies outside the range of the reciprocal root, or is nothing at all.
NEIGHBOURS = [(1e16, 1e-6), (float("inf"), 1e-6), (float("nan"), 1e-6), (0.0, 0.0)]


def _with_values(count, n_kv, value, seed):
    rng = np.random.RandomState(seed)
    row = lambda *shape: rng.standard_normal(shape).astype(np.float32)
    k_new, w = synth.f32_to_bf16_bits(row(count, n_kv * D)), synth.f32_to_bf16_bits(1 + 0.02 * row(2 * D))
    return k_new, np.broadcast_to(synth.f32_to_bf16_bits(np.float32([value])), k_new.shape).copy(), w


@pytest.mark.parametrize("value,eps", NEIGHBOURS)
@pytest.mark.parametrize("group", [2, 4, 5])  # (the key row's neighbour: the value row, or the last query row, here all zeros)
def test_a_rows_neighbours_leave_no_trace(dev, group, value, eps):
    n_kv, count = 32, 128
    k_new, v_new, w = _with_values(count, n_kv, value, group)
    got, sin, cos = _append_positions(dev, group * n_kv, n_kv, count, k_new, v_new, w, eps)
    assert np.array_equal(got, _chain(k_new.reshape(count, n_kv, D), w[D:], sin, cos, eps))


@pytest.mark.parametrize("value,eps", NEIGHBOURS)
@pytest.mark.parametrize("chained", [False, True])
def test_a_rows_neighbours_leave_no_trace_in_a_stack(dev, chained, value, eps):
    """The same in the multi-layer launches, whose key rows have a wavefront to themselves: independent layers and a chain. From 300 cached
    positions on, where each is one launch."""
    n_q, n_kv, layers, first, count = 32, 8, 32, 300, 16
    dim, kv_dim = n_q * D, n_kv * D
    k_new, v_new, w = _with_values(count * layers, n_kv, value, 77)
    k_d, v_d, w_d = (to_dev(x, dev) for x in (k_new, v_new, np.tile(w, (layers, 1))))
    kc, vc = (torch.zeros(layers, first + count, kv_dim, dtype=torch.int16, device=dev) for _ in "kv")
    ws = torch.zeros(ops.workspace_bytes(n_q, D, first + count) // 4, dtype=torch.float32, device=dev)
    sin, cos = ops.sincos_table(D, first + count, dev)
    q = torch.full(((layers + 1) * dim,), 0x3F80, dtype=torch.int16, device=dev)
    out = q[dim:] if chained else torch.zeros(layers * dim, dtype=torch.int16, device=dev)
    for i in range(count):
        rows = slice(i * layers, (i + 1) * layers)
        n = ops.mha_decode_append_stack(q, k_d[rows], v_d[rows], w_d, sin, cos, kc, vc, out, ws, layer_id=0, layer_count=layers, pos=first + i,
                                        kv_dim=kv_dim, kv_mul=n_q // n_kv, head_num=n_q, head_dim=D, max_seq_len=first + count,
                                        kv_layout=B.KV_LAYOUT_POS_MAJOR, query_stride=dim, key_new_stride=kv_dim, value_new_stride=kv_dim,
                                        norm_weight_stride=2 * D, output_stride=dim, eps=eps)
        assert n == 1
    torch.cuda.synchronize()
    got = kc[:, first:].cpu().numpy().view(np.uint16).reshape(layers, count, n_kv, D)
    tables = (t.cpu().numpy().reshape(-1, 1, D // 2)[first:] for t in (sin, cos))
    raw = k_new.reshape(count, layers, n_kv, D).transpose(1, 0, 2, 3)
    assert np.array_equal(got, _chain(raw, w[D:], *tables, eps))
