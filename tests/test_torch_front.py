"""The native calls of llminfer_amd.ops: how they take their arguments and refuse wrong ones (no GPU needed: a refused call
reaches neither the C ABI nor the device), and what they hand on where there is a GPU."""
import inspect
import os
import subprocess
import sys

import pytest
import torch

from llminfer_amd import _binding as B
from llminfer_amd import ops

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SCALARS = dict(layer_id=0, pos=5, kv_dim=1024, kv_mul=4, head_num=32, head_dim=128, max_seq_len=64)


def _t(n=8, dtype=torch.bfloat16):
    return torch.zeros(n, dtype=dtype)


@pytest.mark.parametrize("call,error,text", [
    (lambda t: ops.mha_decode(t, t, t, t, t, **SCALARS), ValueError, "query must be a device tensor"),
    (lambda t: ops.mha_decode(t, t, t, t, **SCALARS), TypeError, "workspace"),
    (lambda t: ops.mha_decode(t, t, t, t, t, t, **SCALARS), TypeError, "5 positional"),
    (lambda t: ops.mha_decode(t, t, t, t, t, **{k: v for k, v in SCALARS.items() if k != "pos"}), TypeError, "'pos'"),
    (lambda t: ops.mha_decode(t, t, t, t, t, splits=3, **SCALARS), TypeError, "unexpected keyword argument 'splits'"),
    (lambda t: ops.mha_decode(t, t, t, t, t, eps=1e-6, **SCALARS), TypeError, "unexpected keyword argument 'eps'"),
    (lambda t: ops.mha_decode(t, t, t, t, t, query=t, **SCALARS), TypeError, "multiple values for argument 'query'"),
    (lambda t: ops.mha_decode(query=None, key_cache=t, value_cache=t, output=t, workspace=None, **SCALARS), ValueError, "key_cache must be"),
    (lambda t: ops.mha_decode(None, None, None, None, None, **dict(SCALARS, pos=1.5)), TypeError, "integer"),
    (lambda t: ops.gemv(None, None, None, mode="f32"), TypeError, "integer"),
    (lambda t: ops.gemv(None, None, None), ValueError, "weight"),
    (lambda t: ops.kv_restride(t, t, layer_num=1, max_seq_len=1, kv_dim=1024, head_dim=128), TypeError, "num_pos"),
    (lambda t: ops.mha_decode_append_stack(*[None] * 10, **SCALARS), TypeError, "layer_count"),
])
def test_refused_arguments(call, error, text):
    with pytest.raises(error, match=text):
        call(_t())


def test_tensors_without_storage_raise():
    """Under vmap (over tensors that only claim to be the device's) torch refuses to give an address: an error like any other."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        x = torch.empty((4, 128), dtype=torch.bfloat16, device="cuda")
        w = torch.empty((16, 128), dtype=torch.bfloat16, device="cuda")
        with pytest.raises(RuntimeError, match="data pointer"):
            torch.vmap(lambda row: ops.gemv(row, w, w[0, :16]))(x)
        with pytest.raises(RuntimeError, match="data pointer"):
            torch.vmap(lambda row: ops.mha_decode(None, None, None, None, None, pos_device=row, **SCALARS))(x)


def test_signatures_are_the_documented_ones():
    sig = inspect.signature(ops.mha_decode_append)
    assert list(sig.parameters)[:10] == ["query_raw", "key_new", "value_new", "norm_weight", "sin_cache", "cos_cache", "key_cache",
                                         "value_cache", "output", "workspace"]
    assert sig.parameters["eps"].default == 1e-6 and sig.parameters["one_launch"].default is False
    assert inspect.signature(ops.gemv).parameters["mode"].default == B.GEMV_OUT_BF16
    assert inspect.signature(ops.mha_decode).parameters["kv_layout"].default == B.KV_LAYOUT_POS_MAJOR


def test_import_needs_nothing_built():
    """Importing the module, its argument helpers and the names of its calls load no library; what is missing is said by the call."""
    code = ("from llminfer_amd import _binding as B, ops\n"
            "from llminfer_amd.ops import *\n"
            "assert B._lib is None\n"
            "a = ops.make_mha_args(16, 16, 16, 16, None, **%r)\n"
            "assert a.head_num == 32 and 'gemv' in dir(ops) and callable(gemv) and callable(ops.mha_decode)\n"
            "for f in (ops.gemv, kv_restride):\n"
            "    try:\n"
            "        f(None, None, None)\n"
            "    except RuntimeError as e:\n"
            "        assert 'is not built' in str(e), e\n"
            "    else:\n"
            "        raise SystemExit('no error')\n" % SCALARS)
    env = dict(os.environ, LLMI_HIP_LIBRARY=os.path.join(ROOT, "no_such_library.so"))
    subprocess.run([sys.executable, "-c", code], check=True, env=env, cwd=ROOT)
    with pytest.raises(AttributeError, match="no attribute 'gemm'"):
        ops.gemm


@pytest.mark.gpu
def test_calls_on_the_device(dev):
    n, k = 33, 520
    gen = torch.Generator(device=dev)
    gen.manual_seed(3)
    x = torch.randn(k, generator=gen, device=dev).to(torch.bfloat16)
    w = torch.randn((n, k), generator=gen, device=dev).to(torch.bfloat16)
    want = torch.empty(n, device=dev)
    assert ops.gemv(x, w, want, mode=B.GEMV_OUT_F32) is want
    side, got = torch.cuda.Stream(), torch.empty(n, device=dev)
    side.wait_stream(torch.cuda.current_stream())
    for stream in (side, side.cuda_stream, None):  # a stream, its number, the current one
        got.zero_()
        torch.cuda.synchronize()
        if stream is None:
            with torch.cuda.stream(side):
                ops.gemv(input=x, weight=w, output=got, mode=B.GEMV_OUT_F32, stream=None)
        else:
            ops.gemv(x, w, got, mode=B.GEMV_OUT_F32, stream=stream)
        side.synchronize()
        assert torch.equal(got, want)
    # strides are refused, dtypes are checked by mode
    with pytest.raises(ValueError, match="weight must be contiguous"):
        ops.gemv(x[:n], w.t(), want, mode=B.GEMV_OUT_F32)
    with pytest.raises(ValueError, match="output has dtype torch.float32"):
        ops.gemv(x, w, want)
    with pytest.raises(AssertionError):
        ops.qkv_gemv(x, w, x[:16], x[:8], x[:16])
    # a status of the C ABI arrives as LlmiError with its own text
    with pytest.raises(B.LlmiError) as e:
        ops.mha_decode(x, x, x, x, None, **dict(SCALARS, pos=64))
    assert e.value.status == B.STATUS["POS_RANGE"] and "llmi_hip_mha_decode" in str(e.value)
    with pytest.raises(B.LlmiError) as e:
        ops.mha_decode(x, x, x, x, None, **dict(SCALARS, layer_id=2**31))  # (wraps to a negative layer, as in the C struct)
    assert e.value.status == B.STATUS["INVALID_ARG"]
