"""Torch-tensor front end of the C ABI. PyTorch is only used for device memory
and streams: each function reads data_ptr()s and calls libllmi_hip.so. The calls
of a decode step are native (csrc/front/torch_ops.cpp): their own cost on the host
is what an eager step costs."""
import ctypes

import torch

from . import _binding as B

_BF16_DTYPES = (torch.bfloat16, torch.uint16, torch.int16)


def _ptr(t):
    return None if t is None else t.data_ptr()


def _stream_handle(stream):
    if stream is None:
        stream = torch.cuda.current_stream()
    return stream.cuda_stream if hasattr(stream, "cuda_stream") else int(stream)


def _check_dev(name, t, dtypes):
    if t is None:
        return
    if not t.is_cuda:
        raise ValueError("%s must be a device tensor" % name)
    if t.dtype not in dtypes:
        raise ValueError("%s has dtype %s, expected one of %s" % (name, t.dtype, dtypes))
    if not t.is_contiguous():
        raise ValueError("%s must be contiguous" % name)


def workspace_bytes(head_num, head_dim, max_seq_len):
    return int(B.lib().llmi_hip_mha_workspace_bytes(head_num, head_dim, max_seq_len))


def make_mha_args(query, key_cache, value_cache, output, workspace, *, layer_id, pos, kv_dim, kv_mul,
                  head_num, head_dim, max_seq_len, kv_layout=B.KV_LAYOUT_POS_MAJOR, force_path=B.PATH_AUTO,
                  num_splits=0, waves_per_group=0, output_f32=None, stream=None, pos_device=None, workspace_side=0):
    """Fills an llmi_mha_args from torch tensors (or raw integer addresses)."""
    def addr(x):
        return x if (x is None or isinstance(x, int)) else x.data_ptr()

    a = B.MhaArgs()
    a.query = addr(query)
    a.key_cache = addr(key_cache)
    a.value_cache = addr(value_cache)
    a.workspace = addr(workspace)
    if workspace is None:
        a.workspace_bytes = 0
    elif isinstance(workspace, int):
        raise ValueError("pass workspace as a tensor so its size is known")
    else:
        a.workspace_bytes = workspace.numel() * workspace.element_size()
    a.output = addr(output)
    a.output_f32 = addr(output_f32)
    a.layer_id, a.pos, a.kv_dim, a.kv_mul = layer_id, pos, kv_dim, kv_mul
    a.head_num, a.head_dim, a.max_seq_len = head_num, head_dim, max_seq_len
    a.kv_layout, a.force_path, a.num_splits, a.waves_per_group = kv_layout, force_path, num_splits, waves_per_group
    a.stream = stream
    a.pos_device = addr(pos_device)
    a.workspace_side = workspace_side
    return a


def workspace_side(workspace, stream=None):
    """Which 8 KiB blocks of `workspace` lie near which side of the package (llmi_hip_mha_workspace_side): 0, 1 or 2,
    to be passed as workspace_side with this workspace. Overwrites its first 32 KiB and synchronises the stream."""
    _check_dev("workspace", workspace, (torch.float32,))
    side = ctypes.c_int32(0)
    s = stream if stream is not None else torch.cuda.current_stream(workspace.device).cuda_stream
    B.check(B.lib().llmi_hip_mha_workspace_side(workspace.data_ptr(), workspace.numel() * workspace.element_size(), s,
                                                ctypes.byref(side)), "llmi_hip_mha_workspace_side")
    return side.value


def mha_plan(args):
    plan = B.MhaPlan()
    B.check(B.lib().llmi_hip_mha_plan(ctypes.byref(args), ctypes.byref(plan)), "llmi_hip_mha_plan")
    return plan


def mha_decode_raw(args):
    """Calls llmi_hip_mha_decode on a prepared llmi_mha_args; returns the status."""
    return int(B.lib().llmi_hip_mha_decode(ctypes.byref(args)))


def sincos_table(head_dim, max_seq_len, device="cuda", stream=None):
    sin = torch.empty((max_seq_len, head_dim // 2), dtype=torch.float32, device=device)
    cos = torch.empty_like(sin)
    B.check(B.lib().llmi_hip_sincos_table(sin.data_ptr(), cos.data_ptr(), head_dim, max_seq_len,
                                          _stream_handle(stream)), "llmi_hip_sincos_table")
    return sin, cos


def _native():
    """The extension, bound to the loaded library's functions. Raises if it has not been built."""
    try:
        from . import _torch_ops as native
    except ImportError as e:
        raise RuntimeError("the torch front end is not built (%s); run `python -m llminfer_amd.build`. "
                           "There is no fallback implementation." % e) from e
    lib = B.lib()
    names = ("llmi_hip_mha_decode", "llmi_hip_mha_decode_append", "llmi_hip_mha_decode_append_oproj", "llmi_hip_mha_oproj_launches",
             "llmi_hip_mha_decode_append_stack", "llmi_hip_mha_stack_launches", "llmi_hip_qk_norm_rope_append", "llmi_hip_kv_restride",
             "llmi_hip_gemv", "llmi_hip_qkv_gemv")
    addresses = {n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in names}
    abi = native.bind(addresses, torch._C._cuda_getDevice, torch._C._cuda_getCurrentRawStream, _check_dev, B.check, _BF16_DTYPES,
                      (torch.float32,))
    if abi != lib.llmi_hip_abi_version():
        raise RuntimeError("the torch front end was built against ABI %d, the library is %d" % (abi, lib.llmi_hip_abi_version()))
    return native


# The native calls by name. They take their places in this module when the first of them is asked for: importing it, and its argument
# helpers, need nothing built.
_CALLS = ("mha_decode", "mha_decode_append", "mha_decode_append_stack", "qk_norm_rope_append", "kv_restride", "gemv", "qkv_gemv")
__all__ = ["workspace_bytes", "make_mha_args", "workspace_side", "mha_plan", "mha_decode_raw", "sincos_table", *_CALLS]


def _bind_calls():
    native = _native()
    globals().update({name: getattr(native, name) for name in _CALLS})
    return native


def _unbuilt(name):
    """What stands for a native call while there is none: the call says what is missing."""
    def call(*args, **kw):
        return getattr(_bind_calls(), name)(*args, **kw)
    call.__name__ = call.__qualname__ = name
    return call


def __getattr__(name):
    if name not in _CALLS:
        raise AttributeError("module %r has no attribute %r" % (__name__, name))
    try:
        return getattr(_bind_calls(), name)
    except (RuntimeError, OSError):
        return _unbuilt(name)


def __dir__():
    return sorted(set(globals()) | set(_CALLS))
