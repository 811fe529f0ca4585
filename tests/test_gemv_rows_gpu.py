"""GPU tests of the GEMV at the edges of its kernels: every step count (rows of 512 elements a step, whole and part steps), the
long-row loop behind the last of them, and both sides of the row count at which workgroups grow to four wavefronts."""
import numpy as np
import pytest
import torch

from llminfer_amd import _binding as B
from llminfer_amd import ops

from helpers import to_dev
from test_gemv_gpu import _case, _gate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [8, 512, 520] + [512 * s + d for s in range(2, 20) for d in (0, 8)] + [10232, 10240, 10248] + [512 * s + d for s in range(21, 34) for d in (-8, 0, 8)] + [21000])
def test_every_step_count(oracle, dev, k):
    n = 7
    x, w, sumabs = _case(k, n, k)
    out = torch.full((n + 1,), float("nan"), dtype=torch.float32, device=dev)
    ops.gemv(to_dev(x, dev), to_dev(w, dev), out[:n], mode=B.GEMV_OUT_F32)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    _gate(got[:n], oracle.gemv_bf16(x, w), sumabs, False, "k = %d" % k)
    assert np.isnan(got[n])


@pytest.mark.parametrize("n", [1, 3, 6143, 6144, 6145, 6147])
@pytest.mark.parametrize("k", [264, 10248])
def test_row_counts(oracle, dev, n, k):
    x, w, sumabs = _case(n, n, k)
    out = torch.full((n + 4,), float("nan"), dtype=torch.float32, device=dev)
    ops.gemv(to_dev(x, dev), to_dev(w, dev), out[:n], mode=B.GEMV_OUT_F32)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    _gate(got[:n], oracle.gemv_bf16(x, w), sumabs, False, "n = %d" % n)
    assert np.all(np.isnan(got[n:]))  # nothing written past the last row


@pytest.mark.parametrize("n,k", [(n, k) for n in (1024, 1025, 2048, 2049, 2560, 2561) for k in (4096, 4104, 6144, 6152, 8192, 10232, 10240, 12288, 12296)] +
                         [(24575, 4096), (24576, 4096), (24577, 4088)])
def test_kernels_by_row_count(oracle, dev, n, k):
    """Batches of four, windows of four and ten, on either side of the row counts between them."""
    test_row_counts(oracle, dev, n, k)
