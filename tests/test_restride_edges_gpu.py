"""Cache conversion at the edges of its blocks (16 head rows), against torch's own copy: rows behind num_pos stay as they are."""
import pytest
import torch

from llminfer_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers,n_kv,num_pos,max_seq_len", [
    (1, 1, 1, 1), (2, 3, 5, 9), (3, 8, 2, 2), (2, 5, 16, 33), (4, 16, 1, 7), (70, 2, 8, 8), (1, 1, 4097, 5000),
])
def test_restride_moves_exactly_the_positions_asked_for(dev, layers, n_kv, num_pos, max_seq_len):
    src = torch.randint(-2 ** 15, 2 ** 15, (layers, max_seq_len, n_kv, 128), dtype=torch.int16, device=dev)
    dst = torch.full((layers, n_kv, max_seq_len, 128), 77, dtype=torch.int16, device=dev)
    want = dst.clone()
    want[:, :, :num_pos] = src[:, :num_pos].transpose(1, 2)
    ops.kv_restride(src, dst, layer_num=layers, max_seq_len=max_seq_len, kv_dim=n_kv * 128, head_dim=128, num_pos=num_pos)
    assert torch.equal(dst, want)
