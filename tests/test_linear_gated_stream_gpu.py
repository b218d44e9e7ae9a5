"""The ReLU gate of the streaming Linear (linear_stream.hip), read in the order in which the result is stored: the ungated launch's bits
where the gate is above zero, zeros elsewhere - at ragged row tiles and column blocks, from gates whose rows are only 8-byte aligned."""
import pytest
import torch

from beatsaberrl_amd import ops
from test_ops_gpu import _rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,K,M", [(8192, 192, 768), (8209, 192, 200), (9000, 128, 512), (8193, 128, 136), (20011, 256, 264), (8224, 256, 8)])
@pytest.mark.parametrize("offset,pad", [(0, 0), (4, 4), (4, 12)])
def test_gate_keeps_the_ungated_bits(rows, K, M, offset, pad, dtype):
    g, w = _rand(rows, K, dtype=dtype, seed=1), _rand(M, K, dtype=dtype, seed=2, scale=K ** -0.5)
    buf = _rand(rows * (M + pad) + offset, dtype=dtype, seed=3)
    buf[::7] = 0
    buf[3::97] = float("nan")
    buf[5::89] = float("inf")
    buf[11::83] = torch.finfo(dtype).smallest_normal / 4
    gate = buf[offset:].view(rows, M + pad)[:, :M]
    out = ops.linear_gated(g, w, gate)
    assert torch.equal(out, torch.where(gate > 0, ops.linear(g, w, None), 0))
