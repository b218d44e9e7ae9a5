"""Where the block tail's loops over hidden chunks and projection stages go round in pairs (block_tail.h): an odd number of chunks gives
the bits of the next even one whose last 32 hidden features are zero, and the fewest projected columns those of the most."""
import math

import pytest
import torch

from beatsaberrl_amd import ops
from test_ops_gpu import _rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("act", ["relu", "gelu"])
@pytest.mark.parametrize("d", [192, 256, 384])
@pytest.mark.parametrize("rows", [1, 515, 20001])
def test_odd_chunk_counts_and_the_fewest_columns(rows, d, act, dtype):
    att, x = _rand(rows, d, dtype=dtype, seed=1), _rand(rows, d, dtype=dtype, seed=2)
    wo, bo = _rand(d, d, dtype=dtype, seed=3, scale=1 / math.sqrt(d)), 0.3 * _rand(d, seed=4)
    wn, bn = _rand(3 * d, d, dtype=dtype, seed=5, scale=1 / math.sqrt(d)), 0.3 * _rand(3 * d, seed=6)
    l2, l1 = (1 + 0.2 * _rand(d, seed=7), 0.2 * _rand(d, seed=8), 1e-5), (1 + 0.2 * _rand(d, seed=9), 0.2 * _rand(d, seed=10), 1e-5)
    for F in (96, 544):
        w0, b0, w2 = _rand(F + 32, d, dtype=dtype, seed=11, scale=0.06), 0.3 * _rand(F + 32, seed=12), _rand(d, F + 32, dtype=dtype, seed=13, scale=0.05)
        b2 = 0.3 * _rand(d, seed=14)
        w0[F:], b0[F:], w2[:, F:] = 0, 0, 0
        out = []
        for f, n_next in ((F, 64), (F, 3 * d), (F + 32, 3 * d)):
            assert ops.block_tail_supported(d, f, dtype, n_next)
            img = ops.block_tail_pack(wo, bo, w0[:f].contiguous(), b0[:f].contiguous(), w2[:, :f].contiguous(), b2, wn[:n_next].contiguous(), bn[:n_next].contiguous())
            out.append(ops.block_tail(att, x, img, f, l2, l1, n_next, rows, None, act))
        for got in out[:2]:
            assert torch.equal(got[0], out[2][0]) and torch.equal(got[1], out[2][1])
            assert torch.equal(got[2], out[2][2][:, :got[2].shape[1]])
