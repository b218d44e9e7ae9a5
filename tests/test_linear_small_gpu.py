"""The latency Linear kernels (direct fragments, operands shared through LDS, fp32 on the matrix pipe) and the fp32 attention
at the edges of their tiles, against fp32 / fp64 closed forms on the same operands."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

from beatsaberrl_amd import ops  # noqa: E402

DEV = "cuda"


def _rand(*s, dtype=torch.float32, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*s, generator=g) * scale).to(dtype).to(DEV)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 33, 65, 1000, 4100])
@pytest.mark.parametrize("K,M", [(64, 7), (100, 128), (16, 33), (192, 192), (320, 576), (768, 200), (960, 384), (24, 1026)])
def test_small_linear(dtype, rows, K, M):
    x, w, b = _rand(rows, K, dtype=dtype, seed=1), _rand(M, K, dtype=dtype, seed=2, scale=K ** -0.5), _rand(M, seed=3)
    res = _rand(rows, M, dtype=dtype, seed=4)
    y0 = F.linear(x.double(), w.double(), b.double())
    u = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7, torch.float32: 2.0 ** -17}[dtype]
    ok = lambda got, want, k: bool(((got.double() - want).abs() <= k * u * want.abs().clamp_min(1.0)).all())
    assert ok(ops.linear(x, w, b), y0, 1.0)
    assert ok(ops.linear(x, w, b, act="relu"), y0.relu(), 1.0)
    assert ok(ops.linear(x, w, b, act="gelu"), F.gelu(y0), 1.0)
    assert ok(ops.linear(x, w, b, residual=res), y0 + res.double(), 2.0)
    assert ok(ops.linear(x, w, b, out_dtype=torch.float32), y0, 1.0)
    if M > 3:
        p, q = ops.linear(x, w, b, out_dtype=torch.float32, split=M - 3)
        assert ok(torch.cat([p, q], 1), y0, 1.0)
    if rows % 5 == 0:
        big = torch.zeros(rows // 5, 9, M, device=DEV, dtype=dtype)
        ops.linear(x, w, b, out=big[:, 2:7])
        assert ok(big[:, 2:7].reshape(rows, M), y0, 1.0) and not bool(big[:, :2].any()) and not bool(big[:, 7:].any())
    # a row's bits do not depend on how many there are
    n = (rows + 1) // 2
    assert torch.equal(ops.linear(x[:n], w, b, residual=res[:n]), ops.linear(x, w, b, residual=res)[:n])


@pytest.mark.parametrize("B,T,TQ,H,dh", [(1, 16, 16, 4, 32), (3, 48, 48, 12, 32), (7, 29, 5, 4, 48), (5, 1, 1, 2, 64), (9, 33, 1, 3, 64), (257, 16, 16, 4, 32)])
def test_fp32_attention(B, T, TQ, H, dh):
    d = H * dh
    qkv = _rand(B, T, 3 * d, seed=5)
    q, k, v = qkv[:, :TQ, :d], qkv[..., d:2 * d], qkv[..., 2 * d:]
    g = torch.Generator().manual_seed(6)
    nv = torch.randint(0, T, (B,), generator=g, dtype=torch.int32).to(DEV)
    bias = torch.zeros(B, T, device=DEV)
    bias[torch.arange(T, device=DEV)[None] > nv[:, None]] = -16384.0
    hd = lambda t: t.double().reshape(B, -1, H, dh).transpose(1, 2)
    s = hd(q) @ hd(k).transpose(-1, -2) / dh ** 0.5 + bias.double()[:, None, None]
    ref = (s.softmax(-1) @ hd(v)).transpose(1, 2).reshape(B, TQ, d)
    for kw in ({"n_valid": nv}, {"key_bias": bias}):
        assert (ops.attn_fwd(q, k, v, H, **kw).double() - ref).abs().max() <= 4e-6
    noff = ops.token_offsets(nv, B, T - 1, torch.device(DEV))
    rows = torch.cat([qkv[:, 0], torch.cat([qkv[b, 1:1 + int(nv[b])] for b in range(B)])])
    out = ops.attn_ragged(rows[:B, :d], rows[:, d:2 * d], rows[:, 2 * d:], noff, B, 1, T - 1, H, lead_only=True)
    assert (out.double() - ref[:, 0]).abs().max() <= 4e-6


@pytest.mark.parametrize("T,TQ,H,dh", [(16, 16, 4, 32), (48, 48, 2, 32), (29, 5, 4, 48), (33, 1, 3, 64)])
@pytest.mark.parametrize("junk", [float("nan"), float("inf"), 3e38])
def test_fp32_attention_never_looks_at_masked_keys(T, TQ, H, dh, junk):
    B, d = 9, H * dh
    qkv = _rand(B, T, 3 * d, seed=5)
    nv = torch.arange(B, dtype=torch.int32) * T // B
    q = qkv[:, :TQ, :d].clone()
    want = ops.attn_fwd(q, qkv[..., d:2 * d], qkv[..., 2 * d:], H, n_valid=nv.to(DEV))
    for b in range(B):
        qkv[b, int(nv[b]) + 1:, d:] = junk
    got = ops.attn_fwd(q, qkv[..., d:2 * d], qkv[..., 2 * d:], H, n_valid=nv.to(DEV))
    assert torch.equal(got, want) and torch.isfinite(got).all()
