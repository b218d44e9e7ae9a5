"""The compacted token stream: offsets, tokenizer, attention and the one-kernel block tail on ragged batches, and the
ConfigPolicy route built on them, against torch closed forms and the CPU oracle."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

from beatsaberrl_amd import ops  # noqa: E402
from beatsaberrl_amd.config_policy import ConfigPolicy  # noqa: E402
from oracle import config_model as cm  # noqa: E402

DEV = "cuda"


def _rand(*s, dtype=torch.float32, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*s, generator=g) * scale).to(dtype).to(DEV)


def _counts(B, opt, seed=3):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, opt + 1, (B,), generator=g, dtype=torch.int32)


@pytest.mark.parametrize("B", [1, 3, 64, 1023, 1024, 4097, 70001])
def test_token_offsets(B):
    n = _counts(B, 47) * 2 - 20                      # some below 0, some above the bound: clamped
    noff = ops.token_offsets(n.to(DEV), B, 47, torch.device(DEV)).cpu()
    want = torch.cat([torch.zeros(1, dtype=torch.int64), n.clamp(0, 47).long().cumsum(0)])
    assert torch.equal(noff.long(), want)
    full = ops.token_offsets(None, B, 31, torch.device(DEV)).cpu()
    assert torch.equal(full.long(), torch.arange(B + 1) * 31)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lead,opt,H,dh", [(1, 31, 8, 32), (1, 47, 12, 32), (5, 24, 4, 48), (1, 3, 4, 32)])
def test_attn_ragged(dtype, lead, opt, H, dh):
    B, d = 37, H * dh
    n = _counts(B, opt)
    n[0], n[1] = 0, opt
    noff = ops.token_offsets(n.to(DEV), B, opt, torch.device(DEV))
    rows = lead * B + int(n.sum())
    qkv = _rand(B * (lead + opt), 3 * d, dtype=dtype, seed=5)
    qkv[rows:] = float("nan")                        # rows past the stream are never read
    q, k, v = qkv[:, :d], qkv[:, d:2 * d], qkv[:, 2 * d:]
    bias = (_rand(B * opt, dtype=dtype, seed=6) * 0.5) if lead == 5 else None
    out = ops.attn_ragged(q, k, v, noff, B, lead, opt, H, opt_bias=bias)
    outl = ops.attn_ragged(q[:lead * B], k, v, noff, B, lead, opt, H, lead_only=True, opt_bias=bias)
    off = noff.cpu().tolist()
    tol = 2e-3 if dtype is torch.float16 else 1.6e-2
    for b in range(B):
        idx = list(range(lead * b, lead * b + lead)) + list(range(lead * B + off[b], lead * B + off[b + 1]))
        i = torch.tensor(idx, device=DEV)
        qq, kk, vv = (t[i].float().view(len(idx), H, dh).transpose(0, 1) for t in (q, k, v))
        s = qq @ kk.transpose(1, 2) / dh ** 0.5
        if bias is not None:
            s[:, :, lead:] += bias[off[b]:off[b + 1]].float()
        ref = (torch.softmax(s, -1) @ vv).transpose(0, 1).reshape(len(idx), d)
        assert (out[i].float() - ref).abs().max() <= tol
        assert (outl[lead * b:lead * b + lead].float() - ref[:lead]).abs().max() <= tol


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d,Fh,act", [(192, 768, "relu"), (256, 1024, "gelu"), (384, 1536, "gelu"), (192, 64, "gelu"), (256, 96, "relu")])
@pytest.mark.parametrize("n", [1, 63, 700, 35000])
def test_block_tail(dtype, d, Fh, act, n):
    if n == 35000 and Fh in (64, 96):
        pytest.skip("the small hidden widths are covered at the small row counts")
    if not ops.block_tail_supported(d, Fh, dtype, 3 * d):
        pytest.skip("image shorter than the ring")
    mk = lambda *s, seed, scale=1.0, dt=torch.float32: _rand(*s, seed=seed, scale=scale, dtype=dt)
    lead = (n + 3) // 4
    pad = 50
    x, att = mk(n + pad, d, seed=1, dt=dtype), mk(n + pad, d, seed=2, dt=dtype)
    wo, w0, w2, wn = (mk(d, d, seed=3, scale=d ** -0.5, dt=dtype), mk(Fh, d, seed=4, scale=d ** -0.5, dt=dtype),
                      mk(d, Fh, seed=5, scale=Fh ** -0.5, dt=dtype), mk(3 * d, d, seed=6, scale=d ** -0.5, dt=dtype))
    bo, b0, b2, bn = mk(d, seed=7), mk(Fh, seed=8), mk(d, seed=9), mk(3 * d, seed=10)
    l2, l1 = (mk(d, seed=11) + 1, mk(d, seed=12), 1e-5), (mk(d, seed=13) + 1, mk(d, seed=14), 1e-5)
    img = ops.block_tail_pack(wo, bo, w0, b0, w2, b2, wn, bn)
    extra = torch.tensor([n - lead], dtype=torch.int32, device=DEV)
    xo, ho, qo = ops.block_tail(att, x, img, Fh, l2, l1, 3 * d, lead, extra, act, ho_rows=lead)
    xd, hd, qd = ops.block_tail(att[:n], x[:n], img, Fh, l2, l1, 3 * d, n, None, act)
    assert torch.equal(xo[:n], xd) and torch.equal(ho, hd[:lead]) and torch.equal(qo[:n], qd)
    r = lambda t: t.to(dtype).float()
    x1 = r(x[:n].float() + att[:n].float() @ wo.float().t() + bo)
    h2 = r(F.layer_norm(x1, (d,), *l2))
    hid = h2 @ w0.float().t() + b0
    hid = r(F.gelu(hid) if act == "gelu" else F.relu(hid))
    ref = x1 + hid @ w2.float().t() + b2
    u = 2.0 ** -10 if dtype is torch.float16 else 2.0 ** -7
    lim = lambda got, want, k: ((got.float() - want).abs() <= k * u * want.abs().clamp_min(1.0)).all()
    # an ulp of x1, h2 or a hidden value moves with the summation order now and then: few values, by a few ulps
    assert lim(xd, ref, 8.0) and (xd.float() - ref).square().mean().sqrt() <= u, (xd.float() - ref).abs().max()
    href = F.layer_norm(xd.float(), (d,), *l1)
    assert lim(hd, href, 2.0), (hd.float() - href).abs().max()
    qref = hd.float() @ wn.float().t() + bn
    assert lim(qd, qref, 2.0), (qd.float() - qref).abs().max()
    img0 = ops.block_tail_pack(None, None, None, None, None, None, wn, bn)
    _, hl, ql = ops.block_tail(None, x, img0, 0, None, l1, 3 * d, lead, extra, None, ho_rows=lead)
    hr = F.layer_norm(x[:n].float(), (d,), *l1)
    assert lim(hl, hr[:lead], 2.0)
    assert lim(ql[:n], r(hr) @ wn.float().t() + bn, 12.0)
    if n <= 700:        # without a LayerNorm behind: the same rows
        img1 = ops.block_tail_pack(wo, bo, w0, b0, w2, b2)
        xl, h_none, q_none = ops.block_tail(att[:n], x[:n], img1, Fh, l2, None, 0, n, None, act)
        assert h_none is None and q_none is None and torch.equal(xl, xd)


@pytest.mark.parametrize("arch,dtype,ceil", [
    ((4, 256, 8, 1024, 32), "bf16", (9.6e-2, 6.8e-2)), ((4, 256, 8, 1024, 32), "f16", (1.2e-2, 8e-3)),
    ((6, 384, 12, 1536, 48), "f16", (2.0e-2, 1.4e-2)), ((1, 192, 4, 768, 29), "f16", (6e-3, 5e-3)), ((2, 192, 6, 384, 17), "bf16", (6e-2, 4e-2))])
@pytest.mark.parametrize("mask", ["uniform", "quarter_empty", "none"])
def test_ragged_route(arch, dtype, ceil, mask):
    L, d, H, ffn, T = arch
    spec = cm.ConfigSpec(L, d, H, ffn, T, act="gelu", final_ln=True)
    p = cm.init_params(spec, 41, randomize_affine=True)
    m = ConfigPolicy.from_spec(spec, dtype=dtype)
    m.load_state_dict(p)
    m = m.to(DEV)
    B = 131
    obs, k = cm.make_inputs(spec, B, 42, mask)
    lg, v = m.forward_stacked(obs.to(DEV), None if mask == "none" else k.to(DEV), route="ragged")
    ref, rv = cm.forward(p, spec, obs, k)
    em, ev = cm.forward(p, spec, obs, k, emulate=dtype, round_residual=True)
    e = [(lg.cpu() - ref).abs().max().item(), (lg.cpu() - em).abs().max().item(), (v.cpu() - ev).abs().max().item()]
    print(f"\nGATE16 ragged {arch} {dtype} {mask} fp32={e[0]:.3e} class={e[1]:.3e} value={e[2]:.3e}")
    assert e[0] <= ceil[0] and max(e[1:]) <= ceil[1], e
    # what a masked slot holds cannot reach an output, an env's bits do not depend on its neighbours, and the pruned final
    # block is the full one's token 0
    if mask != "none":
        junk = obs.clone()
        for b in range(B):
            junk[b, spec.prop_dim + int(k[b]) * spec.obj_dim:] = float("nan")
        lg2, v2 = m.forward_stacked(junk.to(DEV), k.to(DEV), route="ragged")
        assert torch.equal(lg, lg2) and torch.equal(v, v2)
        lg3, v3 = m.forward_stacked(obs[40:77].to(DEV), k[40:77].to(DEV), route="ragged")
        assert torch.equal(lg[40:77], lg3) and torch.equal(v[40:77], v3)
    m.prune_final = False
    lg4, _ = m.forward_stacked(obs.to(DEV), None if mask == "none" else k.to(DEV), route="ragged")
    assert (lg4 - lg).abs().max().item() <= ceil[1]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("act,Fh", [("gelu", 1024), ("relu", 96)])
@pytest.mark.parametrize("n", [1, 63, 700, 35000])
@pytest.mark.parametrize("form", ["into", "along", "out of"])
def test_block_tail_fp32_stream(dtype, act, Fh, n, form):
    """The forms that carry the residual stream in fp32 (d = 256): into it (16-bit x), along it, out of it (no LayerNorm behind).
    Neither x1 nor an fp32 xo is rounded; h2, the hidden, ho and qo are."""
    d = 256
    mk = lambda *s, seed, scale=1.0, dt=torch.float32: _rand(*s, seed=seed, scale=scale, dtype=dt)
    lead, last = (n + 3) // 4, form == "out of"
    x, att = mk(n + 5, d, seed=1, dt=dtype if form == "into" else torch.float32), mk(n + 5, d, seed=2, dt=dtype)
    wo, w0, w2, wn = (mk(d, d, seed=3, scale=d ** -0.5, dt=dtype), mk(Fh, d, seed=4, scale=d ** -0.5, dt=dtype),
                      mk(d, Fh, seed=5, scale=Fh ** -0.5, dt=dtype), mk(3 * d, d, seed=6, scale=d ** -0.5, dt=dtype))
    bo, b0, b2, bn = mk(d, seed=7), mk(Fh, seed=8), mk(d, seed=9), mk(3 * d, seed=10)
    l2, l1 = (mk(d, seed=11) + 1, mk(d, seed=12), 1e-5), (mk(d, seed=13) + 1, mk(d, seed=14), 1e-5)
    img = ops.block_tail_pack(wo, bo, w0, b0, w2, b2, *(() if last else (wn, bn)))
    extra = torch.tensor([n - lead], dtype=torch.int32, device=DEV)
    xo, ho, qo = ops.block_tail(att, x, img, Fh, l2, None if last else l1, 0 if last else 3 * d, lead, extra, act, ho_rows=lead,
                                xo_dtype=dtype if last else torch.float32)
    r = lambda t: t.to(dtype).float()
    u = 2.0 ** -10 if dtype is torch.float16 else 2.0 ** -7
    x1 = x[:n].float() + att[:n].float() @ wo.float().t() + bo
    h2 = F.layer_norm(x1, (d,), *l2)
    hid = r(h2) @ w0.float().t() + b0
    hid = r(F.gelu(hid) if act == "gelu" else F.relu(hid))
    ref = x1 + hid @ w2.float().t() + b2
    lim = lambda got, want, k: ((got.float() - want).abs() <= k * u * want.abs().clamp_min(1.0)).all()
    e = (xo[:n].float() - ref).abs()
    if last:
        assert lim(xo[:n], ref, 8.0)
    else:
        # fp32 out: what is left are single ulps of h2 and of the hidden that moved with the summation order.  One of h2
        # (u h2 at most) reaches xo through two matrices of unit gain; the typical value has none and shows fp32 sums
        assert e.max() <= 8.0 * u and e.median() <= 0.2 * u, (e.max().item(), e.median().item())
        hr = F.layer_norm(xo[:n], (d,), *l1)                      # both LayerNorms see unrounded rows
        assert lim(ho, hr[:lead], 1.0) and lim(qo[:n], r(hr) @ wn.float().t() + bn, 12.0)
