"""ConfigPolicy on either side of the lines at which `auto` changes its route or the form of the compacted one: precision,
agreement with the oracle, and the forms that only large batches take."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from beatsaberrl_amd.config_policy import ConfigPolicy  # noqa: E402
from oracle import config_model as cm  # noqa: E402

DEV = "cuda"


def _model(arch, dtype, seed=5, **kw):
    spec = cm.ConfigSpec(*arch, **kw)
    p = cm.init_params(spec, seed, randomize_affine=True)
    m = ConfigPolicy.from_spec(spec, dtype=dtype)
    m.load_state_dict(p)
    return spec, p, m.to(DEV)


def _out(r):
    return torch.cat([r[0].reshape(r[0].shape[0], -1), r[1][:, None]], 1).float().cpu()


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("arch", [(4, 256, 8, 1024, 32), (1, 256, 8, 1024, 32), (2, 256, 8, 512, 16), (3, 192, 4, 768, 29)])
def test_no_batch_size_rounds_the_residual_stream(arch, dtype):
    """Where the block-stack kernel covers the model, `auto` is as close to the fp32 oracle as that kernel (fp32 residual) at
    every batch size: 0.99 to 1.01 of its distance measured, 1.06 to 1.19 with a 16-bit stream."""
    spec, p, m = _model(arch, dtype)
    B = 700
    obs, k = cm.make_inputs(spec, B, 6, "uniform")
    ref = _out(cm.forward(p, spec, obs, k))
    obs, k = obs.to(DEV), k.to(DEV)
    err = lambda r: ((_out(r) - ref[:r[1].shape[0]]).norm() / ref[:r[1].shape[0]].norm()).item()
    for n in (200, 300, 512, 513, B):
        mine, blocks = err(m.forward_stacked(obs[:n], k[:n])), err(m.forward_stacked(obs[:n], k[:n], route="blocks"))
        assert mine <= 1.03 * blocks, (n, mine, blocks)


@pytest.mark.parametrize("arch,dtype", [((2, 128, 4, 512, 16), "f32"), ((2, 384, 12, 1536, 48), "f16")])
def test_masters_of_another_type_place_or_shape_are_refused(arch, dtype):
    """By pointer go LayerNorm masters in fp32 on the device and weights of the descriptor's shapes: the checks of ops.ln_fwd and
    ops.linear, which the route calls no more."""
    spec, _, m = _model(arch, dtype)
    obs, k = cm.make_inputs(spec, 9, 6, "uniform")
    obs, k = obs.to(DEV), k.to(DEV)
    m.forward_stacked(obs, k)
    m.half()
    with pytest.raises((RuntimeError, TypeError)):
        m.forward_stacked(obs, k)
    m.float().blocks[1].ln_ffn.cpu()
    m.bump_weights_version()
    with pytest.raises((RuntimeError, TypeError)):
        m.forward_stacked(obs, k)
    m.to(DEV)
    m.forward_stacked(obs, k)
    m.blocks[1].ffn[0], m.blocks[1].ffn[2] = torch.nn.Linear(m.d, 96).to(DEV), torch.nn.Linear(96, m.d).to(DEV)
    m.bump_weights_version()
    with pytest.raises(RuntimeError):
        m.forward_stacked(obs, k, route="ragged")
    if dtype == "f32":          # its op-by-op route takes any hidden width
        assert torch.equal(m.forward_stacked(obs, k)[0], m.forward_stacked(obs, k, route="ops")[0])


@pytest.mark.parametrize("arch,dtype", [((2, 128, 4, 512, 16), "f32"), ((2, 384, 12, 1536, 48), "f16")])
def test_another_eps_reaches_the_forward(arch, dtype):
    spec, _, m = _model(arch, dtype)
    obs, k = cm.make_inputs(spec, 9, 6, "uniform")
    obs, k = obs.to(DEV), k.to(DEV)
    want = m.forward_stacked(obs, k)
    for blk in m.blocks:
        blk.ln_attn.eps = blk.ln_ffn.eps = 0.5
    got = m.forward_stacked(obs, k)
    assert (got[0] - want[0]).norm() > 0.05 * want[0].norm()
    assert torch.equal(got[0], m.forward_stacked(obs, k, route="ops")[0])


@pytest.mark.parametrize("arch,dtype,B,ceil", [
    ((4, 256, 8, 1024, 32), "bf16", 449, (4.3e-2, 4.1e-2)), ((4, 256, 8, 1024, 32), "f16", 449, (5.0e-3, 6.0e-3)),
    ((6, 384, 12, 1536, 48), "f16", 235, (6.7e-3, 6.2e-3)), ((2, 192, 6, 384, 17), "bf16", 844, (4.2e-2, 2.6e-2))])
@pytest.mark.parametrize("mask", ["uniform", "quarter_empty", "none"])
def test_block_tail_form_of_the_compacted_route(arch, dtype, B, ceil, mask):
    """The first batch that takes the form (config wide's and config deep's, d = 192): distance to the fp32 oracle and to the
    rounding-emulating one (ceilings: 1.3 times the largest measured over the masks), and agreement with the form and the routes
    on the other side of the line, which are as far from that oracle."""
    spec, p, m = _model(arch, dtype, seed=41, act="gelu", final_ln=True)
    assert (B - 1) * spec.T <= m._rows_by_op(torch.float16) < B * spec.T
    obs, k = cm.make_inputs(spec, B, 42, mask)
    o, kk = obs.to(DEV), None if mask == "none" else k.to(DEV)
    got = _out(m.forward_stacked(o, kk, route="ragged"))
    ref = _out(cm.forward(p, spec, obs, k))
    em = _out(cm.forward(p, spec, obs, k, emulate=dtype, round_residual=spec.d != 256))
    e = [(got - ref).abs().max().item(), (got - em).abs().max().item()]
    print(f"\nGATE16 tail {arch} {dtype} {mask} fp32={e[0]:.3e} class={e[1]:.3e}")
    assert e[0] <= ceil[0] and e[1] <= ceil[1], e
    less = [m.forward_stacked(o[:-1], None if kk is None else kk[:-1], route=r) for r in ("ragged", "ops", None)]      # by op
    for other in less:
        assert (_out(other) - got[:-1]).abs().max().item() <= 2 * ceil[1]
    if mask != "none":      # what a masked slot holds cannot reach an output
        junk = o.clone()
        for b in range(B):
            junk[b, spec.prop_dim + int(k[b]) * spec.obj_dim:] = float("nan")
        assert torch.equal(_out(m.forward_stacked(junk, kk, route="ragged")), got)
        perm = torch.randperm(B)            # an env's bits do not depend on its neighbours
        assert torch.equal(_out(m.forward_stacked(o[perm], kk[perm], route="ragged")), got[perm])
    m.prune_final = False
    assert (_out(m.forward_stacked(o, kk, route="ragged")) - got).abs().max().item() <= 2 * ceil[1]


@pytest.mark.parametrize("arch,dtype,sizes", [((2, 256, 8, 1024, 32), "bf16", (500, 1100, 3000)), ((2, 384, 12, 1536, 48), "f16", (250, 345, 1500))])
def test_one_set_of_bits_per_form(arch, dtype, sizes):
    """Inside a form (here the tail, over its tile sizes), and on the route that covers every batch size, an env's bits do not
    depend on the batch."""
    spec, _, m = _model(arch, dtype)
    obs, k = cm.make_inputs(spec, sizes[-1], 6, "uniform")
    obs, k = obs.to(DEV), k.to(DEV)
    tails = [_out(m.forward_stacked(obs[:n], k[:n], route="ragged")) for n in sizes]
    assert all(n * spec.T > m._rows_by_op(torch.float16) for n in sizes) and all(torch.equal(t, tails[-1][:n]) for n, t in zip(sizes, tails))
    route = "blocks" if spec.d == 256 else "ops"
    whole = _out(m.forward_stacked(obs, k, route=route))
    assert all(torch.equal(_out(m.forward_stacked(obs[:n], k[:n], route=route)), whole[:n]) for n in (1, 9, *sizes[:2]))


@pytest.mark.parametrize("arch,dtype,B", [((2, 128, 4, 512, 16), "f32", 65), ((2, 256, 8, 1024, 32), "bf16", 300), ((2, 256, 8, 1024, 32), "bf16", 600),
                                          ((2, 384, 12, 1536, 48), "f16", 40), ((2, 384, 12, 1536, 48), "f16", 400)])
def test_compacted_route_replays_from_a_captured_graph(arch, dtype, B):
    """The row count stays on the device: one graph serves every mask of its batch size."""
    spec, _, m = _model(arch, dtype)
    obs, k = cm.make_inputs(spec, B, 1, "uniform")
    obs, k = obs.to(DEV), k.to(DEV)
    assert m.auto_route(B) == "ragged"
    m.forward_stacked(obs, k)                                    # replicas and images
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        lg, v = m.forward_stacked(obs, k)
    for seed, mask in ((2, "uniform"), (3, "none"), (4, "quarter_empty")):
        o, kk = cm.make_inputs(spec, B, seed, mask)
        obs.copy_(o.to(DEV)); k.copy_(kk.to(DEV))
        g.replay()
        got = (lg.clone(), v.clone())
        want = m.forward_stacked(o.to(DEV), kk.to(DEV))          # eager work between the replays
        torch.cuda.synchronize()
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), mask


@pytest.mark.parametrize("dtype,tol", [("f16", 4e-3), ("bf16", 2e-2)])
@pytest.mark.parametrize("B", [1, 2, 5, 17, 33, 64, 129])
def test_by_op_fp32_stream_at_the_edges_of_its_tiles(B, dtype, tol):
    """1 to ~2000 rows with every remainder of the 16-, 32- and 64-row tiles among them, against the block-stack kernel (the same
    rounding points; tolerance: both are within the type's class of the fp32 model)."""
    spec, _, m = _model((3, 256, 8, 544, 32), dtype)
    obs, k = cm.make_inputs(spec, B, B, "uniform")
    obs, k = obs.to(DEV), k.to(DEV)
    a, b = _out(m.forward_stacked(obs, k, route="ragged")), _out(m.forward_stacked(obs, k, route="blocks"))
    assert (a - b).norm() <= tol * b.norm()
    full = _out(m.forward_stacked(obs, None, route="ragged"))
    m.prune_final = False
    assert (_out(m.forward_stacked(obs, None, route="ragged")) - full).norm() <= tol * full.norm()
