"""The few-envs form of the compacted route at d = 384 (csrc/cfg_env_rows.hip): precision, the edges of its row tiles, and every form of
input that it accepts."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from beatsaberrl_amd.config_policy import ConfigPolicy  # noqa: E402
from oracle import config_model as cm  # noqa: E402

DEV = "cuda"
# both sides round at the same points: their distance stays below what either has to the fp32 model (9e-4 | 7.4e-3 at six blocks)
CLASS = {"f16": 1.5e-3, "bf16": 1.2e-2}


def _model(n_layers=2, T=48, dtype="f16", seed=5, **kw):
    spec = cm.ConfigSpec(n_layers, 384, 12, 1536, T, **kw)
    p = cm.init_params(spec, seed, randomize_affine=True)
    m = ConfigPolicy.from_spec(spec, dtype=dtype)
    m.load_state_dict(p)
    return spec, p, m.to(DEV)


def _out(r):
    return torch.cat([r[0].reshape(r[0].shape[0], -1), r[1][:, None]], 1).float().cpu()


def _rel(a, b):
    return ((a - b).norm() / b.norm()).item()


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("kw", [{"n_layers": 6}, {"act": "relu", "final_ln": True, "n_layers": 1}, {"n_layers": 3, "T": 17, "n_gears": 9, "prop_dim": 132},
                                {"T": 33, "prop_dim": 21, "obj_dim": 5}, {"T": 2, "n_gears": 1, "obj_dim": 32}])
def test_two_launches_per_block_against_the_oracle(kw, dtype):
    spec, p, m = _model(dtype=dtype, **kw)
    B = 61
    obs, k = cm.make_inputs(spec, B, 6, "uniform")
    ref = _out(cm.forward(p, spec, obs, k))
    o, kk = obs.to(DEV), k.to(DEV)
    got, ops = _out(m.forward_stacked(o, kk)), _out(m.forward_stacked(o, kk, route="ops"))
    assert _rel(got, ref) <= 1.15 * _rel(ops, ref), (_rel(got, ref), _rel(ops, ref))
    assert _rel(got, ops) <= CLASS[dtype]
    m.prune_final = False                                                    # every row of the final block: one kernel per op
    assert _rel(got, _out(m.forward_stacked(o, kk))) <= CLASS[dtype]


@pytest.mark.parametrize("B", [1, 2, 31, 32, 33, 97])
def test_edges_of_the_row_tiles(B):
    """Envs of 1, 15 .. 17, 31 .. 33 and 47 / 48 rows; totals around multiples of 32; an env's bits do not depend on its neighbours,
    and what a masked slot holds cannot reach an output."""
    spec, _, m = _model(3, act="gelu", final_ln=True)
    obs, k = cm.make_inputs(spec, B, B, "uniform")
    for i, n in enumerate([0, 15, 16, 14, 31, 32, 30, 47, 46][:B]):
        k[i] = n
    o, kk = obs.to(DEV), k.to(DEV)
    got = _out(m.forward_stacked(o, kk))
    assert _rel(got, _out(m.forward_stacked(o, kk, route="ops"))) <= CLASS["f16"]
    junk = o.clone()
    for b in range(B):
        junk[b, spec.prop_dim + int(k[b]) * spec.obj_dim:] = float("nan" if b % 2 else "inf")
    assert torch.equal(_out(m.forward_stacked(junk, kk)), got)
    perm = torch.randperm(B)
    assert torch.equal(_out(m.forward_stacked(o[perm], kk[perm])), got[perm])
    assert all(torch.equal(_out(m.forward_stacked(o[b:b + 1], kk[b:b + 1])), got[b:b + 1]) for b in range(min(B, 9)))
    full = _out(m.forward_stacked(o))
    assert torch.equal(_out(m.forward_stacked(o, torch.full_like(kk, spec.T + 3))), full)      # counts are clamped to the slots
    assert torch.equal(_out(m.forward_stacked(o, torch.full_like(kk, spec.T - 1))), full)


def test_strides_and_types_of_the_observations():
    spec, _, m = _model()
    B = 40
    obs, k = cm.make_inputs(spec, B, 4, "quarter_empty")
    o, kk = obs.half().float().to(DEV), k.to(DEV)
    want = _out(m.forward_stacked(o, kk))
    assert torch.equal(_out(m.forward_stacked(o.half(), kk)), want) and torch.equal(_out(m.forward_stacked(o.double(), kk)), want)
    wide = torch.full((B, spec.obs_dim + 3), float("nan"), device=DEV)
    wide[:, 1:1 + spec.obs_dim] = o
    assert torch.equal(_out(m.forward_stacked(wide[:, 1:1 + spec.obs_dim], kk)), want)
    assert torch.equal(_out(m.forward_stacked(o.t().contiguous().t(), kk)), want)


def test_lines_of_auto():
    """`auto` keeps the form past the line of route="ragged"; both sides of its own lines agree, and its bits are one set below them."""
    spec, _, m = _model()
    with_counts = m.FEW_ENVS
    obs, k = cm.make_inputs(spec, with_counts + 1, 3, "uniform")
    o, kk = obs.to(DEV), k.to(DEV)
    few = _out(m.forward_stacked(o[:with_counts], kk[:with_counts]))
    assert torch.equal(_out(m.forward_stacked(o[:234], kk[:234], route="ragged")), few[:234])
    assert torch.equal(_out(m.forward_stacked(o[:301], kk[:301])), few[:301])
    assert _rel(_out(m.forward_stacked(o, kk))[:with_counts], few) <= CLASS["f16"]
    assert _rel(_out(m.forward_stacked(o[:235]))[:234], _out(m.forward_stacked(o[:234]))) <= CLASS["f16"]


def test_masters_off_a_16_byte_grid():
    """Vectors that the kernels cannot read in 16-byte pieces: one kernel per op."""
    spec, _, m = _model()
    obs, k = cm.make_inputs(spec, 9, 6, "uniform")
    want = _out(m.forward_stacked(obs.to(DEV), k.to(DEV)))
    flat = torch.empty(spec.d + 1, device=DEV)
    flat[1:] = m.blocks[1].ln_ffn.weight.detach()
    m.blocks[1].ln_ffn.weight.data = flat[1:]
    m.bump_weights_version()
    assert _rel(_out(m.forward_stacked(obs.to(DEV), k.to(DEV))), want) <= CLASS["f16"]
