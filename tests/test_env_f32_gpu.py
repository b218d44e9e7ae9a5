"""The fp32 forward in one launch (csrc/cfg_env_f32.hip): against the fp32 oracle and the launches it replaces, at the edges of its
workgroups, over every form of model and input that it accepts."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from beatsaberrl_amd.config_policy import ConfigPolicy  # noqa: E402
from oracle import config_model as cm  # noqa: E402

DEV = "cuda"
TOL = 2e-6      # both sides are 3e-7 to 5e-7 from the model in 64 bits


def _model(n_layers=2, T=16, seed=5, **kw):
    spec = cm.ConfigSpec(n_layers, 128, 4, 512, T, **kw)
    p = cm.init_params(spec, seed, randomize_affine=True)
    m = ConfigPolicy.from_spec(spec, dtype="f32")
    m.load_state_dict(p)
    return spec, p, m.to(DEV)


def _out(r):
    return torch.cat([r[0].reshape(r[0].shape[0], -1), r[1][:, None]], 1).cpu()


def _close(a, b):
    assert a.shape == b.shape and (a - b).norm() <= TOL * b.norm(), ((a - b).norm() / b.norm()).item()


@pytest.mark.parametrize("mask", ["none", "uniform", "quarter_empty"])
@pytest.mark.parametrize("kw", [{}, {"act": "relu", "final_ln": True, "n_layers": 1}, {"n_layers": 3, "T": 9, "n_gears": 9}, {"T": 2, "n_gears": 1, "prop_dim": 20},
                                {"n_layers": 8, "prop_dim": 132, "obj_dim": 32}, {"prop_dim": 4, "obj_dim": 4}])
def test_one_launch_against_the_oracle(kw, mask):
    spec, p, m = _model(**kw)
    B = 37
    obs, k = cm.make_inputs(spec, B, 6, mask)
    k = torch.full_like(k, spec.T - 1) if mask == "none" else k
    got = _out(m.forward_stacked(obs.to(DEV), None if mask == "none" else k.to(DEV)))
    _close(got, _out(cm.forward(p, spec, obs, k)))
    _close(got, _out(m.forward_stacked(obs.to(DEV), k.to(DEV), route="ops")))


def test_an_envs_bits_do_not_depend_on_its_batch():
    """One and two envs per workgroup, several rounds, odd batches; the launches take over for large masked batches."""
    spec, _, m = _model()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    top = 10 * cus
    obs, k = cm.make_inputs(spec, top + 1, 3, "uniform")
    obs, k = obs.to(DEV), k.to(DEV)
    whole = _out(m.forward_stacked(obs[:top], k[:top]))
    for n in (1, 2, 3, cus - 1, cus, cus + 1, 2 * cus, 2 * cus + 1, 3 * cus + 5, top - 1):
        assert torch.equal(_out(m.forward_stacked(obs[:n], k[:n])), whole[:n]), n
    perm = torch.randperm(top, device=DEV)
    assert torch.equal(_out(m.forward_stacked(obs[:top][perm], k[:top][perm])), whole[perm.cpu()])
    _close(_out(m.forward_stacked(obs, k))[:top], whole)                       # one more env: one kernel per op
    _close(_out(m.forward_stacked(obs[:top], k[:top], route="ops")), whole)


@pytest.mark.parametrize("B", [5, 300])
def test_masked_slots_strides_and_counts(B):
    spec, _, m = _model()
    obs, k = cm.make_inputs(spec, B, 4, "uniform")
    k[0], k[1] = 0, spec.T - 1
    o, kk = obs.to(DEV), k.to(DEV)
    want = _out(m.forward_stacked(o, kk))
    junk = o.clone()
    for b in range(B):
        junk[b, spec.prop_dim + int(k[b]) * spec.obj_dim:] = float("nan" if b % 2 else "inf")
    assert torch.equal(_out(m.forward_stacked(junk, kk)), want)                # what a masked slot holds cannot reach an output
    wide = torch.full((B, spec.obs_dim + 3), float("nan"), device=DEV)
    wide[:, 1:1 + spec.obs_dim] = o                                            # rows off every 16-byte grid
    assert torch.equal(_out(m.forward_stacked(wide[:, 1:1 + spec.obs_dim], kk)), want)
    assert torch.equal(_out(m.forward_stacked(o.t().contiguous().t(), kk)), want)
    odd = torch.stack([kk, kk], 1).reshape(-1)[::2]                            # a strided count tensor
    assert torch.equal(_out(m.forward_stacked(o, odd)), want)
    past = kk.clone()
    past[0], past[1] = -3, spec.T + 5                                          # counts are clamped to the slots
    assert torch.equal(_out(m.forward_stacked(o, past)), want)


def test_new_weights_reach_the_image():
    spec, p, m = _model()
    obs, k = cm.make_inputs(spec, 9, 6, "uniform")
    m.forward_stacked(obs.to(DEV), k.to(DEV))
    q = cm.init_params(spec, 77, randomize_affine=True)
    m.load_state_dict(q)
    _close(_out(m.forward_stacked(obs.to(DEV), k.to(DEV))), _out(cm.forward(q, spec, obs, k)))
    m.prune_final = False                                                      # every row of the final block: one kernel per op
    _close(_out(m.forward_stacked(obs.to(DEV), k.to(DEV))), _out(cm.forward(q, spec, obs, k)))
