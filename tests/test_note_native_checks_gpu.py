"""What NotePolicy's native forward and update must leave to the op-by-op ones: parameters that are not plain fp32 masters,
modules that somebody listens to or has replaced."""
import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu

from beatsaberrl_amd import fp16_linear as fl  # noqa: E402
from beatsaberrl_amd.policy import NotePolicy  # noqa: E402
from oracle import note_policy_ref as nr  # noqa: E402

DEV = "cuda"


def _policy(**kw):
    torch.manual_seed(4)
    m = NotePolicy(**{**dict(embed=128, trunk_dim=256, n_blocks=2, n_heads=4, n_gears=5), **kw}).to(DEV)
    m.fp16 = True
    return m


def _obs(B=40):
    g = torch.Generator().manual_seed(B)
    obs = 0.7 * torch.randn(B, nr.OBS_DIM, generator=g)
    obs[:, nr.OFF_MASK:nr.OFF_MASK + 24] = (torch.rand(B, 24, generator=g) < 0.6).float()
    return obs.to(DEV)


def _grads(m, obs):
    m.zero_grad(set_to_none=True)
    lg, v = m.forward_stacked(obs)
    (256.0 * ((lg ** 2).mean() + (v ** 2).mean())).backward()
    return {n: p.grad for n, p in m.named_parameters()}


def test_parametrized_and_biasless_linears():
    """weight_norm holds the same weights: the same outputs to 16-bit rounding, and gradients reach what it is made of."""
    m, w, obs = _policy(), _policy(), _obs()
    with torch.no_grad():
        m.trunk_fc1.bias.zero_()
    w.load_state_dict(m.state_dict())
    want = _grads(m, obs)
    ref = m.forward_stacked(obs)
    for lin in (w.trunk_fc2, w.critic_mlp[0]):
        torch.nn.utils.parametrizations.weight_norm(lin)
    w.trunk_fc1.bias = None
    fl.bump_weights_version()
    got = _grads(w, obs)
    for a, b in zip(w.forward_stacked(obs), ref):
        assert (a - b).norm() <= 4e-3 * b.norm()
    for n in ("trunk_fc2", "critic_mlp.0"):
        assert got[f"{n}.parametrizations.weight.original1"].abs().sum() > 0
    for n in ("trunk_fc1.weight", "note_mlp.0.weight", "blocks.0.q_proj.weight"):
        assert (got[n] - want[n]).norm() <= 2e-2 * want[n].norm()


def test_masters_of_another_type_or_place_are_refused():
    """By the op-by-op forward's own checks, as before the native calls: their pointers never reach a kernel."""
    obs = _obs()
    for change in (lambda m: m.half(), lambda m: m.critic_mlp[2].cpu(), lambda m: m.critic_mlp.__setitem__(2, nn.Linear(64, 256).to(DEV))):
        m = _policy()
        _grads(m, obs)                                           # image and plan are there
        change(m)
        with pytest.raises((RuntimeError, TypeError)):
            _grads(m, obs)
        fl.bump_weights_version()
        with pytest.raises((RuntimeError, TypeError)), torch.no_grad():
            m.forward_stacked(obs)
    m = _policy()
    m.critic_mlp[1] = nn.Tanh()
    with pytest.raises(RuntimeError):
        _grads(m, obs)


def test_settings_changed_after_a_forward_are_followed():
    obs = _obs()
    m = _policy(note_geo=True)
    before = _grads(m, obs)
    lg, v = m.forward_stacked(obs)
    m.z_asinh, fresh = 3.0, _policy(note_geo=True, z_asinh=3.0)
    fresh.load_state_dict(m.state_dict())
    want = fresh.forward_stacked(obs)
    assert all(torch.equal(a, b) for a, b in zip(m.forward_stacked(obs), want)) and not torch.equal(want[0], lg)
    with torch.no_grad():
        assert torch.equal(m.forward_stacked(obs)[0], want[0])
    after, ref = _grads(m, obs), _grads(fresh, obs)
    assert all(torch.equal(after[n], ref[n]) for n in ref) and any(not torch.equal(after[n], before[n]) for n in ref)


@pytest.mark.parametrize("k", ["trunk_ln1", "trunk_ln2", "critic_ln"])
def test_layernorms_that_are_called_as_modules_keep_their_hooks_and_class(k):
    m, obs, seen = _policy(), _obs(), []
    want = [t.detach() for t in m.forward_stacked(obs)]
    h = getattr(m, k).register_forward_hook(lambda *a: seen.append(1))
    with torch.no_grad():
        m.forward_stacked(obs)
    n = len(seen)
    _grads(m, obs)                                               # the rollout's forward and the update's own
    assert n == 1 and len(seen) == 3
    h.remove()
    assert all(torch.equal(a, b) for a, b in zip(m.forward_stacked(obs), want)) and len(seen) == 3

    class Shifted(type(getattr(m, k))):
        def forward(self, x):
            return super().forward(x) + 1

    getattr(m, k).__class__ = Shifted
    assert not torch.equal(m.forward_stacked(obs)[1], want[1])
