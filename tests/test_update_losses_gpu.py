"""The update's loss kernels at inputs and under transforms where they could part from torch's expression."""
import pytest
import torch
import torch.autograd.forward_ad  # noqa: F401
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

from beatsaberrl_amd.policy import hl_loss, hl_target  # noqa: E402

DEV = "cuda"


def _bins(B, K, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    centers = torch.linspace(-6.0, 6.0, K, device=DEV)
    return (2.0 * torch.randn(B, K, generator=g, device=DEV)).requires_grad_(True), 4.0 * torch.randn(B, generator=g, device=DEV), centers, 0.75 * 12.0 / (K - 1)


def _hl_torch(logits, v, centers, sigma):
    return -(hl_target(v, centers, sigma) * F.log_softmax(logits.float(), dim=-1)).sum(-1).mean()


@pytest.mark.parametrize("K", [2, 101, 129, 512])
def test_hl_loss_of_returns_that_are_not_finite(K):
    """NaN reaches the loss and its row's gradient, as in torch's expression; the infinities are clamped into the support."""
    x, v, centers, sigma = _bins(7, K)
    v[0], v[1] = float("inf"), float("-inf")
    loss = hl_loss(x, v, centers, sigma)
    want = _hl_torch(x, v, centers, sigma)
    assert torch.isfinite(loss) and abs(loss.item() - want.item()) <= 2e-5 * abs(want.item())
    v[3] = float("nan")
    loss = hl_loss(x, v, centers, sigma)
    assert torch.isnan(loss) and torch.isnan(_hl_torch(x, v, centers, sigma))
    g, = torch.autograd.grad(loss, x)
    assert torch.isnan(g).any(-1).tolist() == [i == 3 for i in range(7)]


def test_hl_loss_arguments_the_kernel_does_not_cover():
    """A tensor on the host is refused, never handed to the kernel; other shapes get torch's broadcasting and errors."""
    x, v, centers, sigma = _bins(6, 101)
    for args in ((x, v.cpu(), centers, sigma), (x, v, centers.cpu(), sigma), (x, v, centers[:50], sigma), (x, v[:5], centers, sigma)):
        with pytest.raises(RuntimeError):
            hl_loss(*args)
    one = x[:, :1].detach()
    assert torch.equal(hl_loss(one, v, centers, sigma), _hl_torch(one, v, centers, sigma))            # logits broadcast over the bins
    s = torch.tensor(sigma, device=DEV, requires_grad=True)                                           # a width that is learned
    g, = torch.autograd.grad(hl_loss(x, v, centers, s), s)
    assert torch.isfinite(g) and g.item() != 0.0
    assert torch.isnan(hl_loss(x[:0], v[:0], centers, sigma))


def test_hl_loss_differentiated_twice_and_under_transforms():
    """What torch's expression gives: a Hessian-vector product, grad / vmap / jvp of torch.func, a forward-mode tangent."""
    x, v, centers, sigma = _bins(9, 101)
    u = torch.randn(9, 101, device=DEV)
    hvp = []
    for f in (hl_loss, _hl_torch):
        g, = torch.autograd.grad(f(x, v, centers, sigma), x, create_graph=True)
        hvp.append((g.detach(), torch.autograd.grad((g * u).sum(), x)[0]))
    for got, want in zip(*hvp):         # fp32 softmax, erf and their differences: a few ulp of values up to 1 / B
        assert torch.allclose(got, want, atol=3e-5 / 9)
    f, t = (lambda a: hl_loss(a, v, centers, sigma)), (lambda a: _hl_torch(a, v, centers, sigma))
    y = x.detach()
    assert torch.equal(torch.func.grad(f)(y), torch.func.grad(t)(y))
    batch = torch.stack([y, 2 * y, -y])
    assert torch.equal(torch.func.vmap(f)(batch), torch.func.vmap(t)(batch))
    assert all(torch.equal(a, b) for a, b in zip(torch.func.jvp(f, (y,), (u,)), torch.func.jvp(t, (y,), (u,))))
    with torch.autograd.forward_ad.dual_level():
        d = torch.autograd.forward_ad.make_dual(y, u)
        a, b = (torch.autograd.forward_ad.unpack_dual(g(d)).tangent for g in (f, t))
        assert torch.equal(a, b)


def test_heads_logp_differentiated_twice():
    from beatsaberrl_amd.autograd_ops import HeadsLogpFn

    def torch_form(x, a):
        ls = torch.log_softmax(x, -1)
        return ls.gather(-1, a.unsqueeze(-1)).squeeze(-1).sum(-1), -(ls.exp() * ls).sum(-1).sum(-1)

    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(5, 29, 7, generator=g, device=DEV).transpose(0, 1).contiguous().transpose(0, 1).requires_grad_(True)      # rows out of order
    a, w, u = (torch.randint(0, 7, (5, 29), generator=g, device=DEV), torch.randn(2, 5, generator=g, device=DEV),
               torch.randn(5, 29, 7, generator=g, device=DEV))
    out = []
    for f in (lambda x, a: HeadsLogpFn.apply(x, a)[:2], torch_form):
        lp, ent = f(x, a)
        d, = torch.autograd.grad((w[0] * lp + w[1] * ent).sum(), x, create_graph=True)
        d1, = torch.autograd.grad(lp.sum(), x, retain_graph=True)
        out.append((d.detach(), d1, torch.autograd.grad((d * u).sum(), x, retain_graph=True)[0],
                    torch.autograd.grad(lp, x, torch.eye(5, device=DEV), retain_graph=True, is_grads_batched=True)[0]))
    for got, want in zip(*out):
        assert torch.allclose(got, want, atol=1e-5)


@pytest.mark.parametrize("bad", [-1, 5, 2 ** 32 + 1, -2 ** 40])
def test_update_of_an_action_outside_its_head(bad):
    """NaN log-probability and gradient for that env alone; fewer rows of actions are torch's case, as before the kernels."""
    from beatsaberrl_amd.autograd_ops import HeadsLogpFn
    x = torch.randn(6, 29, 5, device=DEV, requires_grad=True)
    a = torch.randint(0, 5, (6, 29), device=DEV)
    a[2, 11] = bad
    lp, ent, _ = HeadsLogpFn.apply(x, a)
    assert torch.isnan(lp).tolist() == [i == 2 for i in range(6)] and torch.isfinite(ent).all()
    g, = torch.autograd.grad(lp.sum() + ent.sum(), x)
    assert torch.isnan(g[2, 11]).all() and torch.isnan(g).sum() == 5


def test_update_actions_of_other_shapes():
    from beatsaberrl_amd.policy import NotePolicy
    from oracle import note_policy_ref as nr
    m = NotePolicy(embed=128, trunk_dim=64, n_blocks=1, n_heads=4, n_gears=5).to(DEV)
    m.fp16 = True
    obs, a = torch.randn(6, nr.OBS_DIM, device=DEV), torch.randint(0, 5, (6, 29), device=DEV)
    _, lp, ent, _ = m.get_action_and_value(obs, a)
    _, lp4, ent4, _ = m.get_action_and_value(obs, a[:4])
    assert lp4.shape == (4,) and torch.allclose(lp4, lp[:4], atol=1e-5) and torch.allclose(ent4, ent, atol=1e-5)
    assert lp4.requires_grad
    for wrong in (a.cpu(), a[:, :, None].expand(6, 29, 2), torch.zeros(7, 29, device=DEV)):
        with pytest.raises((RuntimeError, TypeError)):
            m.get_action_and_value(obs, wrong)
