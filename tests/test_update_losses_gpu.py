"""The update's loss kernels at inputs where they could part from torch's expression: returns that are not numbers."""
import pytest
import torch
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
