"""The fused config forward with no more packed tiles than SIMDs, one to a wave (cfg_forward.hip): an env's bits are those it has in a batch
of many rounds, on both sides of the line and whatever the tiles hold."""
import pytest
import torch

from beatsaberrl_amd.config_policy import ConfigPolicy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", ["gelu", "relu"])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_an_env_keeps_its_bits(dtype, act):
    torch.manual_seed(5)
    simds = 4 * torch.cuda.get_device_properties(0).multi_processor_count
    with torch.device("cuda"):
        m = ConfigPolicy(act=act, dtype=dtype)
    many = 12 * simds
    obs = torch.randn(many, m.obs_dim, device="cuda")
    for low, high, batches in ((0, 16, (simds + 1, simds + 3, 3 * simds // 2, 7 * simds // 4)), (15, 16, (simds + 1, 2 * simds)),
                               (0, 1, (simds + 5, 4 * simds - 1, 4 * simds, 4 * simds + 1)), (4, 8, (2 * simds, 2 * simds + 1))):
        n_valid = torch.randint(low, high, (many,), device="cuda", dtype=torch.int32)
        with torch.no_grad():
            want = m.forward_stacked(obs, n_valid)
            for B in batches:
                got = m.forward_stacked(obs[:B], n_valid[:B].contiguous())
                for g, w in zip(got, want):
                    assert torch.equal(g, w[:B]), (low, high, B)
