"""Host-side contract of ConfigPolicy, no GPU."""
import torch

from beatsaberrl_amd.config_policy import ConfigPolicy


def test_workspace_query_belongs_to_the_descriptor():
    m = ConfigPolicy()
    m._desc(torch.float16)
    m._ws_rows = (64, 1 << 20)              # as a forward of 64 envs leaves it
    m._desc(torch.float16)
    assert m._ws_rows == (64, 1 << 20)
    m.pack_short = False
    m._desc(torch.float16)
    assert m._ws_rows[0] != 64


def test_compacted_route_leaves_another_eps_to_the_ops():
    for arch in (dict(dtype="f32"), dict(n_layers=3, d=384, n_heads=12, ffn=1536, T=48, final_ln=True)):
        m = ConfigPolicy(**arch)
        assert m.ragged_supported()
        for ln in (m.blocks[1].ln_attn, m.blocks[0].ln_ffn, m.final_ln):
            if ln is not None:
                ln.eps = 1e-6
                assert not m.ragged_supported()
                ln.eps = 1e-5
        assert m.ragged_supported()
