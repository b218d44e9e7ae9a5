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
