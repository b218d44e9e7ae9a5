"""Two envs per wave (blocks_pair.hip): a large batch's forward at d = 192 against the same envs in batches that the one-env kernels take.
The same bits, whatever the share of attendable notes makes of the pairs: two to a wave, one to a wave, or all of it left to the other
kernel; at the edges of the chunks in which envs are paired; and an env whose values are not finite stays alone with that."""
import pytest
import torch

from beatsaberrl_amd.obs_layout import N_NOTE_SLOTS, OBS_DIM, OFF_NOTE_MASK
from beatsaberrl_amd.policy import NotePolicy

pytestmark = pytest.mark.gpu


def _share(kind, B):
    rows = torch.rand(B, 1, device="cuda")
    return {"none": 0 * rows, "all": 0 * rows + 1, "usual": 0 * rows + 0.6, "some alone": 0 * rows + 0.75, "mixed": rows.round()}[kind]


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("blocks,ffn", [(1, 2), (2, 4), (3, 1)])
def test_pairs_give_each_env_its_bits(blocks, ffn, dtype):
    torch.manual_seed(blocks)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    with torch.device("cuda"):
        m = NotePolicy(embed=192, trunk_dim=384, n_blocks=blocks, n_heads=4, n_gears=5, ffn_mult=ffn)
    with torch.no_grad():
        for p in m.parameters():
            if p.dim() == 1:
                p.add_(0.1 * torch.randn_like(p))
    m.fp16, m.stream_dtype = True, torch.float16 if dtype == "f16" else torch.bfloat16
    m.flatten_fp16()
    step = 2 * cus
    for kind, extra in (("usual", 1), ("usual", 63), ("usual", 4 * cus + 1), ("mixed", 130), ("some alone", 8 * cus + 7), ("none", 64), ("all", 65), ("usual", 12 * cus + 2)):
        B = 4 * cus + extra
        obs = 0.7 * torch.randn(B, OBS_DIM, device="cuda")
        obs[:, OFF_NOTE_MASK:OFF_NOTE_MASK + N_NOTE_SLOTS] = (torch.rand(B, N_NOTE_SLOTS, device="cuda") < _share(kind, B)).float()
        bad = torch.arange(7, B, 211, device="cuda")
        obs[bad, 0] = float("nan")
        obs[bad + 1 if bad[-1] + 1 < B else bad - 1, 1] = float("inf")
        with torch.no_grad():
            got = m.forward_stacked(obs)
            want = [torch.cat(w) for w in zip(*(m.forward_stacked(o) for o in obs.split(step)))]
        for g, w in zip(got, want):
            assert torch.equal(g.isnan(), w.isnan()), (kind, B)
            assert torch.equal(g.nan_to_num(), w.nan_to_num()), (kind, B, (g - w).abs().nan_to_num().max().item())
