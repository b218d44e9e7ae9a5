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


def test_auto_routes_by_shape_and_batch(monkeypatch):
    """Which route and form `auto` takes on either side of its lines: no batch size gives up the fp32 residual stream that the
    block-stack kernel has, and the forms change where they were measured to cross."""
    got = []
    for n in ("fused", "blocks", "rows", "ops"):
        monkeypatch.setattr(ConfigPolicy, f"_forward_{n}", lambda s, o, k, dt, tail=None, w=None, n=n: got.append(n if n != "rows" else "tail" if tail else "by op"))
    monkeypatch.setattr(ConfigPolicy, "_replicas", lambda *a: None)
    monkeypatch.setattr(ConfigPolicy, "_rows_weights", lambda *a: None)

    class Obs:          # a batch on the GPU, as far as the choice of a route looks at it
        is_cuda, device = True, "cuda"

        def __init__(self, *shape):
            self.shape = shape

        def dim(self):
            return 2

    def route(B, **kw):
        m = ConfigPolicy(**kw)
        got.clear()
        m.forward_stacked(Obs(B, m.obs_dim))
        return got[0]

    wide, deep = dict(n_layers=4, d=256, n_heads=8, ffn=1024, T=32), dict(n_layers=6, d=384, n_heads=12, ffn=1536, T=48)
    assert [route(B, **wide) for B in (1, 256, 257, 448, 449, 32768)] == ["blocks", "blocks", "by op", "by op", "tail", "tail"]
    assert [route(B, **{**wide, "n_layers": 1}) for B in (256, 257, 4096)] == ["blocks", "by op", "by op"]
    assert [route(B, **{**wide, "T": 40}) for B in (1, 358, 359)] == ["by op", "by op", "tail"]
    assert [route(B, **deep) for B in (1, 234, 235, 65536)] == ["by op", "by op", "tail", "tail"]
    assert {route(B, n_layers=3, d=192, n_heads=4, ffn=768, T=29) for B in (1, 300, 9000)} == {"blocks"}
    assert [route(B, n_layers=3, d=192, n_heads=6, ffn=768, T=29) for B in (1, 494, 495)] == ["by op", "by op", "tail"]
    assert route(8, **deep, prop_dim=4096) == "by op" and route(8, **deep, prop_dim=4100) == "ops" and route(8, **deep, obj_dim=36) == "ops"
    assert {route(B, dtype="f32") for B in (1, 20000)} == {"by op"} and {route(B) for B in (1, 20000)} == {"fused"}


def test_copies_and_pickles_leave_the_native_structs_behind():
    import copy
    import pickle

    from beatsaberrl_amd import _lib
    m = ConfigPolicy()
    m._desc(torch.float16)
    m._replica = (("key",), {("rows", True, True): (_lib.CfgRowsWeights(), [])})          # as a forward leaves it
    for c in (copy.deepcopy(m), pickle.loads(pickle.dumps(m))):
        assert c._replica is None and c._desc_cache is None and torch.equal(c.heads.weight, m.heads.weight)
    assert m._replica is not None
    for k in ("_desc_cache", "_ws_rows"):           # a file written before the module had them
        del m.__dict__[k]
    assert m.fused_supported()
