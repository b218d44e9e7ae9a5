"""torch.autograd Functions over the kernel ops: the update (training) side of the op layer.

Each Function pairs a forward kernel with its backward kernels, the way the reference's op layer
does (python/fused_ln.py:56-112 `_LnFn` / `_LnAddFn`; python/fp16_linear.py:442-640 the Linear
Functions with `wgrad` / `wgrad_bgrad` / `dgrad_drelu`; :930-1000 the attention Functions over
`attn29_bwd`).  Gradients of weights and biases are fp32 (they feed fp32 masters), activations'
gradients are in the stream dtype.

What runs where in a backward pass:
  * LayerNorm: `ops.ln_bwd` (dx with the residual-path gradient folded in, dw, db, folded-bias dbb);
  * Linear data gradient: `ops.linear` against the transposed replica, or `ops.linear_gated` when the
    Linear follows a ReLU (the mask rides the GEMM epilogue);
  * Linear weight / bias gradient: `ops.wgrad` on the 16-bit stream (MFMA, LDS transpose loads); on the
    fp32 stream the vendor GEMM through torch (`g.t() @ x`), as the reference does;
  * attention: `ops.attn_bwd`, writing dq | dk | dv into one packed gradient buffer;
  * block FFN with the fused forward kernel (`FusedFfnFn`): the chain's backward over the hidden the kernel wrote, or over
    a recomputed one;
  * the whole NotePolicy update (`NoteTrainFn`): one native call each way.
"""
from __future__ import annotations

import ctypes

import torch
import torch.nn.functional as F
from torch.autograd import forward_ad

from . import _lib
from . import fp16_linear as _fl
from . import ops


def _w_for(w: torch.Tensor, dtype):
    """The weight in the stream dtype: fp32 masters are cast per call here (the update path casts once per
    forward; the rollout path's in-place replicas live in fp16_linear)."""
    w = w.detach()
    return w.contiguous() if w.dtype is dtype else w.to(dtype).contiguous()


def _wgrad(g2, x2, need_w, need_b):
    """(dW, db) fp32 for dy = g2 (rows, M), x = x2 (rows, K)."""
    if not (need_w or need_b):
        return None, None
    if g2.dtype is torch.float32:
        dw = g2.t() @ x2 if need_w else None
        db = g2.sum(0) if need_b else None
        return dw, db
    if need_w:
        dw, db = ops.wgrad(g2, x2, want_db=need_b)
        return dw, db
    return None, g2.sum(0, dtype=torch.float32)


def _rows(t):
    return t.reshape(-1, t.shape[-1])


class LnFn(torch.autograd.Function):
    """y = LayerNorm(x) (reference python/fused_ln.py:56-68)."""

    @staticmethod
    def forward(ctx, x, weight, bias, eps):
        y, mean, rstd = ops.ln_fwd(x, weight.detach(), bias.detach(), eps, want_stats=True)
        ctx.save_for_backward(x, weight, mean, rstd)
        return y

    @staticmethod
    def backward(ctx, dy):
        x, weight, mean, rstd = ctx.saved_tensors
        dx, dw, db = ops.ln_bwd(x, dy.contiguous(), weight.detach(), mean, rstd)
        return dx, dw, db, None


class LnResFn(torch.autograd.Function):
    """(x, LayerNorm(x)) for a pre-LN residual stream: x is handed back as it came so that the residual branch
    hangs off this node, and the backward forms grad(x) + LN's dx in ln_bwd's store loop (one rounding, no
    separate add pass over the stream) - the saving the reference takes through `_LnAddFn`
    (python/fused_ln.py:71-108) on its deferred-residual block layout."""

    @staticmethod
    def forward(ctx, x, weight, bias, eps):
        y, mean, rstd = ops.ln_fwd(x, weight.detach(), bias.detach(), eps, want_stats=True)
        ctx.save_for_backward(x, weight, mean, rstd)
        return x.view_as(x), y

    @staticmethod
    def backward(ctx, gx, gy):
        x, weight, mean, rstd = ctx.saved_tensors
        dx, dw, db = ops.ln_bwd(x, gy.contiguous(), weight.detach(), mean, rstd, gx=gx.contiguous())
        return dx, dw, db, None


class LnAddFn(torch.autograd.Function):
    """(x, y) = (a + b (+ b_bias), LayerNorm(x)) (reference python/fused_ln.py:71-108): d/da == d/db ==
    grad(x) + LN's dx, formed in one rounding inside ln_bwd; d/d(b_bias) = its column sums."""

    @staticmethod
    def forward(ctx, a, b, weight, bias, eps, b_bias):
        x, y, mean, rstd = ops.ln_fwd_add(a, b, weight.detach(), bias.detach(), eps,
                                          None if b_bias is None else b_bias.detach(), want_stats=True)
        ctx.save_for_backward(x, weight, mean, rstd)
        return x, y

    @staticmethod
    def backward(ctx, gx, gy):
        x, weight, mean, rstd = ctx.saved_tensors
        want = ctx.needs_input_grad[5]
        r = ops.ln_bwd(x, gy.contiguous(), weight.detach(), mean, rstd, gx=gx.contiguous(), want_dbb=want)
        dx, dw, db = r[:3]
        return dx, dx, dw, db, None, (r[3] if want else None)


class LinearFn(torch.autograd.Function):
    """act(x @ w.T + b) (+ residual), act in {None, "relu"}; w (M, K) and b fp32 masters or any tensors
    autograd tracks (a torch.cat of several masters for a packed projection)."""

    @staticmethod
    def forward(ctx, x, w, b, act, residual, out_f32=False):
        if act not in (None, "relu"):
            raise NotImplementedError("training path: only ReLU epilogues have a backward")
        if act == "relu" and residual is not None:
            raise NotImplementedError("relu + residual epilogue has no backward here")
        w16 = _w_for(w, x.dtype)
        bias = None if b is None else b.detach().float().contiguous()
        y = ops.linear(x, w16, bias, act=act, residual=residual, out_dtype=torch.float32 if out_f32 else None)
        ctx.act = act
        ctx.has_b = b is not None
        ctx.save_for_backward(x, w16, y if act == "relu" else None)
        return y

    @staticmethod
    def backward(ctx, g):
        x, w16, y = ctx.saved_tensors
        g = g.to(x.dtype).contiguous()                         # an fp32 output's gradient re-enters the stream dtype
        if ctx.act == "relu":
            g = ops.relu_bwd(g, y)
        need_x, need_w, need_b, _, need_r = ctx.needs_input_grad[:5]
        dx = ops.linear(g, w16.t().contiguous()) if need_x else None
        dw, db = _wgrad(_rows(g), _rows(x), need_w, need_b and ctx.has_b)
        return dx, dw, db, None, (g if need_r else None), None


class ChainFn(torch.autograd.Function):
    """Linear (ReLU Linear)+ with every ReLU in a GEMM epilogue (reference python/fp16_linear.py:668-767
    `_chain_forward` / backward): forward keeps the post-ReLU hiddens; backward runs, last layer first,
    (dW, db) = wgrad(g, input) and g = (g @ W) * [hidden > 0] as ONE gated GEMM per layer."""

    @staticmethod
    def forward(ctx, x, residual, out_f32, *wb):
        n = len(wb) // 2
        ws = [_w_for(w, x.dtype) for w in wb[0::2]]
        hs = [x]
        h = x
        for i in range(n):
            last = i == n - 1
            bias = wb[2 * i + 1]
            bias = None if bias is None else bias.detach().float().contiguous()
            h = ops.linear(h, ws[i], bias, act=None if last else "relu", residual=residual if last else None,
                           out_dtype=torch.float32 if (last and out_f32) else None)
            if not last:
                hs.append(h)
        ctx.n = n
        ctx.has_b = [wb[2 * i + 1] is not None for i in range(n)]
        ctx.save_for_backward(*hs, *ws)
        return h

    @staticmethod
    def backward(ctx, g):
        n = ctx.n
        hs, ws = ctx.saved_tensors[:n], ctx.saved_tensors[n:]
        g = g.to(hs[0].dtype).contiguous()
        need = ctx.needs_input_grad
        grads = [None] * (2 * n)
        g_res = g if need[1] else None
        for i in range(n - 1, -1, -1):
            dw, db = _wgrad(_rows(g), _rows(hs[i]), need[3 + 2 * i], need[4 + 2 * i] and ctx.has_b[i])
            grads[2 * i], grads[2 * i + 1] = dw, db
            wt = ws[i].t().contiguous()                       # (K_in, M_out): the data gradient is g @ W
            if i > 0:
                g = ops.linear_gated(g, wt, hs[i])             # through the ReLU that produced hs[i]
            elif need[0]:
                g = ops.linear(g, wt)
            else:
                g = None
        return (g, g_res, None, *grads)


class FusedFfnFn(torch.autograd.Function):
    """x + W2 relu(W0 h2 + b0) + b2 with the forward as ONE kernel, the block FFN of the update path when the
    fused FFN is on (reference python/fp16_linear.py:1197-1251 `_FusedFfn`).  The backward is the unfused chain's:
    (dW2, db2) = wgrad(g, hidden), gm = (g @ W2) * [hidden > 0] as one gated GEMM, (dW0, db0) = wgrad(gm, h2),
    dh2 = gm @ W0, dx = g.  save_hidden: the forward kernel also writes the activated hidden for the backward, as the
    reference's does (its mask is hidden > 0); otherwise the forward keeps h2 only and the backward recomputes the
    hidden with the Linear kernel (one more rows x d x F GEMM per step, rows x F activations less held between
    forward and backward).  Shapes without the packed-image kernel always recompute."""

    @staticmethod
    def _image(w0, b0, w2, b2, w0h, b0f, w2h, b2f):
        """The packed kernel's weight image for the update path: one buffer per FFN (held on its first master
        weight), repacked only when a master has changed - torch's in-place counters of the four masters (every
        optimizer step and load moves them) and the global weights version make the key - instead of once per
        forward call from the freshly cast copies."""
        if not ops.ffn_pack_supported(w0h.shape[1], w0h.shape[0], w0h.dtype):
            return None
        key = (_fl._weights_version, w0._version, b0._version, w2._version, b2._version, w0h.dtype, str(w0h.device))
        cache = getattr(w0, "_bsrl_ffn_image_train", None)
        if cache is None:
            cache = w0._bsrl_ffn_image_train = [None, None]
        if cache[0] != key:
            cache[1] = ops.ffn_pack_into(cache[1], w0h, b0f, w2h, b2f)
            cache[0] = key
        return cache[1]

    @staticmethod
    def forward(ctx, x, h2, w0, b0, w2, b2, save_hidden=False):
        w0h, w2h = _w_for(w0, x.dtype), _w_for(w2, x.dtype)
        b0f, b2f = b0.detach().float().contiguous(), b2.detach().float().contiguous()
        xc, hc = x.contiguous(), h2.contiguous()
        img = FusedFfnFn._image(w0, b0, w2, b2, w0h, b0f, w2h, b2f)
        r = ops.ffn_fused(xc, hc, w0h, b0f, w2h, b2f, act="relu", want_hidden=True, image=img) if save_hidden else None
        hid = None
        if r is not None:
            hid = r[2]
        else:
            r = ops.ffn_fused(xc, hc, w0h, b0f, w2h, b2f, act="relu", image=img)
        if r is None:
            raise ops.Unsupported(f"fused FFN d={x.shape[-1]} F={w0.shape[0]} dtype={x.dtype}")
        ctx.has_hid = hid is not None
        if hid is not None:
            ctx.save_for_backward(h2, w0h, w2h, b0f, hid)
        else:
            ctx.save_for_backward(h2, w0h, w2h, b0f)
        return r[0]

    @staticmethod
    def backward(ctx, g):
        if ctx.has_hid:
            h2, w0h, w2h, b0f, hid = ctx.saved_tensors
        else:
            h2, w0h, w2h, b0f = ctx.saved_tensors
            hid = ops.linear(h2, w0h, b0f, act="relu")
        need = ctx.needs_input_grad                              # x, h2, w0, b0, w2, b2
        g = g.contiguous()
        dw2, db2 = _wgrad(_rows(g), _rows(hid), need[4], need[5])
        gm = ops.linear_gated(g, w2h.t().contiguous(), hid)
        del hid
        dw0, db0 = _wgrad(_rows(gm), _rows(h2), need[2], need[3])
        dh2 = ops.linear(gm, w0h.t().contiguous()) if need[1] else None
        return (g if need[0] else None), dh2, dw0, db0, dw2, db2, None


class AttnPackedFn(torch.autograd.Function):
    """Self-attention off the packed (B, T, 3d) projection (reference python/fp16_linear.py:930-965
    `_Attn29Packed`): ONE packed gradient comes back."""

    @staticmethod
    def forward(ctx, qkv, key_bias, n_heads):
        d = qkv.shape[-1] // 3
        out = ops.attn_fwd(qkv[..., :d], qkv[..., d:2 * d], qkv[..., 2 * d:], n_heads, key_bias=key_bias)
        ctx.n_heads = n_heads
        ctx.save_for_backward(qkv, key_bias)
        return out

    @staticmethod
    def backward(ctx, dout):
        qkv, key_bias = ctx.saved_tensors
        d = qkv.shape[-1] // 3
        dqkv = torch.empty_like(qkv)
        ops.attn_bwd(qkv[..., :d], qkv[..., d:2 * d], qkv[..., 2 * d:], dout.contiguous(), ctx.n_heads, key_bias=key_bias,
                     out=(dqkv[..., :d], dqkv[..., d:2 * d], dqkv[..., 2 * d:]))
        return dqkv, None, None


class AttnQKVFn(torch.autograd.Function):
    """q (B, TQ, d) over the packed (B, T, 2d) k|v projection (reference python/fp16_linear.py:967-1000
    `_Attn29QKV`): the final block's lead queries and the critic's single query."""

    @staticmethod
    def forward(ctx, q, kv, key_bias, n_heads):
        d = q.shape[-1]
        out = ops.attn_fwd(q, kv[..., :d], kv[..., d:], n_heads, key_bias=key_bias)
        ctx.n_heads = n_heads
        ctx.save_for_backward(q, kv, key_bias)
        return out

    @staticmethod
    def backward(ctx, dout):
        q, kv, key_bias = ctx.saved_tensors
        d = q.shape[-1]
        dq = torch.empty_like(q)
        dkv = torch.empty_like(kv)
        ops.attn_bwd(q, kv[..., :d], kv[..., d:], dout.contiguous(), ctx.n_heads, key_bias=key_bias,
                     out=(dq, dkv[..., :d], dkv[..., d:]))
        return dq, dkv, None, None


def _plain_eager(*ts) -> bool:
    """No transform is watching: nothing of torch.func, forward-mode AD, a batch of gradients or a dispatch mode (tracing, fake
    tensors), which would not see a launch through ctypes, and no tensor subclass."""
    return (not torch._C._are_functorch_transforms_active() and forward_ad._current_level < 0 and torch._C._len_torch_dispatch_stack() == 0
            and all(type(t) in (torch.Tensor, torch.nn.Parameter) and not torch._C._functorch.is_legacy_batchedtensor(t) for t in ts))


def heads_logp(logits, action):
    """(logprob, entropy, per-head entropy) of given actions, in torch ops."""
    logsm = torch.log_softmax(logits, dim=-1)
    ent_h = -(logsm.exp() * logsm).sum(-1)
    return logsm.gather(-1, action.unsqueeze(-1)).squeeze(-1).sum(-1), ent_h.sum(-1), ent_h.detach()


class HeadsLogpFn(torch.autograd.Function):
    """`heads_logp` on fp32 logits (B, n_heads, K) and one action per head: the sampling kernel's evaluation forward, one kernel
    back.  An action outside its head makes log-probability and gradient of its env NaN: torch's gather would refuse it, and
    nothing here waits for the device.  A backward that is itself differentiated is torch's."""

    @staticmethod
    def forward(ctx, logits, action):
        _, logprob, entropy, ent_h, _ = ops.sample_heads(logits.contiguous(), action=action.contiguous(), want_ent_h=True, strict=True)
        ctx.save_for_backward(logits, action)
        ctx.mark_non_differentiable(ent_h)
        ctx.set_materialize_grads(False)
        return logprob, entropy, ent_h

    @staticmethod
    def backward(ctx, glp, gent, _):
        logits, action = ctx.saved_tensors
        if glp is None and gent is None:
            return None, None
        if torch.is_grad_enabled() or not _plain_eager(logits, *(g for g in (glp, gent) if g is not None)):
            logsm = torch.log_softmax(logits, dim=-1)
            p, d = logsm.exp(), 0.0
            if glp is not None:
                d = glp[:, None, None] * (F.one_hot(action, logits.shape[-1]) - p)
            if gent is not None:
                d = d - gent[:, None, None] * p * (logsm - (p * logsm).sum(-1, keepdim=True))
            return d, None
        c = lambda g: None if g is None else g.contiguous()
        return ops.heads_logp_bwd(c(logits), c(action), c(glp), c(gent)), None


class HlLossFn(torch.autograd.Function):
    """Batch mean of the HL-Gauss critic loss on fp32 bin logits; the row kernel leaves its gradient, softmax(logits) - target,
    beside the loss."""

    @staticmethod
    def forward(ctx, logits, v_tgt, centers, sigma):
        loss, grad = ops.hl_loss_rows(logits, v_tgt, centers, sigma)
        ctx.save_for_backward(grad, logits)
        return loss.mean()

    @staticmethod
    def backward(ctx, g):
        grad, logits = ctx.saved_tensors
        if torch.is_grad_enabled():                            # to be differentiated again: the softmax as a function of the logits
            p = torch.softmax(logits, dim=-1)
            grad = p - (p.detach() - grad)
        return grad * (g / grad.shape[0]), None, None, None


class NoteTrainPlan:
    """What bsrl_note_train_* need to know about a policy's shape: the descriptor, and where every parameter's gradient lies in
    the flat buffer that the backward writes."""

    def __init__(self, desc: dict, shapes):
        self.desc = _lib.NoteDesc(**desc)
        offsets = (ctypes.c_int64 * len(shapes))()
        self.total = _lib.load().bsrl_note_train_layout(self.desc, offsets, len(shapes))
        self.supported = self.total > 0
        # the gradients as one split of the flat buffer (gaps are alignment): where parameter i's piece is, and its shape
        n = [int(torch.Size(s).numel()) for s in shapes]
        order = sorted(range(len(n)), key=lambda i: offsets[i])
        self.sizes, self.at, end = [], [0] * len(n), 0
        for i in order if self.supported else ():
            if offsets[i] > end:
                self.sizes.append(offsets[i] - end)
            self.at[i] = len(self.sizes)
            self.sizes.append(n[i])
            end = offsets[i] + n[i]
        if self.total > end:
            self.sizes.append(self.total - end)
        self.shapes = [tuple(s) if len(s) > 1 else None for s in shapes]
        self.heads, self.critic = range(16 + 16 * self.desc.n_blocks + 10, len(shapes) - 16), range(len(shapes) - 16, len(shapes))
        # the masters that the backward reads (its matrices are the forward's 16-bit copies): the LayerNorm scales
        L = self.desc.n_blocks
        trunk, critic = 16 + 16 * L, len(shapes) - 16
        self.bwd_params = [i for b in range(L) for i in (16 + 16 * b, 26 + 16 * b)] + [trunk + 2, trunk + 8, critic]

    def pointers(self, params):
        return (ctypes.c_void_p * len(params))(*[p.data_ptr() for p in params])

    def saves(self, B, device):
        """Whether the update of B envs takes its block stack from the rollout forward (the size rule is the library's)."""
        with torch.cuda.device(device):
            return bool(_lib.load().bsrl_note_train_saves(self.desc, B))

    def begin(self, params, obs, saber_idx, body_idx):
        """The update's saved activations with everything in front of the block stack in them, for a rollout forward that writes
        the blocks'; None where the update computes them itself."""
        lib, B = _lib.load(), obs.shape[0]
        if not lib.bsrl_note_train_saves(self.desc, B):
            return None
        saved = torch.empty(lib.bsrl_note_train_size(self.desc, B, 0), dtype=torch.uint8, device=obs.device)
        rc = lib.bsrl_note_train_begin(self.desc, self.pointers(params), obs.data_ptr(), obs.stride(0), ops.dt_code(obs.dtype), saber_idx.data_ptr(),
                                       body_idx.data_ptr(), B, saved.data_ptr(), saved.numel(), ops._stream(obs))
        if not _lib.check(rc, "bsrl_note_train_begin"):
            raise ops.Unsupported("bsrl_note_train_begin")
        return saved

    def bwd_pointers(self, tensors):
        ptrs = (ctypes.c_void_p * len(self.shapes))()
        for i, t in zip(self.bwd_params, tensors):
            ptrs[i] = t.data_ptr()
        return ptrs


class NoteTrainFn(torch.autograd.Function):
    """(logits, value, bin logits) of the NotePolicy update: forward and backward are one native call each over the compacted
    token stream.  The bin logits are this forward's own; logits and value are the rollout's (`r_logits`, `r_value`), whose
    gradients enter where this forward's would: value = softmax(bin logits) @ centers.  `saved`: what the rollout has left of this
    forward (`NoteTrainPlan.begin`), or None.  Notes that attention cannot see are
    never computed: their weight in every softmax is exactly zero."""

    @staticmethod
    def forward(ctx, plan, obs, saber_idx, body_idx, centers, r_logits, r_value, saved, *params):
        lib, B, dev = _lib.load(), obs.shape[0], obs.device
        vlogits = torch.empty(B, plan.desc.bins, dtype=torch.float32, device=dev)
        with torch.cuda.device(dev):
            if saved is not None:                      # the rollout's block stack has left its activations there
                rc = lib.bsrl_note_train_end(plan.desc, plan.pointers(params), vlogits.data_ptr(), B, saved.data_ptr(), saved.numel(), ops._stream(obs))
            else:
                size = lib.bsrl_note_train_size(plan.desc, B, 0)
                if size <= 0:
                    raise ops.Unsupported(f"note_train B={B}")
                saved = torch.empty(size, dtype=torch.uint8, device=dev)
                rc = lib.bsrl_note_train_forward(plan.desc, plan.pointers(params), obs.data_ptr(), obs.stride(0), ops.dt_code(obs.dtype),
                                                 saber_idx.data_ptr(), body_idx.data_ptr(), vlogits.data_ptr(), B, saved.data_ptr(),
                                                 size, ops._stream(obs))
        if not _lib.check(rc, "bsrl_note_train_forward"):
            raise ops.Unsupported("bsrl_note_train_forward")
        ctx.plan, ctx.logits_shape = plan, r_logits.shape
        ctx.set_materialize_grads(False)
        ctx.save_for_backward(saved, vlogits, centers, *[params[i] for i in plan.bwd_params])
        return r_logits.clone(), r_value.clone(), vlogits

    @staticmethod
    def backward(ctx, g_logits, g_value, g_vlogits):
        saved, vlogits, centers, *scales = ctx.saved_tensors
        plan, lib, dev, B = ctx.plan, _lib.load(), saved.device, vlogits.shape[0]
        n_pass = 8                                             # inputs ahead of the parameters
        # what no output in the loss depends on has no gradient, rather than a zero that an optimizer would step on
        unused = set(plan.heads if g_logits is None else ()) | set(plan.critic if g_value is None and g_vlogits is None else ())
        if g_value is not None:                                # through the expectation over the bins
            p = torch.softmax(vlogits, dim=-1)
            gv = g_value.float().unsqueeze(1) * p * (centers - (p @ centers).unsqueeze(1))
            g_vlogits = gv if g_vlogits is None else g_vlogits + gv
        if g_logits is None:
            g_logits = torch.zeros(ctx.logits_shape, dtype=torch.float32, device=dev)
        if g_vlogits is None:
            g_vlogits = torch.zeros_like(vlogits)
        g_logits, g_vlogits = g_logits.float().contiguous(), g_vlogits.float().contiguous()
        flat = torch.empty(plan.total, dtype=torch.float32, device=dev)
        n_scratch = lib.bsrl_note_train_size(plan.desc, B, 1)
        scratch = torch.empty(n_scratch, dtype=torch.uint8, device=dev)
        with torch.cuda.device(dev):
            rc = lib.bsrl_note_train_backward(plan.desc, plan.bwd_pointers(scales), g_logits.data_ptr(), g_vlogits.data_ptr(), flat.data_ptr(),
                                              B, saved.data_ptr(), saved.numel(), scratch.data_ptr(), n_scratch, ops._stream(saved))
        if not _lib.check(rc, "bsrl_note_train_backward"):
            raise ops.Unsupported("bsrl_note_train_backward")
        need = ctx.needs_input_grad
        pieces = flat.split_with_sizes(plan.sizes)
        grads = [None if not need[n_pass + i] or i in unused else pieces[at] if s is None else pieces[at].view(s)
                 for i, (at, s) in enumerate(zip(plan.at, plan.shapes))]
        del pieces
        return (None,) * n_pass + tuple(grads)
