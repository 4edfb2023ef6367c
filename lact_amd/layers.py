"""Drop-ins for the reference's layer classes around the TTT operation, with the reference's constructor
arguments and parameter names (a state_dict moves over unchanged):

  BidirectionalLaCTSwiGLU                minimal_implementations/bidirectional_lact_layer.py:171-270
  CausalLaCTSwiGLUWithSlidingWindowAttn  minimal_implementations/causal_lact_with_sliding_window_attn.py:222-391
  FastWeightGluMLPMultihead              lact_nvs/lact_ttt.py:150-258

The projections are torch.nn.Linear: their large products run in hipBLASLt, the weight gradients of plain ones and the
small maps of the layer's input (learning rates, momentum, gates) in liblact_hip.so, as does everything between: one kernel turns
the to_qkv output into the operation's q, k, v (silu, per-head L2 norm, head layout), one makes the learning rates
and the momentum, the operation itself, and one kernel turns its output into the o_proj input (per-head RMSNorm,
per-head gate, head layout) -- each with a hand-written backward.  The sliding-window attention of the causal
layer (flash_attn_func in the reference) is a pair of kernels for bf16 heads of 64 and 128, whose inputs the first
kernel writes and whose output the last one adds; other types and head sizes go through torch's
scaled_dot_product_attention over blocks of the window size, which bounds the mask to [window, 2*window] per block.
"""
from __future__ import annotations

import ctypes
import math
from typing import Optional

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad as fwad
from torch.utils._python_dispatch import _get_current_dispatch_mode

from . import _lib
from ._autograd import once_differentiable
from ._lib import LACT_BF16, LACT_F32
from .minimal import _bidirectional, inv_softplus
from .nvs import fast_weight_swish_glu_weight_norm_mini_batch_apply
from .ttt_operation import _block_causal


def _ptr(t: Optional[torch.Tensor]):
    return ctypes.c_void_p(0 if t is None else t.data_ptr())


def _stream(t: torch.Tensor):
    return ctypes.c_void_p(torch.cuda.current_stream(t.device).cuda_stream)


def _act(t: torch.Tensor):
    if not t.is_cuda:
        raise RuntimeError(f"lact_amd runs on an MI355X only: tensors must be on a HIP device (no CPU path), got one on {t.device}")
    if t.dtype == torch.bfloat16:
        return LACT_BF16
    if t.dtype == torch.float32:
        return LACT_F32
    raise TypeError(f"unsupported activation dtype {t.dtype}: bf16 or fp32")


def _expect(t: Optional[torch.Tensor], device: torch.device, shape, name: str):
    """The kernels take raw pointers: a tensor elsewhere, or of another shape, has to be refused here."""
    if t is None:
        return
    if t.device != device:
        raise RuntimeError(f"expected all tensors to be on the same device: {name} is on {t.device}, not on {device}")
    if tuple(t.shape) != tuple(shape):
        raise ValueError(f"{name}: expected shape {tuple(shape)}, got {tuple(t.shape)}")


class _PreFn(torch.autograd.Function):
    """qkv [B, L, 3*H*hd] -> q, k, v [(B H), L, hd]."""

    @staticmethod
    def forward(ctx, qkv, H, hd, l2norm):
        qkv, act = qkv.contiguous(), _act(qkv)
        B, L, _ = qkv.shape
        _expect(qkv, qkv.device, (B, L, 3 * H * hd), "qkv")
        q, k, v = (torch.empty((B * H, L, hd), dtype=qkv.dtype, device=qkv.device) for _ in range(3))
        with torch.cuda.device(qkv.device):
            _lib.check(_lib.lib().lact_layer_pre_forward(act, B, L, H, hd, int(l2norm), _ptr(qkv), _ptr(q), _ptr(k),
                                                         _ptr(v), _stream(qkv)))
        ctx.save_for_backward(qkv)
        ctx.dims = (B, L, H, hd, int(l2norm))
        return q, k, v

    @staticmethod
    @once_differentiable
    def backward(ctx, dq, dk, dv):
        (qkv,) = ctx.saved_tensors
        B, L, H, hd, l2norm = ctx.dims
        zeros = lambda: torch.zeros((B * H, L, hd), dtype=qkv.dtype, device=qkv.device)
        dq, dk, dv = (zeros() if g is None else g.to(qkv.dtype).contiguous() for g in (dq, dk, dv))
        dqkv = torch.empty_like(qkv)
        with torch.cuda.device(qkv.device):
            _lib.check(_lib.lib().lact_layer_pre_backward(_act(qkv), B, L, H, hd, l2norm, _ptr(qkv), _ptr(dq), _ptr(dk),
                                                          _ptr(dv), _ptr(dqkv), _stream(qkv)))
        return dqkv, None, None, None


class _PreAttnFn(torch.autograd.Function):
    """qkv [B, L, 3*H*hd], qk_scale, qk_offset [H*hd, 2] -> q, k, v [(B H), L, hd] as _PreFn, and the attention's rescaled q and
    k and its v, [B, L, H*hd] each."""

    @staticmethod
    def forward(ctx, qkv, qk_scale, qk_offset, H, hd, l2norm):
        qkv, act = qkv.contiguous(), _act(qkv)
        B, L, _ = qkv.shape
        _expect(qkv, qkv.device, (B, L, 3 * H * hd), "qkv")
        _expect(qk_scale, qkv.device, (H * hd, 2), "qk_scale")
        _expect(qk_offset, qkv.device, (H * hd, 2), "qk_offset")
        scale, offset = qk_scale.detach().float().contiguous(), qk_offset.detach().float().contiguous()
        outs = [torch.empty((B * H, L, hd), dtype=qkv.dtype, device=qkv.device) for _ in range(3)]
        att = [torch.empty((B, L, H * hd), dtype=qkv.dtype, device=qkv.device) for _ in range(3)]
        with torch.cuda.device(qkv.device):
            _lib.check(_lib.lib().lact_layer_pre_attn_forward(
                act, B, L, H, hd, int(l2norm), int(qk_scale.dtype == qkv.dtype), _ptr(qkv), _ptr(scale), _ptr(offset),
                *[_ptr(t) for t in outs], *[_ptr(t) for t in att], _stream(qkv)))
        ctx.save_for_backward(qkv, scale)
        ctx.dims, ctx.dtypes = (B, L, H, hd, int(l2norm)), (qk_scale.dtype, qk_offset.dtype)
        return (*outs, *att)

    @staticmethod
    @once_differentiable
    def backward(ctx, *grads):
        qkv, scale = ctx.saved_tensors
        B, L, H, hd, l2norm = ctx.dims
        shapes = [(B * H, L, hd)] * 3 + [(B, L, H * hd)] * 3
        grads = [torch.zeros(s, dtype=qkv.dtype, device=qkv.device) if g is None else g.to(qkv.dtype).contiguous() for g, s in zip(grads, shapes)]
        lib = _lib.lib()
        dqkv, dscale, doffset = torch.empty_like(qkv), torch.empty_like(scale), torch.empty_like(scale)
        part = torch.empty(lib.lact_layer_pre_attn_part_rows(B, L, H) * 4 * H * hd, dtype=torch.float32, device=qkv.device)
        with torch.cuda.device(qkv.device):
            _lib.check(lib.lact_layer_pre_attn_backward(_act(qkv), B, L, H, hd, l2norm, _ptr(qkv), _ptr(scale), *[_ptr(g) for g in grads],
                                                        _ptr(dqkv), _ptr(part), _ptr(dscale), _ptr(doffset), _stream(qkv)))
        return dqkv, dscale.to(ctx.dtypes[0]), doffset.to(ctx.dtypes[1]), None, None, None


class _LrFn(torch.autograd.Function):
    """lr_raw [B, L, 3*H] (head-major with three rates per head, or rate-major when rates_major), momentum_raw
    [B, L, H] or None -> lr0, lr1, lr2, momentum [(B H), L, 1] fp32."""

    @staticmethod
    def forward(ctx, lr_raw, mom_raw, H, base_lr_inv, rates_major=False):
        lr_raw = lr_raw.float().contiguous()
        _act(lr_raw)
        mom_c = None if mom_raw is None else mom_raw.float().contiguous()
        B, L, _ = lr_raw.shape
        _expect(lr_raw, lr_raw.device, (B, L, 3 * H), "lr_raw")
        _expect(mom_c, lr_raw.device, (B, L, H), "momentum_raw")
        outs = [torch.empty((B * H, L, 1), dtype=torch.float32, device=lr_raw.device) for _ in range(3)]
        mom = torch.empty((B * H, L, 1), dtype=torch.float32, device=lr_raw.device) if mom_c is not None else None
        with torch.cuda.device(lr_raw.device):
            _lib.check(_lib.lib().lact_layer_lr_forward(B, L, H, int(rates_major), float(base_lr_inv), _ptr(lr_raw), _ptr(outs[0]),
                                                        _ptr(outs[1]), _ptr(outs[2]), _ptr(mom_c), _ptr(mom),
                                                        _stream(lr_raw)))
        ctx.save_for_backward(lr_raw, mom_c)
        ctx.dims = (B, L, H, float(base_lr_inv), int(rates_major))
        ctx.mom_dtype = None if mom_raw is None else mom_raw.dtype
        if mom is None:
            return outs[0], outs[1], outs[2]
        return outs[0], outs[1], outs[2], mom

    @staticmethod
    @once_differentiable
    def backward(ctx, d0, d1, d2, dm=None):
        lr_raw, mom_c = ctx.saved_tensors
        B, L, H, base, rates_major = ctx.dims
        c = lambda g: None if g is None else g.float().contiguous()
        d0, d1, d2, dm = c(d0), c(d1), c(d2), c(dm)
        dlr_raw = torch.empty_like(lr_raw)
        dmom_raw = torch.empty_like(mom_c) if mom_c is not None else None
        with torch.cuda.device(lr_raw.device):
            _lib.check(_lib.lib().lact_layer_lr_backward(B, L, H, rates_major, base, _ptr(lr_raw), _ptr(d0), _ptr(d1), _ptr(d2),
                                                         _ptr(dlr_raw), _ptr(mom_c), _ptr(dm), _ptr(dmom_raw),
                                                         _stream(lr_raw)))
        return dlr_raw, (None if dmom_raw is None else dmom_raw.to(ctx.mom_dtype)), None, None, None


class _PostFn(torch.autograd.Function):
    """o [(B H), L, hd] -> y [B, L, H*hd]: RMSNorm(weight) per head if weight is given or use_norm, times
    silu(gate_raw [B, L, H]) if given, plus add [B, L, H*hd] if given."""

    @staticmethod
    def forward(ctx, o, weight, gate_raw, B, H, use_norm, eps, add=None):
        o, act = o.contiguous(), _act(o)
        _, L, hd = o.shape
        _expect(o, o.device, (B * H, L, hd), "o")
        _expect(weight, o.device, (hd,), "weight")
        _expect(gate_raw, o.device, (B, L, H), "gate_raw")
        _expect(add, o.device, (B, L, H * hd), "add")
        w = None if weight is None else weight.float().contiguous()
        g = None if gate_raw is None else gate_raw.to(o.dtype).contiguous()
        add_c = None if add is None else add.to(o.dtype).contiguous()
        y = torch.empty((B, L, H * hd), dtype=o.dtype, device=o.device)
        with torch.cuda.device(o.device):
            _lib.check(_lib.lib().lact_layer_post_add_forward(act, B, L, H, hd, int(use_norm), float(eps), _ptr(o), _ptr(w),
                                                          _ptr(g), _ptr(add_c), _ptr(y), _stream(o)))
        ctx.save_for_backward(o, w, g)
        ctx.add_dtype = None if add is None else add.dtype
        ctx.dims = (B, L, H, hd, int(use_norm), float(eps))
        ctx.dtypes = (None if weight is None else weight.dtype, None if gate_raw is None else gate_raw.dtype)
        return y

    @staticmethod
    @once_differentiable
    def backward(ctx, dy):
        o, w, g = ctx.saved_tensors
        B, L, H, hd, use_norm, eps = ctx.dims
        lib = _lib.lib()
        dy = dy.to(o.dtype).contiguous()
        d_o = torch.empty_like(o)
        dg = torch.empty_like(g) if g is not None else None
        rows = lib.lact_layer_post_dw_rows(B, L, H)
        dw_part = torch.empty((rows, hd), dtype=torch.float32, device=o.device) if (use_norm and w is not None) else None
        with torch.cuda.device(o.device):
            _lib.check(lib.lact_layer_post_backward(_act(o), B, L, H, hd, use_norm, eps, _ptr(o), _ptr(w), _ptr(g), _ptr(dy),
                                                    _ptr(d_o), _ptr(dg), _ptr(dw_part), _stream(o)))
        wd, gd = ctx.dtypes
        dw = None if dw_part is None else dw_part.sum(dim=0).to(wd)
        return d_o, dw, (None if dg is None else dg.to(gd)), None, None, None, None, (None if ctx.add_dtype is None else dy.to(ctx.add_dtype))


def _plain(*ts) -> bool:
    """Whether the host module's functions may take a call: plain tensors, and nobody around who wants to see Python functions or
    tensor operations (compilation and tracing, function transforms, forward mode, modes, subclasses).  Others get the functions
    above and the modules themselves."""
    return (all(t is None or type(t) in (torch.Tensor, nn.Parameter) for t in ts)
            and not (torch.compiler.is_compiling() or torch.jit.is_tracing() or torch._C._are_functorch_transforms_active()
                     or torch._C._len_torch_function_stack() > 0 or _get_current_dispatch_mode() is not None or fwad._current_level >= 0
                     or any(torch._C._functorch.is_legacy_batchedtensor(t) for t in ts if t is not None)))


def _pre(qkv, H, hd, l2norm):
    return _lib.host().layer_pre(qkv, H, hd, l2norm) if _plain(qkv) else _PreFn.apply(qkv, H, hd, l2norm)


def _pre_attn(qkv, scale, offset, H, hd, l2norm):
    fn = _lib.host().layer_pre_attn if _plain(qkv, scale, offset) else _PreAttnFn.apply
    return fn(qkv, scale, offset, H, hd, l2norm)


def _rates(lr_raw, mom_raw, H, base_lr_inv, rates_major=False):
    fn = _lib.host().layer_lr if _plain(lr_raw, mom_raw) else _LrFn.apply
    return fn(lr_raw, mom_raw, H, base_lr_inv, rates_major)


def _post(o, weight, gate_raw, B, H, use_norm, eps, add=None):
    fn = _lib.host().layer_post if _plain(o, weight, gate_raw, add) else _PostFn.apply
    return fn(o, weight, gate_raw, B, H, use_norm, eps, add)


def _plain_linear(m: nn.Module) -> bool:
    """An nn.Linear in fp32 whose call is F.linear and nothing else: no subclass, hook, parametrisation or replaced forward."""
    return (type(m) is nn.Linear and "forward" not in m.__dict__
            and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks)
            and all(t is None or (t.is_cuda and t.dtype == torch.float32) for t in (m.weight, m.bias)))


def _fused_linears(x: torch.Tensor, *mods: nn.Module) -> bool:
    """Whether the host module may evaluate linear maps of x instead of their modules: plain fp32 ones under bf16 autocast."""
    return (x.is_cuda and x.dim() == 3 and x.numel() > 0 and torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") == torch.bfloat16
            and all(_plain_linear(m) and m.weight.device == x.device and m.in_features == x.shape[-1] for m in mods)
            and not nn.modules.module._has_any_global_hook() and _plain(x, *[t for m in mods for t in (m.weight, m.bias)]))


def _linear(m: nn.Module, x: torch.Tensor) -> torch.Tensor:
    """m(x); the gradient of a fused map's weight comes from csrc/gemm_dma_kernels.h, summed and returned in fp32."""
    return _lib.host().linear(x, m.weight) if m.bias is None and _fused_linears(x, m) else m(x)


MAX_LR_OUTPUTS, MAX_BF16_OUTPUTS = 24, 16      # registers of the kernels in csrc/layer_kernels.h


def _input_projections(x, to_qkv, lr_proj, momentum=None, gate=None):
    """to_qkv(x), lr_proj(x) outside autocast, momentum(x), gate(x) (either may be absent: None)."""
    mods = [m for m in (to_qkv, lr_proj, momentum, gate) if m is not None]
    if (x.dtype == torch.float32 and to_qkv.bias is None and _fused_linears(x, *mods) and x.shape[-1] % 8 == 0 and x.shape[:-1].numel() < 1 << 31
            and 0 < lr_proj.out_features <= MAX_LR_OUTPUTS and sum(m.out_features for m in mods[2:]) <= MAX_BF16_OUTPUTS):
        maps = [t for m in (lr_proj, momentum, gate) for t in ((None, None) if m is None else (m.weight, m.bias))]
        qkv, lr_raw, *rest = _lib.host().layer_in(x, to_qkv.weight, *maps)
        return qkv, lr_raw, None if momentum is None else rest[0], None if gate is None else rest[-1]
    qkv = _linear(to_qkv, x)
    with torch.autocast(device_type="cuda", enabled=False):      # the reference keeps the rates out of autocast (:247-249)
        lr_raw = lr_proj(x)
    return qkv, lr_raw, None if momentum is None else momentum(x), None if gate is None else gate(x)


def _fast_weights(layer, B):
    """[nh, ...] parameters -> [(B nh), ...] (bidirectional_lact_layer.py:259-261)."""
    return tuple(w.repeat(B, 1, 1) for w in (layer.w0, layer.w1, layer.w2))


def _shared_weights(layer, B):
    """The fast weights of a batch, and whether they are the parameters themselves, which the operation takes for every sequence (three
    copies, and three sums behind the backward, less: 618 -> 522 us a step at 3 x 2500 tokens, 8 heads of 96)."""
    w = (layer.w0, layer.w1, layer.w2)
    return (w, True) if _plain(*w) else (_fast_weights(layer, B), False)


def _norm_args(o_norm):
    if isinstance(o_norm, nn.RMSNorm):
        return o_norm.weight, True, (o_norm.eps if o_norm.eps is not None else 1e-5)
    return None, False, 1e-5


class BidirectionalLaCTSwiGLU(nn.Module):
    """bidirectional_lact_layer.py:171-270."""

    def __init__(self, dim: int, head_dim: int, inter_multi: float = 1, use_o_norm: bool = True,
                 qk_l2_norm: bool = True, use_muon: bool = True, base_lr: float = 1e-2):
        super().__init__()
        self.dim, self.head_dim, self.inter_multi = dim, head_dim, inter_multi
        self.use_o_norm, self.qk_l2_norm, self.use_muon = use_o_norm, qk_l2_norm, use_muon
        self.num_heads = dim // head_dim
        self.to_qkv = nn.Linear(dim, 3 * dim, bias=False)
        self.o_proj = nn.Linear(dim, dim, bias=False)
        self.lr_dim = 1
        self.lr_proj = nn.Linear(dim, self.lr_dim * 3 * self.num_heads, bias=False)
        self.base_lr = base_lr
        self.base_lr_inv = inv_softplus(base_lr)
        d_in, d_out, d_h = head_dim, head_dim, int(head_dim * inter_multi)
        self.w0 = nn.Parameter(torch.randn(self.num_heads, d_h, d_in) / math.sqrt(d_in))
        self.w1 = nn.Parameter(torch.randn(self.num_heads, d_out, d_h) / math.sqrt(d_h))
        self.w2 = nn.Parameter(torch.randn(self.num_heads, d_h, d_in) / math.sqrt(d_in))
        self.o_norm = nn.RMSNorm(head_dim, eps=1e-5, elementwise_affine=True) if use_o_norm else nn.Identity()

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        """x: [b, l, d] -> [b, l, d]"""
        B = x.shape[0]
        qkv, lr_raw, _, _ = _input_projections(x, self.to_qkv, self.lr_proj)
        q, k, v = _pre(qkv, self.num_heads, self.head_dim, self.qk_l2_norm)
        lr0, lr1, lr2 = _rates(lr_raw, None, self.num_heads, self.base_lr_inv)
        w, shared = _shared_weights(self, B)
        o = _bidirectional(*w, q, k, v, lr0, lr1, lr2, self.use_muon, shared_weights=shared)
        weight, use_norm, eps = _norm_args(self.o_norm)
        return _linear(self.o_proj, _post(o, weight, None, B, self.num_heads, use_norm, eps))


MAX_TOKEN_STRIDE = 1 << 24     # elements; the kernels' offsets inside a tile are 32-bit


def _head_rows(t: torch.Tensor) -> torch.Tensor:
    """[b, l, h, d] whose heads lie next to each other inside a token, 16-byte aligned."""
    ok = (t.stride(3) == 1 and t.stride(2) == t.shape[3] and t.stride(1) % 8 == 0 and t.stride(0) % 8 == 0
          and t.shape[2] * t.shape[3] <= t.stride(1) <= MAX_TOKEN_STRIDE and t.data_ptr() % 16 == 0)
    # clone: contiguous() hands back what merely starts off a 16-byte boundary or has odd strides in dimensions of size 1
    return t if ok else t.clone(memory_format=torch.contiguous_format)


def _torch_window_attention(q, k, v, window):
    l = q.shape[1]
    q, k, v = (t.transpose(1, 2) for t in (q, k, v))              # [b, h, l, d]
    if window is None or window >= l:
        return F.scaled_dot_product_attention(q, k, v, is_causal=True).transpose(1, 2)
    outs = []
    for s in range(0, l, window):
        e = min(s + window, l)
        ks = max(0, s - window + 1)
        qi = torch.arange(s, e, device=q.device)[:, None]
        kj = torch.arange(ks, e, device=q.device)[None, :]
        mask = (kj <= qi) & (kj >= qi - (window - 1))
        outs.append(F.scaled_dot_product_attention(q[:, :, s:e], k[:, :, ks:e], v[:, :, ks:e], attn_mask=mask))
    return torch.cat(outs, dim=2).transpose(1, 2)


def _on_window_kernels(q, k, v) -> bool:
    """Whether csrc/window_attention.h takes the call: its type, head sizes and limits, on plain tensors.  What sees the call as
    tensor operations (vmap and the other function transforms, forward-mode differentiation, dispatch modes, tensor subclasses,
    autocast to another type) gets them."""
    b, l, h, d = q.shape
    if not (q.is_cuda and d in (64, 128) and b * l * h > 0 and q.device == k.device == v.device and q.shape == k.shape == v.shape
            and q.dtype == k.dtype == v.dtype == torch.bfloat16):
        return False
    if b * h > 1 << 20 or l * h * d > 1 << 31 or h * d > MAX_TOKEN_STRIDE:
        return False
    if torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") != torch.bfloat16:
        return False
    return torch.compiler.is_compiling() or not (
        torch._C._are_functorch_transforms_active() or torch.jit.is_tracing() or _get_current_dispatch_mode() is not None
        or any(type(t) not in (torch.Tensor, nn.Parameter) or torch._C._functorch.is_legacy_batchedtensor(t) for t in (q, k, v))
        or (fwad._current_level >= 0 and any(fwad.unpack_dual(t).tangent is not None for t in (q, k, v))))


def _window_forward(q, k, v, window):
    B, L, H, D = q.shape
    out = torch.empty((B, L, H, D), dtype=q.dtype, device=q.device)
    lse = torch.empty((B, H, L), dtype=torch.float32, device=q.device)
    with torch.cuda.device(q.device):
        _lib.check(_lib.lib().lact_window_attention_forward(
            B, L, H, D, window, _ptr(q), q.stride(1), q.stride(0), _ptr(k), k.stride(1), k.stride(0), _ptr(v), v.stride(1), v.stride(0),
            _ptr(out), _ptr(lse), _stream(q)))
    return out, lse


def _window_backward(g, q, k, v, out, lse, window):
    B, L, H, D = q.shape
    g = _head_rows(g.to(q.dtype))
    dq, dk, dv = (torch.empty((B, L, H, D), dtype=q.dtype, device=q.device) for _ in range(3))
    delta = torch.empty_like(lse)
    with torch.cuda.device(q.device):
        _lib.check(_lib.lib().lact_window_attention_backward(
            B, L, H, D, window, _ptr(q), q.stride(1), q.stride(0), _ptr(k), k.stride(1), k.stride(0), _ptr(v), v.stride(1), v.stride(0),
            _ptr(out), _ptr(lse), _ptr(g), g.stride(1), g.stride(0), _ptr(delta), _ptr(dq), _ptr(dk), _ptr(dv), _stream(q)))
    return dq, dk, dv


class _WindowAttentionFn(torch.autograd.Function):
    """bf16 sliding-window attention on [b, l, h, d], d = 64 or 128 (csrc/window_attention.h)."""

    @staticmethod
    def forward(ctx, q, k, v, window):
        q, k, v = _head_rows(q), _head_rows(k), _head_rows(v)
        out, lse = _window_forward(q, k, v, window)
        ctx.save_for_backward(q, k, v, out, lse)
        ctx.window = window
        return out

    @staticmethod
    @once_differentiable
    def backward(ctx, g):
        q, k, v, out, lse = ctx.saved_tensors
        if torch._C._functorch.is_legacy_batchedtensor(g):      # is_grads_batched: the batch is torch's business
            with torch.enable_grad():
                x = [t.detach().requires_grad_() for t in (q, k, v)]
                return (*torch.autograd.grad(_torch_window_attention(*x, ctx.window), x, g), None)
        return (*_window_backward(g, q, k, v, out, lse, ctx.window), None)


# The same as operators, which torch.compile traces through (their dispatch costs an eager call more than the function above).
@torch.library.custom_op("lact_amd::window_attention", mutates_args=(), schema="(Tensor q, Tensor k, Tensor v, int window) -> (Tensor, Tensor)")
def _window_attention_op(q, k, v, window):
    return _window_forward(_head_rows(q), _head_rows(k), _head_rows(v), window)


@_window_attention_op.register_fake
def _(q, k, v, window):
    b, l, h, _ = q.shape
    return q.new_empty(q.shape), q.new_empty((b, h, l), dtype=torch.float32)


@torch.library.custom_op("lact_amd::window_attention_backward", mutates_args=(),
                         schema="(Tensor g, Tensor q, Tensor k, Tensor v, Tensor out, Tensor lse, int window) -> (Tensor, Tensor, Tensor)")
def _window_attention_backward_op(g, q, k, v, out, lse, window):
    return _window_backward(g, _head_rows(q), _head_rows(k), _head_rows(v), out.contiguous(), lse.contiguous(), window)


@_window_attention_backward_op.register_fake
def _(g, q, k, v, out, lse, window):
    return q.new_empty(q.shape), q.new_empty(q.shape), q.new_empty(q.shape)


def _window_attention_setup(ctx, inputs, output):
    ctx.save_for_backward(*inputs[:3], *output)
    ctx.window = inputs[3]
    ctx.mark_non_differentiable(output[1])


def _window_attention_vjp(ctx, g, _):
    return (*_window_attention_backward_op(g, *ctx.saved_tensors, ctx.window), None)


_window_attention_op.register_autograd(_window_attention_vjp, setup_context=_window_attention_setup)


def sliding_window_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, window: Optional[int]) -> torch.Tensor:
    """q, k, v: [b, l, h, d].  Causal attention where query i sees keys i-(window-1) .. i -- what the reference asks
    of flash_attn_func(causal=True, window_size=(window-1, 0)) (causal_lact_with_sliding_window_attn.py:371-375).
    bf16 with heads of 64 or 128 runs in this library's kernels; other types and head sizes through torch's attention, where
    query blocks of `window` rows attend to their own and the previous block under a band mask."""
    if _on_window_kernels(q, k, v):
        width = q.shape[1] if window is None else min(window, q.shape[1])
        return _window_attention_op(q, k, v, width)[0] if torch.compiler.is_compiling() else _WindowAttentionFn.apply(q, k, v, width)
    return _torch_window_attention(q, k, v, window)


class CausalLaCTSwiGLUWithSlidingWindowAttn(nn.Module):
    """causal_lact_with_sliding_window_attn.py:222-391."""

    def __init__(self, dim: int, head_dim: int, attn_head_dim: int, lact_chunk_size: int = 2048, window_size: int = 2048,
                 inter_multi: float = 1, use_o_norm: bool = True, use_momentum: bool = True, use_muon: bool = True,
                 base_lr: float = 1e-2, ttt_scale_before_sum: bool = True):
        super().__init__()
        self.dim, self.head_dim, self.attn_head_dim, self.inter_multi = dim, head_dim, attn_head_dim, inter_multi
        self.lact_chunk_size, self.window_size, self.use_o_norm = lact_chunk_size, window_size, use_o_norm
        self.num_ttt_heads, self.num_attn_heads = dim // head_dim, dim // attn_head_dim
        self.to_qkv = nn.Linear(dim, 3 * dim, bias=False)
        self.o_proj = nn.Linear(dim, dim, bias=False)
        self.lr_dim = 1
        self.lr_proj = nn.Linear(dim, self.lr_dim * 3 * self.num_ttt_heads, bias=False)
        self.base_lr = base_lr
        self.base_lr_inv = inv_softplus(base_lr)
        d_in, d_out, d_h = head_dim, head_dim, int(head_dim * inter_multi)
        self.w0 = nn.Parameter(torch.randn(self.num_ttt_heads, d_h, d_in) / math.sqrt(d_in))
        self.w1 = nn.Parameter(torch.randn(self.num_ttt_heads, d_out, d_h) / math.sqrt(d_h))
        self.w2 = nn.Parameter(torch.randn(self.num_ttt_heads, d_h, d_in) / math.sqrt(d_in))
        self.use_muon, self.use_momentum = use_muon, use_momentum
        if use_momentum:
            self.momentum_proj = nn.Sequential(nn.Linear(dim, self.num_ttt_heads), nn.Sigmoid())
        self.o_norm = nn.RMSNorm(head_dim, eps=1e-5, elementwise_affine=True) if use_o_norm else nn.Identity()
        self.qk_scale = nn.Parameter(torch.ones(dim, 2))
        self.qk_offset = nn.Parameter(torch.zeros(dim, 2))
        # the reference creates this only when ttt_scale_before_sum, and its forward always uses it (:348)
        self.ttt_scale_proj = nn.Linear(dim, self.num_ttt_heads)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        """x: [b, l, d] -> [b, l, d]"""
        B, L, _ = x.shape
        H = self.num_ttt_heads
        # the Sigmoid of momentum_proj is in the kernel behind this
        qkv, lr_raw, mom_raw, gate_raw = _input_projections(x, self.to_qkv, self.lr_proj, self.momentum_proj[0] if self.use_momentum else None,
                                                            self.ttt_scale_proj)
        q, k, v, aq, ak, av = _pre_attn(qkv, self.qk_scale, self.qk_offset, H, self.head_dim, True)
        res = _rates(lr_raw, mom_raw, H, self.base_lr_inv)
        lr0, lr1, lr2 = res[:3]
        momentum = res[3] if self.use_momentum else None
        w, shared = _shared_weights(self, B)
        o = _block_causal(*w, q, k, v, lr0, lr1, lr2, self.lact_chunk_size, self.use_muon, momentum, False, shared_weights=shared)
        sh = lambda t: t.reshape(B, L, self.num_attn_heads, self.attn_head_dim)
        attn = sliding_window_attention(sh(aq), sh(ak), sh(av), self.window_size).reshape(B, L, -1)
        weight, use_norm, eps = _norm_args(self.o_norm)
        return _linear(self.o_proj, _post(o, weight, gate_raw, B, H, use_norm, eps, attn))


class FastWeightGluMLPMultihead(nn.Module):
    """lact_nvs/lact_ttt.py:150-258: the layer of the novel-view-synthesis model.  Fast weights in the transposed
    layout (w0, w2: [nh, d, dh]; w1: [nh, dh, d]); `info["ttt_op_order"]` is the list of TTTOperator steps and
    `info["w0"/"w1"/"w2"]`, when present, are the fast weights a previous call returned (state carried from the
    reconstruction pass into the rendering pass, lact_nvs/model.py:272-384)."""

    def __init__(self, dim: int, head_dim: int, inter_multi: int = 1, bias: bool = False, base_lr: float = 0.01,
                 muon_update_steps: int = 0):
        super().__init__()
        assert dim % head_dim == 0
        self.dim, self.num_heads, self.muon_update_steps = dim, dim // head_dim, muon_update_steps
        self.head_dim = head_dim
        d_in = d_out = head_dim
        d_h = int(head_dim * inter_multi)
        gain = math.sqrt(2)
        self.w0 = nn.Parameter(torch.randn(self.num_heads, d_in, d_h) * gain / math.sqrt(d_in))
        self.w1 = nn.Parameter(torch.randn(self.num_heads, d_h, d_out) * gain / math.sqrt(d_h))
        self.w2 = nn.Parameter(torch.randn(self.num_heads, d_in, d_h) * gain / math.sqrt(d_in))
        self.to_qkv = nn.Linear(dim, 3 * dim, bias=bias)
        self.c_proj = nn.Linear(dim, dim, bias=bias)
        self.lr_dim = self.num_heads
        self.lr_fc = nn.Linear(dim, self.lr_dim * 3)
        self.base_lr_inv = inv_softplus(base_lr)
        self.o_norm = nn.RMSNorm(head_dim, eps=1e-5, elementwise_affine=True)

    def forward(self, x: torch.Tensor, info={}, *args):
        """x: [b, l, d] -> ([b, l', d], {"w0", "w1", "w2"}) with l' the rows of the apply steps in program order."""
        B = x.shape[0]
        if x.dtype == torch.float32:                                                         # :203-213
            qkv, lr_raw, _, _ = _input_projections(x, self.to_qkv, self.lr_fc)
        else:
            qkv = _linear(self.to_qkv, x)
            with torch.autocast(device_type="cuda", enabled=False):
                lr_raw = self.lr_fc(x.float())
        q, k, v = _pre(qkv, self.num_heads, self.head_dim, True)
        lr0, lr1, lr2 = _rates(lr_raw, None, self.num_heads, self.base_lr_inv, True)    # '(lrs h d)', :215-219
        if "w0" in info:                                                                      # :221-229
            assert "w1" in info and "w2" in info
            w0, w1, w2 = info["w0"], info["w1"], info["w2"]
        else:
            w0, w1, w2 = _fast_weights(self, B)
        o, w0, w1, w2 = fast_weight_swish_glu_weight_norm_mini_batch_apply(
            w0, w1, w2, q, k, v, lr0, lr1, lr2, info["ttt_op_order"], muon_update_steps=self.muon_update_steps)
        weight, use_norm, eps = _norm_args(self.o_norm)
        y = _post(o, weight, None, B, self.num_heads, use_norm, eps)
        return _linear(self.c_proj, y), {"w0": w0, "w1": w1, "w2": w2}
