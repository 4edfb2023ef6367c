"""Host side of the TTT operation: schedules as the C ABI's step programs.  The native host module
(csrc/torch_host.cpp) checks and allocates the tensors, owns the autograd boundary and calls liblact_hip.so on the
current HIP stream.

PyTorch is used for device memory, streams and autograd bookkeeping only; all arithmetic of the
operation runs in the HIP kernels.  There is no fallback path.
"""
from __future__ import annotations

import ctypes
from dataclasses import dataclass
from typing import Optional, Sequence, Tuple

import torch

from . import _lib
from ._autograd import once_differentiable
from ._lib import LACT_APPLY, LACT_UPDATE

# lact_llm/lact_model/ttt_operation.py:51-57
NS5_COEFFS: Tuple[Tuple[float, float, float], ...] = (
    (4.0848, -6.8946, 2.9270),
    (3.9505, -6.3029, 2.6377),
    (3.7418, -5.5913, 2.3037),
    (2.8769, -3.1427, 1.2046),
    (2.8366, -3.0525, 1.2012),
)
# lact_nvs/lact_ttt.py:51 and lact_ar_video/minVid/models/blocks/functions.py:56
NS_CLASSIC: Tuple[float, float, float] = (3.4445, -4.7750, 2.0315)


@dataclass(frozen=True)
class Program:
    """A test-time-training schedule: steps are (kind, start, end, out_start)."""
    steps: Tuple[Tuple[int, int, int, int], ...]
    out_len: int
    ns_coeffs: Optional[Tuple[Tuple[float, float, float], ...]] = None   # None: Muon off
    prenorm: bool = False
    weight_norm: bool = True
    detach_norms: bool = False
    muon_replaces_weight: bool = False
    ns_mode: int = 0   # 0: bf16 GEMMs + fp32 iterate (autocast), 1: bf16 iterate (no autocast), 2: fp32 (exact)
    # fused-kernel variant (lact_llm/lact_model/ttt_operation_fused_kernel.py): Newton-Schulz on the stacked
    # gradient cat(dw0, dw2); eps inside the sqrt of the row renorm
    muon_stacked: bool = False
    renorm_eps_in_sqrt: bool = False
    # callers that only use the output (the block-causal and bidirectional functions) spare the copies of the final
    # fast weights and momentum states: run_program then returns None in their places
    return_state: bool = True

    def native(self):
        """The schedule in the native host module's form, made on first use."""
        h = self.__dict__.get("_native")
        if h is None:
            flat = None if self.ns_coeffs is None else [float(x) for tr in self.ns_coeffs for x in tr]
            h = _lib.host().Schedule([list(s) for s in self.steps], self.out_len, flat, self.prenorm, self.weight_norm, self.detach_norms,
                                     self.muon_replaces_weight, int(self.ns_mode), self.muon_stacked, self.renorm_eps_in_sqrt, self.return_state)
            object.__setattr__(self, "_native", h)
        return h

    def __getstate__(self):      # copies and pickles make their own
        return {k: v for k, v in self.__dict__.items() if k != "_native"}

    @property
    def n_updates(self) -> int:
        return sum(1 for s in self.steps if s[0] == LACT_UPDATE)


def block_causal_steps(seq_len: int, chunk_size: int):
    """Apply chunk i with the weights of chunks < i, then update on chunk i; the last chunk is
    apply-only (lact_llm/lact_model/ttt_operation.py:121-212)."""
    steps, e = [], 0
    for s in range(0, seq_len - chunk_size, chunk_size):
        e = s + chunk_size
        steps.append((LACT_APPLY, s, e, s))
        steps.append((LACT_UPDATE, s, e, 0))
    steps.append((LACT_APPLY, e, seq_len, e))
    return tuple(steps)


def _ptr(t: Optional[torch.Tensor]):
    return ctypes.c_void_p(0 if t is None else t.data_ptr())


@torch.compiler.disable
def run_program(prog: Program, w0, w1, w2, q, k, v, lr0, lr1, lr2, momentum=None, momentum_state=None, shared_weights=False):
    """Runs `prog`.  Returns (out, (w0, w1, w2) after the last update, (m0, m1, m2) momentum states; None each
    without momentum).
    `shared_weights`: w0, w1, w2 hold fewer matrices than q has batch entries, and entry i starts from matrix i modulo their number.
    `momentum_state` = the (m0, m1, m2) of an earlier call: the first update continues from it (inference only)."""
    m0, m1, m2 = momentum_state if momentum_state is not None else (None, None, None)
    res = _lib.host().run_program(prog.native(), w0, w1, w2, q, k, v, lr0, lr1, lr2, momentum, m0, m1, m2, shared_weights)
    return res[0], res[1:4], res[4:7]


NS_AUTOCAST, NS_PLAIN_BF16, NS_FP32 = 0, 1, 2
_ns_mode_override: Optional[int] = None


class newton_schulz_mode:
    """Context manager forcing the Newton-Schulz numerics of every operation called inside it
    (NS_FP32 = fp32 MFMA, no bf16 rounding: the exact-arithmetic check of the Muon path)."""

    def __init__(self, mode: Optional[int]):
        self.mode = mode

    def __enter__(self):
        global _ns_mode_override
        self.prev, _ns_mode_override = _ns_mode_override, self.mode
        return self

    def __exit__(self, *exc):
        global _ns_mode_override
        _ns_mode_override = self.prev
        return False


def _ns_mode(q: torch.Tensor) -> int:
    """Without autocast and with fp32 activations the reference keeps the whole Newton-Schulz
    iterate in bf16 (ttt_operation.py:45 casts, nothing casts back)."""
    if _ns_mode_override is not None:
        return _ns_mode_override
    return NS_PLAIN_BF16 if (q.dtype == torch.float32 and not torch.is_autocast_enabled()) else NS_AUTOCAST


class _NewtonSchulzFn(torch.autograd.Function):
    """zeropower_via_newtonschulz5 with its closed-form backward (lact_newton_schulz / lact_newton_schulz_backward)."""

    @staticmethod
    def forward(ctx, G, coeffs, ns_mode):
        L = _lib.lib()
        n, rows, cols = G.shape
        g = G.detach().float().contiguous()
        out = torch.empty_like(g)
        ws = torch.empty(L.lact_newton_schulz_workspace_bytes(n, rows, cols, len(coeffs)), dtype=torch.uint8, device=G.device)
        flat = [float(x) for tr in coeffs for x in tr]
        arr = (ctypes.c_float * max(1, len(flat)))(*flat)
        stream = ctypes.c_void_p(torch.cuda.current_stream(G.device).cuda_stream)
        with torch.cuda.device(G.device):
            _lib.check(L.lact_newton_schulz(n, rows, cols, _ptr(g), _ptr(out), len(coeffs), arr, int(ns_mode), _ptr(ws), stream))
        ctx.save_for_backward(g)
        ctx.coeffs, ctx.ns_mode, ctx.in_dtype = tuple(coeffs), int(ns_mode), G.dtype
        return out.to(torch.bfloat16) if ns_mode == NS_PLAIN_BF16 else out

    @staticmethod
    @once_differentiable
    def backward(ctx, dout):
        (g,) = ctx.saved_tensors
        L = _lib.lib()
        n, rows, cols = g.shape
        do = dout.detach().float().contiguous()
        dg = torch.empty_like(g)
        steps = len(ctx.coeffs)
        ws = torch.empty(L.lact_newton_schulz_backward_workspace_bytes(n, rows, cols, steps), dtype=torch.uint8, device=g.device)
        flat = [float(x) for tr in ctx.coeffs for x in tr]
        arr = (ctypes.c_float * max(1, len(flat)))(*flat)
        stream = ctypes.c_void_p(torch.cuda.current_stream(g.device).cuda_stream)
        with torch.cuda.device(g.device):
            _lib.check(L.lact_newton_schulz_backward(n, rows, cols, _ptr(g), _ptr(do), _ptr(dg), steps, arr, ctx.ns_mode, _ptr(ws), stream))
        return dg.to(ctx.in_dtype), None, None


@torch.compiler.disable
def newton_schulz(G: torch.Tensor, coeffs: Sequence[Tuple[float, float, float]], ns_mode: int = NS_PLAIN_BF16) -> torch.Tensor:
    """zeropower_via_newtonschulz5 on [n, rows, cols] (ttt_operation.py:30-66; lact_ttt.py:33-67), differentiable."""
    if G.dim() != 3:
        raise AssertionError("expected a 3-D tensor")          # ttt_operation.py:44
    if not G.is_cuda:
        raise RuntimeError("lact_amd runs on an MI355X only (no CPU path)")
    return _NewtonSchulzFn.apply(G, tuple(tuple(c) for c in coeffs), int(ns_mode))


def check_async_error() -> None:
    """Raises if a barrier wait of the fused Newton-Schulz kernel timed out on the current device since the last check
    (the results of those steps are NaN).  Synchronises the device; call it at a point where the host waits anyway."""
    torch.cuda.synchronize()
    n = _lib.lib().lact_check_async_error()
    if n != 0:
        raise RuntimeError("liblact_hip: " + _lib.lib().lact_last_error().decode())
