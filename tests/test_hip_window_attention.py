"""The sliding-window attention kernels (csrc/window_attention.h) against the float64 oracle attention, output and gradients,
at the edges of their 32-row waves, 64-row tiles and 128 / 256-row blocks, with q, k, v as views of one packed projection."""
import pytest
import torch

from oracle import lact_layers_oracle as LO
from oracle.lact_oracle import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,l,h,d,window", [
    (1, 5, 1, 64, 2), (1, 64, 1, 128, 64), (2, 129, 3, 128, 33), (1, 257, 2, 64, 65), (2, 777, 4, 128, 200), (1, 300, 5, 64, None),
    (2, 1030, 26, 128, 256)])      # the last one is large enough for 256-row blocks
def test_window_attention_against_oracle(b, l, h, d, window):
    print("[gpu-test] window attention", b, l, h, d, window, flush=True)
    from lact_amd import layers as HL
    g = torch.Generator().manual_seed(6)
    packed = torch.randn(b, l, 3 * h * d, generator=g).bfloat16()
    go = torch.randn(b, l, h, d, generator=g).bfloat16()
    x = packed.to("cuda").requires_grad_(True)
    out = HL.sliding_window_attention(*[t.reshape(b, l, h, d) for t in x.chunk(3, dim=-1)], window)
    gx, = torch.autograd.grad(out, [x], go.to("cuda"))
    x64 = packed.double().requires_grad_(True)
    ref = LO.sliding_window_attention(*[t.reshape(b, l, h, d) for t in x64.chunk(3, dim=-1)], window)
    gr, = torch.autograd.grad(ref, [x64], go.double())
    assert out.dtype == torch.bfloat16 and rel_l2(out, ref) < 5e-3
    for i, (a, r) in enumerate(zip(gx.chunk(3, dim=-1), gr.chunk(3, dim=-1))):
        assert rel_l2(a, r) < 1e-2, i
