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


@pytest.mark.parametrize("b,l,h,d,window,growth", [
    (1, 70, 2, 128, 1, 1.0),        # every query sees itself alone
    (2, 300, 64, 64, 64, 1.0),      # 256-row blocks of heads of 64, the window one tile
    (1, 515, 3, 128, 190, 40.0),    # scores that grow along the sequence: the rows' maxima follow them from tile to tile
    (2, 600, 70, 128, 600, 300.0),
    (1, 70, 2, 64, 1, 1.0),         # heads of 64 walk their tiles one after the other
    (1, 515, 3, 64, 190, 40.0),
    (2, 600, 70, 64, 600, 300.0)])
def test_window_attention_scores_and_window_edges(b, l, h, d, window, growth):
    """The scores of a tile are formed one step ahead of their exponentials: window edges inside and on the tiles, and maxima that grow
    from tile to tile by far more than exp2 reaches.  Grown scores leave a handful of probabilities per row, which bf16 rounds to 2^-9
    each and the kernel's output once more; gradients pass through their differences: twice the bounds of the test above."""
    print("[gpu-test] window attention edges", b, l, h, d, window, growth, flush=True)
    from lact_amd import layers as HL
    g = torch.Generator().manual_seed(8)
    q, k, v, go = [torch.randn(b, l, h, d, generator=g) for _ in range(4)]
    k = k * torch.linspace(1.0, growth, l).view(1, l, 1, 1)
    q, k, v, go = [t.bfloat16() for t in (q, k, v, go)]
    dev = [t.to("cuda").requires_grad_(True) for t in (q, k, v)]
    out = HL.sliding_window_attention(*dev, window)
    grads = torch.autograd.grad(out, dev, go.to("cuda"))
    ref_in = [t.double().requires_grad_(True) for t in (q, k, v)]
    ref = LO.sliding_window_attention(*ref_in, window)
    ref_grads = torch.autograd.grad(ref, ref_in, go.double())
    assert rel_l2(out, ref) < 1e-2
    for i, (a, r) in enumerate(zip(grads, ref_grads)):
        assert bool(torch.isfinite(a).all()), i
        if float(r.norm()) > 1e-6 * float(go.double().norm()):      # one visible key: the probabilities are constant
            assert rel_l2(a, r) < 2e-2, i


@pytest.mark.parametrize("dtype,B,L,H,hd", [(torch.float32, 2, 37, 3, 16), (torch.float32, 1, 5, 2, 520), (torch.bfloat16, 1, 4099, 2, 384),
                                             # blocks of the backward by the chunks a lane holds: one and four of bf16, more heads than blocks
                                             (torch.bfloat16, 2, 700, 24, 64), (torch.bfloat16, 1, 2100, 1, 1024), (torch.float32, 1, 9, 600, 136)])
def test_pre_attention_kernel_against_torch(dtype, B, L, H, hd):
    """The layer's pre-processing with the attention's inputs: outputs, and the gradients of the projection and of the rescaling."""
    print("[gpu-test] layer pre with attention", dtype, B, L, H, hd, flush=True)
    from lact_amd import layers as HL
    g = torch.Generator().manual_seed(7)
    qkv = torch.randn(B, L, 3 * H * hd, generator=g).to(dtype)
    scale, offset = torch.rand(H * hd, 2, generator=g) + 0.5, torch.randn(H * hd, 2, generator=g)
    gos = [torch.randn(B * H, L, hd, generator=g).to(dtype) for _ in range(3)] + [torch.randn(B, L, H * hd, generator=g).to(dtype) for _ in range(3)]

    def reference(t, s, o):
        raw = t.chunk(3, dim=-1)
        heads = [torch.nn.functional.silu(r).reshape(B, L, H, hd).transpose(1, 2).reshape(B * H, L, hd) for r in raw]
        norm = lambda x: x / (x.norm(dim=-1, keepdim=True) + 1e-5)
        return [norm(heads[0]), norm(heads[1]), heads[2], raw[0] * s[:, 0] + o[:, 0], raw[1] * s[:, 1] + o[:, 1], raw[2]]

    ref_in = [t.double().requires_grad_(True) for t in (qkv, scale, offset)]
    ref = reference(*ref_in)
    ref_grads = torch.autograd.grad(ref, ref_in, [t.double() for t in gos])
    dev_in = [t.to("cuda").requires_grad_(True) for t in (qkv, scale, offset)]
    out = HL._PreAttnFn.apply(*dev_in, H, hd, True)
    grads = torch.autograd.grad(out, dev_in, [t.to("cuda") for t in gos])
    tol = 1e-5 if dtype == torch.float32 else 6e-3
    for a, r in zip(list(out) + list(grads), list(ref) + list(ref_grads)):
        assert a.shape == r.shape and rel_l2(a, r) < tol
