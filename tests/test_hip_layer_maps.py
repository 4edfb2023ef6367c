"""The linear maps of a layer's input and output under bf16 autocast: the fused functions of the host module against float64,
against the modules they stand in for, and their way back to the modules."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from lact_amd import _lib
from lact_amd import layers as HL
from oracle.lact_oracle import rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda"


def maps(dim, n_lr, n_mom, n_gate, bias, seed=3):
    torch.manual_seed(seed)
    mods = [nn.Linear(dim, 3 * dim, bias=False), nn.Linear(dim, n_lr, bias=bias)] + [nn.Linear(dim, n) if n else None for n in (n_mom, n_gate)]
    return [m.to(DEV) if m is not None else None for m in mods]


# numbers of outputs at the edges of the kernels' groups of four (8, 12, 16, 24; 8, 16), token counts at the edges of a wave's four,
# a block's 16 and 32 and of the weight gradient's 64 and 128 (16 tokens a wave below 512 blocks, 32 from there), channels at
# the edges of a wave's 256
@pytest.mark.parametrize("B,L,dim,n_lr,n_mom,n_gate,bias", [
    (1, 1, 8, 1, 1, 0, False), (1, 63, 256, 8, 0, 1, True), (2, 32, 264, 9, 4, 4, False), (1, 65, 520, 12, 8, 1, True),
    (3, 43, 768, 13, 0, 0, True), (1, 129, 1032, 16, 8, 8, False), (2, 2100, 384, 24, 16, 0, False), (1, 16400, 1024, 17, 5, 5, True),
])
def test_input_maps_against_float64(B, L, dim, n_lr, n_mom, n_gate, bias):
    """Sums of rounded operands in fp32: 2^-9 relative per rounding of x, of a weight, of a gradient and of a result, so a few 1e-3
    in norm (5e-3 asserted; 1e-2 for the few values of a bias gradient); what stays in fp32 (the rates and their gradients) 1e-5."""
    print("[gpu-test] input maps", B, L, dim, n_lr, n_mom, n_gate, bias, flush=True)
    mods = maps(dim, n_lr, n_mom, n_gate, bias)
    x = torch.randn(B, L, dim, device=DEV, requires_grad=True)
    params = [p for m in mods if m is not None for p in m.parameters()]
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert HL._fused_linears(x, *[m for m in mods if m is not None])
        outs = [o for o in HL._input_projections(x, *mods) if o is not None]
    go = [torch.randn(o.shape, device=DEV).to(o.dtype) for o in outs]
    grads = torch.autograd.grad(outs, [x] + params, go)
    xd, pd = x.detach().double().requires_grad_(True), [p.detach().double().requires_grad_(True) for p in params]
    it, ref = iter(pd), []
    for m in mods:
        if m is not None:
            ref.append(F.linear(xd, next(it), next(it) if m.bias is not None else None))
    ref_grads = torch.autograd.grad(ref, [xd] + pd, [g.double() for g in go])
    names = ["qkv", "lr"] + ["mom"] * (n_mom > 0) + ["gate"] * (n_gate > 0)
    for n, a, r in zip(names, outs, ref):
        assert rel_l2(a, r) < (1e-5 if n == "lr" else 5e-3), n
    exact = {id(p) for p in mods[1].parameters()}
    for p, g, r in zip([x] + params, grads, ref_grads):
        assert g.dtype == torch.float32 and g.shape == p.shape
        assert rel_l2(g, r) < (1e-5 if id(p) in exact else 1e-2 if p.dim() == 1 else 5e-3), p.shape


# token counts around one K-step of 64 and around the split's 1024 tokens, tiles of 192 (48 or more of them) and of 128 with ragged
# edges
@pytest.mark.parametrize("T,m,n", [(64, 8, 8), (63, 72, 136), (65, 128, 128), (1000, 136, 264), (2049, 768, 384), (3333, 1344, 1344), (2048, 4608, 192), (5000, 1000, 512)])
def test_weight_gradient_against_float64(T, m, n):
    """Products of bf16 values are exact in fp32; a sum of T of them in fp32 blocks of 16 is good for sqrt(T) 2^-24: 1e-5."""
    print("[gpu-test] weight gradient", T, m, n, flush=True)
    lin = nn.Linear(n, m, bias=False).to(DEV)
    x = torch.randn(1, T, n, device=DEV).bfloat16().requires_grad_(True)
    go = torch.randn(1, T, m, device=DEV).bfloat16()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = HL._linear(lin, x)
    dx, dw = torch.autograd.grad(y, [x, lin.weight], go)
    wb = lin.weight.detach().bfloat16().double()
    assert dw.dtype == torch.float32 and rel_l2(dw, go[0].double().t() @ x.detach()[0].double()) < 1e-5
    assert dx.dtype == torch.bfloat16 and rel_l2(dx, go.double() @ wb) < 4e-3 and rel_l2(y, x.detach().double() @ wb.t()) < 4e-3
    with torch.autocast("cuda", dtype=torch.bfloat16):      # a backward inside the region: the same bits
        inside = torch.autograd.grad(HL._linear(lin, x), [x, lin.weight], go)
    assert torch.equal(inside[0], dx) and torch.equal(inside[1], dw)


def test_partial_gradients_and_unused_outputs():
    """Frozen parameters get no gradient, outputs that nobody uses count as zero, and nothing needs an input that is a leaf of data."""
    print("[gpu-test] partial gradients", flush=True)
    mods = maps(128, 6, 2, 2, True)
    mods[0].weight.requires_grad_(False)
    mods[2].bias.requires_grad_(False)
    x = torch.randn(2, 50, 128, device=DEV)
    wanted = [p for m in mods for p in m.parameters() if p.requires_grad]
    with torch.autocast("cuda", dtype=torch.bfloat16):
        outs = HL._input_projections(x, *mods)
        full = torch.autograd.grad(sum(o.float().sum() for o in outs[1:]), wanted, retain_graph=True)
        some = torch.autograd.grad(outs[1].sum(), wanted, allow_unused=True)
    assert all(g is not None for g in full)
    assert torch.equal(some[0], full[0]) and torch.equal(some[1], full[1])
    assert all(g is None or not g.any() for g in some[2:])
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        again = HL._input_projections(x, *mods)
    assert all(torch.equal(a, b) for a, b in zip(outs, again)) and not again[0].requires_grad


def test_weights_are_cast_once_in_an_autocast_region():
    """As autocast does for the modules: a layer that is called several times in one region keeps one bf16 copy of each weight."""
    print("[gpu-test] casts of the weights", flush=True)
    layer = HL.BidirectionalLaCTSwiGLU(64, 32, use_muon=False).to(DEV)
    x = torch.randn(1, 70, 64, device=DEV)
    copies = {layer.to_qkv.weight: [], layer.o_proj.weight: []}

    def pack(t):
        for w, seen in copies.items():
            if t.dtype == torch.bfloat16 and t.shape == w.shape and torch.equal(t, w.detach().bfloat16()):
                seen.append(t)
        return t

    def step(regions):
        before = {w: len(seen) for w, seen in copies.items()}
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
            for _ in range(regions):
                with torch.autocast("cuda", dtype=torch.bfloat16):
                    y = layer(x) + layer(x)
        assert all(len(seen) == before[w] + 2 * regions for w, seen in copies.items())
        return y

    first = torch.autograd.grad(step(1).float().square().sum(), [layer.to_qkv.weight, layer.o_proj.weight])
    assert all(seen[0].data_ptr() == seen[1].data_ptr() for seen in copies.values())
    with torch.no_grad():
        for w in copies:
            w.mul_(-1)
    again = torch.autograd.grad(step(1).float().square().sum(), [layer.to_qkv.weight, layer.o_proj.weight])   # the next region casts anew
    assert all(not torch.equal(a, b) for a, b in zip(first, again))


def test_second_derivatives_of_the_input_maps_are_refused():
    """(What follows them has none either.)"""
    print("[gpu-test] second derivative of the maps", flush=True)
    mods = maps(64, 3, 1, 1, False)
    x = torch.randn(1, 70, 64, device=DEV, requires_grad=True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        outs = HL._input_projections(x, *mods)
        g = torch.autograd.grad(sum(o.float().sum() for o in outs), x, create_graph=True)[0]
        with pytest.raises(RuntimeError, match="once_differentiable"):
            torch.autograd.grad(g.square().sum() + x.sum(), x)


@pytest.mark.parametrize("T,dtype", [(70, torch.bfloat16), (63, torch.bfloat16), (200, torch.float32)])
def test_output_projection_differentiates_twice(T, dtype):
    """Like the module it stands in for: gradients with a graph are the gradients without one (the weight's summed in fp32 in another
    order: 1e-5), and their derivatives those of float64 within a few bf16 roundings of factors (2^-9 each: 1e-2)."""
    print("[gpu-test] output projection twice", T, dtype, flush=True)
    torch.manual_seed(7)
    lin = nn.Linear(96, 64, bias=False).to(DEV)
    x = torch.randn(2, T, 96, device=DEV).to(dtype).requires_grad_(True)
    go, c = torch.randn(2, T, 64, device=DEV).bfloat16(), torch.randn(64, 96, device=DEV)
    e = torch.randn(2, T, 96, device=DEV)

    def derivatives(f, x, w, go, c, e):
        y = f(x)
        once = torch.autograd.grad(y, [x, w], go, retain_graph=True)
        twice = torch.autograd.grad(y.pow(2), [x, w], go, create_graph=True)
        return y, once, twice, torch.autograd.grad((twice[0] * e).sum() + (twice[1] * c).sum(), [x, w])

    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert HL._fused_linears(x, lin)
        y, once, twice, second = derivatives(lambda t: HL._linear(lin, t), x, lin.weight, go, c, e)
        graph = torch.autograd.grad(HL._linear(lin, x), [x, lin.weight], go, create_graph=True)
    xd, wd = x.detach().double().requires_grad_(True), lin.weight.detach().double().requires_grad_(True)
    _, once_d, twice_d, second_d = derivatives(lambda t: F.linear(t, wd), xd, wd, go.double(), c.double(), e.double())
    assert once[1].dtype == graph[1].dtype == torch.float32 and torch.equal(once[0], graph[0]) and rel_l2(once[1], graph[1]) < 1e-5
    for a, r in zip([*once, *twice, *second], [*once_d, *twice_d, *second_d]):
        assert rel_l2(a, r) < 1e-2


def test_output_projection_takes_batches_of_gradients():
    print("[gpu-test] batches of gradients", flush=True)
    lin = nn.Linear(96, 64, bias=False).to(DEV)
    x = torch.randn(2, 70, 96, device=DEV).bfloat16().requires_grad_(True)
    go = torch.randn(3, 2, 70, 64, device=DEV).bfloat16()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = HL._linear(lin, x)
    batch = torch.autograd.grad(y, [x, lin.weight], go, retain_graph=True, is_grads_batched=True)
    mapped = torch.func.vmap(lambda g: torch.autograd.grad(y, [x, lin.weight], g, retain_graph=True))(go)
    for i in range(3):
        single = torch.autograd.grad(y, [x, lin.weight], go[i], retain_graph=True)
        for got in (batch, mapped):      # sums in another order in front of dx's rounding: one in a hundred lands beside it
            assert rel_l2(got[0][i], single[0]) < 1e-3 and rel_l2(got[1][i], single[1]) < 1e-5


def test_gradient_penalty_on_the_output_projection():
    """|d loss / d o_proj.weight|^2 as part of a loss: a second derivative through o_proj and first ones through everything else."""
    print("[gpu-test] gradient penalty", flush=True)
    torch.manual_seed(9)
    layer = HL.BidirectionalLaCTSwiGLU(64, 32, use_muon=False).to(DEV)
    x = torch.randn(1, 90, 64, device=DEV)

    def penalty():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = layer(x)
        g = torch.autograd.grad(y.float().square().mean(), layer.o_proj.weight, create_graph=True)[0]
        return torch.autograd.grad(g.square().sum(), [layer.o_proj.weight, layer.o_norm.weight, layer.to_qkv.weight, layer.w1])

    fused = penalty()
    layer.o_proj.register_forward_hook(lambda m, a, o: None)
    for a, r in zip(fused, penalty()):      # the module rounds the weight's gradient, and its gradient's, to bf16
        assert rel_l2(a, r) < 2e-2


def test_modules_are_called_where_someone_may_look():
    """Hooks, subclasses, replaced forwards, other types, no autocast: the modules run, as they did."""
    print("[gpu-test] modules that are looked at", flush=True)
    x = torch.randn(1, 70, 64, device=DEV)

    def fused(mods, x=x, dtype=torch.bfloat16, enabled=True):
        with torch.autocast("cuda", dtype=dtype, enabled=enabled):
            return HL._fused_linears(x, *mods)
    plain = [nn.Linear(64, 8).to(DEV)]
    assert fused(plain) and not fused(plain, dtype=torch.float16) and not fused(plain, enabled=False) and not fused(plain, x=x[0])
    seen = []
    hooked = nn.Linear(64, 8).to(DEV)
    hooked.register_forward_hook(lambda m, a, o: seen.append(o))
    sub = type("Sub", (nn.Linear,), {})(64, 8).to(DEV)
    replaced = nn.Linear(64, 8).to(DEV)
    replaced.forward = lambda t: t
    half = nn.Linear(64, 8).to(DEV).bfloat16()
    assert not any(fused([m]) for m in (hooked, sub, replaced, half))
    layer = HL.BidirectionalLaCTSwiGLU(64, 32, use_muon=False).to(DEV)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = layer(x)
        layer.lr_proj.register_forward_hook(lambda m, a, o: seen.append(o))
        close = layer(x)
        assert len(seen) == 1 and rel_l2(close, y) < 1e-2
        assert not torch.func.functional_call(layer, {n: p.detach() for n, p in layer.named_parameters()}, (x,)).requires_grad


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_native_and_python_functions_agree(dtype):
    """The layer functions of the host module and their Python counterparts launch the same kernels: same bits, same gradients (the
    RMSNorm weight's sums over partial rows in another order: 1e-5)."""
    print("[gpu-test] native functions", dtype, flush=True)
    B, L, H, hd = 2, 37, 3, 32
    r = lambda *s, d=dtype: torch.randn(*s, device=DEV).to(d).requires_grad_(True)
    qkv, scale, offset = r(B, L, 3 * H * hd), r(H * hd, 2, d=torch.float32), r(H * hd, 2, d=torch.float32)
    lr, mom = r(B, L, 3 * H, d=torch.float32), r(B, L, H)
    o, w, gate, add = r(B * H, L, hd), r(hd, d=torch.float32), r(B, L, H), r(B, L, H * hd)
    host = _lib.host()
    for native, python, args, consts in (
            (host.layer_pre, HL._PreFn.apply, (qkv,), (H, hd, True)),
            (host.layer_pre_attn, HL._PreAttnFn.apply, (qkv, scale, offset), (H, hd, True)),
            (host.layer_lr, HL._LrFn.apply, (lr, mom), (H, 0.3, True)),
            (lambda a, b, c, d, *k: host.layer_post(a, b, c, *k, d), lambda a, b, c, d, *k: HL._PostFn.apply(a, b, c, *k, d), (o, w, gate, add), (B, H, True, 1e-5))):
        res = []
        for fn in (native, python):
            out = fn(*args, *consts)
            out = [out] if isinstance(out, torch.Tensor) else list(out)
            torch.manual_seed(5)
            res.append(out + list(torch.autograd.grad(out, args, [torch.randn_like(t) for t in out])))
        for a, b in zip(*res):
            assert a.dtype == b.dtype and a.shape == b.shape
            assert torch.equal(a, b) or (a.shape == w.shape and rel_l2(a, b) < 1e-5)


# head sizes at both sides of every change of lanes and chunks; a token count that no wave's rows divide
@pytest.mark.parametrize("hd", [4, 64, 68, 96, 100, 128, 132, 192, 196, 384, 388, 512, 516, 768, 772, 1024])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_of_every_head_size_against_float64(hd, dtype):
    """silu, L2 norm, rescaling, RMSNorm and gate over rows of hd elements: a few roundings of the type per value."""
    print("[gpu-test] rows", hd, dtype, flush=True)
    B, L, H, tol = 2, 19, 3, 1e-2 if dtype == torch.bfloat16 else 1e-5
    g = torch.Generator().manual_seed(hd)
    r = lambda *s, t=dtype: torch.randn(*s, generator=g).to(t)
    args = {"qkv": r(B, L, 3 * H * hd), "scale": r(H * hd, 2, t=torch.float32), "offset": r(H * hd, 2, t=torch.float32)}
    post = {"o": r(B * H, L, hd), "w": r(hd, t=torch.float32), "gate": r(B, L, H), "add": r(B, L, H * hd)}

    def ref_pre(qkv, scale, offset):
        x = qkv.view(B, L, 3, H, hd).permute(2, 0, 3, 1, 4)
        y = F.silu(x)
        heads = lambda t: t.reshape(B * H, L, hd)
        normed = [heads(y[i] / (y[i].norm(dim=-1, keepdim=True) + 1e-5)) for i in (0, 1)]
        flat = qkv.view(B, L, 3, H * hd)
        return (*normed, heads(y[2]), flat[:, :, 0] * scale[:, 0] + offset[:, 0], flat[:, :, 1] * scale[:, 1] + offset[:, 1], flat[:, :, 2])

    def ref_post(o, w, gate, add):
        n = o * torch.rsqrt(o.square().mean(dim=-1, keepdim=True) + 1e-5) * w
        return (n.view(B, H, L, hd).transpose(1, 2) * F.silu(gate).unsqueeze(-1)).reshape(B, L, H * hd) + add,

    host = _lib.host()
    for fn, ref, inp in ((lambda qkv, scale, offset: host.layer_pre_attn(qkv, scale, offset, H, hd, True), ref_pre, args),
                         (lambda qkv, **k: host.layer_pre(qkv, H, hd, True), lambda qkv, **k: ref_pre(qkv, **k)[:3], args),
                         (lambda o, w, gate, add: [host.layer_post(o, w, gate, B, H, True, 1e-5, add)], ref_post, post)):
        a = {n: t.to(DEV).requires_grad_(True) for n, t in inp.items()}
        d = {n: t.double().requires_grad_(True) for n, t in inp.items()}
        out, want = fn(**a), ref(**d)
        assert all(rel_l2(x, y) < tol for x, y in zip(out, want))
        go = [r(*t.shape) for t in want]
        got = torch.autograd.grad(out, list(a.values()), [t.to(DEV) for t in go], allow_unused=True)
        exact = torch.autograd.grad(want, list(d.values()), [t.double() for t in go], allow_unused=True)
        for n, x, y in zip(inp, got, exact):
            assert y is None or not y.any() or rel_l2(x, y) < tol, n


# more rows than the blocks of one pass take (2048 blocks of 4 waves forward, 1024 backward), ending inside a wave's rows: four, eight and
# two rows a wave, fp32
@pytest.mark.parametrize("L,H,hd,dtype", [(16390, 2, 64, torch.bfloat16), (32773, 2, 96, torch.bfloat16), (16411, 1, 384, torch.bfloat16), (16399, 2, 36, torch.float32)])
def test_rows_beyond_one_pass_of_the_waves(L, H, hd, dtype):
    """RMSNorm, gate and sum over many rows: every row's result and gradients are those of a call on a part of the rows (the same
    arithmetic per row, hence the same bits; the weight's gradient, a sum over all rows, against float64)."""
    print("[gpu-test] many rows", L, H, hd, dtype, flush=True)
    g = torch.Generator().manual_seed(hd)
    r = lambda *s, t=dtype: torch.randn(*s, generator=g).to(t).to(DEV)
    o, w, gate, add, dy = r(H, L, hd), r(hd, t=torch.float32), r(1, L, H), r(1, L, H * hd), r(1, L, H * hd)
    host = _lib.host()

    def run(rows):
        x = [o[:, rows].contiguous().requires_grad_(True), w.clone().requires_grad_(True), gate[:, rows].contiguous().requires_grad_(True),
             add[:, rows].contiguous().requires_grad_(True)]
        y = host.layer_post(*x[:3], 1, H, True, 1e-5, x[3])
        return [y.detach(), *torch.autograd.grad(y, x, dy[:, rows].contiguous())]

    whole, parts = run(slice(0, L)), [run(slice(a, min(a + 4000, L))) for a in range(0, L, 4000)]
    for i in (0, 1, 3, 4):     # y, do, dgate, dadd
        assert torch.equal(whole[i], torch.cat([p[i] for p in parts], dim=1)), i
    n = o.double() * torch.rsqrt(o.double().square().mean(-1, keepdim=True) + 1e-5)
    dt = (dy.double().view(L, H, hd) * F.silu(gate.double()).to(dtype).double().view(L, H, 1)).transpose(0, 1)
    # fp32 sums (some thousand roundings of 2^-24 that mostly cancel); a bf16 gate that rounds the other way here is 2^-9 of one addend
    assert rel_l2(whole[2], (dt * n).sum((0, 1))) < (1e-5 if dtype == torch.float32 else 1e-4)
