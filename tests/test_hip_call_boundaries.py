"""What the layer functions around the operation do at the edges of an ordinary call: gradients that are differentiated again,
transforms, tensors of other devices and shapes, views that start anywhere in memory."""
import pytest
import torch

from lact_amd import layers as HL
from lact_amd import ops
from oracle import lact_oracle as O
from oracle.lact_oracle import rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda"


def randn(*shape, dtype=torch.float32, seed=1, grad=True):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype).to(DEV).requires_grad_(grad)


PROGRAM = ops.Program(steps=((ops.LACT_UPDATE, 0, 24, 0), (ops.LACT_APPLY, 0, 24, 0)), out_len=24)


def operands(b, L, d, dh):
    shapes = [(b, dh, d), (b, d, dh), (b, dh, d)] + [(b, L, d)] * 3 + [(b, L, 1)] * 3
    return [randn(*s, seed=i) for i, s in enumerate(shapes)]


CALLS = {
    "pre": lambda: (lambda x: HL._PreFn.apply(x, 2, 16, True), [randn(1, 5, 96)]),
    "pre_attn": lambda: (lambda x, s, o: HL._PreAttnFn.apply(x, s, o, 2, 16, True), [randn(1, 5, 96), randn(32, 2), randn(32, 2)]),
    "lr": lambda: (lambda x, m: HL._LrFn.apply(x, m, 2, 0.1), [randn(1, 5, 6), randn(1, 5, 2)]),
    "post": lambda: (lambda o, w, g, a: HL._PostFn.apply(o, w, g, 1, 2, True, 1e-5, a), [randn(2, 5, 16), randn(16), randn(1, 5, 2), randn(1, 5, 32)]),
    "newton_schulz": lambda: (lambda x: ops.newton_schulz(x, ops.NS5_COEFFS), [randn(1, 16, 24)]),
    "operation": lambda: (lambda *x: ops.run_program(PROGRAM, *x)[0], operands(1, 24, 16, 24)),
    "window": lambda: (lambda q, k, v: HL.sliding_window_attention(q, k, v, 3), [randn(1, 5, 2, 64, dtype=torch.bfloat16, seed=i) for i in range(3)]),
}


@pytest.mark.parametrize("name", CALLS)
def test_second_derivatives_are_refused(name):
    """The kernels' gradients have no gradient of their own: differentiating them is an error, not a silent constant."""
    print("[gpu-test] second derivative", name, flush=True)
    fn, args = CALLS[name]()
    outs = fn(*args)
    outs = outs if isinstance(outs, tuple) else (outs,)
    grads = torch.autograd.grad(outs, args, [torch.ones_like(o) for o in outs], create_graph=True)   # constants: only the saved tensors depend on the inputs
    first = torch.autograd.grad(fn(*args), args, [torch.ones_like(o) for o in outs])
    assert all(torch.equal(a, b) for a, b in zip(grads, first))
    assert all(g.requires_grad for g in grads)
    penalty = sum(g.float().square().sum() for g in grads)
    with pytest.raises(RuntimeError, match="once_differentiable"):
        torch.autograd.grad(penalty + sum(x.float().sum() for x in args), args, retain_graph=True)
    with pytest.raises(RuntimeError, match="once_differentiable"):
        penalty.backward()


def test_tensors_on_another_device_or_of_another_shape_are_refused():
    """Before anything is launched: the kernels would read them through their addresses."""
    print("[gpu-test] devices and shapes", flush=True)
    for name, changes in (("pre_attn", {1: (64, 2), 2: (32, 1)}), ("lr", {0: (1, 5, 5), 1: (1, 4, 2)}),
                          ("post", {0: (4, 5, 16), 1: (32,), 2: (1, 5, 4), 3: (1, 1, 32)}), ("pre", {0: (1, 5, 48)})):
        for i, shape in changes.items():
            fn, args = CALLS[name]()
            with pytest.raises(ValueError, match="expected shape"):
                fn(*[randn(*shape) if j == i else a for j, a in enumerate(args)])
            if i > 0:
                with pytest.raises(RuntimeError, match="same device"):
                    fn(*[a.detach().cpu() if j == i else a for j, a in enumerate(args)])
    fn, args = CALLS["window"]()
    for i in (1, 2):
        with pytest.raises(RuntimeError, match="device"):
            fn(*[a.detach().cpu() if j == i else a for j, a in enumerate(args)])


@pytest.mark.parametrize("grad", [False, True])
def test_operands_on_another_device_or_of_another_shape_are_refused(grad):
    print("[gpu-test] operands", grad, flush=True)
    args = [t.detach().requires_grad_(grad) for t in operands(2, 24, 16, 24)]
    swap = lambda i, t: [t if j == i else a for j, a in enumerate(args)]
    for i in [0, 1, 2, 4, 5, 6, 7, 8]:
        with pytest.raises(RuntimeError, match="same device"):
            ops.run_program(PROGRAM, *swap(i, args[i].detach().cpu()))
    for i in (3, 4, 5):
        for shape in ((1, 24, 16), (2, 24, 8), (2, 24, 24), (2, 24)) + (((2, 23, 16),) if i == 5 else ()):
            with pytest.raises(ValueError, match="expected q, k, v"):
                ops.run_program(PROGRAM, *swap(i, randn(*shape)))
    with pytest.raises(RuntimeError, match="same device"):
        ops.run_program(PROGRAM, *args, torch.rand(2, 24, 1))
    state = [torch.zeros_like(w) for w in args[:3]]
    with torch.no_grad(), pytest.raises(RuntimeError, match="same device"):
        ops.run_program(PROGRAM, *args, randn(2, 24, 1), (state[0], state[1].cpu(), state[2]))


def window_args(shape=(2, 70, 2, 64), seed=0):
    return [randn(*shape, dtype=torch.bfloat16, seed=seed + i) for i in range(3)]


def close(a, b):
    """Two bf16 attentions of the same inputs, each within a few bf16 roundings of the exact one."""
    assert a.shape == b.shape and rel_l2(a, b) < 1e-2


def test_function_transforms_reach_the_window_attention():
    """vmap, reverse and forward mode of torch.func, batched gradients: what sees tensor operations gets them."""
    print("[gpu-test] window attention under transforms", flush=True)
    attend = lambda *x: HL.sliding_window_attention(*x, 17)
    x = [torch.stack([a, b]).detach() for a, b in zip(window_args(), window_args(seed=3))]
    ref = torch.stack([attend(*[t[i] for t in x]) for i in (0, 1)])
    close(torch.vmap(attend)(*x), ref)
    one = [t[0].clone().requires_grad_() for t in x]
    go = torch.stack([randn(2, 70, 2, 64, dtype=torch.bfloat16, seed=s, grad=False) for s in (7, 8)])
    loops = [torch.autograd.grad(attend(*one), one, g) for g in go]
    for i, a in enumerate(torch.autograd.grad(attend(*one), one, go, is_grads_batched=True)):
        close(a, torch.stack([l[i] for l in loops]))
    pulled = torch.func.vjp(attend, *[t.detach() for t in one])[1](go[0])
    for a, b in zip(pulled, loops[0]):
        close(a, b)
    with torch.autocast("cuda", dtype=torch.float16):
        assert attend(*one).dtype == torch.float16


def test_window_attention_takes_views_that_start_anywhere():
    """Off a 16-byte boundary, with odd strides in dimensions of size one, or with rows further apart than the kernels' limit."""
    print("[gpu-test] window attention views", flush=True)
    for shape in ((2, 70, 2, 64), (1, 1, 2, 64)):
        n = torch.Size(shape).numel()
        ref = [randn(*shape, dtype=torch.bfloat16, seed=i, grad=False) for i in range(3)]
        flat = torch.zeros(n + 1, dtype=torch.bfloat16, device=DEV)
        flat[1:] = ref[0].flatten()
        off = flat[1:].view(shape)
        wide = torch.zeros(shape[0], shape[1], 3 * 128 + 1, dtype=torch.bfloat16, device=DEV)
        wide[..., :128] = ref[1].flatten(2)
        odd = wide[..., :128].unflatten(2, (2, 64))
        assert torch.equal(HL.sliding_window_attention(off, odd, ref[2], 9), HL.sliding_window_attention(*ref, 9))
    far = torch.zeros(2, (1 << 24) + 8, dtype=torch.bfloat16, device=DEV)
    rows = randn(1, 2, 1, 64, dtype=torch.bfloat16, grad=False)
    far[:, :64] = rows[0, :, 0]
    view = far[:, :64].view(1, 2, 1, 64)
    assert torch.equal(HL.sliding_window_attention(view, view, view, None), HL.sliding_window_attention(rows, rows, rows, None))


def test_window_attention_beyond_the_kernel_limits_and_compiled():
    print("[gpu-test] window attention limits", flush=True)
    many = torch.randn(59000, 1, 18, 64, dtype=torch.bfloat16, device=DEV)      # batch entries times heads beyond 2^20
    assert not HL._on_window_kernels(many, many, many) and torch.equal(HL.sliding_window_attention(many, many, many, None), many)
    x = window_args()
    fn = torch.compile(lambda *t: HL.sliding_window_attention(*t, 17), fullgraph=True, backend="aot_eager")
    go = torch.ones(2, 70, 2, 64, dtype=torch.bfloat16, device=DEV)
    for call in (fn, lambda *t: HL.sliding_window_attention(*t, 17)):
        out = call(*x)
        res = [out] + list(torch.autograd.grad(out, x, go))
        first = res if call is fn else first
    assert all(torch.equal(a, b) for a, b in zip(first, res))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_operands_may_start_anywhere(dtype):
    """Contiguous views off a 16-byte boundary, and odd strides in the batch dimension of one entry: the same bits."""
    print("[gpu-test] operands that start anywhere", dtype, flush=True)

    def shifted(t):
        flat = torch.zeros(t.numel() + 1, dtype=t.dtype, device=DEV)
        flat[1:] = t.flatten()
        view = flat[1:].view(t.shape)
        assert view.is_contiguous() and view.data_ptr() % 16
        return view
    args = [t.detach() for t in operands(1, 24, 16, 24)]
    args[3:6] = [t.to(dtype) for t in args[3:6]]
    for i in (3, 4, 5):      # a batch stride that no vector divides
        args[i] = args[i].as_strided(args[i].shape, (24 * 16 + 1, 16, 1))
    ref_args = [t.clone(memory_format=torch.contiguous_format) for t in args]
    go = shifted(randn(1, 24, 16, dtype=dtype, seed=9, grad=False))
    res = []
    for xs in (ref_args, [shifted(t) for t in args], args):
        x = [t.detach().requires_grad_() for t in xs]
        out, ws, _ = ops.run_program(PROGRAM, *x)
        res.append([out, *ws] + list(torch.autograd.grad([out, *ws], x, [go, *[torch.ones_like(w) for w in ws]])))
    for other in res[1:]:
        assert all(torch.equal(a, b) for a, b in zip(other, res[0]))


def test_rows_further_apart_than_the_kernels_reach_are_copied():
    print("[gpu-test] distant rows", flush=True)
    args = [t.detach() for t in operands(1, 24, 16, 24)]
    args[3:6] = [t.bfloat16() for t in args[3:6]]
    far = torch.zeros(24, 1 << 23, dtype=torch.bfloat16, device=DEV)
    far[:, :16] = args[3][0]
    apart = list(args)
    apart[3] = far[:, :16].unsqueeze(0)
    with torch.no_grad():
        assert torch.equal(ops.run_program(PROGRAM, *apart)[0], ops.run_program(PROGRAM, *args)[0])


@pytest.mark.parametrize("dtype,nw,b,d,dh,L,C,muon,momentum", [
    (torch.bfloat16, 3, 6, 64, 96, 300, 130, True, True), (torch.bfloat16, 1, 5, 128, 40, 250, 200, False, False),
    (torch.float32, 2, 2, 40, 72, 150, 60, False, True), (torch.float32, 4, 12, 128, 32, 90, 40, True, False),
    # 16 and 8 threads to a quad of a gradient: 33 entries and 5; quads that end inside a block
    (torch.float32, 1, 33, 40, 24, 50, 30, False, False), (torch.bfloat16, 2, 10, 72, 104, 130, 70, False, True)])
@pytest.mark.parametrize("transposed", [False, True])
def test_shared_weights_are_repeated_ones(dtype, nw, b, d, dh, L, C, muon, momentum, transposed):
    """Batch entries that share initial weights: the bits of a call with the weights repeated, its weight gradients summed over the
    entries (in fp32, one order against another: b / nw roundings of 2^-24 of the sum of magnitudes)."""
    print("[gpu-test] shared weights", dtype, nw, b, d, dh, L, C, muon, momentum, transposed, flush=True)
    inp = {n: t.to("cuda") for n, t in O.make_inputs(b, L, d, dh, seed=51, act_dtype=dtype).items()}
    ws = [inp[n][:nw].clone() for n in ("w0", "w1", "w2")]
    if transposed:
        ws = [w.transpose(1, 2).contiguous().transpose(1, 2) for w in ws]
    rest = [inp[n] for n in ("q", "k", "v", "lr0", "lr1", "lr2")] + ([inp["momentum"]] if momentum else [])
    go = torch.randn(b, L, d, generator=torch.Generator().manual_seed(5)).to(dtype).to("cuda")
    prog = ops.Program(steps=ops.block_causal_steps(L, C), out_len=L, return_state=False, ns_coeffs=ops.NS5_COEFFS if muon else None)
    res = []
    for shared in (True, False):
        x = [w.detach().requires_grad_(True) for w in ws] + [t.clone().requires_grad_(True) for t in rest]
        w = x[:3] if shared else [t.repeat(b // nw, 1, 1) for t in x[:3]]
        if not shared and transposed:     # the layout of the other call's weights, and so the order of their row norms
            w = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in w]
        out, _, _ = ops.run_program(prog, *w, *x[3:], shared_weights=shared)
        with torch.no_grad():
            again, _, _ = ops.run_program(prog, *w, *x[3:], shared_weights=shared)
        if not shared:
            for t in w:
                t.retain_grad()
        out.backward(go)
        res.append(([out.detach(), again] + [t.grad for t in x[3:]], [t.grad for t in x[:3]], None if shared else [t.grad for t in w]))
    for a, r in zip(res[0][0], res[1][0]):
        assert torch.equal(a, r)
    for a, each in zip(res[0][1], res[1][2]):
        each = each.reshape(b // nw, nw, *each.shape[1:]).double()
        assert a.dtype == torch.float32
        assert bool(((a.double() - each.sum(0)).abs() <= b // nw * 2.0 ** -24 * each.abs().sum(0)).all())


def test_shared_weights_are_refused_where_they_do_not_fit():
    inp = {n: t.to("cuda") for n, t in O.make_inputs(4, 60, 32, 32, seed=52, act_dtype=torch.float32).items()}
    rest = [inp[n] for n in ("q", "k", "v", "lr0", "lr1", "lr2")]
    prog = ops.Program(steps=ops.block_causal_steps(60, 30), out_len=60, return_state=False)
    with pytest.raises(ValueError):      # three matrices for four entries
        ops.run_program(prog, *[inp[n][:3] for n in ("w0", "w1", "w2")], *rest, shared_weights=True)
    with pytest.raises(ValueError):      # not asked for
        ops.run_program(prog, *[inp[n][:2] for n in ("w0", "w1", "w2")], *rest)
    with pytest.raises(ValueError):      # the state has one matrix per entry
        ops.run_program(ops.Program(steps=prog.steps, out_len=60), *[inp[n][:2] for n in ("w0", "w1", "w2")], *rest, shared_weights=True)
