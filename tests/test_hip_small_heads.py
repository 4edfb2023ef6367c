"""The kernels that run a whole step of small bf16 heads (csrc/small_heads.h) against the ones that run it in pieces."""
import pytest
import torch
from launches import kernels

from lact_amd import _lib, ops
from lact_amd._lib import LACT_APPLY, LACT_UPDATE
from oracle import lact_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
ORDER = ("w0", "w1", "w2", "q", "k", "v", "lr0", "lr1", "lr2")


def in_pieces(fn):
    prev = _lib.lib().lact_set_option(_lib.OPT_PERSISTENT_TILES, 0)
    try:
        return fn()
    finally:
        _lib.lib().lact_set_option(_lib.OPT_PERSISTENT_TILES, prev)


# both sides of the line: hidden units at few tokens, tokens at many hidden units, whole blocks
@pytest.mark.parametrize("b,T,d,dh,one", [
    (1, 64, 128, 256, True), (1, 64, 128, 288, False), (6, 1024, 128, 320, True), (2, 1024, 128, 320, False), (1, 64, 64, 384, True),
    (1, 64, 64, 512, False), (1, 64, 96, 320, True), (2, 129, 96, 512, False), (6, 1024, 128, 512, False), (20, 1024, 128, 512, True),
    (1, 1, 64, 2048, False), (33, 1024, 96, 1024, True), (260, 64, 128, 1024, True)])
def test_apply_takes_the_faster_kernels(b, T, d, dh, one):
    """A wave of the one kernel walks all hidden units, however few tokens there are: few tokens with many of them go in pieces."""
    print("[gpu-test] apply's rule", b, T, d, dh, one, flush=True)
    t = {n: x.to(DEV) for n, x in O.make_inputs(b, T, d, dh, seed=60, act_dtype=torch.bfloat16).items()}
    prog = ops.Program(steps=((LACT_APPLY, 0, T, 0),), out_len=T)
    with torch.no_grad():
        out, names = kernels(lambda: ops.run_program(prog, *[t[n] for n in ORDER])[0])
        ref, pieces = kernels(lambda: in_pieces(lambda: ops.run_program(prog, *[t[n] for n in ORDER])[0]))
    assert ("k_apply_fused" in names) == one and "k_apply_fused" not in pieces
    assert O.rel_l2(out, ref) < 1e-3


# tokens at the edges of a wave's 32, of a split block's 128 and of a block's 256; the hidden size in halves of a stage; more than
# 256 split blocks, which is where whole blocks begin; several steps in one launch
@pytest.mark.parametrize("b,T,d,dh,steps", [
    (1, 1, 64, 32, 1), (2, 33, 64, 96, 1), (3, 127, 96, 64, 1), (2, 129, 96, 160, 1), (5, 300, 128, 32, 1), (30, 257, 128, 288, 1), (3, 128, 128, 128, 3),
    (90, 300, 64, 160, 1), (129, 200, 96, 96, 1), (65, 513, 128, 96, 1), (40, 300, 128, 64, 3)])
def test_apply_in_one_kernel(b, T, d, dh, steps):
    """The same rounded hidden values, summed in another order: a result differs by a rounding where its sum lies next to one (2^-9 of
    a value, rarely: 1e-3 in norm is generous)."""
    print("[gpu-test] apply in one kernel", b, T, d, dh, steps, flush=True)
    L = T * steps
    t = {n: x.to(DEV) for n, x in O.make_inputs(b, L, d, dh, seed=61, act_dtype=torch.bfloat16).items()}
    wide = torch.zeros(b, L, d + 24, dtype=torch.bfloat16, device=DEV)
    wide[..., 8:d + 8] = t["q"]
    args = [t[n] for n in ORDER]
    # several steps on their own weight versions share a launch: an update between any two of them
    prog = []
    for i in range(steps):
        prog.append((LACT_APPLY, i * T, (i + 1) * T, i * T))
        if i + 1 < steps:
            prog.append((LACT_UPDATE, i * T, (i + 1) * T, 0))
    prog = ops.Program(steps=tuple(prog), out_len=L)
    run = lambda q: ops.run_program(prog, *args[:3], q, *args[4:])[0]
    with torch.no_grad():
        (out, names), view, ref = kernels(lambda: run(t["q"])), run(wide[..., 8:d + 8]), in_pieces(lambda: run(t["q"]))
    assert "k_apply_fused" in names and torch.equal(out, view) and torch.isfinite(out.float()).all()
    assert O.rel_l2(out, ref) < (1e-3 if steps == 1 else 1e-2)
    assert torch.equal(out[:, :T], run(t["q"])[:, :T])


def test_infinite_queries_stay_in_their_rows():
    print("[gpu-test] infinite queries", flush=True)
    t = {n: x.to(DEV) for n, x in O.make_inputs(2, 70, 96, 96, seed=62, act_dtype=torch.bfloat16).items()}
    t["q"][0, 40] = float("inf")
    prog = ops.Program(steps=((LACT_APPLY, 0, 70, 0),), out_len=70)
    with torch.no_grad():
        run = lambda: ops.run_program(prog, *[t[n] for n in ORDER])[0]
        out, ref = run(), in_pieces(run)
    rows = torch.isfinite(out.float()).all(dim=-1)
    assert torch.equal(rows, torch.isfinite(ref.float()).all(dim=-1)) and int((~rows).sum()) == 1 and not rows[0, 40]


# tokens at the edges of a wave's 32, of a block's round of 128 and of its splits (down to the 64 that the kernel takes); one and many
# slices of 32 hidden units; more blocks than the chip holds at once; a step that starts inside the sequence, with tokens around
# it that nothing may read
@pytest.mark.parametrize("b,T,d,dh", [(1, 64, 64, 32), (2, 65, 96, 96), (1, 95, 128, 160), (3, 127, 64, 128), (8, 129, 128, 32), (2, 255, 96, 64),
                                      (1, 1500, 128, 256), (5, 1025, 64, 96), (70, 130, 128, 128), (24, 777, 96, 96)])
def test_update_in_one_kernel(b, T, d, dh):
    """The gradients of a step (the momentum states, when there is no earlier one) and the weights it leaves: the same products of the same
    rounded values, summed in another order and rounded to bf16.  A sum is 1e-6 to 1e-5 off, so that one in 1e2 to 1e3 lands on the
    other side of a rounding and moves by 2^-8: 4e-4 in norm at most; 1e-3."""
    print("[gpu-test] update in one kernel", b, T, d, dh, flush=True)
    at, L = 7, T + 40
    t = {n: x.to(DEV) for n, x in O.make_inputs(b, L, d, dh, seed=63, act_dtype=torch.bfloat16).items()}
    for n in ("k", "v", "lr0", "lr1", "lr2"):
        t[n] = t[n].clone()
        t[n][:, :at] = t[n][:, at + T:] = float("nan")
    momentum = torch.full((b, L, 1), 0.9, device=DEV)
    wide = torch.full((b, L, 2 * d + 16), float("nan"), dtype=torch.bfloat16, device=DEV)
    wide[..., 8:d + 8], wide[..., d + 8:2 * d + 8] = t["k"], t["v"]
    prog = ops.Program(steps=((LACT_UPDATE, at, at + T, 0), (LACT_UPDATE, at, at + T, 0), (LACT_APPLY, 0, 32, 0)), out_len=32)
    args = [t[n] for n in ORDER]

    def run(k, v):
        out, w, m = ops.run_program(prog, *args[:4], k, v, *args[6:], momentum=momentum)
        return [out, *w, *m]

    with torch.no_grad():
        (whole, names), view, ref = kernels(lambda: run(t["k"], t["v"])), run(wide[..., 8:d + 8], wide[..., d + 8:2 * d + 8]), in_pieces(lambda: run(t["k"], t["v"]))
    assert "k_update_fused" in names
    for i, (a, c, r) in enumerate(zip(whole, view, ref)):
        assert torch.equal(a, c) and torch.isfinite(a.float()).all()
        assert O.rel_l2(a, r) < 1e-3, (i, O.rel_l2(a, r))


@pytest.mark.parametrize("token", [0, 30, 31, 66, 69])
def test_infinite_tokens_stay_in_their_head(token):
    """70 tokens: the last patch starts at token 38 and clears the 26 that the patch before it holds as well."""
    print("[gpu-test] infinite tokens of an update", token, flush=True)
    t = {n: x.to(DEV) for n, x in O.make_inputs(3, 70, 128, 64, seed=64, act_dtype=torch.bfloat16).items()}
    t["v"][1, token] = float("inf")
    prog = ops.Program(steps=((LACT_UPDATE, 0, 70, 0), (LACT_APPLY, 0, 70, 0)), out_len=70)

    def run():
        out, w, _ = ops.run_program(prog, *[t[n] for n in ORDER])
        return [out, *w]

    with torch.no_grad():
        for a, r in zip(run(), in_pieces(run)):
            fine = torch.isfinite(a.float()).flatten(1).all(dim=1)
            assert torch.equal(fine, torch.isfinite(r.float()).flatten(1).all(dim=1)) and fine.tolist() == [True, False, True]


# tokens at the edges of a wave's 32 and a block's 128 or 256; one and several stages of 32 hidden units (the rings have two and three
# places); all with batch enough that the kernels are taken
@pytest.mark.parametrize("b,T,d,dh", [(255, 127, 64, 32), (128, 129, 64, 64), (5, 4700, 64, 96), (90, 200, 96, 96), (100, 127, 128, 64), (120, 129, 128, 96),
                                      (250, 100, 128, 160), (250, 63, 128, 256)])
def test_tokens_gradients_in_one_kernel(b, T, d, dh):
    """Gradients of a program of two updates: the same products of the same rounded values in another order, on top of weights that the
    forward's kernels sum in another order too (an entry in 1e2 to 1e3 moved by 2^-8, 4e-4 in norm, through a chain of a few
    products; 3e-3).  Rows around the steps stay zero."""
    print("[gpu-test] tokens' gradients in one kernel", b, T, d, dh, flush=True)
    at, L = 5, 2 * T + 9
    inp = {n: x.to(DEV) for n, x in O.make_inputs(b, L, d, dh, seed=65, act_dtype=torch.bfloat16).items()}
    inp["momentum"] = torch.full((b, L, 1), 0.7, device=DEV)
    wide = torch.zeros(b, L, 2 * d + 8, dtype=torch.bfloat16, device=DEV)
    wide[..., 8:d + 8], wide[..., d + 8:] = inp["k"], inp["v"]
    prog = ops.Program(steps=((LACT_UPDATE, at, at + T, 0), (LACT_APPLY, 0, T, 0), (LACT_UPDATE, at + T, at + 2 * T, 0), (LACT_APPLY, T, L, T)), out_len=L)
    go = torch.randn(b, L, d, generator=torch.Generator().manual_seed(3)).bfloat16().to(DEV)
    names = list(ORDER) + ["momentum"]

    def run(views):
        t = {n: x.clone().requires_grad_(True) for n, x in inp.items() if n in names}
        if views:
            packed = wide.clone().requires_grad_(True)
            k, v = packed[..., 8:d + 8], packed[..., d + 8:]
        else:
            k, v = t["k"], t["v"]
        out, ws, _ = ops.run_program(prog, *[t[n] for n in ORDER[:4]], k, v, *[t[n] for n in ORDER[6:]], momentum=t["momentum"])
        loss = [out] + list(ws)
        seeds = [go] + [torch.ones_like(w) * 0.01 for w in ws]
        wanted = [t[n] for n in names if n not in ("k", "v")] + ([packed] if views else [t["k"], t["v"]])
        g = list(torch.autograd.grad(loss, wanted, seeds))
        if views:
            p = g.pop()
            assert float(p[..., :8].float().abs().max()) == 0
            g += [p[..., 8:d + 8], p[..., d + 8:]]
        return g

    (whole, launched), view, ref = kernels(lambda: run(False)), run(True), in_pieces(lambda: run(False))
    assert "k_update_bwd_fused" in launched
    for n, a, c, r in zip([n for n in names if n not in ("k", "v")] + ["k", "v"], whole, view, ref):
        assert torch.isfinite(a.float()).all() and torch.equal(a, c), n
        assert O.rel_l2(a, r) < 3e-3, (n, O.rel_l2(a, r))
        if n in ("k", "v", "lr0", "lr1", "lr2"):
            assert float(a[:, :at].float().abs().max()) == 0 and float(a[:, at + 2 * T:].float().abs().max()) == 0


# three applies between updates: two of them share launches; small steps, which only the apply's kernel takes
@pytest.mark.parametrize("b,T,d,dh", [(1, 1, 64, 32), (2, 33, 96, 64), (3, 127, 128, 96), (24, 257, 128, 160), (2, 300, 64, 96)])
def test_queries_gradients_in_one_kernel(b, T, d, dh):
    print("[gpu-test] queries' gradients in one kernel", b, T, d, dh, flush=True)
    L = 3 * T
    inp = {n: x.to(DEV) for n, x in O.make_inputs(b, L, d, dh, seed=66, act_dtype=torch.bfloat16).items()}
    prog = ops.Program(steps=tuple(s for i in range(3) for s in ((LACT_APPLY, i * T, (i + 1) * T, i * T), (LACT_UPDATE, i * T, (i + 1) * T, 0))), out_len=L)
    go = torch.randn(b, L, d + 8, generator=torch.Generator().manual_seed(3)).bfloat16().to(DEV)[..., :d]      # (rows with a stride)

    def run():
        t = [inp[n].clone().requires_grad_(True) for n in ORDER]
        return torch.autograd.grad(ops.run_program(prog, *t)[0], t, go)

    whole, names = kernels(run)
    assert "k_apply_bwd_fused" in names
    for n, a, r in zip(ORDER, whole, in_pieces(run)):
        assert torch.isfinite(a.float()).all() and O.rel_l2(a, r) < 3e-3, (n, O.rel_l2(a, r))


# the first and the last token of a wave's 32, the last one of a ragged block (whose surplus lanes repeat it)
@pytest.mark.parametrize("token", [0, 31, 32, 69])
def test_infinities_in_the_backward(token):
    """An infinite token of an update spoils its head's gradients, an infinite row of an apply's gradient that head's first weights and its
    own query: nothing else, and the same places as in pieces."""
    print("[gpu-test] infinities in the backward", token, flush=True)
    b, T, d, dh = 200, 70, 64, 32
    inp = {n: x.to(DEV) for n, x in O.make_inputs(b, 2 * T, d, dh, seed=67, act_dtype=torch.bfloat16).items()}
    inp["v"][1, token] = float("inf")
    prog = ops.Program(steps=((LACT_APPLY, 0, T, 0), (LACT_UPDATE, 0, T, 0), (LACT_APPLY, T, 2 * T, T)), out_len=2 * T)
    go = torch.randn(b, 2 * T, d, generator=torch.Generator().manual_seed(3)).bfloat16().to(DEV)
    go[3, token] = float("inf")

    def run():
        t = [inp[n].clone().requires_grad_(True) for n in ORDER]
        return torch.autograd.grad(ops.run_program(prog, *t)[0], t, go)

    whole, names = kernels(run)
    assert {"k_update_bwd_fused", "k_apply_bwd_fused"} <= names
    for n, a, r in zip(ORDER, whole, in_pieces(run)):
        fine = torch.isfinite(a.float())
        assert torch.equal(fine, torch.isfinite(r.float())), n
        heads = set(range(b)) - {1} - ({3} if n in ("w0", "w1", "w2", "q") else set())
        assert fine[sorted(heads)].all() and not fine[1].all(), n
        if n == "q":
            rows = fine[3].all(dim=-1)
            assert int((~rows).sum()) == 1 and not rows[token]
        elif n in ("w0", "w1", "w2"):
            assert not fine[3].all()
        a, r = a.float()[sorted(heads)], r.float()[sorted(heads)]
        assert O.rel_l2(a, r) < 3e-3, n
