"""The small-tile pipeline (csrc/gemm_async.h) at the edges of its 64 x 64 tiles and 32 / 64-element K-steps: whole forward and
backward passes of the operation against the oracle, fp32 and bf16 with head sizes that are no multiple of 16."""
import pytest
import torch
from launches import kernels

from oracle import lact_oracle as O

pytestmark = pytest.mark.gpu
ORDER = ("w0", "w1", "w2", "q", "k", "v", "lr0", "lr1", "lr2", "momentum")


@pytest.mark.parametrize("dtype,b,L,d,dh,C", [
    (torch.float32, 1, 33, 8, 8, 16), (torch.float32, 2, 150, 64, 64, 65), (torch.float32, 2, 200, 72, 40, 63),
    (torch.float32, 1, 2 * 2100, 32, 96, 2100),      # token reductions in several splits, forward and backward
    (torch.bfloat16, 2, 150, 24, 72, 65), (torch.bfloat16, 1, 90, 8, 136, 40)])
def test_small_tiles_against_oracle(dtype, b, L, d, dh, C):
    print("[gpu-test] small tiles", dtype, b, L, d, dh, C, flush=True)
    import lact_amd
    inp = O.make_inputs(b, L, d, dh, seed=31, act_dtype=dtype)
    num = O.Numerics(autocast=dtype == torch.bfloat16)
    cpu = {n: inp[n].clone().requires_grad_(True) for n in ORDER}
    dev = {n: inp[n].to("cuda").requires_grad_(True) for n in ORDER}
    ref = O.block_causal_lact_swiglu(*[cpu[n] for n in ORDER[:9]], C, False, cpu["momentum"], num=num)
    out = lact_amd.block_causal_lact_swiglu(*[dev[n] for n in ORDER[:9]], C, False, dev["momentum"])
    go = torch.randn(ref.shape, generator=torch.Generator().manual_seed(3)).to(dtype)
    gr = torch.autograd.grad(ref, [cpu[n] for n in ORDER], go)
    gh = torch.autograd.grad(out, [dev[n] for n in ORDER], go.to("cuda"))
    tol = 1e-4 if dtype == torch.float32 else 1e-2
    assert O.rel_l2(out, ref) < tol
    for n, a, r in zip(ORDER, gh, gr):
        if float(r.double().norm()) > 0:
            # one dot product per head and chunk: held to a looser bound in bf16, as everywhere
            assert O.rel_l2(a, r) < (tol if n != "momentum" or dtype == torch.float32 else 3e-2), n


@pytest.mark.parametrize("b,L,d,dh,C", [(2, 300, 96, 96, 130), (1, 200, 16, 48, 100), (2, 290, 80, 112, 129), (3, 260, 160, 224, 128)])
def test_partial_k_steps_against_oracle(b, L, d, dh, C):
    """bf16 head sizes that end inside a K-step of the dedicated-loader kernels (one, two or three of its four sub-steps)."""
    test_small_tiles_against_oracle(torch.bfloat16, b, L, d, dh, C)


@pytest.mark.parametrize("dtype,b,L,d,dh,C", [(torch.bfloat16, 1, 3 * 2112, 64, 1088, 2112), (torch.bfloat16, 2, 3 * 2100, 48, 32, 2100),
                                              (torch.float32, 1, 600, 16, 1040, 200)])
def test_partial_sums_are_read_by_the_row_kernels(dtype, b, L, d, dh, C):
    """Three chunks whose token reductions run in several splits (the row kernels add them up, with the momentum step on the way),
    and rows longer than what a wave keeps in registers (1024 columns)."""
    test_small_tiles_against_oracle(dtype, b, L, d, dh, C)


@pytest.mark.parametrize("dtype,C", [(torch.float32, 300), (torch.bfloat16, 2200)])
def test_several_apply_steps_on_one_weight_version(dtype, C):
    """Two apply steps where one would do, on the newest and on an earlier version: the gradients are those of the one step."""
    print("[gpu-test] several applies", dtype, C, flush=True)
    from lact_amd import ops
    from lact_amd._lib import LACT_APPLY, LACT_UPDATE
    inp = {n: t.to("cuda") for n, t in O.make_inputs(1, 2 * C, 64, 32, seed=35, act_dtype=dtype).items()}
    go = torch.randn(1, 4 * C, 64, generator=torch.Generator().manual_seed(5)).to(dtype).to("cuda")
    U = [(LACT_UPDATE, 0, C, 0), (LACT_UPDATE, C, 2 * C, 0)]
    one = (U[0], (LACT_APPLY, 0, 2 * C, 0), U[1], (LACT_APPLY, 0, 2 * C, 2 * C))
    two = (U[0], (LACT_APPLY, 0, C, 0), (LACT_APPLY, C, 2 * C, C), U[1], (LACT_APPLY, 0, C, 2 * C), (LACT_APPLY, C, 2 * C, 3 * C))
    res = []
    for steps in (one, two):
        x = [inp[n].clone().requires_grad_(True) for n in ORDER]
        out, _, _ = ops.run_program(ops.Program(steps=steps, out_len=4 * C), *x)
        res.append([out] + list(torch.autograd.grad(out, x, go)))
    for n, a, r in zip(("out",) + ORDER, res[1], res[0]):
        assert O.rel_l2(a, r) < (1e-5 if dtype == torch.float32 else 1e-2), n


@pytest.mark.parametrize("dtype,b,C,order", [(torch.float32, 2, 72, (0, 1, 2, 3, 4)), (torch.bfloat16, 3, 136, (4, 3, 2, 1, 0)),
                                             (torch.bfloat16, 1, 64, (0, 2, 4, 1, 3)), (torch.float32, 1, 40, (2, 2, 2, 1, 0))])
def test_apply_steps_of_several_versions_in_one_launch(dtype, b, C, order):
    """Apply steps on consecutive weight versions, equally spaced (ascending, descending, in two runs) or on the same rows, against
    the same steps cut in halves, which no launch covers together: outputs and gradients agree."""
    print("[gpu-test] grouped applies", dtype, b, C, order, flush=True)
    from lact_amd import ops
    from lact_amd._lib import LACT_APPLY, LACT_UPDATE
    n = len(order)
    inp = {k: t.to("cuda") for k, t in O.make_inputs(b, n * C, 48, 80, seed=36, act_dtype=dtype).items()}
    go = torch.randn(b, n * C, 48, generator=torch.Generator().manual_seed(6)).to(dtype).to("cuda")
    res = []
    for parts in (1, 2):
        steps, h = [], C // parts
        for i, a in enumerate(order):
            steps += [(LACT_APPLY, a * C + p * h, a * C + (p + 1) * h, i * C + p * h) for p in range(parts)]
            steps.append((LACT_UPDATE, i * C, (i + 1) * C, 0))
        x = [inp[k].clone().requires_grad_(True) for k in ORDER]
        out, _, _ = ops.run_program(ops.Program(steps=tuple(steps), out_len=n * C), *x)
        res.append([out] + list(torch.autograd.grad(out, x, go)))
    for k, a, r in zip(("out",) + ORDER, *res):
        assert O.rel_l2(a, r) < (1e-5 if dtype == torch.float32 else 1e-2), k


@pytest.mark.parametrize("dtype,b,d,update,apply", [(torch.float32, 2, 64, 1100, 1024), (torch.float32, 1, 40, 2049, 2048),
                                                     (torch.bfloat16, 2, 48, 1100, 1024), (torch.bfloat16, 2, 64, 1664, 1600)])
def test_grouped_apply_steps_shorter_than_the_updates(dtype, b, d, update, apply):
    """Apply steps that one launch covers, of fewer tokens than the updates and cut into at least as many splits (the buffers are
    sized for the launch, not for the longest step): outputs and gradients against the oracle."""
    print("[gpu-test] grouped applies, shorter than the updates", dtype, b, d, update, apply, flush=True)
    from lact_amd import ops
    from lact_amd._lib import LACT_APPLY, LACT_UPDATE
    L, rounds = 4 * update, range(0, 4 * update, update)
    inp = O.make_inputs(b, L, d, 64, seed=38, act_dtype=dtype)
    go = torch.randn(b, L, d, generator=torch.Generator().manual_seed(8)).to(dtype)
    prog = ops.Program(steps=tuple(st for r in rounds for st in ((LACT_UPDATE, r, r + update, 0), (LACT_APPLY, r, r + apply, r))), out_len=L)
    steps = [st for r in rounds for st in (O.Step(O.UPDATE, r, r + update), O.Step(O.APPLY, r, r + apply))]
    dev = [inp[n].to("cuda").requires_grad_(True) for n in ORDER]
    out, _, _ = ops.run_program(prog, *dev)
    res = [out] + list(torch.autograd.grad(out, dev, go.to("cuda")))
    cpu = [inp[n].clone().requires_grad_(True) for n in ORDER]
    ref, _, _ = O.run_program(*cpu[:9], steps, num=O.Numerics(autocast=dtype == torch.bfloat16), momentum=cpu[9])
    refs = [ref] + list(torch.autograd.grad(ref, cpu, go))
    for n, a, r in zip(("out",) + ORDER, res, refs):
        # the bounds of test_small_tiles_against_oracle
        assert O.rel_l2(a, r) < (1e-4 if dtype == torch.float32 else 3e-2 if n == "momentum" else 1e-2), n


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d,dh", [(128, 256), (72, 40), (8, 72)])
def test_transposed_weights_are_read_as_they_lie(dtype, d, dh):
    """Fast weights given as transposed views (read in place) against contiguous ones: the row norms are summed in another
    order, everything else is the same arithmetic.  With and without an update; the returned weights of the latter are exact."""
    print("[gpu-test] transposed weights", dtype, d, dh, flush=True)
    from lact_amd import ops
    from lact_amd._lib import LACT_APPLY, LACT_UPDATE
    b, L = 3, 90
    inp = {n: t.to("cuda") for n, t in O.make_inputs(b, L, d, dh, seed=32, act_dtype=dtype).items()}
    plain = [inp[n] for n in ORDER[:9]]
    views = [w.transpose(1, 2).contiguous().transpose(1, 2) for w in plain[:3]] + plain[3:]
    for steps in (((LACT_APPLY, 0, L, 0),), ((LACT_UPDATE, 0, L, 0), (LACT_APPLY, 0, L, 0))):
        prog = ops.Program(steps=steps, out_len=L)
        (out_p, w_p, _), (out_v, w_v, _) = ops.run_program(prog, *plain), ops.run_program(prog, *views)
        assert O.rel_l2(out_v, out_p) < (2e-6 if dtype == torch.float32 else 1e-3)
        for a, r, w in zip(w_v, w_p, plain[:3]):
            assert O.rel_l2(a, r) < 1e-6
            if len(steps) == 1:
                assert torch.equal(a, w) and torch.equal(r, w)


# rows of one, one and a little, and two and a half passes of 256 columns
@pytest.mark.parametrize("d,dh", [(256, 40), (264, 33 * 8), (640, 72)])
def test_transposed_weights_of_many_columns(d, dh):
    """The weights a call without updates hands back and what it applies, from transposed views and contiguous ones: the same bits."""
    print("[gpu-test] transposed weights, many columns", d, dh, flush=True)
    from lact_amd import ops
    from lact_amd._lib import LACT_APPLY
    inp = {n: t.to("cuda") for n, t in O.make_inputs(2, 40, d, dh, seed=36, act_dtype=torch.bfloat16).items()}
    plain = [inp[n] for n in ORDER[:9]]
    views = [w.transpose(1, 2).contiguous().transpose(1, 2) for w in plain[:3]] + plain[3:]
    prog = ops.Program(steps=((LACT_APPLY, 0, 40, 0),), out_len=40)
    with torch.no_grad():
        (out_p, w_p, _), (out_v, w_v, _) = ops.run_program(prog, *plain), ops.run_program(prog, *views)
    assert torch.equal(out_p, out_v)
    for a, r, w in zip(w_v, w_p, plain[:3]):
        assert torch.equal(a, w) and torch.equal(r, w)


@pytest.mark.parametrize("b,d,dh,L,stacked", [
    (3, 128, 256, 200, False), (2, 64, 64, 100, False), (1, 96, 96, 100, False), (2, 32, 224, 80, False), (2, 256, 64, 130, False),
    (2, 96, 160, 90, False), (5, 128, 128, 90, False), (2, 128, 64, 90, True)])
def test_newton_schulz_in_one_block_is_bit_identical(b, d, dh, L, stacked):
    """Matrices that fit one block (csrc/ns_local.h) against the launches per iteration: the same bits in output, weights and, with
    the iterates that the kernel keeps for it, every gradient."""
    print("[gpu-test] local newton-schulz", b, d, dh, L, stacked, flush=True)
    from lact_amd import _lib, ops
    from lact_amd._lib import LACT_APPLY, LACT_UPDATE
    inp = {n: t.to("cuda") for n, t in O.make_inputs(b, L, d, dh, seed=33, act_dtype=torch.bfloat16).items()}
    go = torch.randn(b, L, d, generator=torch.Generator().manual_seed(4)).bfloat16().to("cuda")
    for coeffs, mode in ((ops.NS5_COEFFS, ops.NS_AUTOCAST), ((ops.NS_CLASSIC,) * 3, ops.NS_PLAIN_BF16)):
        prog = ops.Program(steps=((LACT_UPDATE, 0, L, 0), (LACT_APPLY, 0, L, 0)), out_len=L, ns_coeffs=coeffs, ns_mode=mode, muon_stacked=stacked)
        res = []
        for fused in (1, 0):
            _lib.lib().lact_set_option(_lib.OPT_FUSED_NEWTON_SCHULZ, fused)
            try:
                leaves = [inp[n].clone().requires_grad_(True) for n in ORDER[:9]]
                (out, ws, _), launched = kernels(lambda: ops.run_program(prog, *leaves))
                assert ("k_ns_local" in launched) == (fused == 1)
                grads = torch.autograd.grad(out, leaves, go)
                with torch.no_grad():
                    out_inf, ws_inf, _ = ops.run_program(prog, *[inp[n] for n in ORDER[:9]])
                res.append([out.detach(), *[w.detach() for w in ws], out_inf, *ws_inf, *grads])
            finally:
                _lib.lib().lact_set_option(_lib.OPT_FUSED_NEWTON_SCHULZ, 1)
        for a, r in zip(*res):
            assert torch.equal(a, r)


@pytest.mark.parametrize("scale", [1.0, 2.0 ** -70, 2.0 ** -101, 2.0 ** -118, 2.0 ** 40])
@pytest.mark.parametrize("zeros", [False, True])
def test_normalisation_of_extreme_gradients(scale, zeros):
    """The quotient in front of the iterations: by two fused multiply-adds where nothing leaves the normal range, by a division where an
    entry is zero or below 2^-100 or the norm above 2^25.  The launch of its own always divides: the same bits."""
    print("[gpu-test] normalisation", scale, zeros, flush=True)
    from lact_amd import _lib, ops
    from lact_amd._lib import LACT_APPLY, LACT_UPDATE
    inp = {n: t.to("cuda") for n, t in O.make_inputs(2, 90, 64, 96, seed=35, act_dtype=torch.bfloat16).items()}
    for n in ("lr0", "lr1", "lr2"):
        inp[n] = inp[n] * scale
    if zeros:
        inp["k"][..., 5] = 0
    prog = ops.Program(steps=((LACT_UPDATE, 0, 90, 0), (LACT_APPLY, 0, 90, 0)), out_len=90, ns_coeffs=ops.NS5_COEFFS[:1])
    res = []
    for fused in (1, 0):
        _lib.lib().lact_set_option(_lib.OPT_FUSED_NEWTON_SCHULZ, fused)
        try:
            with torch.no_grad():
                (out, ws, _), launched = kernels(lambda: ops.run_program(prog, *[inp[n] for n in ORDER[:9]]))
            assert ("k_ns_local" in launched) == (fused == 1)
            res.append([out, *ws])
        finally:
            _lib.lib().lact_set_option(_lib.OPT_FUSED_NEWTON_SCHULZ, 1)
    for a, r in zip(*res):
        assert torch.isfinite(a.float()).all() and torch.equal(a, r)


# tokens that end inside a tile of 256 and inside its first half, hidden units inside one of 128; K-steps 6, 7, 12; steps that share a launch
@pytest.mark.parametrize("b,d,dh,T", [(6, 384, 640, 1100), (9, 448, 392, 1000), (4, 768, 832, 1300), (3, 512, 1536, 1152)])
def test_wide_hidden_tiles_have_the_same_bits(b, d, dh, T):
    """The 256 x 128 tiles of an update's and an apply backward's hidden stage (which these shapes take: two rounds of 128 x 128 tiles against
    one) against persistent 128 x 128 tiles: every product over k in the same order."""
    print("[gpu-test] wide tiles", b, d, dh, T, flush=True)
    from lact_amd import _lib, ops
    from lact_amd._lib import LACT_APPLY, LACT_UPDATE
    L = 2 * T
    inp = {n: t.to("cuda") for n, t in O.make_inputs(b, L, d, dh, seed=71, act_dtype=torch.bfloat16).items()}
    go = torch.randn(b, L, d, generator=torch.Generator().manual_seed(5)).bfloat16().to("cuda")
    prog = ops.Program(steps=((LACT_APPLY, 0, T, 0), (LACT_UPDATE, 0, T, 0), (LACT_APPLY, T, L, T), (LACT_UPDATE, T, L, 0)), out_len=L)

    def step():
        leaves = [inp[n].clone().requires_grad_(True) for n in ORDER[:9]]
        out, ws, _ = ops.run_program(prog, *leaves)
        return [out.detach(), *[w.detach() for w in ws], *torch.autograd.grad(out, leaves, go)]

    res = []
    for mask in (1, 7):
        prev = _lib.lib().lact_set_option(_lib.OPT_PERSISTENT_TILES, mask)
        try:
            values, names = kernels(step)
            res.append(values)
            assert ({"k_update_hidden_wide", "k_apply_bwd_hidden_wide"} <= names) == (mask == 1)
            assert ({"k_hidden_persist<update>", "k_hidden_persist<apply_bwd>"} <= names) == (mask == 7)
        finally:
            _lib.lib().lact_set_option(_lib.OPT_PERSISTENT_TILES, prev)
    for a, r in zip(*res):
        assert torch.isfinite(a.float()).all() and torch.equal(a, r)


# 64 x 64 tiles of the hidden stages and of the row GEMMs: 224 and 224, 256 and 256, 255 and 85 (dh = 136: the last half tile holds eight
# units), 270 and 90; an update of 70 tokens among long ones, which takes the tiles of the longest
@pytest.mark.parametrize("b,d,dh,T,last,half", [(14, 128, 128, 512, 512, {"hidden", "rows"}), (16, 128, 128, 512, 70, set()),
                                                (17, 40, 136, 265, 265, {"hidden", "rows"}), (18, 40, 136, 300, 70, {"rows"}),
                                                (3, 72, 104, 333, 70, {"hidden", "rows"})])
def test_half_tiles_against_oracle(b, d, dh, T, last, half):
    """fp32 launches on either side of the number of tiles below which half tiles are taken: forward and backward, the learning rates'
    gradients (sums over the columns of a tile) among them."""
    print("[gpu-test] half tiles", b, d, dh, T, last, flush=True)
    from lact_amd import ops
    from lact_amd._lib import LACT_APPLY, LACT_UPDATE
    L = T + last
    inp = O.make_inputs(b, L, d, dh, seed=39, act_dtype=torch.float32)
    go = torch.randn(b, L, d, generator=torch.Generator().manual_seed(9))
    prog = ops.Program(steps=((LACT_UPDATE, 0, T, 0), (LACT_APPLY, 0, T, 0), (LACT_UPDATE, T, L, 0), (LACT_APPLY, T, L, T)), out_len=L)
    steps = [O.Step(O.UPDATE, 0, T), O.Step(O.APPLY, 0, T), O.Step(O.UPDATE, T, L), O.Step(O.APPLY, T, L)]

    def step():
        dev = [inp[n].to("cuda").requires_grad_(True) for n in ORDER]
        out, _, _ = ops.run_program(prog, *dev)
        return [out] + list(torch.autograd.grad(out, dev, go.to("cuda")))

    res, names = kernels(step)
    assert ("k_update_bwd_hidden<half>" in names) == ("hidden" in half) and ("k_update_bwd_hidden" in names) == ("hidden" not in half)
    # the update's products of the short second one are few whatever the first one's are
    assert any(n.startswith("k_row_gemm<") and n.endswith(",half>") for n in names) == ("rows" in half or last < T)
    cpu = [inp[n].clone().requires_grad_(True) for n in ORDER]
    ref, _, _ = O.run_program(*cpu[:9], steps, num=O.Numerics(autocast=False), momentum=cpu[9])
    refs = [ref] + list(torch.autograd.grad(ref, cpu, go))
    for n, a, r in zip(("out",) + ORDER, res, refs):
        assert O.rel_l2(a, r) < 1e-4, n       # the bound of test_small_tiles_against_oracle


def same_specials(a, r):
    a, r = a.detach().float().cpu(), r.detach().float()
    assert torch.isinf(r).any()
    assert torch.equal(torch.isnan(a), torch.isnan(r)) and torch.equal(torch.isinf(a), torch.isinf(r))
    assert torch.equal(a[torch.isinf(a)], r[torch.isinf(r)])


@pytest.mark.parametrize("dtype,d,T", [(torch.bfloat16, 24, 13), (torch.float32, 40, 13), (torch.bfloat16, 64, 70), (torch.bfloat16, 48, 135)])
def test_infinities_pass_the_ragged_end_of_a_contraction(dtype, d, T):
    """An infinite operand at the last place of a contraction that ends inside a K-step, in the features and in the tokens: what the
    copies bring in past the end must add nothing, not the NaN of zero times infinity."""
    print("[gpu-test] infinities", dtype, d, T, flush=True)
    from lact_amd import ops
    from lact_amd._lib import LACT_APPLY, LACT_UPDATE
    num = O.Numerics(autocast=dtype == torch.bfloat16)
    inp = O.make_inputs(1, T, d, 40, seed=41, act_dtype=dtype)
    inp["q"][..., -1] = 1
    args = [inp[n] for n in ORDER[:9]]
    hot = [t.clone() for t in args]
    hot[0][0, 3, -1] = float("inf")      # the last feature of one row of w0
    out, _, _ = ops.run_program(ops.Program(steps=((LACT_APPLY, 0, T, 0),), out_len=T), *[t.to("cuda") for t in hot])
    same_specials(out, O.run_program(*hot, [O.Step(O.APPLY, 0, T)], num=num)[0])
    hot = [t.clone() for t in args]
    for lr in hot[6:]:
        lr[:, -1] = float("inf")         # the last token of all three gradients, which the momentum states hold
    prog = ops.Program(steps=((LACT_UPDATE, 0, T, 0), (LACT_APPLY, 0, T, 0)), out_len=T)
    _, _, ms = ops.run_program(prog, *[t.to("cuda") for t in hot], inp["momentum"].to("cuda"))
    _, _, refs = O.run_program(*hot, [O.Step(O.UPDATE, 0, T), O.Step(O.APPLY, 0, T)], num=num, momentum=inp["momentum"])
    for a, r in zip(ms, refs):
        same_specials(a, r)
    # without the row norm the weights hold them too
    prog = ops.Program(steps=((LACT_UPDATE, 0, T, 0), (LACT_APPLY, 0, T, 0)), out_len=T, weight_norm=False)
    _, ws, _ = ops.run_program(prog, *[t.to("cuda") for t in hot])
    _, refs, _ = O.run_program(*hot, [O.Step(O.UPDATE, 0, T), O.Step(O.APPLY, 0, T)], num=num, weight_norm=False)
    for a, r in zip(ws, refs):
        same_specials(a, r)


# w0 and w2 held transposed (dh > d), w1 (d > dh); whole tiles of 192 and of 128, tiles that end inside one; one split of the tokens
@pytest.mark.parametrize("b,d,dh,T", [(2, 256, 512, 1000), (1, 384, 192, 700), (3, 208, 328, 130), (1, 392, 144, 90), (1, 192, 576, 64)])
@pytest.mark.parametrize("carried", [False, True])
def test_momentum_step_of_matrices_held_transposed(b, d, dh, T, carried):
    """The momentum step in the epilogue of the token reduction, without Newton-Schulz iterations behind it (they amplify a rounding):
    returned weights and momentum states against the oracle, from a carried state (read where it lies) and without one."""
    print("[gpu-test] folded momentum step", b, d, dh, T, carried, flush=True)
    from lact_amd import ops
    from lact_amd._lib import LACT_APPLY, LACT_UPDATE
    inp = O.make_inputs(b, T, d, dh, seed=61, act_dtype=torch.bfloat16)
    g = torch.Generator().manual_seed(7)
    state = [1e-3 * torch.randn(b, *s, generator=g) for s in ((dh, d), (d, dh), (dh, d))] if carried else None
    num = O.Numerics(autocast=True)
    prog = ops.Program(steps=((LACT_UPDATE, 0, T, 0), (LACT_APPLY, 0, T, 0)), out_len=T, ns_coeffs=())
    dev = [inp[n].to("cuda") for n in ORDER]

    def step():
        with torch.no_grad():
            return ops.run_program(prog, *dev, momentum_state=[m.to("cuda") for m in state] if carried else None)

    (out, ws, ms), names = kernels(step)
    assert "k_momentum_prep" not in names and any(n.startswith("k_token_reduce_dma") for n in names)
    ref, wr, mr = O.run_program(*[inp[n] for n in ORDER[:9]], [O.Step(O.UPDATE, 0, T), O.Step(O.APPLY, 0, T)], num=num, momentum=inp["momentum"],
                                ns_coeffs=(), **({"momentum_state": state} if carried else {}))
    # bounds: a token sum rounded to bf16 after the roundings of its operands (test_small_tiles_against_oracle); the weights take the
    # gradient's direction at the norm of one
    for a, r in zip([out, *ws, *ms], [ref, *wr, *mr]):
        assert O.rel_l2(a, r) < 1e-2


@pytest.mark.parametrize("dtype,muon,kernel", [(torch.bfloat16, True, None), (torch.float32, True, "k_momentum_prep"), (torch.bfloat16, False, None)])
@pytest.mark.parametrize("where", ["aligned", "unaligned", "in place"])
def test_carried_momentum_states_anywhere_in_memory(dtype, muon, kernel, where):
    """The library reads a carried state where it lies, or, where 16-byte loads do not reach it, a copy; a caller may have the new state
    written over it.  The bits of a call on aligned states of its own: in the epilogue of the token reduction, in the momentum kernel, and
    in the row norm's."""
    print("[gpu-test] carried states in memory", dtype, muon, where, flush=True)
    import ctypes
    from lact_amd import _lib, ops
    from lact_amd._lib import LACT_APPLY, LACT_UPDATE
    b, L, d, dh = 2, 100, 64, 128
    inp = O.make_inputs(b, L, d, dh, seed=62, act_dtype=dtype)
    dev = [inp[n].to("cuda").contiguous() for n in ORDER]
    g = torch.Generator().manual_seed(8)
    state = [1e-3 * torch.randn(b, *s, generator=g).to("cuda") for s in ((dh, d), (d, dh), (dh, d))]
    steps = ((LACT_UPDATE, 0, L, 0), (LACT_APPLY, 0, L, 0))
    prog = ops.Program(steps=steps, out_len=L, ns_coeffs=ops.NS5_COEFFS if muon else None)
    with torch.no_grad():
        out, ws, ms = ops.run_program(prog, *dev, momentum_state=[m.clone() for m in state])

    lib, keep = _lib.lib(), []
    D = _lib.Desc()
    D.b, D.d, D.dh, D.q_len, D.kv_len, D.out_len, D.act_dtype = b, d, dh, L, L, L, _lib.LACT_BF16 if dtype == torch.bfloat16 else _lib.LACT_F32
    arr, coeffs = (_lib.Step * 2)(*[_lib.Step(*s) for s in steps]), (ctypes.c_float * 15)(*[x for t in ops.NS5_COEFFS for x in t])
    D.n_steps, D.steps, D.ns_steps, D.weight_norm = 2, ctypes.cast(arr, ctypes.POINTER(_lib.Step)), 5 if muon else -1, 1
    if muon:
        D.ns_coeffs = ctypes.cast(coeffs, ctypes.POINTER(ctypes.c_float))
    D.use_momentum = D.forward_only = D.momentum_state_in = 1
    for n in ("q", "k", "v", "o", "do"):
        setattr(D, n + "_ld", d)
        setattr(D, n + "_bs", L * d)
    saved, scratch = ctypes.c_size_t(), ctypes.c_size_t()
    _lib.check(lib.lact_query_sizes(ctypes.byref(D), ctypes.byref(saved), ctypes.byref(scratch)))
    buffers = [torch.empty(n.value, dtype=torch.uint8, device="cuda") for n in (saved, scratch)]

    def lies(t):
        room = torch.zeros(t.numel() + 4, device="cuda")
        keep.append(room)
        at = room[where == "unaligned":][:t.numel()].view(t.shape)
        assert (at.data_ptr() % 16 != 0) == (where == "unaligned")
        return at.copy_(t)
    m_in = [lies(m) for m in state]
    m_out = m_in if where == "in place" else [torch.empty_like(m) for m in state]
    w_out, o = [torch.empty_like(w) for w in state], torch.empty_like(dev[3])
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    three = lambda ts: (ctypes.c_void_p * 3)(*[t.data_ptr() for t in ts])
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    call = lambda: _lib.check(lib.lact_forward_from_state(ctypes.byref(D), *[ptr(t) for t in dev], three(m_in), ptr(o), three(w_out), three(m_out),
                                                          *[ptr(t) for t in buffers], stream))
    _, names = kernels(call)
    assert kernel is None or kernel in names
    for a, r in zip([o, *w_out, *m_out], [out, *ws, *ms]):
        assert torch.equal(a, r)
