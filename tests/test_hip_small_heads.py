"""The kernels that run a whole step of small bf16 heads (csrc/small_heads.h) against the ones that run it in pieces."""
import pytest
import torch

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


# tokens at the edges of a wave's 32, of a split block's 128 and of a block's 256; the hidden size in halves of a stage; more than
# 256 split blocks, which is where whole blocks begin; several steps in one launch
@pytest.mark.parametrize("b,T,d,dh,steps", [
    (1, 1, 64, 32, 1), (2, 33, 64, 96, 1), (3, 127, 96, 64, 1), (2, 129, 96, 160, 1), (5, 300, 128, 32, 1), (2, 257, 128, 288, 1), (3, 128, 128, 128, 3),
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
        out, view, ref = run(t["q"]), run(wide[..., 8:d + 8]), in_pieces(lambda: run(t["q"]))
    assert torch.equal(out, view) and torch.isfinite(out.float()).all()
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
