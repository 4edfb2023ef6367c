"""CPU-side checks of the C ABI: the library loads, exports every symbol the header declares, and its
host-side validation and buffer sizing behave (no kernel is launched)."""
import ctypes
import os
import re

import pytest

from lact_amd import _lib, ops
from lact_amd._lib import LACT_APPLY, LACT_UPDATE
from oracle import lact_oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def header_functions():
    text = open(os.path.join(ROOT, "include", "lact_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(lact_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    L = _lib.lib()
    names = header_functions()
    assert set(names) == set(_lib.EXPORTS)
    for n in names:
        assert getattr(L, n) is not None
    assert L.lact_version() >= 1


def make_desc(steps, b=2, d=64, dh=64, L=256, **kw):
    arr = (_lib.Step * len(steps))(*[_lib.Step(*s) for s in steps])
    D = _lib.Desc()
    D.b, D.d, D.dh, D.q_len, D.kv_len, D.out_len = b, d, dh, L, L, L
    D.act_dtype, D.n_steps, D.steps = 0, len(steps), ctypes.cast(arr, ctypes.POINTER(_lib.Step))
    D.ns_steps, D.weight_norm = -1, 1
    for name in ("q", "k", "v", "o", "do"):
        setattr(D, name + "_ld", d)
        setattr(D, name + "_bs", L * d)
    for k_, v_ in kw.items():
        setattr(D, k_, v_)
    D._keep = arr
    return D


def sizes(D):
    a, s = ctypes.c_size_t(0), ctypes.c_size_t(0)
    rc = _lib.lib().lact_query_sizes(ctypes.byref(D), ctypes.byref(a), ctypes.byref(s))
    return rc, a.value, s.value


def test_query_sizes_and_validation_messages():
    L = _lib.lib()
    ok = make_desc(ops.block_causal_steps(256, 64))
    rc, saved, scratch = sizes(ok)
    assert rc == 0 and saved > 0 and scratch > 0
    # more updates -> more saved state; Muon adds the Newton-Schulz iterates
    rc, saved2, _ = sizes(make_desc(ops.block_causal_steps(256, 32)))
    assert rc == 0 and saved2 > saved
    coeffs = (ctypes.c_float * 15)(*[x for t in ops.NS5_COEFFS for x in t])
    rc, saved3, _ = sizes(make_desc(ops.block_causal_steps(256, 64), ns_steps=5,
                                    ns_coeffs=ctypes.cast(coeffs, ctypes.POINTER(ctypes.c_float))))
    assert rc == 0 and saved3 > saved

    def err(D):
        rc, _, _ = sizes(D)
        assert rc != 0
        return L.lact_last_error().decode()

    assert "multiples of 8" in err(make_desc(ops.block_causal_steps(256, 64), d=60))
    assert "exceeds kv_len" in err(make_desc(((LACT_UPDATE, 0, 300, 0),)))
    assert "exceeds q_len" in err(make_desc(((LACT_APPLY, 0, 300, 0),)))
    assert "out_len" in err(make_desc(((LACT_APPLY, 0, 256, 8),)))
    assert "empty" in err(make_desc(((LACT_APPLY, 5, 5, 0),)))
    assert "kind" in err(make_desc(((7, 0, 5, 0),)))
    assert "ns_coeffs" in err(make_desc(ops.block_causal_steps(256, 64), ns_steps=5))
    assert "alignment" in err(make_desc(ops.block_causal_steps(256, 64), q_ld=68))
    assert "act_dtype" in err(make_desc(ops.block_causal_steps(256, 64), act_dtype=3))
    for name in ("q_ld", "k_ld", "v_ld", "o_ld"):      # offsets inside a tile are 24-bit products
        assert "too large" in err(make_desc(ops.block_causal_steps(256, 64), **{name: 1 << 23}))
        assert sizes(make_desc(ops.block_causal_steps(256, 64), **{name: (1 << 23) - 8}))[0] == 0
    # a forward-only descriptor keeps less for the backward, and the backward entry point refuses it (before it
    # looks at any pointer: no GPU is needed for this check)
    # (at d = 256: the update's pre-activations are kept for the backward only above d = 128)
    rc, saved_bw, _ = sizes(make_desc(ops.block_causal_steps(256, 64), d=256, dh=256))
    rc_fo, saved_fo, _ = sizes(make_desc(ops.block_causal_steps(256, 64), d=256, dh=256, forward_only=1))
    assert rc == 0 and rc_fo == 0 and saved_fo < saved_bw
    null = ctypes.c_void_p(0)
    fo = make_desc(ops.block_causal_steps(256, 64), forward_only=1)
    assert L.lact_backward(ctypes.byref(fo), *([null] * 22)) != 0
    assert "forward_only" in L.lact_last_error().decode()
    # a carried momentum state is an inference feature: needs use_momentum and forward_only, and costs one more
    # state array in `saved`
    assert "momentum_state_in" in err(make_desc(ops.block_causal_steps(256, 64), momentum_state_in=1, use_momentum=1))
    assert "momentum_state_in" in err(make_desc(ops.block_causal_steps(256, 64), momentum_state_in=1, forward_only=1))
    rc, saved_mo, _ = sizes(make_desc(ops.block_causal_steps(256, 64), forward_only=1, use_momentum=1))
    rc2, saved_st, _ = sizes(make_desc(ops.block_causal_steps(256, 64), forward_only=1, use_momentum=1, momentum_state_in=1))
    assert rc == 0 and rc2 == 0 and saved_st > saved_mo
    assert L.lact_query_sizes(None, None, None) != 0 and "null" in L.lact_last_error().decode()
    assert L.lact_newton_schulz_workspace_bytes(4, 64, 128, 5) > 0
    assert L.lact_newton_schulz_workspace_bytes(0, 64, 128, 5) == 0


@pytest.mark.parametrize("L,C", [(64, 16), (70, 16), (16, 16), (10, 16), (17, 16), (4096, 2048), (32760, 4680)])
def test_schedule_builder_matches_oracle(L, C):
    mine = ops.block_causal_steps(L, C)
    ref = O.block_causal_steps(L, C)
    assert [(s[0], s[1], s[2]) for s in mine] == [(0 if s.kind == O.UPDATE else 1, s.start, s.end) for s in ref]
    assert all(s[3] == s[1] for s in mine if s[0] == LACT_APPLY)


def test_ar_video_schedule_matches_oracle():
    """The video step lists against the oracle's, which the oracle tests pin against the reference's loop bounds: the
    documented case and 300 random argument sets (defaults by -1, cut last windows, updates that stop early,
    repeats).  The oracle slices tensors (a range past the end is cut there); the builder states the cut ranges."""
    import numpy as np
    from lact_amd import ar_video
    cases = [(60, 10, 60, 20, 2)]
    rng = np.random.default_rng(7)
    for _ in range(300):
        L = int(rng.integers(8, 400))
        mb = int(rng.choice([-1, int(rng.integers(1, L + 1))]))
        ul = int(rng.choice([-1, int(rng.integers(1, L + 1))]))
        eff_mb = (L if ul == -1 else ul) if mb == -1 else mb
        ue = int(rng.choice([-1, eff_mb + int(rng.integers(1, L + 40))]))      # the first window may exceed the sequence
        cases.append((L, mb, ul, ue, int(rng.integers(1, 4))))
    for L, mb, ul, ue, rep in cases:
        mine = ar_video._ar_steps(L, L, mb, ul, ue, rep)
        ref = O.ar_video_steps(L, mb, ul, ue, rep)
        cut = [(0 if s.kind == O.UPDATE else 1, min(s.start, L), min(s.end, L)) for s in ref]
        assert [(s[0], s[1], s[2]) for s in mine] == cut, (L, mb, ul, ue, rep)
        assert all(s[2] > s[1] for s in mine), (L, mb, ul, ue, rep)      # no empty range reaches the library


def test_cpu_tensors_are_refused():
    import torch
    w = torch.zeros(1, 8, 8)
    x = torch.zeros(1, 4, 8)
    lr = torch.zeros(1, 4, 1)
    with pytest.raises(RuntimeError, match="no CPU path"):
        from lact_amd import block_causal_lact_swiglu
        block_causal_lact_swiglu(w, w, w, x, x, x, lr, lr, lr, 2)


def cpu_call(**changed):
    """run_program on CPU tensors: whatever it refuses for another reason comes before the device's."""
    import torch
    b, L, d = 1, 8, 8
    t = {n: torch.randn(b, d, d) for n in ("w0", "w1", "w2")} | {n: torch.randn(b, L, d) for n in "qkv"} | {n: torch.rand(b, L, 1) for n in ("lr0", "lr1", "lr2")}
    prog = ops.Program(steps=((LACT_UPDATE, 0, L, 0), (LACT_APPLY, 0, L, 0)), out_len=L)
    return ops.run_program(prog, **(t | changed))


@pytest.mark.parametrize("name", ["w1", "q", "v", "lr2"])
def test_forward_mode_tangents_are_refused(name):
    """Also where nothing requires a gradient and the autograd function is passed by."""
    import torch
    import torch.autograd.forward_ad as fwad
    shape = {"w1": (1, 8, 8), "lr2": (1, 8, 1)}.get(name, (1, 8, 8))
    with fwad.dual_level():
        with pytest.raises(NotImplementedError, match="jvp"):
            cpu_call(**{name: fwad.make_dual(torch.randn(shape), torch.randn(shape))})
    with pytest.raises(RuntimeError, match="HIP device"):
        cpu_call()


@pytest.mark.parametrize("missing", [0, 1, 2])
def test_incomplete_momentum_states_are_refused(missing):
    """Continuing from two of the three states would restart the momentum without a word."""
    import torch
    state = [torch.zeros(1, 8, 8) for _ in range(3)]
    state[missing] = None
    with pytest.raises(ValueError, match="three tensors"):
        cpu_call(momentum=torch.rand(1, 8, 1), momentum_state=tuple(state))
    with pytest.raises(RuntimeError, match="HIP device"):      # nothing reads it without a momentum
        cpu_call(momentum_state=tuple(state))


def test_scratch_grows_with_what_the_steps_hold():
    """Many short steps beside one long one: the buffers of the steps that share a launch are as long as those, not as the longest."""
    def steps(rounds):
        short = [st for i in range(rounds) for st in ((LACT_UPDATE, 64 * i, 64 * (i + 1), 0), (LACT_APPLY, 64 * i, 64 * (i + 1), 64 * i))]
        return short + [(LACT_APPLY, 0, 100000, 64 * rounds)]
    need = lambda rounds, **kw: sizes(make_desc(steps(rounds), b=6, d=128, dh=256, L=110000, **kw))[2]
    per_update = 6 * 3 * 128 * 256 * 4
    assert need(64) < need(2) + 62 * 2 * per_update      # a gradient per version, and row sums and dot products per update
    assert need(64, forward_only=1) < need(64) // 3


def test_programs_are_copied_and_pickled_after_use():
    import copy
    import pickle
    prog = ops.Program(steps=((LACT_UPDATE, 0, 8, 0), (LACT_APPLY, 0, 8, 0)), out_len=8, ns_coeffs=ops.NS5_COEFFS)
    prog.native()
    for other in (copy.deepcopy(prog), copy.copy(prog), pickle.loads(pickle.dumps(prog))):
        assert other == prog and hash(other) == hash(prog) and other.native() is not None


def test_fractional_sizes_are_refused():
    """Also after a call with the whole number, whose schedule is kept."""
    import torch
    from lact_amd import ar_video, nvs, ttt_operation
    t = {n: torch.randn(1, 8, 8) for n in ("w0", "w1", "w2", "q", "k", "v")} | {n: torch.rand(1, 8, 1) for n in ("lr0", "lr1", "lr2")}
    args = list(t.values())
    calls = (lambda x: ttt_operation.block_causal_lact_swiglu(*args, chunk_size=x),
             lambda x: nvs.fast_weight_swish_glu_weight_norm_mini_batch_apply(*args, [(0, x, True, False), (0, 4, False, True)]),
             lambda x: nvs.fast_weight_swish_glu_weight_norm_mini_batch_apply(*args, [(0, 4, True, True)], muon_update_steps=x),
             lambda x: ar_video.ar_fast_weight_swish_glu_weight_norm_mini_batch(*args, 1.0, mini_batch_size=x),
             lambda x: ar_video.ar_fast_weight_swish_glu_weight_norm_mini_batch_inference(*args, 1.0, num_repeat=x, do_update=True))
    for call in calls:
        with pytest.raises(RuntimeError, match="HIP device"):
            call(4)
        for x in (4.0, 4.5):
            with pytest.raises(TypeError):
                call(x)


def test_layer_functions_refuse_cpu_tensors_by_name():
    """The host module's and their Python counterparts: the reason and the device, not an error of a device guard."""
    import torch
    from lact_amd import layers as HL
    host, r = _lib.host(), torch.randn
    pre, scale = (r(1, 5, 96), r(32, 2), r(32, 2)), (1, 32, True)
    post = (r(2, 5, 32), None, None, 1, 2, True, 1e-5, None)
    calls = [(host.layer_pre, (pre[0], *scale)), (host.layer_pre_attn, (*pre, *scale)), (host.layer_lr, (r(1, 5, 3), None, 1, 0.1, False)),
             (host.layer_post, post), (host.linear, (r(1, 5, 32), r(8, 32))), (host.layer_in, (r(1, 5, 32), r(96, 32), r(3, 32), None, None, None, None, None)),
             (HL._PreFn.apply, (pre[0], *scale)), (HL._PreAttnFn.apply, (*pre, *scale)), (HL._LrFn.apply, (r(1, 5, 3), None, 1, 0.1, False)),
             (HL._PostFn.apply, post), (HL.BidirectionalLaCTSwiGLU(32, 16), (r(1, 5, 32),))]
    for fn, args in calls:
        with pytest.raises(RuntimeError, match="runs on an MI355X only.*cpu"):
            fn(*args)
