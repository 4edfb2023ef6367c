"""The work a program hands to this framework, as cases that can be timed and compared.

Every case is one call of a public entry point over inputs that are already on the GPU: the block-causal operation of the
language model (training), the update/apply program of view synthesis (reconstruction and rendering), the interleaved
operation of the video model (training) and its inference step, the bidirectional operation, and the layer classes around
them.  `listed` names one case per use at the sizes of the repository's configurations, `draw` gives others of the same
ranges.
"""
import math

import torch
import torch.nn.functional as F

from lact_amd import layers, minimal, nvs, ttt_operation
from lact_amd.ar_video import (ar_fast_weight_swish_glu_weight_norm_mini_batch_inference_with_momentum,
                               ar_fast_weight_swish_glu_weight_norm_mini_batch_with_momentum)

ORDER = ("w0", "w1", "w2", "q", "k", "v", "lr0", "lr1", "lr2")
LARGEST_FLOPS = 2.0e12


def listed():
    return [
        # Training step of the language model's operation at the 760M shape: 4 sequences x 4 heads, two chunks.
        dict(name="llm train 760M", path="block_causal", b=16, tokens=4096, d=384, dh=384, chunk=2048, muon=True, momentum=True,
             dtype="bf16"),
        # The same operation on one long sequence: sixteen chunks one after the other, few heads.
        dict(name="llm train long context", path="block_causal", b=4, tokens=32768, d=384, dh=384, chunk=2048, muon=False,
             momentum=True, dtype="bf16"),
        # The operation with its default switches (no Muon, no momentum) on a sequence that no chunk or tile divides.
        dict(name="llm train ragged", path="block_causal", b=6, tokens=5003, d=256, dh=512, chunk=1000, muon=False, momentum=False,
             dtype="bf16"),
        # Full precision training of the operation at a small model's head.
        dict(name="llm train fp32", path="block_causal", b=8, tokens=2048, d=128, dh=128, chunk=512, muon=False, momentum=True,
             dtype="fp32"),
        # View synthesis: fast weights from 8 input views of 1024 tokens, then one target view.
        dict(name="nvs reconstruct", path="nvs", b=6, update=8192, apply=1024, d=128, dh=256, iters=5, dtype="bf16"),
        # Rendering one more view with the fast weights of the reconstruction: apply only, the smallest call.
        dict(name="nvs render", path="nvs", b=6, update=0, apply=1024, d=128, dh=256, iters=5, dtype="bf16"),
        # Video model, block-causal training step at the Wan 1.3B shape: 21 latent frames of 1560 tokens, 12 heads.
        dict(name="video train 12 heads", path="block_causal", b=12, tokens=32760, d=128, dh=256, chunk=4680, muon=False,
             momentum=True, dtype="bf16"),
        # Video model, interleaved operation of the 3-frame-chunk configuration: clean and noisy chunk per window, wide heads.
        dict(name="video train wide heads", path="video", b=2, tokens=60840, d=768, dh=1536, chunk=4680, muon=False, dtype="bf16"),
        # One denoising call of the video model that also writes its chunk into the fast weights, states carried along.
        dict(name="video inference step", path="video_step", b=2, tokens=4680, d=768, dh=1536, update=True, muon=True, dtype="bf16"),
        # The bidirectional operation at the size of its example configuration, full precision, forward.
        dict(name="bidirectional small fp32", path="bidirectional", b=2, tokens=1024, d=64, dh=64, muon=True, dtype="fp32"),
        # The causal layer with window attention, training step under bf16 autocast at the 760M width.
        dict(name="causal layer train", path="causal_layer", batch=4, tokens=4096, dim=1536, head=384, attn_head=128, chunk=2048,
             window=2048),
        # The bidirectional layer in a transformer of width 768 with 8 heads, ragged token count.
        dict(name="bidirectional layer train", path="bidirectional_layer", batch=3, tokens=2500, dim=768, head=96),
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        case = _draw(rng)
        # a 32-bit product costs some 25 times one of bf16
        if work(case)["flops"] * (25 if case.get("dtype") == "fp32" else 1) <= LARGEST_FLOPS:
            return case


def _draw(rng):
    path = rng.choice(("block_causal", "block_causal", "block_causal_fp32", "nvs", "nvs", "video", "video_step", "bidirectional",
                       "causal_layer", "bidirectional_layer"))
    d, dh = rng.choice(((64, 64), (64, 128), (96, 96), (128, 128), (128, 256), (192, 192), (256, 256), (256, 512), (384, 384), (512, 512)))
    if path == "block_causal":
        chunk = _spread(rng, 256, 5000)
        muon = rng.random() < 0.5 and d >= 128
        # Muon: the bf16 Newton-Schulz iterations of an update amplify one rounding to percents of what follows, more so at small
        # matrices and in chains of updates, which no two implementations share: one update and heads of 128 or more here
        chunks = 1 + rng.random() if muon else rng.uniform(1.5, 8)
        return dict(path=path, b=_spread(rng, 2, 48), tokens=int(chunk * chunks) + 1, d=d, dh=dh, chunk=chunk, muon=muon,
                    momentum=rng.random() < 0.5, dtype="bf16")
    if path == "block_causal_fp32":
        chunk = _spread(rng, 128, 1024)
        return dict(path="block_causal", b=_spread(rng, 1, 16), tokens=int(chunk * rng.uniform(1.5, 5)), d=min(d, 256), dh=min(dh, 256),
                    chunk=chunk, muon=False, momentum=rng.random() < 0.5, dtype="fp32")
    if path == "nvs":
        tokens = _spread(rng, 200, 4096)
        return dict(path=path, b=_spread(rng, 2, 48), update=tokens * rng.choice((0, 1, 4, 8)), apply=tokens, d=d, dh=dh, iters=5,
                    dtype="bf16")
    if path == "video":
        d, dh = rng.choice(((128, 256), (256, 512), (384, 768), (768, 1536)))
        chunk = _spread(rng, 600, 4680)
        return dict(path=path, b=_spread(rng, 1, 12), tokens=chunk * (2 * rng.randint(1, 6) + 1), d=d, dh=dh, chunk=chunk, muon=False,
                    dtype="bf16")
    if path == "video_step":
        d, dh = rng.choice(((128, 256), (256, 512), (384, 768), (768, 1536)))
        return dict(path=path, b=_spread(rng, 1, 24), tokens=_spread(rng, 390, 9360), d=d, dh=dh, update=rng.random() < 0.5,
                    muon=rng.random() < 0.5, dtype="bf16")
    if path == "bidirectional":
        dtype = rng.choice(("bf16", "fp32"))
        return dict(path=path, b=_spread(rng, 1, 16), tokens=_spread(rng, 200, 4096), d=min(d, 256), dh=min(dh, 256),
                    muon=rng.random() < 0.5, dtype=dtype)
    if path == "causal_layer":
        head = rng.choice((128, 256, 384, 512))
        chunk = _spread(rng, 256, 2048)
        return dict(path=path, batch=_spread(rng, 1, 4), tokens=int(chunk * rng.uniform(1.1, 2)), dim=head * rng.randint(1, 4),
                    head=head, attn_head=rng.choice((64, 128)), chunk=chunk, window=rng.choice((chunk, 512, 2048)))
    head = rng.choice((64, 96, 128, 192, 256))
    return dict(path=path, batch=_spread(rng, 1, 4), tokens=_spread(rng, 200, 4096), dim=head * rng.randint(2, 8), head=head)


# ---- inputs -----------------------------------------------------------------------------------------------------------
def _operation_inputs(b, tokens, d, dh, dtype, seed, transposed=False, queries=None):
    """Fast weights ~ N(0, 1/fan-in), q and k of unit length, v ~ N(0, 1), rates softplus(N(0, 1) - 3), one per token."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    act = torch.bfloat16 if dtype == "bf16" else torch.float32
    randn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    t = {"w0": randn(b, dh, d) / math.sqrt(d), "w1": randn(b, d, dh) / math.sqrt(dh), "w2": randn(b, dh, d) / math.sqrt(d)}
    if transposed:
        t = {n: (w * math.sqrt(2.0)).transpose(1, 2).contiguous() for n, w in t.items()}
    t["q"] = F.normalize(randn(b, tokens if queries is None else queries, d), dim=-1).to(act)
    t["k"] = F.normalize(randn(b, tokens, d), dim=-1).to(act)
    t["v"] = randn(b, tokens, d).to(act)
    for n in ("lr0", "lr1", "lr2"):
        t[n] = F.softplus(randn(b, tokens, 1) - 3.0)
    t["momentum"] = torch.sigmoid(randn(b, tokens, 1) + 2.2)
    t["go"] = randn(b, tokens, d).to(act)
    return t


def prepare(case, seed):
    c, path = case, case["path"]
    if path in ("causal_layer", "bidirectional_layer"):
        torch.manual_seed(seed)
        with torch.device("cuda"):
            if path == "causal_layer":
                layer = layers.CausalLaCTSwiGLUWithSlidingWindowAttn(c["dim"], c["head"], c["attn_head"], lact_chunk_size=c["chunk"],
                                                                     window_size=c["window"])
            else:
                layer = layers.BidirectionalLaCTSwiGLU(c["dim"], c["head"], use_muon=False)
        g = torch.Generator(device="cuda").manual_seed(seed + 1)
        x = torch.randn(c["batch"], c["tokens"], c["dim"], generator=g, device="cuda").requires_grad_(True)
        go = torch.randn(c["batch"], c["tokens"], c["dim"], generator=g, device="cuda").bfloat16()
        return {"case": c, "layer": layer, "x": x, "go": go, "wanted": [x] + list(layer.parameters())}
    if path == "nvs":
        total = c["update"] + c["apply"]
        t = _operation_inputs(c["b"], total, c["d"], c["dh"], c["dtype"], seed, transposed=True)
        program = [nvs.TTTOperator(0, c["update"], True, False)] if c["update"] else []
        program.append(nvs.TTTOperator(c["update"], total, False, True))
        return {"case": c, "args": [t[n] for n in ORDER], "program": program}
    t = _operation_inputs(c["b"], c["tokens"], c["d"], c["dh"], c["dtype"], seed)
    state = {"case": c, "momentum": t["momentum"], "go": t["go"], "args": [t[n] for n in ORDER]}
    if path == "video_step":
        # momentum states as an earlier update leaves them: sums over a chunk of rate-weighted outer products
        g = torch.Generator(device="cuda").manual_seed(seed + 1)
        scale = math.sqrt(c["tokens"] / c["d"]) * 0.02
        state["carried"] = [torch.randn(w.shape, generator=g, device="cuda") * scale for w in state["args"][:3]]
    if path in ("block_causal", "video"):
        leaves = state["args"] + ([t["momentum"]] if c.get("momentum", True) else [])
        state["wanted"] = [x.requires_grad_(True) for x in leaves]
    return state


def run(state):
    c, path = state["case"], state["case"]["path"]
    if path in ("causal_layer", "bidirectional_layer"):
        with torch.autocast(device_type="cuda", dtype=torch.bfloat16):
            out = state["layer"](state["x"])
        return [out.detach()] + list(torch.autograd.grad(out, state["wanted"], state["go"]))
    if path == "nvs":
        with torch.no_grad():
            return nvs.fast_weight_swish_glu_weight_norm_mini_batch_apply(*state["args"], state["program"], c["iters"])
    if path == "bidirectional":
        with torch.no_grad():
            return minimal.bidirectional_lact_swiglu(*state["args"], c["muon"])
    if path == "video_step":
        with torch.no_grad():
            return ar_fast_weight_swish_glu_weight_norm_mini_batch_inference_with_momentum(
                *state["args"], 1.0, do_update=c["update"], use_moun=c["muon"], fw_momentum=state["momentum"],
                dw0_momentum=state["carried"][0], dw1_momentum=state["carried"][1], dw2_momentum=state["carried"][2],
                use_momentum=True)
    if path == "video":
        out, *weights = ar_fast_weight_swish_glu_weight_norm_mini_batch_with_momentum(
            *state["args"], 1.0, mini_batch_size=c["chunk"], update_every=2 * c["chunk"], use_moun=c["muon"],
            fw_momentum=state["momentum"], use_momentum=True)
    else:
        out = ttt_operation.block_causal_lact_swiglu(*state["args"], c["chunk"], c["muon"], state["momentum"] if c["momentum"] else None)
        weights = []
    grads = torch.autograd.grad(out, state["wanted"], state["go"])
    return [out.detach()] + [w.detach() for w in weights] + list(grads)


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------
def _newton_schulz_flops(b, d, dh, iters):
    r, c = min(d, dh), max(d, dh)
    return 3.0 * iters * (4.0 * r * r * c + 2.0 * r ** 3) * b


def work(case):
    c, path = case, case["path"]
    if path in ("causal_layer", "bidirectional_layer"):
        n, dim, head = c["batch"] * c["tokens"], c["dim"], c["head"]
        heads = dim // head
        flops = 2.0 * n * dim * (4 * dim + 3 * heads)                          # to_qkv, o_proj and the rates
        if path == "causal_layer":
            flops += 2.0 * n * dim * 2 * heads                                 # momentum and gate
            updated = c["chunk"] if c["tokens"] > c["chunk"] else 0
            flops += c["batch"] * heads * (6.0 * head * head * c["tokens"] + 12.0 * head * head * updated)
            flops += _newton_schulz_flops(c["batch"] * heads, head, head, 5) * (1 if updated else 0)
            w = min(c["window"], c["tokens"])
            pairs = c["tokens"] * w - w * (w - 1) / 2.0
            flops += 4.0 * c["batch"] * dim * pairs
        else:
            flops += c["batch"] * heads * 18.0 * head * head * c["tokens"]
        params = 4.0 * dim * dim + 3.0 * dim * head
        return {"bytes": 4.0 * n * dim * 2 + 2.0 * n * dim * 2 + 8.0 * params, "flops": 3.0 * flops}
    b, d, dh = c["b"], c["d"], c["dh"]
    size = 2 if c["dtype"] == "bf16" else 4
    apply_tokens, update_tokens, updates, iters = c.get("tokens", 0), 0, 0, 0
    if path == "block_causal":
        updates = max(0, math.ceil(c["tokens"] / c["chunk"]) - 1)
        update_tokens, iters = updates * c["chunk"], 5 if c["muon"] else 0
    elif path == "video":
        updates = len(range(c["chunk"], c["tokens"], 2 * c["chunk"]))
        update_tokens = updates * c["chunk"]
    elif path == "video_step":
        updates = 1 if c["update"] else 0
        update_tokens, iters = updates * c["tokens"], 3 if c["muon"] else 0
    elif path == "nvs":
        apply_tokens, update_tokens, updates, iters = c["apply"], c["update"], 1 if c["update"] else 0, c["iters"]
    else:
        updates, update_tokens, iters = 1, c["tokens"], 5 if c["muon"] else 0
    flops = b * d * dh * (6.0 * apply_tokens + 12.0 * update_tokens) + updates * _newton_schulz_flops(b, d, dh, iters)
    moved = b * (2.0 * apply_tokens * d * size + update_tokens * (2.0 * d * size + 16)) + 12.0 * b * d * dh
    if path in ("nvs", "video_step", "video"):
        moved += 12.0 * b * d * dh                                              # the fast weights come back
    if path == "video_step" and updates:
        moved += 24.0 * b * d * dh                                              # and the momentum states go in and out
    if path in ("block_causal", "video"):                                       # the backward reads the gradient, writes ten
        moved += b * (2.0 * apply_tokens * d * size + update_tokens * (2.0 * d * size + 16)) + 12.0 * b * d * dh
        flops *= 3.0
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    c = case
    if c["path"] == "causal_layer" or c.get("muon") or (c["path"] == "nvs" and c["update"]):
        # five bf16 Newton-Schulz iterations amplify one flipped rounding of the gradient to percents of what follows from it
        return {"rel": 0.03, "max": 0.99}
    if c.get("dtype") == "fp32":
        return {"rel": 1e-4, "max": 1e-2}
    chain = c["tokens"] / c["chunk"] if c["path"] == "block_causal" else 1
    # every update reads the weights that the one before it wrote: a long chain of them adds its roundings up
    return {"rel": 2e-2 if chain > 8 else 1e-2, "max": 0.5}
