"""The work a user of this package has it do, as timed cases: single BitLinear
calls from one token to a long prompt, the weight packer, and the 2B decoder's
prompt pass, greedy decode loop and whole generations.

listed() names the standing cases, draw(rng) gives further ones of the same
ranges, prepare(case, seed) makes what a program holds before the call, run()
is one pass through the public entry points, work() the bytes and operations
that a pass cannot do without, tolerance() how far another correct
implementation's results may be off.
"""
import math

import numpy as np
import torch

from bitnet_amd import bitlinear, decoder, pack_weight

# (N, K) of the 2B decoder's four products and of the larger shapes in kernel_test.REFERENCE_SHAPES
MODEL_SHAPES = (
    (3840, 2560), (2560, 2560), (13824, 2560), (2560, 6912),
    (3200, 3200), (4800, 3200), (3200, 10240), (20480, 3200),
)
# output rows of the sub-tensors of a fused weight, where the shape is one of the decoder's fused ones
SEGMENTS = {(3840, 2560): (2560, 3200, 3840), (13824, 2560): (6912, 13824)}
VOCAB = 128256
EOS = VOCAB - 1


def listed():
    return [
        # one token through one BitLinear module: the unit of every eager decode loop (config 0)
        {"name": "forward 1 x 2560 x 2560", "kind": "forward", "m": 1, "n": 2560, "k": 2560, "segments": False},
        # a batch of eight sequences, the down projection (config 2)
        {"name": "forward 8 x 2560 x 6912", "kind": "forward", "m": 8, "n": 2560, "k": 6912, "segments": False},
        # a short prompt of ragged length, fused q/k/v with the converter's scale per sub-tensor
        {"name": "forward 101 x 3840 x 2560 seg", "kind": "forward", "m": 101, "n": 3840, "k": 2560, "segments": True},
        # a long prompt, gate and up projection (config 3)
        {"name": "forward 2048 x 13824 x 2560", "kind": "forward", "m": 2048, "n": 13824, "k": 2560, "segments": False},
        # the drop-in product on int8 rows into the caller's buffer, as the reference's test calls it, at its largest shape
        {"name": "product 1 x 20480 x 3200", "kind": "product", "m": 1, "n": 20480, "k": 3200, "quantize": False, "mode": 0},
        # quantizer and product as two calls, as a program written against the reference's shim makes them
        {"name": "product 333 x 4800 x 3200", "kind": "product", "m": 333, "n": 4800, "k": 3200, "quantize": True, "mode": 1},
        # loading a model: one fused weight into the packed layout, on the device
        {"name": "pack 13824 x 2560", "kind": "pack", "n": 13824, "k": 2560},
        # the greedy decode loop behind a 512-token prompt, one sequence and a batch (config 4)
        {"name": "decode 1 x 512 + 32", "kind": "decode", "batch": 1, "prompt": 512, "steps": 32},
        {"name": "decode 8 x 512 + 32", "kind": "decode", "batch": 8, "prompt": 512, "steps": 32},
        # a prompt alone: time to the first token
        {"name": "prefill 1 x 512", "kind": "prefill", "batch": 1, "prompt": 512},
        # whole answers from token ids: ragged prompts in a batch, greedy, stopping at an end token
        {"name": "generate 3 x 200 + 24 greedy", "kind": "generate", "batch": 3, "prompt": 200, "steps": 24, "sample": False},
        # a chat answer: one sequence, temperature and nucleus sampling, stopping at an end token
        {"name": "generate 1 x 64 + 24 sampled", "kind": "generate", "batch": 1, "prompt": 64, "steps": 24, "sample": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("forward", "product", "pack", "unpack", "decode", "prefill", "generate"), (7, 5, 2, 1, 2, 2, 2))[0]
    if kind in ("forward", "product", "pack", "unpack"):
        if rng.random() < 0.5:
            n, k = rng.choice(MODEL_SHAPES)
        else:  # other models' layers: any multiple of the layout's tile
            n, k = 16 * _log_int(rng, 16, 1280), 128 * _log_int(rng, 2, 80)
        case = {"kind": kind, "n": n, "k": k}
        if kind in ("forward", "product"):
            case["m"] = max(1, min(_log_int(rng, 1, 2048), 2048 * 13824 * 2560 // (n * k)))
        if kind == "forward":
            case["segments"] = (n, k) in SEGMENTS and rng.random() < 0.5
        if kind == "product":
            case["quantize"] = rng.random() < 0.5
            case["mode"] = rng.choice((0, 1)) if case["quantize"] else 0
        if kind in ("pack", "unpack"):
            case["n"] = min(n, 13824 * 2560 // k // 16 * 16)
        return case
    if kind == "decode":
        return {"kind": kind, "batch": rng.randint(1, 8), "prompt": _log_int(rng, 16, 700), "steps": rng.randint(8, 32)}
    if kind == "prefill":
        batch = rng.randint(1, 4)
        return {"kind": kind, "batch": batch, "prompt": _log_int(rng, 16, 1024 // batch)}
    return {"kind": kind, "batch": rng.randint(1, 4), "prompt": _log_int(rng, 8, 300), "steps": rng.randint(6, 24),
            "sample": rng.random() < 0.5}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _ternary(n, k, gen):
    """P(0) = 0.4, P(+-1) = 0.3 each, as BASELINE.json's configurations draw them."""
    u = torch.rand(n, k, generator=gen, device="cuda")
    return (u >= 0.7).to(torch.int8) - (u < 0.3).to(torch.int8)


def _activations(m, k, gen):
    """Standard normal rows; prompt-sized blocks carry 1 % outliers of 20 times the size (config 3)."""
    x = torch.randn(m, k, generator=gen, device="cuda")
    if m >= 64:
        x = torch.where(torch.rand(m, k, generator=gen, device="cuda") < 0.01, x * 20.0, x)
    return x.to(torch.bfloat16)


def _scales(count, gen):
    """A vector of mean |w| of N(0, 0.02^2) sources, one slot per sub-tensor (unused slots of the usual four zero)."""
    ws = torch.zeros(max(4, count), device="cuda")
    ws[:count] = 0.016 * (1.0 + 0.2 * torch.rand(count, generator=gen, device="cuda"))
    return ws.to(torch.bfloat16)


def _model(seed):
    """The 2B decoder with random weights, in bf16 on the GPU."""
    prev = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device("cuda"):
            model = decoder.Transformer(decoder.ModelArgs())
    finally:
        torch.set_default_dtype(prev)
    return decoder.random_init_(model, seed=int(seed))


def prepare(case, seed):
    kind, gen = case["kind"], _gen(seed)
    if kind in ("pack", "unpack"):
        w = _ternary(case["n"], case["k"], gen)
        return {"kind": kind, "w": w if kind == "pack" else pack_weight.convert_weight_int8_to_int2(w, keep_device=True)}
    if kind in ("forward", "product"):
        m, n, k = case["m"], case["n"], case["k"]
        slots = 6 if (n, k) == (4800, 3200) else 4  # that shape's fused weight has more sub-tensors
        packed = pack_weight.convert_weight_int8_to_int2(_ternary(n, k, gen), keep_device=True)
        x = _activations(m, k, gen)
        if kind == "forward":
            ends = SEGMENTS[(n, k)] if case["segments"] else None
            mod = bitlinear.BitLinearKernel(k, n, seg_ends=ends).cuda()
            mod.weight.data = packed
            mod.weight_scale.data = _scales(len(ends) if ends else slots, gen)
            return {"kind": kind, "mod": mod, "x": x}
        state = {"kind": kind, "packed": packed, "ws": _scales(slots, gen), "mode": case["mode"]}
        if case["quantize"]:
            state["x"] = x
        else:
            q, s = bitlinear.quant_input(x)
            state.update(q=q, s=s.view(-1), out=torch.empty(m, n, dtype=torch.bfloat16, device="cuda"))
        return state
    B, P, steps = case["batch"], case["prompt"], case.get("steps", 1)
    model = _model(seed)
    g = decoder.Generator(model, B, P + steps + 1)
    prompt = torch.randint(0, VOCAB, (B, P), generator=gen, device="cuda")
    first = g.prefill(prompt)  # the captured prompt pass of this length, and the cache a decode loop starts from
    state = {"kind": kind, "gen": g, "prompt": prompt}
    if kind == "decode":
        g.decode(first, P, 1)  # captures the step
        state.update(first=first, start=P, steps=steps)
    if kind == "generate":
        # lengths from half the longest to the longest
        ids = prompt.tolist()
        state["prompts"] = [row[: P - (b * P // (2 * B))] for b, row in enumerate(ids)]
        state.update(steps=steps, sample=case["sample"], seed=int(seed), rng=_gen(seed))
        run(state)  # a serving program has answered before: every captured pass exists
    return state


def _answers(answers):
    return {"tokens": np.array([t for a in answers for t in a], dtype=np.int64),
            "lengths": np.array([len(a) for a in answers], dtype=np.int64)}


def run(state):
    kind = state["kind"]
    if kind == "forward":
        return state["mod"](state["x"])
    if kind == "product":
        if "x" in state:
            q, s = bitlinear.quant_input(state["x"], state["mode"])
            return {"q": q, "s": s, "out": bitlinear.bitnet_int8xint2_linear(q, state["packed"], s, state["ws"])}
        return bitlinear.bitnet_int8xint2_linear(state["q"], state["packed"], state["s"], state["ws"], out=state["out"])
    if kind == "pack":
        return pack_weight.convert_weight_int8_to_int2(state["w"], keep_device=True)
    if kind == "unpack":
        return pack_weight.convert_weight_int2_to_int8(state["w"])
    g = state["gen"]
    if kind == "decode":
        tokens = g.decode(state["first"], state["start"], state["steps"])
        end = state["start"] + state["steps"]
        k, v = g.cache[-1]  # the rows that are in use: the last layer's depend on everything in front of them
        return {"tokens": tokens, "k": k[:, :end], "v": v[:, :end]}
    if kind == "prefill":
        P = state["prompt"].shape[1]
        token = g.prefill(state["prompt"])
        k, v = g.cache[-1]
        return {"token": token, "k": k[:, :P], "v": v[:, :P]}
    if not state["sample"]:
        return _answers(g.generate_all(state["prompts"], state["steps"], eos_id=EOS))
    state["rng"].manual_seed(state["seed"])
    return _answers(g.generate_all(state["prompts"], state["steps"], use_sampling=True, eos_id=EOS, rng=state["rng"]))


def _decoder_work(batch, prompt, steps):
    """(bytes, flops) of a prompt pass over `prompt` tokens (0: none) and `steps` decode steps behind position `start`."""
    a = decoder.ModelArgs()
    hd = a.dim // a.n_heads
    kv = 2 * a.n_kv_heads * hd
    per_layer = (a.dim + kv) * a.dim + a.dim * a.dim + 3 * a.ffn_dim * a.dim
    weights, head = a.n_layers * per_layer // 4, a.vocab_size * a.dim * 2
    token_flops = 2 * a.n_layers * per_layer
    passes = steps + (1 if prompt["tokens"] else 0)
    total = passes * (weights + head)
    flops = batch * (steps * (token_flops + 2 * a.vocab_size * a.dim))
    if prompt["tokens"]:
        T = prompt["tokens"]
        flops += batch * (T * token_flops + 2 * a.vocab_size * a.dim + a.n_layers * 4 * a.n_heads * hd * T * (T + 1) // 2)
        total += batch * T * (a.dim * 2 + a.n_layers * kv * 2)  # embedding rows read, cache rows written
    for i in range(steps):
        rows = prompt["start"] + i + 1
        total += batch * a.n_layers * kv * 2 * rows
        flops += batch * a.n_layers * 4 * a.n_heads * hd * rows
    return {"bytes": total, "flops": flops}


def work(case):
    kind = case["kind"]
    if kind in ("pack", "unpack"):
        n, k = case["n"], case["k"]
        return {"bytes": n * k + n * k // 4, "flops": 0}
    if kind in ("forward", "product"):
        m, n, k = case["m"], case["n"], case["k"]
        rows = m * k * 2 if kind == "forward" else m * k + m * 2
        if kind == "product" and case["quantize"]:
            rows = m * k * 2 + m * k + m * 2  # the int8 rows and their scales are results here
        return {"bytes": rows + n * k // 4 + m * n * 2 + 8, "flops": 2 * m * n * k}
    B, P = case["batch"], case["prompt"]
    if kind == "decode":
        return _decoder_work(B, {"tokens": 0, "start": P}, case["steps"])
    if kind == "prefill":
        return _decoder_work(B, {"tokens": P, "start": P}, 0)
    return _decoder_work(B, {"tokens": P, "start": P}, case["steps"] - 1)


def tolerance(case):
    kind = case["kind"]
    if kind in ("pack", "unpack", "generate"):
        return "exact"  # bytes, and token ids
    if kind in ("forward", "product"):
        return {"rel": 4e-3, "max": 8e-3, "differ": 0.0}  # exact int32 sums, one rounding to bf16
    return {"rel": 1e-2, "max": 0.3, "differ": 0.0}  # bf16 cache rows behind 30 layers; the token ids are the same
