"""The work that programs have this framework do, as cases that can be timed and compared.

Five kinds, each through the public entry points:

  linear    one call of a ternary linear module (`SpBitLinear`, `SpBitLinearBF16`) on fresh activations: what a
            transformer written against the reference's `model.py` does 120 times per forward pass
  prompt    `Transformer.forward` over the new tokens of one or several prompts: the prefill of a request
  decode    one single-token step of `Transformer.forward`, captured once in a graph and replayed, as
            `greedy_decode` and any serving loop run it
  generate  `greedy_decode`, a whole request: prompt pass, graph capture, greedy steps
  encode    `compress_weight` on one matrix: what converting a checkpoint spends its time on (host data)

The sizes are those of the 2B-shaped model that the benchmark and the tests use, and generic ones.
"""
import torch

import ternainfer_amd as T
from ternainfer_amd import _lib
from ternainfer_amd.model import ModelArgs, Transformer, greedy_decode

DIM, FFN, QKV, LAYERS, HEADS, KV_HEADS, HEAD_DIM, VOCAB = 2560, 6912, 3840, 30, 20, 5, 128, 128256
#: (out_features, in_features, number of weight scales): QKV, O, gate+up and down projection
SHAPES = [(QKV, DIM, 3), (DIM, DIM, 1), (2 * FFN, DIM, 2), (DIM, FFN, 1)]
P_ZERO = 0.40                                   # share of zero weights
FORMAT_BYTES = 1 / 8 + (1 - P_ZERO) / 8 + (4 + 6) / 4096      # reference format, bytes per weight: bitmap, signs, offsets
P2_BYTES = 0.25                                 # the model's weights as `Transformer` keeps them


def _linear(name, module, batch, tokens, n, k, scales):
    return dict(name=name, kind="linear", module=module, batch=batch, tokens=tokens, n=n, k=k, scales=scales)


def listed():
    return [
        # one token through the O projection, module called eagerly: launches and host work are everything
        _linear("linear_int8_1", "int8", 0, 1, DIM, DIM, 1),
        # a few dozen rows (a batch of decode requests), bf16 activations, the deep matrix
        _linear("linear_bf16_37", "bf16", 0, 37, DIM, FFN, 1),
        # three prompts of 100 tokens, 3-D activations, weight repacked at load time
        _linear("linear_repacked_3x100", "int8_repacked", 3, 100, QKV, DIM, 3),
        # the benchmark's prefill size on its widest matrix
        _linear("linear_bf16_2048", "bf16", 0, 2048, 2 * FFN, DIM, 2),
        # a long batch of prompt tokens whose number is no power of two, reference format, the deep matrix
        _linear("linear_int8_5000", "int8", 0, 5000, DIM, FFN, 1),
        # the prefill of a short chat turn and of a long document
        dict(name="prompt_1x100", kind="prompt", batch=1, tokens=100),
        dict(name="prompt_1x1920", kind="prompt", batch=1, tokens=1920),
        # one user; a small server with requests of different lengths; a busy one
        dict(name="decode_1", kind="decode", batch=1, slots=384, filled=0.66, ragged=False),
        dict(name="decode_8_long", kind="decode", batch=8, slots=1528, filled=0.9, ragged=True),
        dict(name="decode_32", kind="decode", batch=32, slots=512, filled=0.6, ragged=True),
        # three requests answered from the start to the last token
        dict(name="generate_3x77", kind="generate", batch=3, tokens=77, gen=24),
        # the widest matrix of a block
        dict(name="encode_gate_up", kind="encode", n=2 * FFN, k=DIM),
    ]


def _spread(rng, low, high):
    """An integer of [low, high], uniform over its logarithm."""
    return max(low, min(high, round(low * (high / low) ** rng.random())))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "prompt", "prompt", "decode", "decode", "decode", "generate", "encode"])
    if kind == "linear":
        n, k, scales = rng.choice(SHAPES) if rng.random() < 0.7 else (64 * _spread(rng, 4, 128), 64 * _spread(rng, 4, 64), 1)
        rows = _spread(rng, 1, 8192)
        batch = rng.choice([0, 0, 2, 3])
        if batch and rows >= 8:
            return dict(kind=kind, module=rng.choice(["int8", "int8_repacked", "bf16"]), batch=batch, tokens=max(1, rows // batch), n=n, k=k, scales=scales)
        return dict(kind=kind, module=rng.choice(["int8", "int8_repacked", "bf16"]), batch=0, tokens=rows, n=n, k=k, scales=scales)
    if kind == "prompt":
        total = _spread(rng, 16, 4096)
        batch = min(_spread(rng, 1, 8), max(1, total // 16))
        return dict(kind=kind, batch=batch, tokens=min(2048, total // batch))
    if kind == "decode":
        batch = _spread(rng, 1, 64)
        return dict(kind=kind, batch=batch, slots=min(_spread(rng, 64, 4096), 65536 // batch), filled=round(rng.uniform(0.05, 1.0), 3),
                    ragged=rng.random() < 0.5)
    if kind == "generate":
        return dict(kind=kind, batch=_spread(rng, 1, 8), tokens=_spread(rng, 16, 256), gen=_spread(rng, 8, 32))
    return dict(kind=kind, n=64 * _spread(rng, 4, 216), k=64 * _spread(rng, 4, 40))


def _ternary(n, k, gen, device):
    u = torch.rand((n, k), generator=gen, device=device)
    w = torch.zeros((n, k), dtype=torch.int8, device=device)
    w[u >= P_ZERO] = 1
    w[u >= P_ZERO + (1 - P_ZERO) / 2] = -1
    return w


def _position(case, sequence):
    """Cache slot of the new token: the same for all sequences, or shorter prefixes for the later ones."""
    last = max(0, min(case["slots"] - 1, int(case["filled"] * case["slots"]) - 1))
    return last - (last * sequence) // (2 * case["batch"]) if case["ragged"] else last


def _cache(batch, slots):
    """The keys and values of all blocks in one tensor, and the pairs of views that `Transformer.forward` takes."""
    whole = torch.zeros((LAYERS, 2, batch, KV_HEADS, slots, HEAD_DIM), dtype=torch.bfloat16, device="cuda")
    return whole, [(whole[i, 0], whole[i, 1]) for i in range(LAYERS)]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "encode":
        # every 64 x 64 tile has as many zeros whatever the seed, in other places: the length of the sign stream is the same
        n, k = case["n"], case["k"]
        zero = _ternary(n, k, torch.Generator(device="cuda").manual_seed(n * k), "cuda") == 0
        zero = zero.view(n // 64, 64, k // 64, 64)[:, torch.randperm(64, generator=gen, device="cuda")]
        zero = zero[..., torch.randperm(64, generator=gen, device="cuda")].reshape(n, k)
        sign = 1 - 2 * torch.randint(0, 2, (n, k), generator=gen, device="cuda", dtype=torch.int8)
        return {"kind": kind, "w": sign.masked_fill_(zero, 0).cpu()}
    if kind == "linear":
        n, k, scales = case["n"], case["k"], case["scales"]
        vals, offsets, median, bitmap = T.compress_weight(_ternary(n, k, gen, "cuda").cpu())
        entry = {"l.weight_compressed_val": vals, "l.weight_TileOffsets_global": offsets, "l.weight_TileOffsets_median": median,
                 "l.weight_bitmap": bitmap, "l.weight_scale": T.pack_weight_scale([torch.tensor(0.75 + 0.25 * i) for i in range(scales)])}
        _lib.load().ternaspmm_repack_cache_clear()          # weights were loaded: as the header asks of a program that does
        module = T.SpBitLinearBF16(k, n, entry, "l") if case["module"] == "bf16" else \
            T.SpBitLinear(k, n, entry, "l", repack=case["module"] == "int8_repacked")
        rows = (case["batch"], case["tokens"]) if case["batch"] else (case["tokens"],)
        x = torch.randn(rows + (k,), generator=gen, device="cuda")
        x[..., torch.randperm(k, generator=gen, device="cuda")[:max(1, k // 100)]] *= 20      # the outlier channels that activations have
        return {"kind": kind, "module": module, "x": x.to(torch.bfloat16)}
    model = Transformer(ModelArgs(), seed=seed)
    batch = case["batch"]
    state = {"kind": kind, "model": model}
    if kind == "decode":
        whole, cache = _cache(batch, case["slots"])
        whole.normal_(generator=gen)
        tokens = torch.randint(0, VOCAB, (batch, 1), generator=gen, device="cuda")
        at = [_position(case, b) for b in range(batch)]
        pos = torch.tensor([[p] for p in at] if case["ragged"] else at[:1], dtype=torch.int64, device="cuda")
        with torch.inference_mode():
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                model.forward(tokens, cache, pos)
            torch.cuda.current_stream().wait_stream(side)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                logits = model.forward(tokens, cache, pos)
        return dict(state, graph=graph, logits=logits, whole=whole, inputs=(tokens, cache, pos))
    state["prompt"] = torch.randint(0, VOCAB, (batch, case["tokens"]), generator=gen, device="cuda")
    if kind == "prompt":
        whole, cache = _cache(batch, case["tokens"])
        return dict(state, whole=whole, cache=cache, slots=torch.arange(case["tokens"], device="cuda"))
    return dict(state, gen=case["gen"])


def run(state):
    kind = state["kind"]
    if kind == "encode":
        return T.compress_weight(state["w"])
    if kind == "generate":
        return greedy_decode(state["model"], state["prompt"], state["gen"])[0]
    with torch.inference_mode():
        if kind == "linear":
            return state["module"](state["x"])
        if kind == "prompt":
            return {"logits": state["model"].forward(state["prompt"], state["cache"], state["slots"]), "cache": state["whole"]}
        state["graph"].replay()
        return {"logits": state["logits"], "cache": state["whole"]}


def _step_work(rows, attended, logits):
    """Bytes and operations of one pass of the model over `rows` tokens, of which `logits` go through the LM head.
    `attended` = (cache slots read, each once; pairs of a query and a slot)."""
    weights = sum(n * k for n, k, _ in SHAPES) * LAYERS
    slots, pairs = attended
    kv = 2 * KV_HEADS * HEAD_DIM * 2 * LAYERS
    return {"bytes": weights * P2_BYTES + VOCAB * DIM * 2 + logits * VOCAB * 2 + rows * DIM * 2 + (slots + rows) * kv,
            "flops": 2 * rows * weights + 2 * logits * VOCAB * DIM + 4 * pairs * HEADS * HEAD_DIM * LAYERS}


def work(case):
    kind = case["kind"]
    if kind == "encode":
        weights = case["n"] * case["k"]
        return {"bytes": weights * (1 + FORMAT_BYTES), "flops": 0}
    if kind == "linear":
        n, k = case["n"], case["k"]
        m = max(1, case["batch"]) * case["tokens"]
        held = P2_BYTES if case["module"] == "int8_repacked" else FORMAT_BYTES
        return {"bytes": n * k * held + 2 * m * (n + k), "flops": 2 * m * n * k}
    batch = case["batch"]
    if kind == "decode":
        seen = sum(_position(case, b) + 1 for b in range(batch))
        return _step_work(batch, (seen, seen), batch)
    t = case["tokens"]
    first = _step_work(batch * t, (batch * t, batch * t * (t + 1) // 2), batch)
    if kind == "prompt":
        return first
    total = dict(first)
    for i in range(case["gen"]):
        seen = batch * (t + i + 1)
        for key, value in _step_work(batch, (seen, seen), batch).items():
            total[key] += value
    return total


def tolerance(case):
    kind = case["kind"]
    if kind in ("encode", "generate"):
        return "exact"                          # bits of the format; token ids
    if kind == "linear":
        return {"rel": 5e-3}                    # bf16 results (2^-9 a rounding) of exact or 32-bit sums
    # bf16 stream, 30 blocks deep; in front of every linear the activations are rounded to 8 bits, and an input that moves by
    # one bf16 step moves one of them by a whole step now and then
    return {"rel": 2e-2}
