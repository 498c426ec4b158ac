"""The work that stands for this framework's use: what its speed is measured on.

Five kinds of calls, each through the entry point a program uses:

``linear``  ``CompressedLinear.forward``: the ``nn.Linear``-shaped seat of a packed matrix, on one
            token (decode), a few (a short turn, a small batch) or a prompt
``encode``  ``nf4_quantize``: fp32 weights into packed codes and scales
``decode``  ``nf4_dequant``: packed codes and scales back into fp32
``step``    decode tokens of a resident model, each id given (scoring a known continuation):
            ``recorded`` replays the captured step, otherwise ``teacher_force_token`` launches it
``prompt``  ``DecodeV2Loop.prefill_from``: a prompt, or the next turn behind a cached prefix

The architectures are the ones the decoder's own configurations describe, with random-init
weights; matrix sizes are theirs or lie around them.
"""

import math

import torch

from deepfold_amd import decodev2 as dv2
from deepfold_amd.chr0.loader import ChrMatrix
from deepfold_amd.host.linear import CompressedLinear
from deepfold_amd.nf4 import nf4_dequant, nf4_quantize
from deepfold_amd.nf4.plan import k_pad

ARCHS = {
    "3b": dv2.QWEN25_3B,
    "14b": dv2.QWEN25_14B,
    "20b": dv2.INTERNLM25_20B,
    "32b": dv2.QWEN25_32B,
}
#: tokens of one pass of a ``step`` case
STEPS = 4


def listed():
    return [
        # one token through the smallest full matrix of a 3B layer, bias as q/k/v have it
        {"name": "linear_1_2048x2048", "kind": "linear", "m": 2048, "k": 2048, "tokens": 1, "bias": True},
        # a short odd turn through a 14B o projection: the few-column tiles, no whole vectors
        {"name": "linear_17_5120x5120", "kind": "linear", "m": 5120, "k": 5120, "tokens": 17, "bias": False},
        # a mid-size prompt through a 3B gate, with a bias and an odd token count
        {"name": "linear_333_11008x2048", "kind": "linear", "m": 11008, "k": 2048, "tokens": 333, "bias": True},
        # a long prompt through a 14B down projection: the largest linear call
        {"name": "linear_1024_5120x13824", "kind": "linear", "m": 5120, "k": 13824, "tokens": 1024, "bias": False},
        # quantising a 14B gate on load
        {"name": "encode_13824x5120", "kind": "encode", "m": 13824, "k": 5120},
        # dense weights out of a small ragged matrix and out of a 32B down projection
        {"name": "decode_1000x1111", "kind": "decode", "m": 1000, "k": 1111},
        {"name": "decode_5120x27648", "kind": "decode", "m": 5120, "k": 27648},
        # scoring without a recorded graph, behind the 3B benchmark prompt: host and launches
        {"name": "step_3b_at_512", "kind": "step", "arch": "3b", "ctx": 512, "recorded": False},
        # the 14B decode step as it is served, and the 20B one near the end of its cache
        {"name": "step_14b_at_640", "kind": "step", "arch": "14b", "ctx": 640, "recorded": True},
        {"name": "step_20b_at_1920", "kind": "step", "arch": "20b", "ctx": 1920, "recorded": True},
        # the 14B benchmark prompt
        {"name": "prompt_14b_512", "kind": "prompt", "arch": "14b", "start": 0, "tokens": 512},
        # the 32B benchmark prompt, the longest and largest of all
        {"name": "prompt_32b_1791", "kind": "prompt", "arch": "32b", "start": 0, "tokens": 1791},
    ]


def _between(rng, lo, hi):
    """A whole number of lo..hi, spread evenly over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def _features(rng, lo, hi):
    """A feature count: whole groups of 64 as models have them, or any number."""
    n = _between(rng, lo, hi)
    return max(64, n // 64 * 64) if rng.random() < 0.7 else n


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "encode", "decode", "step", "prompt", "prompt"])
    if kind == "linear":
        tokens = 1 if rng.random() < 0.25 else _between(rng, 2, 2048)
        return {"kind": kind, "m": _features(rng, 256, 28672), "k": _features(rng, 256, 28672),
                "tokens": tokens, "bias": rng.random() < 0.5}
    if kind in ("encode", "decode"):
        m = _features(rng, 64, 28672)
        return {"kind": kind, "m": m, "k": _features(rng, 64, min(28672, 150_000_000 // m))}
    arch = rng.choice(sorted(ARCHS))
    room = ARCHS[arch].max_seq
    if kind == "step":
        return {"kind": kind, "arch": arch, "ctx": _between(rng, 8, room - STEPS - 1),
                "recorded": rng.random() < 0.6}
    tokens = _between(rng, 2, 1791)
    # a first prompt, or a turn appended behind what the cache already holds
    start = 0 if rng.random() < 0.5 else rng.randrange(0, room - tokens)
    return {"kind": kind, "arch": arch, "start": start, "tokens": tokens}


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _gauss(g, *shape, sigma=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * sigma


def _ids(seed, n, vocab):
    g = torch.Generator(device="cpu")
    g.manual_seed(int(seed))
    return torch.randint(0, vocab, (n,), generator=g).tolist()


def _cached_prefix(kv, length, g):
    """Rows 0..length of every layer's cache as a prompt leaves them (k and v of unit-variance
    hidden states through weights of sigma 0.02)."""
    for cache in (kv.k, kv.v):
        for layer in range(cache.shape[0]):
            cache[layer, :length] = _gauss(g, length, *cache.shape[2:], sigma=0.02 * 5120 ** 0.5).to(cache.dtype)


def prepare(case, seed):
    kind = case["kind"]
    g = _generator(seed)
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["tokens"]
        packed, scale = nf4_quantize(_gauss(g, m, k, sigma=0.02))
        layer = CompressedLinear(k, m, bias=case["bias"], device="cuda")
        layer.attach(ChrMatrix("weight", m, k, k_pad(k), packed, scale))
        if case["bias"]:
            layer.set_bias(_gauss(g, m, sigma=0.1))
        # hidden states: unit variance with a few channels an order of magnitude above the rest
        channels = torch.where(torch.rand(k, generator=g, device="cuda") < 0.005, 12.0, 1.0)
        return {"kind": kind, "layer": layer, "x": (_gauss(g, 1, n, k) * channels).to(torch.bfloat16)}
    if kind == "encode":
        return {"kind": kind, "w": _gauss(g, case["m"], case["k"], sigma=0.02)}
    if kind == "decode":
        packed, scale = nf4_quantize(_gauss(g, case["m"], case["k"], sigma=0.02))
        return {"kind": kind, "packed": packed, "scale": scale, "m": case["m"], "k": case["k"]}
    spec = ARCHS[case["arch"]]
    weights = dv2.DeviceWeights.random(spec, seed)
    loop = dv2.DecodeV2Loop.from_weights(weights)
    loop.warmup()
    if kind == "step":
        ctx = case["ctx"]
        _cached_prefix(loop.state.kv, ctx, g)
        loop.state.position.fill_(ctx)
        loop.state.valid_len.fill_(ctx)
        graph = dv2.capture_greedy(loop.state, weights) if case["recorded"] else None
        return {"kind": kind, "state": loop.state, "weights": weights, "graph": graph, "ctx": ctx,
                "ids": _ids(seed, STEPS, spec.vocab)}
    _cached_prefix(loop.state.kv, case["start"], g)
    return {"kind": kind, "loop": loop, "start": case["start"], "ids": _ids(seed, case["tokens"], spec.vocab)}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "encode":
        return nf4_quantize(state["w"])
    if kind == "decode":
        return nf4_dequant(state["packed"], state["scale"], state["m"], state["k"], k_pad(state["k"]))
    if kind == "step":
        st, weights, graph, ctx = state["state"], state["weights"], state["graph"], state["ctx"]
        st.position.fill_(ctx)
        logits = []
        for token in state["ids"]:
            if graph is None:
                dv2.teacher_force_token(st, weights, token)
            else:
                st.load_token(token)
                graph.replay()
            logits.append(st.arena.logits.clone())
        rows = slice(ctx, ctx + len(logits))
        return {"logits": torch.cat(logits), "k": st.kv.k[:, rows], "v": st.kv.v[:, rows]}
    loop, start, ids = state["loop"], state["start"], state["ids"]
    logits = loop.prefill_from(ids, start)
    rows = slice(start, start + len(ids))
    return {"logits": logits, "k": loop.state.kv.k[:, rows], "v": loop.state.kv.v[:, rows]}


def work(case):
    kind = case["kind"]
    if kind in ("linear", "encode", "decode"):
        m, k = case["m"], case["k"]
        packed = m * k_pad(k) * 17 // 32
        if kind != "linear":
            return {"bytes": packed + 4 * m * k, "flops": m * k}
        n = case["tokens"]
        return {"bytes": packed + 2 * n * (m + k) + (2 * m if case["bias"] else 0), "flops": 2 * m * k * n}
    spec = ARCHS[case["arch"]]
    row = spec.kv_bytes(1)
    if kind == "step":
        ctx = case["ctx"]
        seen = sum(ctx + i + 1 for i in range(STEPS))
        return {"bytes": STEPS * (spec.weight_bytes_per_token() + 2 * spec.vocab) + seen * row,
                "flops": 2 * STEPS * spec.linear_weights() + 4 * spec.n_layers * spec.q_dim * seen}
    n, start = case["tokens"], case["start"]
    seen = n * start + n * (n + 1) // 2
    head = spec.vocab * spec.hidden
    return {"bytes": spec.weight_bytes_per_token() + (start + n) * row + 2 * spec.vocab,
            "flops": 2 * n * (spec.linear_weights() - head) + 2 * head + 4 * spec.n_layers * spec.q_dim * seen}


def tolerance(case):
    kind = case["kind"]
    if kind in ("encode", "decode"):
        return "exact"
    if kind == "linear":
        # one bf16 rounding of the result (two with a bias) and, where the matrix cores take bf16
        # weights, one of every weight: 2.1e-3 .. 2.7e-3 (largest 1.1e-2) against the product in
        # 64 bits
        return {"rel": 1e-2, "max": 5e-2}
    # bf16 hand-overs between the launches of 36 to 64 layers drift apart like a random walk:
    # a step through separate norm and merge launches is 3.1e-2 .. 4.1e-2 (largest 0.21) from the
    # folded one, a prompt through windows of 32 tokens 4.5e-2 .. 6.8e-2 (0.43) from windows of
    # 64, through plain torch operations between the matrix products 0.10 (0.61)
    return {"rel": 0.15, "max": 0.8} if kind == "step" else {"rel": 0.2, "max": 0.95}


#: the sixteen levels, as their binary32 patterns
_LEVEL_BITS = (0xBF800000, 0xBF3239B1, 0xBF066B30, 0xBECA32A0, 0xBE91A24D, 0xBE3D353F, 0xBDBA7871, 0x00000000,
               0x3DA2FAFF, 0x3E24CAE3, 0x3E7C04DD, 0x3EAD033A, 0x3EE1A4B8, 0x3F1007AB, 0x3F3913B3, 0x3F800000)


def _widened(packed, scale, m, k):
    """The matrix the codes and scales stand for, in 64 bits."""
    levels = torch.tensor(_LEVEL_BITS, dtype=torch.int64, device=packed.device).to(torch.int32)
    levels = levels.view(torch.float32).double()
    codes = torch.stack((packed & 15, packed >> 4), dim=-1).reshape(m, -1, 64).long()
    return (levels[codes] * scale.double().reshape(m, -1, 1)).reshape(m, -1)[:, :k]


def exact(case, seed):
    if case["kind"] not in ("linear", "decode"):
        return None  # whole codes; whole models, whose layers carry every rounding along
    state = prepare(case, seed)
    if case["kind"] == "decode":
        return _widened(state["packed"], state["scale"], case["m"], case["k"])
    layer = state["layer"]
    y = state["x"].double() @ _widened(layer.packed, layer.scale, case["m"], case["k"]).t()
    return y + layer.bias.double() if case["bias"] else y
