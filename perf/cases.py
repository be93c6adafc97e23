"""Performance cases: the work a program gives this library, through its public entry points.

A case is one of
  linear   vtq_linear_device on `layers` weight matrices of one shape, one call each
           (decode at batch 1, several sequences or a prompt at larger batches);
  ffn      the two matrices of a feed-forward block, `layers` blocks one after another;
  host     vtq_linear on host arrays, the call that stands in for the engine's linear_dispatch;
  run      vtqrt_run: a prompt, then greedy decoding, with every position's logits.

Decode cases walk over several layers, each with weights of its own, as a
decode step does: one matrix called again and again would stay in a cache.
Every result is defined to the last bit (the reference's operation order), so
every case is compared exactly.
"""
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vitni-tensor_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import vtq  # noqa: E402
from vtq import runtime, synth  # noqa: E402

# weight formats by name: (ggml type, regime)
FORMATS = {
    "q4_k": (vtq.Q4_K, vtq.REGIME_INTEGER),
    "q4_k_float": (vtq.Q4_K, vtq.REGIME_FLOAT_FUSED),  # the reference's default build
    "q6_k": (vtq.Q6_K, vtq.REGIME_INTEGER),
    "q8_0": (vtq.Q8_0, vtq.REGIME_INTEGER),
    "q5_0": (vtq.Q5_0, vtq.REGIME_INTEGER),
    "q4_0": (vtq.Q4_0, vtq.REGIME_INTEGER),
    "f32": (vtq.F32, vtq.REGIME_INTEGER),
}


def _linear(fmt, batch, in_feat, out_feat, layers=1):
    return {"kind": "linear", "format": fmt, "batch": batch, "in_feat": in_feat, "out_feat": out_feat, "layers": layers}


def listed():
    model = dict(synth.LLAMA_1B1)
    return [
        # the smallest call: a key/value projection of a small model whose
        # width is no multiple of 256 (files then hold Q5_0), one token
        {"name": "q5_0_decode_kv_896", **_linear("q5_0", 1, 896, 128)},
        # the engine's own call: one token, host arrays in and out, weights resident
        {"name": "q4_k_host_4096", "kind": "host", "format": "q4_k", "batch": 1, "in_feat": 4096, "out_feat": 4096},
        # decode, attention-sized Q8_0 matrices of a 7B model
        {"name": "q8_0_decode_4096", **_linear("q8_0", 1, 4096, 4096, 8)},
        # decode, the feed-forward pair of a 7B model (the benchmark's step)
        {"name": "q4_k_decode_ffn", "kind": "ffn", "format": "q4_k", "batch": 1, "dim": 4096, "hidden": 11008,
         "layers": 8},
        # decode, the output head
        {"name": "q6_k_decode_head", **_linear("q6_k", 1, 4096, 32000)},
        # eight sequences decoded together
        {"name": "q4_k_batch8", **_linear("q4_k", 8, 4096, 11008, 4)},
        # nineteen sequences, down projection (two chunks of the pinned dot a row)
        {"name": "q4_0_batch19_down", **_linear("q4_0", 19, 11008, 4096)},
        # a prompt of 77 tokens in the reference's default build
        {"name": "q4_k_float_prompt77", **_linear("q4_k_float", 77, 2048, 5632)},
        # a prompt of 128 tokens on Q8_0 weights
        {"name": "q8_0_prompt128", **_linear("q8_0", 128, 4096, 4096)},
        # a prompt of 200 tokens through a Q6_K down projection
        {"name": "q6_k_prompt200_down", **_linear("q6_k", 200, 11008, 4096)},
        # a prompt of 512 tokens, up projection of an 8B model
        {"name": "q4_k_prompt512_up", **_linear("q4_k", 512, 4096, 14336)},
        # the whole engine: 1.1B Llama, 128 prompt ids, 64 new tokens
        {"name": "run_1b1", "kind": "run", **model, "arch": "llama", "prompt": 128, "new": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case: formats by how often files hold them, batch 1 to 512, rows of 256 to
    14336 inputs (any multiple of the format's block), 64 to 32000 outputs; now and then a
    whole run of a smaller model, or a host call."""
    pick = rng.random()
    if pick < 0.12:
        heads = rng.choice([4, 8, 16, 32])
        dim = heads * 64
        return {"kind": "run", "dim": dim, "hidden": max(256, round(dim * rng.uniform(2.0, 4.0) / 256) * 256),
                "layers": rng.randint(2, 10), "heads": heads, "kv_heads": heads // rng.choice([1, 2, 4]),
                "vocab": _log_int(rng, 1000, 32000), "ctx": 1024, "rope_theta": 10000.0, "rms_eps": 1e-5,
                "arch": rng.choice(["llama", "llama", "qwen2"]), "prompt": _log_int(rng, 2, 400),
                "new": _log_int(rng, 1, 40)}
    fmt = rng.choices(["q4_k", "q6_k", "q8_0", "q5_0", "q4_0", "f32", "q4_k_float"], [30, 20, 15, 8, 9, 6, 12])[0]
    block = 256 if fmt in ("q4_k", "q4_k_float", "q6_k") else 1 if fmt == "f32" else 32
    most = 512 * 14336 * 4096 if fmt in ("q4_k", "q6_k") else 512 * 4096 * 2048
    while True:
        batch = 1 if rng.random() < 0.3 else _log_int(rng, 2, 512)
        in_feat = max(block, round(_log_int(rng, 256, 14336) / block) * block)
        out_feat = _log_int(rng, 64, 32000)
        if batch * in_feat * out_feat <= most:
            break
    if pick < 0.22:
        return {"kind": "host", "format": fmt, "batch": batch, "in_feat": in_feat, "out_feat": out_feat}
    return _linear(fmt, batch, in_feat, out_feat)


# ------------------------------------------------------------------ inputs

_context = None


def _ctx():
    """The program's one context."""
    global _context
    if _context is None:
        _context = vtq.Context(0)
    return _context


def _shapes(case):
    """(in_feat, out_feat) of every call of one pass."""
    if case["kind"] == "ffn":
        return [(case["dim"], case["hidden"]), (case["hidden"], case["dim"])] * case["layers"]
    return [(case["in_feat"], case["out_feat"])] * case.get("layers", 1)


def _weights(gen, fmt, out_feat, in_feat):
    """GGUF blocks as synth.weights draws them: scales |N(0, 0.01)| in f16, every code uniform."""
    dev = gen.device
    if fmt == "f32":
        return (0.02 * torch.randn(out_feat * in_feat, generator=gen, device=dev)).view(torch.uint8)
    ggml, _ = FORMATS[fmt]
    numel, nbytes = vtq.BLOCK[ggml]
    n = out_feat * (in_feat // numel)
    w = torch.randint(0, 256, (n, nbytes), generator=gen, device=dev, dtype=torch.uint8)

    def scale():
        return (0.01 * torch.randn(n, generator=gen, device=dev)).abs().half().view(torch.uint8).view(n, 2)

    if ggml == vtq.Q4_K:
        w[:, 0:2] = scale()
        w[:, 2:4] = scale()
    elif ggml == vtq.Q6_K:
        w[:, 192:208] = torch.randint(-64, 64, (n, 16), generator=gen, device=dev, dtype=torch.int8).view(torch.uint8)
        w[:, 208:210] = scale()
    else:
        if ggml == vtq.Q8_0:
            w[:, 2:] = torch.randint(-127, 128, (n, 32), generator=gen, device=dev, dtype=torch.int8).view(torch.uint8)
        w[:, 0:2] = scale()
    return w.view(-1)


def _inputs(case, seed):
    """(x, w) of every call, on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    got = []
    for in_feat, out_feat in _shapes(case):
        x = torch.randn(case["batch"], in_feat, generator=gen, device="cuda")
        got.append((x, _weights(gen, case["format"], out_feat, in_feat)))
    return got


def prepare(case, seed):
    if case["kind"] == "run":
        cfg = {k: case[k] for k in synth.LLAMA_1B1}
        blob = synth.llama_gguf(cfg, seed, arch=case["arch"], qkv_bias=case["arch"] == "qwen2")
        rng = np.random.default_rng(seed)
        return {"model": runtime.Model(blob), "new": case["new"], "weights_hash": rng.bytes(32),
                "prompt": rng.integers(0, case["vocab"], case["prompt"]).astype(np.uint32)}
    ggml, regime = FORMATS[case["format"]]
    batch = case["batch"]
    pairs = _inputs(case, seed)
    if case["kind"] == "host":
        x, w = (t.cpu().numpy() for t in pairs[0])
        y = np.zeros((batch, case["out_feat"]), np.float32)
        # a context of its own: it caches weights by their host address, so it goes when they go
        return {"host": (ggml, regime, x, w, y, batch, case["in_feat"], case["out_feat"]), "context": vtq.Context(0)}
    calls, outs = [], []
    for (x, w), (in_feat, out_feat) in zip(pairs, _shapes(case)):
        y = torch.empty(batch, out_feat, device="cuda")
        calls.append((ggml, regime, x.data_ptr(), w.data_ptr(), w.numel(), y.data_ptr(), batch, in_feat, out_feat))
        outs.append(y)
    return {"calls": calls, "outs": outs, "keep": pairs, "context": _ctx()}


def run(state):
    if "model" in state:
        tokens, digest, logits = state["model"].run(state["prompt"], state["new"], state["weights_hash"])
        return {"tokens": tokens, "digest": np.frombuffer(bytes.fromhex(digest), np.uint8), "logits": logits}
    if "host" in state:
        state["context"].linear(*state["host"])
        return state["host"][4]
    ctx = state["context"]
    stream = torch.cuda.current_stream().cuda_stream
    for call in state["calls"]:
        ctx.linear_device(*call, stream)
    return state["outs"]


def work(case):
    if case["kind"] != "run":
        ggml, _ = FORMATS[case["format"]]
        b = case["batch"]
        return {"bytes": sum(o * vtq.row_bytes(ggml, i) + 4 * b * (i + o) for i, o in _shapes(case)),
                "flops": sum(2 * b * i * o for i, o in _shapes(case))}
    d, h, kv = case["dim"], case["hidden"], case["dim"] // case["heads"] * case["kv_heads"]
    layer = d * (2 * d + 2 * kv) + 3 * d * h  # weights of a layer
    head = d * case["vocab"]
    new, steps = case["new"], case["prompt"] + case["new"]
    cache = 2 * 4 * kv * case["layers"]       # bytes of a cached position
    weights = case["layers"] * layer * 144 // 256 + head * 210 // 256
    # the weights once for the prompt and once for each new token, each step's
    # cached positions, the logits
    attended = sum(range(case["prompt"], steps))
    return {"bytes": weights * (1 + new) + cache * (attended + steps) + 4 * steps * case["vocab"],
            "flops": 2 * steps * (case["layers"] * layer + head) + 4 * d * case["layers"] * steps * (steps + 1) // 2}


def tolerance(case):
    return "exact"  # every result is pinned to the bit, tokens and digest too


# ------------------------------------------------------- 64-bit reference

def _f16(b):
    return b.contiguous().view(torch.float16).double()  # [n, 1]


def _decode(fmt, w, out_feat, in_feat):
    """W[out_feat, in_feat] in 64 bits."""
    if fmt == "f32":
        return w.view(torch.float32).view(out_feat, in_feat).double()
    ggml, _ = FORMATS[fmt]
    w = w.view(-1, vtq.BLOCK[ggml][1])
    n = w.shape[0]
    if ggml == vtq.Q8_0:
        v = _f16(w[:, 0:2]) * w[:, 2:].contiguous().view(torch.int8).double()
    elif ggml == vtq.Q4_0:  # element 2k in byte k's low half, 2k + 1 in its high half
        q = torch.stack((w[:, 2:] & 15, w[:, 2:] >> 4), 2).view(n, 32)
        v = _f16(w[:, 0:2]) * (q.double() - 8)
    elif ggml == vtq.Q5_0:
        bits = (w[:, 2:6].unsqueeze(2) >> torch.arange(8, device=w.device, dtype=torch.uint8)) & 1
        q = torch.cat((w[:, 6:] & 15, w[:, 6:] >> 4), 1) | (bits.view(n, 32) << 4)
        v = _f16(w[:, 0:2]) * (q.double() - 16)
    elif ggml == vtq.Q4_K:
        s = w[:, 4:16]
        sc = torch.cat((s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)), 1).double()
        mn = torch.cat((s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)), 1).double()
        qs = w[:, 16:].reshape(n, 4, 1, 32)
        q = torch.cat((qs & 15, qs >> 4), 2).view(n, 8, 32).double()
        v = _f16(w[:, 0:2]).unsqueeze(2) * sc.unsqueeze(2) * q - (_f16(w[:, 2:4]) * mn).unsqueeze(2)
    else:  # Q6_K: two halves of 128 elements, four runs of 32 each
        ql, qh = w[:, 0:128].reshape(n, 2, 2, 32), w[:, 128:192].reshape(n, 2, 1, 32)
        lo = torch.cat((ql & 15, ql >> 4), 2)
        hi = torch.cat([(qh >> (2 * k)) & 3 for k in range(4)], 2)
        q = ((hi << 4) | lo).view(n, 16, 16).double() - 32
        v = _f16(w[:, 208:210]).unsqueeze(2) * w[:, 192:208].contiguous().view(torch.int8).double().unsqueeze(2) * q
    return v.reshape(out_feat, in_feat)


def _quantized(x):
    """The activations a k-quant dot takes: int8 codes of each 256-block times its scale
    (the codes are the operation's definition and come from 32-bit arithmetic)."""
    b = x.view(x.shape[0], -1, 256)
    d = b.abs().amax(2, keepdim=True) / 127.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    s = b * inv
    q = torch.trunc(s + torch.copysign(torch.full_like(s, 0.5), s)).clamp(-127, 127)
    return (q.double() * d.double()).view(x.shape)


def exact(case, seed):
    if case["kind"] == "run":
        return None  # greedy picks are fed back: in 64 bits the run takes another path at the first near tie
    fmt = case["format"]
    outs = []
    for (x, w), (in_feat, out_feat) in zip(_inputs(case, seed), _shapes(case)):
        xs = _quantized(x) if fmt in ("q4_k", "q6_k") else x.double()
        outs.append(xs @ _decode(fmt, w, out_feat, in_feat).T)
    return outs[0].cpu().numpy() if case["kind"] == "host" else outs
