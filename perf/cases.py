"""The work whose speed is tracked, through the package's public entry points.

Four kinds of case, each a call that a program using this package makes:

  matmul  HipBackend.mat_mul with a resident weight, host activations in and
          host results out (one row: an op-level decode GEMV; several rows: a
          batch of tokens).
  sample  HipBackend.sample: one token drawn from a vocabulary of logits.
  decode  InferenceEngine.process_token: one token at a position of a filled
          KV cache, logits out.
  prompt  InferenceEngine.prefill: a prompt (or a further chat turn behind a
          filled KV cache), the last token's logits out.

Model cases take their dimensions and weight-type mixes from
dotllm_amd.synth.SPECS, most with a few of the layers only: a stack of that
model's own blocks between its embedding and its head.  `tiny` and `small5`
are whole models.  A filled KV cache is the engine's seeded fill (a documented
closed form), so that a step at a long context does not need its prompt.
"""
import math

import numpy as np
import torch

from dotllm_amd import HipBackend, InferenceEngine, LoadedModel, SamplingOptions, synth
from dotllm_amd._lib import Q4_K, Q5_K, Q6_K, Q8_0, byte_count

TYPES = {"q4_k": Q4_K, "q5_k": Q5_K, "q6_k": Q6_K, "q8_0": Q8_0}


def listed():
    return [
        # One op-level projection of the smallest model (tiny's FFN up): launch and copy latency.
        dict(name="matmul_row_q8_0", kind="matmul", type="q8_0", m=1, n=1408, k=512),
        # A ragged handful of token rows through small5's FFN up: the op-level batched product.
        dict(name="matmul_37_rows_q5_k", kind="matmul", type="q5_k", m=37, n=2816, k=1024),
        # The default SamplingOptions over the 1B shape's vocabulary: what an unconfigured caller draws every token with.
        dict(name="sample_top_k", kind="sample", n=128256, top_k=40, top_p=0.95, recent=64),
        # Nucleus sampling without top-k over the 7B shape's vocabulary.
        dict(name="sample_top_p", kind="sample", n=32000, top_k=0, top_p=0.9, recent=64),
        # A whole small model early in a chat: a decode step that is all latency.
        dict(name="decode_tiny", kind="decode", model="tiny", layers=4, pos=100, kv_fp16=True),
        # The 7B shape's blocks at the end of a 4096-token context.
        dict(name="decode_7b_4096", kind="decode", model="mistral7b", layers=4, pos=4095, kv_fp16=True),
        # The Phi-3-mini shape's blocks (Q8_0/Q6_K, one kv head per head) with the reference's fp32 KV cache.
        dict(name="decode_phi_fp32kv", kind="decode", model="phi3mini", layers=4, pos=1003, kv_fp16=False),
        # A short user turn behind a long conversation.
        dict(name="turn_7b_23", kind="prompt", model="mistral7b", layers=2, n=23, pos0=1800, kv_fp16=True),
        # A whole model with the fp32 KV cache: an odd-sized prompt on Q5_K.
        dict(name="prompt_small5_fp32kv", kind="prompt", model="small5", layers=4, n=301, pos0=0, kv_fp16=False),
        # The 1B shape's blocks: a page of text.
        dict(name="prompt_1b_512", kind="prompt", model="llama1b", layers=4, n=512, pos0=0, kv_fp16=True),
        # The Phi-3-mini shape's blocks: an odd-sized prompt on Q8_0 and Q6_K.
        dict(name="prompt_phi_777", kind="prompt", model="phi3mini", layers=2, n=777, pos0=0, kv_fp16=True),
        # The 7B shape's blocks: the longest chunk the engine takes at once.
        dict(name="prompt_7b_2048", kind="prompt", model="mistral7b", layers=2, n=2048, pos0=0, kv_fp16=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["matmul", "sample", "decode", "decode", "prompt", "prompt", "prompt"])
    if kind == "matmul":
        # widths and heights of the models' projections, any number of rows
        return dict(kind=kind, type=rng.choice(sorted(TYPES)), m=_log_int(rng, 1, 300),
                    n=_log_int(rng, 96, 8192), k=256 * rng.choice([2, 4, 8, 11, 12, 16, 32]))
    if kind == "sample":
        n = _log_int(rng, 2000, 128256)
        top_k = rng.choice([0, 0, rng.randint(1, 100)])
        return dict(kind=kind, n=n, top_k=top_k, top_p=round(rng.uniform(0.3, 0.97), 3), recent=rng.randint(0, 200))
    model = rng.choice(["tiny", "small5", "llama1b", "phi3mini", "mistral7b"])
    whole = model in ("tiny", "small5")
    layers = 4 if whole else rng.choice([1, 2])
    kv_fp16 = rng.random() < 0.7
    if kind == "decode":
        return dict(kind=kind, model=model, layers=layers, pos=_log_int(rng, 8, 4095), kv_fp16=kv_fp16)
    n = _log_int(rng, 2, 2048)
    pos0 = _log_int(rng, 16, 4096 - n) if n <= 512 and rng.random() < 0.5 else 0
    return dict(kind=kind, model=model, layers=layers, n=n, pos0=pos0, kv_fp16=kv_fp16)


# ------------------------------------------------------------------ inputs --

def _spec(case):
    return dict(synth.SPECS[case["model"]], layers=case["layers"])


def _positions(case):
    return case["pos"] + 1 if case["kind"] == "decode" else case["pos0"] + case["n"]


def _context(case):
    return max(512, (_positions(case) + 511) // 512 * 512)


def _image(case, seed):
    return synth.build_image(case["model"], seed=seed + 1, spec=_spec(case), context=_context(case))


def _tokens(case, seed):
    n = 1 if case["kind"] == "decode" else case["n"]
    return synth.prompt(_spec(case)["vocab"], n, seed=seed + 17)


def _matmul_inputs(case, seed):
    rng = np.random.default_rng(seed + 3)
    t = TYPES[case["type"]]
    w = np.empty(case["n"] * byte_count(t, case["k"]), dtype=np.uint8)
    synth.synth_tensor(t, case["n"], case["k"], seed + 1, w)
    a = rng.standard_normal(case["m"] * case["k"], dtype=np.float32)   # rows after a norm
    return t, w, a


def _logits(case, seed):
    """Logits of a language model: a broad normal bulk and a few clear favourites."""
    rng = np.random.default_rng(seed + 5)
    x = rng.standard_normal(case["n"], dtype=np.float32) * 1.5
    top = rng.choice(case["n"], size=min(200, case["n"] // 4), replace=False)
    x[top] += rng.uniform(3.0, 9.0, size=top.size).astype(np.float32)
    recent = [int(i) for i in np.concatenate([rng.choice(top, size=case["recent"] // 4),
                                              rng.integers(0, case["n"], case["recent"] - case["recent"] // 4)])]
    return x, recent, float(rng.random(dtype=np.float32))


def prepare(case, seed):
    backend = HipBackend()
    kind = case["kind"]
    if kind == "matmul":
        t, w, a = _matmul_inputs(case, seed)
        backend.upload_weight("w", t, w, case["n"], case["k"])
        return dict(case=case, backend=backend, type=t, a=a, y=np.zeros(case["m"] * case["n"], dtype=np.float32))
    if kind == "sample":
        x, recent, r = _logits(case, seed)
        return dict(case=case, backend=backend, x=x, recent=recent, r=r,
                    options=SamplingOptions(top_k=case["top_k"], top_p=case["top_p"]))
    model = LoadedModel.load(_image(case, seed))
    engine = InferenceEngine(model, backend, kv_fp16=case["kv_fp16"], context=_context(case))
    filled = case["pos"] if kind == "decode" else case["pos0"]
    if filled:
        engine.kv_fill_random(filled, seed + 1)
    return dict(case=case, backend=backend, engine=engine, tokens=_tokens(case, seed))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "matmul":
        state["backend"].mat_mul(state["a"], None, state["y"], state["type"], case["k"], case["n"], "w")
        return state["y"]
    if kind == "sample":
        return state["backend"].sample(state["x"], state["options"], state["recent"], state["r"])
    if kind == "decode":
        return state["engine"].process_token(state["tokens"][0], case["pos"])
    logits, _ = state["engine"].prefill(state["tokens"], case["pos0"])
    return logits


# ------------------------------------------------------- necessary work ----

def work(case):
    kind = case["kind"]
    if kind == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": float(n * byte_count(TYPES[case["type"]], k) + 4 * m * (n + k)), "flops": 2.0 * m * n * k}
    if kind == "sample":
        return {"bytes": 4.0 * case["n"], "flops": 4.0 * case["n"]}
    spec = _spec(case)
    n = 1 if kind == "decode" else case["n"]
    pos0 = _positions(case) - n
    weights = params = head = 0
    for name, r, c, t in synth.tensor_list(spec):
        if name == "token_embd.weight":
            weights += n * byte_count(t, c)
        else:
            weights += r * byte_count(t, c)
            if name == "output.weight":
                head = r * c
            elif r > 1:
                params += r * c
    elt = 2 if case["kv_fp16"] else 4
    kv = 2 * spec["layers"] * (pos0 + n) * spec["kv_heads"] * spec["head_dim"] * elt
    keys = n * pos0 + n * (n + 1) // 2
    attn = 4.0 * keys * spec["heads"] * spec["head_dim"] * spec["layers"]
    return {"bytes": float(weights + kv + 4 * spec["vocab"]), "flops": 2.0 * params * n + 2.0 * head + attn}


def tolerance(case):
    if case["kind"] == "sample":
        return "exact"      # a token id
    if case["kind"] == "matmul":
        return {"rel": 1e-5}   # fp32-level sums over exact block integers
    # fp32-level arithmetic throughout, but two of its steps are discontinuous:
    # ExpApprox jumps by up to 18% where its argument crosses certain values
    # (one SiLU output then moves by up to 5%), and a key or value can land on
    # the other side of an fp16 rounding boundary.  Distance to 64 bits over
    # some seeds: decode steps and fp32-cache prompts 6e-7 to 1.3e-6 with a few
    # in 100 at up to 2.4e-4; prompts into an fp16 cache, where every position
    # rounds, 3e-6 to 4.2e-3 with a median of 3e-4.
    return {"rel": 1e-2} if case["kind"] == "prompt" and case["kv_fp16"] else {"rel": 1e-3}


# --------------------------------------------- the same results in 64 bits --

def _blocks(raw, size, dev):
    return torch.from_numpy(np.ascontiguousarray(raw).reshape(-1, size).copy()).to(dev)


def _half(b, at):
    return b[:, at:at + 2].contiguous().view(torch.float16).double()


def _fields6(b):
    """The 16 six-bit fields of the 12 bytes at 4 (first bit lowest), [blocks, 16]."""
    bits = (b[:, 4:16, None] >> torch.arange(8, device=b.device, dtype=torch.uint8)) & 1
    bits = bits.reshape(b.shape[0], 16, 6).double()
    return bits @ (2.0 ** torch.arange(6, device=b.device, dtype=torch.float64))


def _nibbles(q):
    return torch.stack([q & 15, q >> 4], dim=-1).reshape(q.shape[0], -1)


def _dequant(raw, t, rows, cols, dev):
    if t == Q8_0:
        b = _blocks(raw, 34, dev)
        w = b[:, 2:].contiguous().view(torch.int8).double() * _half(b, 0)
    elif t in (Q4_K, Q5_K):
        b = _blocks(raw, 144 if t == Q4_K else 176, dev)
        f = _fields6(b)
        q = _nibbles(b[:, 16:144] if t == Q4_K else b[:, 48:176]).double()
        off = 8.0
        if t == Q5_K:
            hi = (b[:, 16:48, None] >> torch.arange(8, device=dev, dtype=torch.uint8)) & 1
            q, off = q + 16.0 * hi.reshape(b.shape[0], 256).double(), 16.0
        q = (q - off).reshape(-1, 8, 32)
        w = (_half(b, 0) * f[:, 0::2])[:, :, None] * q - (_half(b, 2) * f[:, 1::2])[:, :, None]
    else:   # Q6_K: two halves of 128: 64 bytes of low nibbles, 32 of high pairs, 8 scales each
        b = _blocks(raw, 210, dev)
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], dim=2)
        high = (qh >> torch.tensor([0, 2, 4, 6], device=dev, dtype=torch.uint8).reshape(1, 1, 4, 1)) & 3
        q = low.double() + 16.0 * high.double() - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).double().reshape(-1, 2, 4, 2, 1)
        w = _half(b, 208)[:, :, None, None, None] * sc * q.reshape(-1, 2, 4, 2, 16)
    return w.reshape(rows, cols)


def _exp_approx(x):
    """The engine's exponential (a polynomial about a truncated power of two), in 64 bits."""
    c = x.clamp(-87.3, 88.4)
    k = torch.trunc(c * 1.4426950408889634 + 0.5)
    y = (c - k * 0.693145751953125) - k * 1.42860677e-6
    cc = y * y * 0.5
    cy = cc * y
    r = (1.0 + y + cc + cy * 0.3333333 + cy * y * 0.2) * torch.exp2(k)
    return torch.where(x < -87.3, torch.zeros_like(r), r)


def _filled_kv(layer, kind, n, dim, seed, dev):
    """The engine's seeded KV fill: SplitMix64 of (layer, kind, position, element), [n, dim]."""
    with np.errstate(over="ignore"):
        key = (np.uint64((2 * layer + kind) << 44) | (np.arange(n, dtype=np.uint64) << np.uint64(20))[:, None]
               | np.arange(dim, dtype=np.uint64)[None, :])
        z = np.uint64(seed) + np.uint64(0x9E3779B97F4A7C15) * (key + np.uint64(1))
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    v = ((z >> np.uint64(40)).astype(np.float32) / np.float32(1 << 24) - np.float32(0.5)) * np.float32(3.0)
    return torch.from_numpy(v).to(dev)


def _rope(spec, p0, n, dev):
    """cos and sin of the positions: the angles are rounded to 32 bits, as the model defines them."""
    hd = spec["head_dim"]
    i = np.arange(hd // 2, dtype=np.float32)
    expo = (np.float32(2.0) * i / np.float32(hd)).astype(np.float64)
    freq = np.float32(1.0) / np.power(float(spec["rope_base"]), expo).astype(np.float32)
    ang = (np.arange(p0, p0 + n, dtype=np.float32)[:, None] * freq[None, :]).astype(np.float64)
    return torch.from_numpy(np.cos(ang)).to(dev)[:, None], torch.from_numpy(np.sin(ang)).to(dev)[:, None]


def _rotate(x, cos, sin):
    a, b = x.chunk(2, dim=-1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _exact_model(case, seed, dev):
    spec = _spec(case)
    model = LoadedModel.load(_image(case, seed))

    def weight(name):
        x = model.tensor(name)
        return _dequant(x.data, x.ggml_type, x.rows, x.cols, dev)

    def norm(x):   # the synthetic norm weights are ones
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + float(np.float32(1e-5)))

    tokens = torch.tensor(_tokens(case, seed), device=dev)
    n, total = tokens.numel(), _positions(case)
    p0 = total - n
    heads, kvh, hd = spec["heads"], spec["kv_heads"], spec["head_dim"]
    cos, sin = _rope(spec, p0, n, dev)
    h = weight("token_embd.weight")[tokens]
    pos = torch.arange(p0, total, device=dev)
    keys = torch.arange(total, device=dev)
    vector = (pos + 1) // 8 * 8   # the engine's softmax takes the keys past the last whole 8 with exp
    for l in range(spec["layers"]):
        p = f"blk.{l}."
        x = norm(h)
        q = _rotate((x @ weight(p + "attn_q.weight").t()).reshape(n, heads, hd), cos, sin)
        k = _rotate((x @ weight(p + "attn_k.weight").t()).reshape(n, kvh, hd), cos, sin)
        v = (x @ weight(p + "attn_v.weight").t()).reshape(n, kvh, hd)
        k = torch.cat([_filled_kv(l, 0, p0, kvh * hd, seed + 1, dev).reshape(p0, kvh, hd).double(), k])
        v = torch.cat([_filled_kv(l, 1, p0, kvh * hd, seed + 1, dev).reshape(p0, kvh, hd).double(), v])
        if case["kv_fp16"]:
            k, v = k.half().double(), v.half().double()
        out = torch.empty(n, heads, hd, dtype=torch.float64, device=dev)
        for i in range(heads):
            j = i // (heads // kvh)
            s = (q[:, i].contiguous() @ k[:, j].t().contiguous()) / math.sqrt(hd)
            s = s.masked_fill(keys[None, :] > pos[:, None], -math.inf)
            s = s - s.max(-1, keepdim=True).values
            e = torch.where(keys[None, :] < vector[:, None], _exp_approx(s), torch.exp(s))
            out[:, i] = (e @ v[:, j].contiguous()) / e.sum(-1, keepdim=True)
        h = h + out.reshape(n, -1) @ weight(p + "attn_output.weight").t()
        x = norm(h)
        g = x @ weight(p + "ffn_gate.weight").t()
        g = g / (1.0 + _exp_approx(-g))
        h = h + (g * (x @ weight(p + "ffn_up.weight").t())) @ weight(p + "ffn_down.weight").t()
    return (weight("output.weight") @ norm(h[-1])).cpu()


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if case["kind"] == "sample":
        return None   # a token id
    if case["kind"] == "matmul":
        t, w, a = _matmul_inputs(case, seed)
        x = torch.from_numpy(a).to(dev).double().reshape(case["m"], case["k"])
        return (x @ _dequant(w, t, case["n"], case["k"], dev).t()).reshape(-1).cpu()
    if case["kind"] == "prompt" and case["kv_fp16"]:
        # Which side of an fp16 rounding boundary each key and value falls on is
        # part of these logits: how far two correct results are from the 64-bit
        # one is chance (3e-6 to 4e-3 from seed to seed).  The products are
        # covered by the matmul cases, the rest by the fp32-cache prompts.
        return None
    return _exact_model(case, seed, dev)
