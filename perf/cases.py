"""The framework's work as performance cases: what they are, how their inputs are made, one pass of
each through the public entry points, the work a pass cannot do without, and the same results in
64 bits by plain torch.

A case is a dict of plain values. `path` says what a pass does with a model of the described shape:
  decode    `steps` tokens of a running session at a context of `ctx` positions: one step
            (HipForwardPass.forward) when steps is 1, else the device-side greedy loop
            (decode_greedy); the logits of the last step come back. When the cache is full the
            session starts again from its prompt.
  sample    one token of a sampled session: forward, repetition penalty, top-k candidates.
  prompt    a prompt of `tokens` tokens into an empty cache (prefill); the last logits come back.
  generate  a whole request: a prompt of `tokens` tokens, `steps` generated tokens (greedy with a
            repetition penalty); the tokens and the last logits come back.
Models have few layers (a layer's work is the same in each) at the widths, head counts, tensor types
and contexts of the named configurations and of generic ones; weights are seeded, zero-mean and
scaled as trained ones are, in the GGUF block formats.
"""
import math

import numpy as np
import torch

import dotnetfoundryllm_amd as F
from dotnetfoundryllm_amd import _native as N

ARCH = {"llama": N.ARCH_LLAMA, "mistral": N.ARCH_MISTRAL, "qwen2": N.ARCH_QWEN2, "gemma2": N.ARCH_GEMMA2}
TYPE = {"f16": N.F16, "q4_0": N.Q4_0, "q8_0": N.Q8_0, "q4_k": N.Q4_K, "q5_k": N.Q5_K, "q6_k": N.Q6_K}
# tensor types of a file: (q, k, o, gate, up), (v, down), output
MIX = {"q4_k_m": ("q4_k", "q6_k", "q6_k"), "q5_k": ("q5_k", "q5_k", "q6_k"), "q8_0": ("q8_0", "q8_0", "q8_0"),
       "q4_0": ("q4_0", "q4_0", "q6_k"), "q4_k": ("q4_k", "q4_k", "q4_k"), "f16": ("f16", "f16", "f16")}

# model shapes: hidden, heads, kv heads, head_dim, ffn, rope base
SHAPE = {
    "tiny": ("llama", 512, 8, 2, 64, 1408, 10000.0),
    "llama-4096": ("llama", 4096, 32, 8, 128, 14336, 500000.0),
    "mistral-4096": ("mistral", 4096, 32, 8, 128, 14336, 10000.0),
    "qwen2-3584": ("qwen2", 3584, 28, 4, 128, 18944, 1000000.0),
    "gemma2-3584": ("gemma2", 3584, 16, 8, 256, 14336, 10000.0),
    "llama-2048": ("llama", 2048, 16, 4, 128, 5632, 10000.0),
    "qwen2-1536": ("qwen2", 1536, 12, 2, 128, 8960, 1000000.0),
    "gemma2-2304": ("gemma2", 2304, 8, 4, 256, 9216, 10000.0),
}


def _case(name, path, shape, mix, layers, vocab, tokens=0, ctx=0, steps=0, window=4096):
    c = dict(path=path, shape=shape, mix=mix, layers=layers, vocab=vocab, tokens=tokens, ctx=ctx, steps=steps,
             window=window)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: one token of the tiny model, all its layers, the host choosing the token
        _case("decode-tiny", "decode", "tiny", "q4_k", 8, 32000, ctx=200, steps=1),
        # an 8B model's layers in the device-side greedy loop, the ordinary chat context
        _case("decode-llama-512", "decode", "llama-4096", "q4_k_m", 2, 2048, ctx=512, steps=16),
        # a Qwen2 model's layers at a longer context, the host taking every token's logits
        _case("decode-qwen2-2k", "decode", "qwen2-3584", "q5_k", 2, 2048, ctx=2049, steps=1),
        # Gemma-2's layers (one windowed, one full) at a long context
        _case("decode-gemma2-6k", "decode", "gemma2-3584", "q8_0", 2, 2048, ctx=6150, steps=8),
        # an unquantized model's layer
        _case("decode-f16", "decode", "llama-4096", "f16", 1, 2048, ctx=301, steps=1),
        # one sampled token over a 152064-entry vocabulary: a layer, the LM head, penalty, top-k 40
        _case("sample-152k", "sample", "qwen2-3584", "q5_k", 1, 152064, ctx=256, steps=1),
        # prompts: a question, a page, a long document, the longest window's document
        _case("prompt-37", "prompt", "llama-4096", "q4_k_m", 2, 2048, tokens=37),
        _case("prompt-511", "prompt", "llama-4096", "q4_k_m", 2, 2048, tokens=511),
        _case("prompt-2047", "prompt", "qwen2-3584", "q5_k", 2, 2048, tokens=2047),
        _case("prompt-6143", "prompt", "gemma2-3584", "q8_0", 2, 2048, tokens=6143),
        # a prompt of a Q4_0 file with the window on every layer
        _case("prompt-q4_0-300", "prompt", "mistral-4096", "q4_0", 1, 2048, tokens=300, window=256),
        # a whole request on the tiny model
        _case("generate-tiny", "generate", "tiny", "q4_k", 8, 32000, tokens=100, steps=24),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["decode", "decode", "prompt", "prompt", "prompt", "sample", "generate"])
    if path == "generate":
        return _case(None, path, "tiny", rng.choice(["q4_k", "q8_0", "q4_0"]), 8, 32000, tokens=_log_int(rng, 2, 400),
                     steps=rng.randint(4, 40))
    if path == "sample":
        return _case(None, path, rng.choice(["llama-2048", "qwen2-1536"]), rng.choice(["q4_k_m", "q8_0", "q5_k"]), 1,
                     rng.choice([32000, 128256, 151936, 152064]), ctx=_log_int(rng, 16, 1500), steps=1)
    shape, mix = rng.choice([("tiny", "q4_k"), ("tiny", "q8_0"), ("llama-4096", "q4_k_m"), ("llama-4096", "q8_0"),
                             ("qwen2-3584", "q5_k"), ("qwen2-3584", "q4_k_m"), ("gemma2-3584", "q8_0"),
                             ("mistral-4096", "q4_0"), ("mistral-4096", "q4_k_m"), ("llama-2048", "q4_k_m"),
                             ("llama-2048", "q5_k"), ("qwen2-1536", "q4_k_m"), ("gemma2-2304", "q8_0"),
                             ("gemma2-2304", "q5_k"), ("llama-2048", "f16")])
    small = shape in ("tiny", "llama-2048", "qwen2-1536", "gemma2-2304")
    layers = 8 if shape == "tiny" else 2
    slow = mix in ("f16", "q4_0")  # the formats without a regrouped layout: shorter prompts
    window = rng.choice([256, 1024, 4096])
    if path == "decode":
        return _case(None, path, shape, mix, layers, 2048, ctx=_log_int(rng, 16, 4000 if shape != "tiny" else 400),
                     steps=rng.choice([1, 1, 8, 16]), window=window)
    return _case(None, path, shape, mix, layers, 2048,
                 tokens=_log_int(rng, 2, 500 if shape == "tiny" else 700 if slow else 5000 if small else 3000),
                 window=window)


# ---- inputs ---------------------------------------------------------------------------------------
def _halves(v):
    return v.to(torch.float16).view(torch.uint8).reshape(v.shape + (2,))


def _blocks(tt, rows, cols, std, gen):
    """Random zero-mean weights of about `std` in GGUF blocks of type tt, as bytes on the GPU."""
    dev = "cuda"

    def bytes_(*shape):
        return torch.randint(0, 256, shape, dtype=torch.uint8, device=dev, generator=gen)

    def spread(n):
        return 0.75 + 0.5 * torch.rand(n, device=dev, generator=gen)

    if tt == N.F16:
        w = torch.randn(rows * cols, device=dev, generator=gen) * std
        return w.to(torch.float16).view(torch.uint8)
    if tt == N.F32:
        return (torch.randn(rows * cols, device=dev, generator=gen) * std).view(torch.uint8)
    if tt in (N.Q4_0, N.Q8_0):
        n = rows * cols // 32
        if tt == N.Q4_0:  # q uniform in 0..15: deviation 4.61
            return torch.cat([_halves(spread(n) * (std / 4.61)), bytes_(n, 16)], 1).reshape(-1)
        q = (torch.randn((n, 32), device=dev, generator=gen) * 40.0).clamp_(-127, 127).round_().to(torch.int8)
        return torch.cat([_halves(spread(n) * (std / 40.0)), q.view(torch.uint8)], 1).reshape(-1)
    n = rows * cols // 256
    if tt == N.Q6_K:  # d * scale * (q - 32): |scale| about 74, q uniform
        sc = torch.randint(20, 128, (n, 16), device=dev, generator=gen)
        sc = torch.where(bytes_(n, 16) < 128, sc, -sc).to(torch.int8).view(torch.uint8)
        return torch.cat([bytes_(n, 192), sc, _halves(spread(n) * (std / (80.0 * 18.5)))], 1).reshape(-1)
    mid, dev_q = (7.5, 4.61) if tt == N.Q4_K else (15.5, 9.23)
    sc = torch.randint(8, 64, (n, 8), device=dev, generator=gen)
    mn = (sc + torch.randint(-3, 4, (n, 8), device=dev, generator=gen)).clamp_(0, 63)
    d = spread(n) * (std / (39.0 * dev_q))
    packed = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6),
                        (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1).to(torch.uint8)
    rest = 128 if tt == N.Q4_K else 160
    return torch.cat([_halves(d), _halves(d * mid), packed, bytes_(n, rest)], 1).reshape(-1)


def _tensors(case, seed):
    """Every tensor of the model: (slot, layer, type, rows, cols, bytes on the GPU), one at a time."""
    arch, H, nh, nkv, hd, ffn, _ = SHAPE[case["shape"]]
    main, wide, out = (TYPE[t] for t in MIX[case["mix"]])
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed * 7919 + 17)
    gemma = arch == "gemma2"

    def mat(slot, layer, tt, rows, cols, std=None):
        return slot, layer, tt, rows, cols, _blocks(tt, rows, cols, std or 1.0 / math.sqrt(cols), gen)

    def norm(slot, layer):
        w = torch.randn(H, device="cuda", generator=gen) * 0.1 + (0.0 if gemma else 1.0)
        return slot, layer, N.F32, 1, H, w.view(torch.uint8)

    emb = N.F32 if case["shape"] == "tiny" else main if case["path"] == "sample" else N.F16
    yield mat(N.SLOT_TOKEN_EMBD, 0, emb, case["vocab"], H, 0.5)
    yield norm(N.SLOT_OUTPUT_NORM, 0)
    yield mat(N.SLOT_OUTPUT, 0, out, case["vocab"], H)
    for l in range(case["layers"]):
        yield norm(N.SLOT_ATTN_NORM, l)
        yield mat(N.SLOT_ATTN_Q, l, main, nh * hd, H)
        yield mat(N.SLOT_ATTN_K, l, main, nkv * hd, H)
        yield mat(N.SLOT_ATTN_V, l, wide, nkv * hd, H)
        yield mat(N.SLOT_ATTN_OUTPUT, l, main, H, nh * hd)
        yield norm(N.SLOT_FFN_NORM, l)
        yield mat(N.SLOT_FFN_GATE, l, main, ffn, H)
        yield mat(N.SLOT_FFN_UP, l, main, ffn, H)
        yield mat(N.SLOT_FFN_DOWN, l, wide, H, ffn)
        if arch == "qwen2":
            for slot, n in ((N.SLOT_ATTN_Q_BIAS, nh * hd), (N.SLOT_ATTN_K_BIAS, nkv * hd), (N.SLOT_ATTN_V_BIAS, nkv * hd)):
                yield mat(slot, l, N.F32, 1, n, 0.1)
        if gemma:
            yield norm(N.SLOT_POST_ATTN_NORM, l)
            yield norm(N.SLOT_POST_FFN_NORM, l)


def _desc(case):
    arch, H, nh, nkv, hd, ffn, base = SHAPE[case["shape"]]
    gemma = arch == "gemma2"
    d = N.ModelDesc()
    d.arch, d.n_layers, d.hidden, d.ffn, d.n_heads, d.n_kv_heads = ARCH[arch], case["layers"], H, ffn, nh, nkv
    d.head_dim, d.vocab, d.max_ctx, d.rope_base, d.rope_scale, d.rope_scaled = hd, case["vocab"], 8192, base, 1.0, 0
    d.norm_eps, d.attn_scale = (1e-6 if gemma else 1e-5), float(np.float32(1.0) / np.sqrt(np.float32(hd)))
    d.attn_softcap, d.final_softcap = (50.0, 30.0) if gemma else (0.0, 0.0)
    d.sliding_window = case["window"] if arch in ("gemma2", "mistral") else 0x7FFFFFFF
    return d


def _prompt(case, seed, n):
    return np.random.default_rng(seed).integers(0, case["vocab"], n).astype(np.int32)


def _capacity(case):
    """Cache positions: the prompt and room for a session's tokens."""
    need = {"decode": case["ctx"] + 512, "sample": case["ctx"] + 512, "prompt": case["tokens"] + 64,
            "generate": case["tokens"] + case["steps"] + 1}[case["path"]]
    return (need + 255) // 256 * 256


_context = []


class _Session:
    """A model on the GPU and one sequence of it, given back when dropped."""

    def __init__(self, case, seed):
        if not _context:
            _context.append(F.Context(0))  # a program keeps one
        self.case = case
        self.model = F.Model(_context[0], _desc(case))
        for slot, layer, tt, _, _, data in _tensors(case, seed):
            self.model.upload(slot, layer, tt, data.cpu().numpy())
        self.model.finalize()
        self.kv = F.HipKvCache(self.model, _capacity(case))
        self.fwd = F.HipForwardPass(self.model)
        self.prompt = _prompt(case, seed, case["ctx"] or case["tokens"])
        self.next = _prompt(case, seed + 1, 4096)  # what the user's session feeds, by position
        self.lm = self.sampler = None

    def begin(self):
        self.kv.clear()
        self.fwd.prefill(self.prompt, 0, self.kv)

    def __del__(self):
        for held in ("sampler", "kv", "model"):
            if getattr(self, held, None) is not None:
                getattr(self, held).close()


PENALTY, TEMPERATURE, TOP_K, RECENT = 1.1, 0.8, 40, 64


def prepare(case, seed):
    s = _Session(case, seed)
    if case["path"] in ("decode", "sample"):
        s.begin()
    if case["path"] == "generate":
        s.lm = F.LlamaLanguageModel(s.model, s.kv)
        s.sampler = F.SamplerPipeline(temperature=0.0)
    return s


def run(s):
    case, kv, fwd = s.case, s.kv, s.fwd
    if case["path"] == "prompt":
        s.begin()
        return {"logits": fwd.logits}
    if case["path"] == "generate":
        tokens, _ = s.lm.generate(s.prompt, case["steps"], s.sampler, stop_at_eos=False, repetition_penalty=PENALTY)
        fwd.forward(int(tokens[-1]), kv.current_length, kv)  # the logits after the last token
        return {"tokens": tokens, "logits": fwd.logits}
    pos = kv.current_length
    if pos + case["steps"] > kv.max_sequence_length:
        s.begin()
        pos = kv.current_length
    token = int(s.next[pos % 4096])
    if case["path"] == "sample":
        fwd.forward(token, pos, kv)
        fwd.penalize(s.next[:RECENT], PENALTY)
        ids, vals = fwd.sample_topk(1.0 / TEMPERATURE, TOP_K)
        return {"ids": ids, "vals": vals}
    if case["steps"] == 1:
        fwd.forward(token, pos, kv)
        return {"logits": fwd.logits}
    tokens = fwd.decode_greedy(token, pos, case["steps"], kv)
    return {"tokens": tokens, "logits": fwd.logits}


# ---- what a pass cannot do without ------------------------------------------------------------------
def _bytes_of(tt, n):
    return n * 4 if tt == N.F32 else n * 2 if tt == N.F16 else N.type_bytes(tt, n)


def work(case):
    arch, H, nh, nkv, hd, ffn, _ = SHAPE[case["shape"]]
    main, wide, out = (TYPE[t] for t in MIX[case["mix"]])
    q, kvd, L = nh * hd, nkv * hd, case["layers"]
    layer_n = 2 * q * H + 2 * kvd * H + 3 * ffn * H
    layer_b = _bytes_of(main, 2 * q * H + kvd * H + 2 * ffn * H) + _bytes_of(wide, kvd * H + ffn * H)
    head_n, head_b = case["vocab"] * H, _bytes_of(out, case["vocab"] * H)

    def spans(lo, hi):  # positions attended, summed over the query positions [lo, hi) and the layers
        full = sum(range(lo + 1, hi + 1))
        cut = sum(min(p, case["window"]) for p in range(lo + 1, hi + 1))
        return {"mistral": L * cut, "gemma2": (L + 1) // 2 * cut + L // 2 * full}.get(arch, L * full)

    def tokens_once(lo, hi):  # the positions' projections and attention, every weight and row once
        n = hi - lo
        return (L * layer_b + head_b + 8.0 * kvd * L * hi + 4.0 * n * H + 4.0 * case["vocab"],
                2.0 * (n * L * layer_n + head_n) + 4.0 * q * spans(lo, hi))

    def steps(lo, n):
        got = [(L * layer_b + head_b + 8.0 * kvd * spans(p, p + 1) + 4.0 * case["vocab"],
                2.0 * (L * layer_n + head_n) + 4.0 * q * spans(p, p + 1)) for p in range(lo, lo + n)]
        return sum(b for b, _ in got), sum(f for _, f in got)

    if case["path"] == "prompt":
        b, f = tokens_once(0, case["tokens"])
    elif case["path"] == "generate":
        b, f = steps(case["tokens"] - 1, case["steps"] + 1)
        if case["tokens"] > 1:
            pb, pf = tokens_once(0, case["tokens"] - 1)
            b, f = b + pb - head_b, f + pf - 2.0 * head_n
    else:
        b, f = steps(case["ctx"], case["steps"])
    return {"bytes": b, "flops": f}


def tolerance(case):
    # float32 sums over operands of 22 to 24 bits: measured against 64 bits 4e-7 to 2.5e-6 of the
    # logits (the 8 layers of the tiny model and Gemma-2's post-norms the most), 1.4e-5 for prompts of
    # the formats without a regrouped layout; a near-tie may change a chosen token
    plain = case["path"] in ("prompt", "generate") and case["mix"] in ("q4_0", "f16")
    return {"rel": 5e-5 if plain else 1e-5, "max": 1e-3 if plain else 2e-4, "differ": 0.01}


# ---- the same in 64 bits ------------------------------------------------------------------------------
def _dequant(tt, raw, rows, cols):
    """Weights of GGUF blocks in float64, [rows][cols]; each format as its definition says."""
    if tt == N.F32:
        return raw.view(torch.float32).double().reshape(rows, cols)
    if tt == N.F16:
        return raw.view(torch.float16).double().reshape(rows, cols)
    nbytes, _ = N.BLOCK[tt]
    b = raw.reshape(-1, nbytes)

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    def nibbles(x):  # low, then high, of each byte
        return torch.stack([x & 15, x >> 4], -1).flatten(1)

    if tt == N.Q4_0:
        q = torch.cat([b[:, 2:18] & 15, b[:, 2:18] >> 4], 1).double() - 8
        return (q * half(0)).reshape(rows, cols)
    if tt == N.Q8_0:
        return (b[:, 2:34].contiguous().view(torch.int8).double() * half(0)).reshape(rows, cols)
    if tt == N.Q6_K:
        hi = torch.stack([(b[:, 128:192] >> s) & 3 for s in (0, 2, 4, 6)], -1).flatten(1)
        q = nibbles(b[:, :128]).double() + 16 * hi.double() - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double().repeat_interleave(16, 1)
        return (half(208) * sc * q).reshape(rows, cols)
    s = b[:, 4:16]
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    q = nibbles(b[:, 16:144] if tt == N.Q4_K else b[:, 48:176]).double()
    if tt == N.Q5_K:
        q = q + 16 * torch.stack([(b[:, 16:48] >> i) & 1 for i in range(8)], -1).flatten(1).double()
    w = (half(0) * sc).repeat_interleave(32, 1) * q - (half(2) * mn).repeat_interleave(32, 1)
    return w.reshape(rows, cols)


class _Exact:
    """The model in float64: feeds tokens, keeps keys and values, gives the last token's logits."""

    def __init__(self, case, seed):
        self.case = case
        self.raw = {(slot, layer): (tt, rows, cols, data) for slot, layer, tt, rows, cols, data in _tensors(case, seed)}
        self.k, self.v, self.n = [None] * case["layers"], [None] * case["layers"], 0
        base, hd = SHAPE[case["shape"]][6], SHAPE[case["shape"]][4]
        # the rotation angles are float32 by definition: pos * (1 / base^(2 i / hd))
        e = (np.float32(2) * np.arange(hd // 2, dtype=np.float32)) / np.float32(hd)
        self.inv = np.float32(1) / np.power(np.float64(base), e.astype(np.float64)).astype(np.float32)

    def vec(self, slot, layer=0):
        return self.raw[slot, layer][3].view(torch.float32).double()

    def mul(self, x, slot, layer=0):
        tt, rows, cols, data = self.raw[slot, layer]
        step = max(256, (1 << 27) // cols // 256 * 256)  # rows at a time
        per = data.numel() // rows
        return torch.cat([x @ _dequant(tt, data[r * per:min(rows, r + step) * per], min(rows, r + step) - r, cols).t()
                          for r in range(0, rows, step)], 1)

    def norm(self, x, slot, layer=0):
        gemma = SHAPE[self.case["shape"]][0] == "gemma2"
        w = self.vec(slot, layer) + (1.0 if gemma else 0.0)
        return x * torch.rsqrt(x.square().mean(1, keepdim=True) + (1e-6 if gemma else float(np.float32(1e-5)))) * w

    def rope(self, x, n):
        hd = SHAPE[self.case["shape"]][4]
        th = np.arange(self.n, self.n + n, dtype=np.float32)[:, None] * self.inv[None, :]
        th = torch.from_numpy(th.astype(np.float64)).cuda()[:, None, :]
        c, s = th.cos(), th.sin()
        x = x.reshape(n, -1, hd // 2, 2)
        return torch.stack([x[..., 0] * c - x[..., 1] * s, x[..., 0] * s + x[..., 1] * c], -1).reshape(n, -1, hd)

    def feed(self, tokens):
        case = self.case
        arch, H, nh, nkv, hd, ffn, _ = SHAPE[case["shape"]]
        gemma, n = arch == "gemma2", len(tokens)
        tt, rows, cols, data = self.raw[N.SLOT_TOKEN_EMBD, 0]
        per = data.numel() // rows
        ids = torch.from_numpy(np.asarray(tokens, dtype=np.int64)).cuda()
        x = _dequant(tt, data.reshape(rows, per)[ids].contiguous().reshape(-1), n, cols)
        for l in range(case["layers"]):
            xn = self.norm(x, N.SLOT_ATTN_NORM, l)
            q, k, v = (self.mul(xn, t, l) for t in (N.SLOT_ATTN_Q, N.SLOT_ATTN_K, N.SLOT_ATTN_V))
            if arch == "qwen2":
                q, k, v = (y + self.vec(t, l) for y, t in
                           ((q, N.SLOT_ATTN_Q_BIAS), (k, N.SLOT_ATTN_K_BIAS), (v, N.SLOT_ATTN_V_BIAS)))
            q, k, v = self.rope(q, n), self.rope(k, n), v.reshape(n, nkv, hd)
            self.k[l] = k if self.n == 0 else torch.cat([self.k[l], k])
            self.v[l] = v if self.n == 0 else torch.cat([self.v[l], v])
            qp = torch.arange(self.n, self.n + n, device="cuda")[:, None]
            kp = torch.arange(self.n + n, device="cuda")[None, :]
            dead = kp > qp
            if arch == "mistral" or (gemma and l % 2 == 0):
                dead = dead | (kp <= qp - case["window"])
            heads = []
            for h in range(nh):
                g = h // (nh // nkv)
                s = q[:, h].contiguous() @ self.k[l][:, g].t().contiguous() * float(np.float32(1.0) / np.sqrt(np.float32(hd)))
                if gemma:
                    s = torch.tanh(s / 50.0) * 50.0
                heads.append(torch.softmax(s.masked_fill_(dead, -math.inf), 1) @ self.v[l][:, g].contiguous())
            o = self.mul(torch.cat(heads, 1), N.SLOT_ATTN_OUTPUT, l)
            x = x + (self.norm(o, N.SLOT_POST_ATTN_NORM, l) if gemma else o)
            xn = self.norm(x, N.SLOT_FFN_NORM, l)
            g, u = self.mul(xn, N.SLOT_FFN_GATE, l), self.mul(xn, N.SLOT_FFN_UP, l)
            if gemma:
                g = 0.5 * g * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (g + 0.044715 * g ** 3)))
            else:
                g = g * torch.sigmoid(g)
            o = self.mul(g * u, N.SLOT_FFN_DOWN, l)
            x = x + (self.norm(o, N.SLOT_POST_FFN_NORM, l) if gemma else o)
        self.n += n
        y = self.mul(self.norm(x[-1:], N.SLOT_OUTPUT_NORM), N.SLOT_OUTPUT)[0]
        return torch.tanh(y / 30.0) * 30.0 if gemma else y


def _penalized(y, ids):
    for i in ids:
        y[i] = y[i] / float(np.float32(PENALTY)) if y[i] > 0 else y[i] * float(np.float32(PENALTY))
    return y


def exact(case, seed):
    m = _Exact(case, seed)
    prompt, following = _prompt(case, seed, case["ctx"] or case["tokens"]), _prompt(case, seed + 1, 4096)
    if case["path"] == "prompt":
        return {"logits": m.feed(prompt)}
    if case["path"] == "generate":
        tokens = []
        y = m.feed(prompt)
        for i in range(case["steps"]):
            y = _penalized(y if i == 0 else m.feed(tokens[-1:]), tokens)
            tokens.append(int(y.argmax()))
        return {"tokens": None, "logits": m.feed(tokens[-1:])}
    m.feed(prompt)
    token = int(following[case["ctx"] % 4096])
    if case["path"] == "sample":
        y = _penalized(m.feed([token]).cpu(), following[:RECENT].tolist()) / float(np.float32(TEMPERATURE))
        ids = torch.sort(torch.topk(y, TOP_K).indices).values
        return {"ids": None, "vals": y[ids]}
    for _ in range(case["steps"]):
        y = m.feed([token])
        token = int(y.argmax())
    return {"tokens": None, "logits": y} if case["steps"] > 1 else {"logits": y}
