"""The work that stands for this framework's use, as cases that a timing harness can run.

Three families, each through the entry points that a program calls:

  matmul     activation rows against one quantized weight (`step_matmul`): a decode step's single row, a batch of decode
             rows, a prompt's rows; q4_0 and q8_0; aion's int8 arithmetic (the default) and the bf16 mode
  attention  one attention step over a KV cache (`step_attention`): a prompt over its own keys and a query token per
             sequence over a long cache, with the cache types, head layouts and windows that models use
  decoder    a decoder-only model (`Decoder`, `SessionDecoder`): a prompt from an empty cache, and a run of greedy tokens
             behind a prompt

`listed()` holds one case per kind of use, `draw()` samples the ranges they stand for.
"""
import math

import numpy as np
import torch

from aion_amd import backend as be
from aion_amd.decoder import Decoder, DecoderConfig, SessionDecoder

WEIGHT = {"q4": be.Q4_0, "q8": be.Q8_0}
CACHE = {"bf16": be.BF16, "f16": be.F16}
TORCH = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
QUERY = {"bf16": be.BF16, "f16": be.F16, "f32": be.F32}
MODE = {"exact": be.GEMM_EXACT_I8, "bf16": be.GEMM_BF16_MFMA}


def listed():
    return [
        # the smallest call: one row against a square q8 projection
        {"name": "matmul_q8_1x2048x2048", "family": "matmul", "weight": "q8", "m": 1, "n": 2048, "k": 2048, "mode": "exact"},
        # the logits of one token over a large vocabulary: the largest weight stream of a decode step
        {"name": "matmul_q4_1x262144x2048", "family": "matmul", "weight": "q4", "m": 1, "n": 262144, "k": 2048, "mode": "exact"},
        # four sequences decoded together, down projection of a mid-sized model
        {"name": "matmul_q4_4x4096x14336", "family": "matmul", "weight": "q4", "m": 4, "n": 4096, "k": 14336, "mode": "exact"},
        # eight sequences decoded together, gate or up projection, q8
        {"name": "matmul_q8_8x14336x4096", "family": "matmul", "weight": "q8", "m": 8, "n": 14336, "k": 4096, "mode": "exact"},
        # a short prompt of odd length against a projection whose width is no power of two
        {"name": "matmul_q8_77x11008x4096", "family": "matmul", "weight": "q8", "m": 77, "n": 11008, "k": 4096, "mode": "exact"},
        # an ordinary prompt, aion's arithmetic
        {"name": "matmul_q4_512x4096x4096", "family": "matmul", "weight": "q4", "m": 512, "n": 4096, "k": 4096, "mode": "exact"},
        # a long prompt in the bf16 mode, the throughput path
        {"name": "matmul_q4_2048x14336x4096_bf16", "family": "matmul", "weight": "q4", "m": 2048, "n": 14336, "k": 4096, "mode": "bf16"},
        # a long prompt over its own keys: 8 query heads on one KV head of size 256
        {"name": "attention_prompt_4096", "family": "attention", "batch": 1, "queries": 4096, "keys": 4096, "heads": 8, "kv_heads": 1,
         "head": 256, "query": "bf16", "cache": "bf16", "window": 0},
        # one token of eight sequences over long caches
        {"name": "attention_token_16384_b8", "family": "attention", "batch": 8, "queries": 1, "keys": 16384, "heads": 8, "kv_heads": 1,
         "head": 256, "query": "bf16", "cache": "bf16", "window": 0},
        # one token over a cache of odd length in the decoder's own types, grouped heads of size 128
        {"name": "attention_token_1531", "family": "attention", "batch": 1, "queries": 1, "keys": 1531, "heads": 32, "kv_heads": 8,
         "head": 128, "query": "f32", "cache": "f16", "window": 0},
        # the time to the first token: a 128-token prompt through 26 blocks and the logits
        {"name": "decoder_prompt_128", "family": "decoder", "entry": "decoder", "layers": 26, "hidden": 2048, "heads": 8, "kv_heads": 1,
         "head": 256, "ffn": 8192, "vocab": 262144, "weight": "q4", "prompt": 128, "tokens": 0},
        # 16 greedy tokens behind it, batch 1
        {"name": "decoder_tokens_16", "family": "decoder", "entry": "decoder", "layers": 26, "hidden": 2048, "heads": 8, "kv_heads": 1,
         "head": 256, "ffn": 8192, "vocab": 262144, "weight": "q4", "prompt": 128, "tokens": 16},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_matmul(rng):
    k = 32 * _log(rng, 16, 448)                                        # 512 .. 14336, any number of quant blocks
    n = _log(rng, 512, 262144 if k <= 4096 else 32768)
    if rng.random() < 0.6:
        n = max(64, n // 64 * 64)                                      # most projections, but not all, are whole tiles wide
    m = 1 if rng.random() < 0.25 else _log(rng, 2, 2048)
    mode = "bf16" if m >= 64 and rng.random() < 0.35 else "exact"
    return {"family": "matmul", "weight": rng.choice(["q4", "q8"]), "m": m, "n": n, "k": k, "mode": mode}


def _draw_attention(rng):
    heads, kv_heads, head = rng.choice([(8, 1, 256), (8, 2, 256), (32, 8, 128), (32, 32, 128), (16, 4, 64)])
    cache = rng.choice(["bf16", "f16"])
    query = cache if rng.random() < 0.5 else "f32"
    window = 0 if rng.random() < 0.75 else _log(rng, 128, 2048)
    if rng.random() < 0.5:
        batch, queries = rng.choice([1, 1, 1, 2, 4]), _log(rng, 16, 4096)
        keys = queries
    else:
        batch, queries, keys = rng.choice([1, 1, 2, 4, 8, 16]), 1, _log(rng, 64, 16384)
    return {"family": "attention", "batch": batch, "queries": queries, "keys": keys, "heads": heads, "kv_heads": kv_heads, "head": head,
            "query": query, "cache": cache, "window": window}


def _draw_decoder(rng):
    head = rng.choice([64, 128, 256])
    hidden = 256 * rng.randint(4, 16)
    heads = hidden // head
    kv_heads = rng.choice([g for g in (1, 2, 4, 8) if heads % g == 0])
    tokens = 0 if rng.random() < 0.5 else rng.randint(4, 16)
    return {"family": "decoder", "entry": "session" if tokens == 0 and rng.random() < 0.4 else "decoder", "layers": rng.randint(2, 26), "hidden": hidden,
            "heads": heads, "kv_heads": kv_heads, "head": head, "ffn": 256 * rng.randint(hidden // 128, hidden // 64),
            "vocab": 256 * _log(rng, 32, 512), "weight": rng.choice(["q4", "q8"]), "prompt": _log(rng, 8, 512), "tokens": tokens}


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        u = rng.random()
        case = _draw_matmul(rng) if u < 0.5 else _draw_attention(rng) if u < 0.8 else _draw_decoder(rng)
        if _cost(case) <= most:
            return case


def _cost(case):
    w = work(case)
    return max(w["bytes"] / 4e12, w["flops"] / 5e14)


# ---------------------------------------------------------------------------------------------------------- what a pass needs
def _weight_bytes(kind, n, k):
    return n * k // 32 * be.BLOCK_BYTES[WEIGHT[kind]]


def _visible(case):
    """Query-key pairs of one (sequence, head) and keys that any query sees, summed over the batch."""
    pairs = keys = 0
    for length in _lengths(case):
        first = length - case["queries"]
        w = case["window"]
        if w == 0:
            pairs += case["queries"] * first + case["queries"] * (case["queries"] + 1) // 2
            keys += length
        else:
            pos = np.arange(first, length)
            pairs += int(np.minimum(pos + 1, w + 1).sum())
            keys += length - max(0, first - w)
    return pairs, keys


def _lengths(case):
    """Keys of each sequence: a prompt fills its cache, sequences that are decoded together are at different lengths."""
    t, b = case["keys"], case["batch"]
    if case["queries"] > 1 or case["window"] == 0 and t % 2 == 0:
        return [t] * b
    return [max(1, t - i * t // (2 * b)) for i in range(b)]


def work(case):
    if case["family"] == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _weight_bytes(case["weight"], n, k) + 4 * m * (n + k), "flops": 2 * m * n * k}
    if case["family"] == "attention":
        pairs, keys = _visible(case)
        size = {"bf16": 2, "f16": 2, "f32": 4}
        rows = case["batch"] * case["queries"] * case["heads"] * case["head"]
        return {"bytes": rows * (size[case["query"]] + 4) + 2 * keys * case["kv_heads"] * case["head"] * 2,
                "flops": 4 * pairs * case["heads"] * case["head"]}
    cfg = _config(case)
    block = cfg.hidden * (2 * cfg.q_dim + 2 * cfg.kv_dim + 3 * cfg.ffn)
    blocks = sum(_weight_bytes(case["weight"], 1, block) for _ in range(cfg.layers))
    head = _weight_bytes(case["weight"], cfg.vocab, cfg.hidden)
    p, t = case["prompt"], case["tokens"]
    if t == 0:
        cache = 2 * cfg.layers * p * cfg.kv_dim * 2
        flops = 2 * p * block * cfg.layers + 2 * cfg.vocab * cfg.hidden + 2 * cfg.layers * p * (p + 1) * cfg.q_dim
        return {"bytes": blocks + head + cache + 4 * p * cfg.hidden + 4 * cfg.vocab, "flops": flops}
    cache = sum(2 * cfg.layers * (p + i + 1) * cfg.kv_dim * 2 for i in range(t))
    flops = t * (2 * block * cfg.layers + 2 * cfg.vocab * cfg.hidden) + 4 * cfg.layers * cfg.q_dim * sum(p + i + 1 for i in range(t))
    return {"bytes": t * (blocks + head + 4 * cfg.hidden + 4 * cfg.vocab) + cache, "flops": flops}


def tolerance(case):
    """Measured: exact matmuls against their integer codes and scales in float64 8e-8 .. 1.2e-7, the bf16 mode against unrounded
    operands 2.3e-3, attention against float64 1.3e-3 (bf16 cache) and 2.5e-4 (f16), a decoder's logits and cache rows with the
    attention's probabilities in half precision against hi + lo parts 4e-3 .. 1.2e-2 (max 0.08)."""
    if case["family"] == "matmul":
        return {"rel": 4e-3} if case["mode"] == "bf16" else {"rel": 8e-7, "max": 2e-5}
    if case["family"] == "attention":
        return {"rel": 5e-3, "max": 0.12} if case["cache"] == "bf16" else {"rel": 1e-3, "max": 0.03}
    return {"rel": 2.5e-2, "max": 0.3}


# ----------------------------------------------------------------------------------------------------------------- the program
_contexts = {}


def _context(mode):
    """One context per GEMM mode for the whole program, as a serving process keeps it."""
    if mode not in _contexts:
        _contexts[mode] = be.HipBackend(0)
        _contexts[mode].set_gemm_mode(MODE[mode])
    return _contexts[mode]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _buffer(gpu, tensor):
    """A torch tensor's memory as an operand of the steps (the tensor keeps owning it)."""
    return be.DeviceBuffer(gpu, tensor.data_ptr(), tensor.numel() * tensor.element_size())


class _Memory:
    def __init__(self, handle, shape, typestr):
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (handle, False), "version": 2}


def _tensor(buffer, shape, typestr):
    """Memory of the framework as a torch tensor."""
    return torch.as_tensor(_Memory(buffer.handle, shape, typestr), device="cuda")


def _blocks(gpu, kind, n, k, values):
    """Device buffer with the packed blocks of an [n, k] weight given as the f32 tensor `values` in the layout of its type:
    q8_0 [n, k] blocked along k, q4_0 [k, n] blocked along k."""
    torch.cuda.synchronize()
    rows, cols, axis = (n, k, 1) if kind == "q8" else (k, n, 0)
    packed = gpu.quantize_device(WEIGHT[kind], _buffer(gpu, values), rows, cols, axis)
    gpu.sync()
    return packed


def _normal(kind, n, k, std, gen):
    return torch.randn((n, k) if kind == "q8" else (k, n), generator=gen, device="cuda").mul_(std)


class _Matmul:
    def __init__(self, case, seed):
        self.gpu, gen = _context(case["mode"]), _generator(seed)
        m, n, k, kind = case["m"], case["n"], case["k"], case["weight"]
        packed = _blocks(self.gpu, kind, n, k, _normal(kind, n, k, 0.02, gen))
        self.weight = self.gpu.weight_from_device(WEIGHT[kind], be.ROWS_NK if kind == "q8" else be.KMAJOR_KN, n, k, packed)
        self.gpu.sync()
        packed.free()
        self.a = torch.randn((m, k), generator=gen, device="cuda")
        self.c = torch.empty((m, n), device="cuda")
        self.m, self.a_buf, self.c_buf = m, _buffer(self.gpu, self.a), _buffer(self.gpu, self.c)
        torch.cuda.synchronize()

    def run(self):
        self.gpu.step_matmul(self.weight, self.a_buf, self.m, self.c_buf)
        return self.c

    def __del__(self):
        if hasattr(self, "weight"):
            self.weight.free()


class _Attention:
    def __init__(self, case, seed):
        self.gpu, gen = _context("exact"), _generator(seed)
        b, l, t, h, g, d = (case[x] for x in ("batch", "queries", "keys", "heads", "kv_heads", "head"))
        make = lambda kind, *shape: torch.randn(shape, generator=gen, device="cuda").to(TORCH[kind])  # noqa: E731
        self.q, self.k, self.v = make(case["query"], b, l, h, d), make(case["cache"], b, t, g, d), make(case["cache"], b, t, g, d)
        lengths = torch.tensor(_lengths(case), dtype=torch.int32, device="cuda")
        positions = (lengths[:, None] - l + torch.arange(l, dtype=torch.int32, device="cuda")).contiguous()
        self.index = (positions, lengths)
        self.out = torch.empty((b, l, h, d), device="cuda")
        self.operands = [_buffer(self.gpu, x) for x in (self.out, self.q, self.k, self.v)]
        self.options = {"q_dtype": QUERY[case["query"]], "kv_dtype": CACHE[case["cache"]],
                        "window": (case["window"], 0, 0) if case["window"] else be.CAUSAL,
                        "query_positions": _buffer(self.gpu, positions), "kv_lengths": _buffer(self.gpu, lengths)}
        self.shape, self.scale = (b, l, t, h, g, d, d), 1.0 / math.sqrt(d)
        torch.cuda.synchronize()

    def run(self):
        self.gpu.step_attention(*self.operands, self.shape, self.scale, **self.options)
        return self.out


def _config(case):
    return DecoderConfig(layers=case["layers"], hidden=case["hidden"], heads=case["heads"], kv_heads=case["kv_heads"], head_dim=case["head"],
                         ffn=case["ffn"], vocab=case["vocab"], max_seq=-(-(case["prompt"] + case["tokens"]) // 256) * 256, wdtype=WEIGHT[case["weight"]])


class _Weights:
    """Weights with two properties of trained ones, so that a run can be compared: the residual stream carries its embedding (the
    projections back into it are scaled by 1 / sqrt(2 layers), as models are initialised), and the logits have a clear maximum (row
    t of the head is the embedding of token t - 1: the model counts up). With N(0, 0.02) throughout, the int8 re-quantization in
    front of every projection makes two correct implementations drift apart by a tenth of the logits over 26 blocks."""

    def __init__(self, gpu, cfg, kind, seed):
        self.gpu, self.cfg, self.kind, self.gen = gpu, cfg, kind, _generator(seed)
        self.table = torch.randn((cfg.vocab, cfg.hidden), generator=self.gen, device="cuda")

    def blocks(self, name):
        c = self.cfg
        if name == "lm_head":
            n, k = c.vocab, c.hidden
            values = self.table.roll(1, 0).mul_(0.02)
            values = values if self.kind == "q8" else values.t().contiguous()
        else:
            n, k = {"wq": (c.q_dim, c.hidden), "wk": (c.kv_dim, c.hidden), "wv": (c.kv_dim, c.hidden), "wo": (c.hidden, c.q_dim),
                    "wgate": (c.ffn, c.hidden), "wup": (c.ffn, c.hidden), "wdown": (c.hidden, c.ffn)}[name.split(".")[1]]
            std = 0.02 / math.sqrt(2 * c.layers) if name.endswith(("wo", "wdown")) else 0.02
            values = _normal(self.kind, n, k, std, self.gen)
        packed = _blocks(self.gpu, self.kind, n, k, values)
        out = packed.numpy(np.uint8)
        packed.free()
        return out

    def embed(self):
        return self.table.cpu().numpy()


class _Decoder:
    def __init__(self, case, seed):
        self.gpu = _context("exact")
        cfg = _config(case)
        weights = _Weights(self.gpu, cfg, case["weight"], seed)
        self.decoder = (SessionDecoder if case["entry"] == "session" else Decoder)(self.gpu, cfg, weights)
        self.prompt = torch.randint(cfg.vocab, (case["prompt"],), generator=weights.gen, device="cuda", dtype=torch.int32).cpu().numpy()
        self.tokens = case["tokens"]
        self.out = {"logits": _tensor(self.decoder.logits, (cfg.vocab,), "<f4"),
                    "keys": [_tensor(b, (cfg.max_seq, cfg.kv_dim), "<f2") for b in self.decoder.kc],
                    "values": [_tensor(b, (cfg.max_seq, cfg.kv_dim), "<f2") for b in self.decoder.vc]}
        if self.tokens:
            self.first = self.decoder.prefill(self.prompt)
            self.decoder.begin_decode(self.first)            # records the step once, as a server does before it serves
        self.gpu.sync()

    def run(self):
        d = self.decoder
        if self.tokens:
            d.pos = self.prompt.size                         # back behind the prompt: the same continuation again
            d.begin_decode(self.first)
            return dict(self.out, tokens=d.decode_run(self.tokens))
        d.pos = 0
        return dict(self.out, token=d.prefill(self.prompt))

    def __del__(self):
        if hasattr(self, "decoder"):
            self.decoder.close()


def prepare(case, seed):
    return {"matmul": _Matmul, "attention": _Attention, "decoder": _Decoder}[case["family"]](case, seed)


def run(state):
    return state.run()
