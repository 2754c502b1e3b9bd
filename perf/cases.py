"""The work that a program has this framework do, as cases that can be timed and checked.

Three kinds of case:

  * ``translate``: one whole call, encoder prefill plus greedy decoding of a batch, through
    ``Translator.encode_cross`` and ``Translator.greedy_top`` (tokens and their logits).
  * ``linear``: one quantized matrix product through the C ABI: ``mlg_gemv`` for the few rows
    it takes, ``mlg_gemm`` / ``mlg_gemm_resid`` above (encoder projections, FFN, LM-head logits).
  * ``attention`` (``mlg_attn_decode``) and ``topk`` (``mlg_logsoftmax_topk``): the two other
    blocks of a decode step that a program can call by themselves.

Weights are quantized blocks drawn from a pool of random blocks (values about N(0, 0.02), as
the benchmark's random-init models), so that a model file is written and a matrix is laid out
quickly.  A model and a vocabulary-wide matrix are loaded once per process, as a serving
program keeps them; everything else follows from the seed.
"""
from __future__ import annotations

import ctypes
import math
import os
import struct
import tempfile
from pathlib import Path

import numpy as np
import torch

import malaga_amd as M
from malaga_amd import _lib

F32, F16, Q8_0, Q4_K, Q5_K, Q6_K = _lib.F32, _lib.F16, _lib.Q8_0, _lib.Q4_K, _lib.Q5_K, _lib.Q6_K
TYPES = {"q4_K": Q4_K, "q5_K": Q5_K, "q6_K": Q6_K, "q8_0": Q8_0, "f16": F16}
BLOCK = {Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210), Q8_0: (32, 34), F16: (32, 64)}
VOCAB = 256206
TGT_LANG = 256100
POOL = 16384

# widths of the two benchmark models; the 3.3B one with 12 + 12 of its 24 + 24 layers
MODELS = {
    "600m": dict(d=1024, ffn=4096, heads=16, layers=12),
    "3b": dict(d=2048, ffn=8192, heads=16, layers=12),
}
PRESETS = {  # (projections, FFN down and embedding)
    "q4_k_m": (Q4_K, Q6_K),
    "q8_0": (Q8_0, Q8_0),
}


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # one projection of one decoding sentence: the smallest call, launch latency
        dict(name="proj_b1_q4k", kind="linear", type="q4_K", N=1024, K=1024, rows=1, bias=True, relu=False, resid=False),
        # LM-head logits of one sentence decoded with four beams
        dict(name="head_b4_q6k", kind="linear", type="q6_K", N=VOCAB, K=1024, rows=4, bias=False, relu=False, resid=False),
        # LM-head logits of eight sentences decoded with four beams
        dict(name="head_b32_q6k", kind="linear", type="q6_K", N=VOCAB, K=1024, rows=32, bias=False, relu=False, resid=False),
        # the encoder's fused QKV projection over a batch of 32 sentences (packed tokens)
        dict(name="enc_qkv_q4k", kind="linear", type="q4_K", N=3072, K=1024, rows=911, bias=True, relu=False, resid=False),
        # the encoder's second FFN projection with its residual add, the same batch
        dict(name="enc_down_q6k", kind="linear", type="q6_K", N=1024, K=4096, rows=911, bias=True, relu=False, resid=True),
        # the 3.3B model's first FFN projection over a batch of 64 sentences
        dict(name="enc_up_3b_q4k", kind="linear", type="q4_K", N=8192, K=2048, rows=1651, bias=True, relu=True, resid=False),
        # the first FFN projection of an 8-bit model over a handful of sentences
        dict(name="enc_up_q8", kind="linear", type="q8_0", N=4096, K=1024, rows=203, bias=True, relu=True, resid=False),
        # self attention of one decode step, a batch of 32 well into its output
        dict(name="attn_b32", kind="attention", rows=32, heads=16, hd=64, L=128),
        # one beam step's log-softmax and candidates, eight sentences with four beams
        dict(name="topk_b32", kind="topk", rows=32, V=VOCAB, k=4),
        # one sentence, the reference's own benchmark shape (21 ids in, 18 tokens out)
        dict(name="one_600m", kind="translate", model="600m", preset="q4_k_m", batch=1, mean=21, spread=0.0, new=18),
        # a batch of 32 sentences of ordinary lengths
        dict(name="batch32_600m", kind="translate", model="600m", preset="q4_k_m", batch=32, mean=28, spread=0.5, new=32),
        # a large serving batch of the large model
        dict(name="batch64_3b", kind="translate", model="3b", preset="q4_k_m", batch=64, mean=28, spread=0.5, new=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.random()
    if what < 0.55:  # a projection of one of the models, over decode rows or packed tokens
        d = rng.choice([1024, 2048])
        n, k, act, res = rng.choice([(3 * d, d, False, False), (d, d, False, True), (4 * d, d, True, False),
                                     (d, 4 * d, False, True), (2 * d, d, False, False)])
        t = rng.choice(["q4_K", "q4_K", "q6_K", "q5_K", "q8_0", "f16"])
        rows = rng.choice([rng.randint(1, 4), _log(rng, 5, 64), _log(rng, 65, 1651), _log(rng, 65, 1651)])
        if rng.random() < 0.15:  # a vocabulary shortlist's head
            return dict(kind="linear", type=rng.choice(["q6_K", "q8_0"]), N=rng.randint(20000, 40000), K=1024,
                        rows=_log(rng, 1, 64), bias=False, relu=False, resid=False)
        return dict(kind="linear", type=t, N=n, K=k, rows=rows, bias=True, relu=act, resid=res and rows > 4)
    if what < 0.65:
        return dict(kind="attention", rows=_log(rng, 1, 64), heads=16, hd=rng.choice([64, 128]), L=_log(rng, 8, 200))
    if what < 0.75:
        return dict(kind="topk", rows=_log(rng, 2, 64), V=rng.choice([VOCAB, VOCAB, rng.randint(20000, 40000)]),
                    k=rng.randint(2, 5))
    return dict(kind="translate", model="600m", preset="q4_k_m", batch=_log(rng, 1, 32), mean=_log(rng, 8, 60),
                spread=rng.choice([0.0, 0.3, 0.5]), new=_log(rng, 6, 32))


# ------------------------------------------------------- random quantized blocks

_POOLS: dict = {}


def _pool(t):
    """POOL random blocks of a type: raw bytes [POOL, block bytes] and their f64 values."""
    if t in _POOLS:
        return _POOLS[t]
    r = np.random.default_rng(1000 + t)
    n, nb = BLOCK[t]
    p = 2 * POOL
    raw = np.zeros((p, nb), np.uint8)

    def f16(v):
        return v.astype(np.float16)

    if t == F16:
        w = f16(r.normal(0, 0.02, (p, n)))
        raw[:] = w.view(np.uint8).reshape(p, nb)
        val = w.astype(np.float64)
    elif t == Q8_0:
        d = f16(r.uniform(0.8, 1.2, p) * 0.02 / 40)
        q = np.clip(np.rint(r.normal(0, 40, (p, n))), -127, 127).astype(np.int8)
        raw[:, :2] = d.view(np.uint8).reshape(p, 2)
        raw[:, 2:] = q.view(np.uint8)
        val = d.astype(np.float64)[:, None] * q
    elif t == Q6_K:
        d = f16(r.uniform(0.8, 1.2, p) * 0.02 / (10 * 96))
        sc = (r.integers(64, 128, (p, 16)) * r.choice([-1, 1], (p, 16))).astype(np.int8)
        q = np.clip(np.rint(r.normal(0, 10, (p, 256))), -32, 31).astype(np.int64)
        u = (q + 32).astype(np.uint8).reshape(p, 2, 4, 32)  # [half][quarter t][l]
        ql = np.zeros((p, 2, 64), np.uint8)
        ql[:, :, :32] = (u[:, :, 0] & 15) | ((u[:, :, 2] & 15) << 4)
        ql[:, :, 32:] = (u[:, :, 1] & 15) | ((u[:, :, 3] & 15) << 4)
        qh = (u[:, :, 0] >> 4) | ((u[:, :, 1] >> 4) << 2) | ((u[:, :, 2] >> 4) << 4) | ((u[:, :, 3] >> 4) << 6)
        raw[:, :128], raw[:, 128:192] = ql.reshape(p, 128), qh.reshape(p, 64)
        raw[:, 192:208], raw[:, 208:] = sc.view(np.uint8), d.view(np.uint8).reshape(p, 2)
        val = d.astype(np.float64)[:, None] * (np.repeat(sc.astype(np.int64), 16, axis=1) * q)
    else:  # q4_K / q5_K: 8 sub-blocks of 32, 6-bit scales and mins
        top, mid, sd = (15, 7.5, 2.8) if t == Q4_K else (31, 15.5, 5.6)
        d = f16(r.uniform(0.8, 1.2, p) * 0.02 / (sd * 48))
        dmin = f16(d.astype(np.float64) * mid)
        sc = r.integers(33, 64, (p, 8)).astype(np.uint8)
        mn = np.clip(sc.astype(np.int64) + r.integers(-2, 3, (p, 8)), 0, 63).astype(np.uint8)
        q = np.clip(np.rint(r.normal(mid, sd, (p, 8, 32))), 0, top).astype(np.uint8)
        packed = np.zeros((p, 12), np.uint8)
        packed[:, 0:4] = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
        packed[:, 4:8] = (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6)
        packed[:, 8:12] = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
        raw[:, :2], raw[:, 2:4], raw[:, 4:16] = d.view(np.uint8).reshape(p, 2), dmin.view(np.uint8).reshape(p, 2), packed
        qs = (q[:, 0::2] & 15) | ((q[:, 1::2] & 15) << 4)  # [pair of sub-blocks][32]
        raw[:, nb - 128:] = qs.reshape(p, 128)
        if t == Q5_K:
            raw[:, 16:48] = sum(((q[:, s] >> 4) << s).astype(np.uint8) for s in range(8))
        val = (d.astype(np.float64)[:, None, None] * sc[:, :, None].astype(np.float64) * q
               - dmin.astype(np.float64)[:, None, None] * mn[:, :, None].astype(np.float64)).reshape(p, 256)
    _POOLS[t] = raw[:POOL], torch.from_numpy(np.ascontiguousarray(val[:POOL]))
    return _POOLS[t]


def _blocks(t, N, K, key):
    """Which pool block every block of an [N, K] matrix is."""
    return np.random.default_rng(key).integers(0, POOL, (N, K // BLOCK[t][0]), dtype=np.int32)


def _rows_bytes(t, idx):
    return np.ascontiguousarray(_pool(t)[0][idx.reshape(-1)])


def _rows_exact(t, idx, device):
    val = _pool(t)[1].to(device)
    return val[torch.from_numpy(idx.reshape(-1).astype(np.int64)).to(device)].reshape(idx.shape[0], -1)


# ------------------------------------------------------------------- model files

def _key(*parts):
    h = 2166136261
    for ch in "/".join(map(str, parts)).encode():
        h = ((h ^ ch) * 16777619) & 0xFFFFFFFF
    return h


def _tensors(model, preset):
    """name -> (shape [N, K] or [n], type, kind) in file order."""
    c, (lin, down) = MODELS[model], PRESETS[preset]
    d, f = c["d"], c["ffn"]
    out = {"token_embd.weight": ((VOCAB, d), down)}
    for side in ("enc", "dec"):
        for i in range(c["layers"]):
            p = "%s.blk.%d." % (side, i)
            mats = [("attn_qkv", 3 * d, d, lin), ("attn_out", d, d, lin), ("ffn_up", f, d, lin), ("ffn_down", d, f, down)]
            norms = ["attn_norm", "ffn_norm"]
            if side == "dec":
                mats += [("cross_attn_q", d, d, lin), ("cross_attn_kv", 2 * d, d, lin), ("cross_attn_out", d, d, lin)]
                norms += ["cross_attn_norm"]
            for n, rows, cols, t in mats:
                out[p + n + ".weight"] = ((rows, cols), t)
                out[p + n + ".bias"] = ((rows,), F32)
            for n in norms:
                out[p + n + ".weight"] = ((d,), F32)
                out[p + n + ".bias"] = ((d,), F32)
        out[side + ".output_norm.weight"] = ((d,), F32)
        out[side + ".output_norm.bias"] = ((d,), F32)
    return out


def _vector(model, name, n):
    r = np.random.default_rng(_key(model, name))
    norm_gain = name.endswith("norm.weight")
    return (r.normal(1.0, 0.1, n) if norm_gain else r.normal(0.0, 0.05, n)).astype(np.float32)


def _model_file(model, preset):
    d = Path(tempfile.gettempdir()) / "malaga_perf_models"
    d.mkdir(parents=True, exist_ok=True)
    path = d / ("%s-%s.gguf" % (model, preset))
    if path.exists():
        return path
    c = MODELS[model]
    meta = [("general.architecture", "nllb"), ("general.name", "random blocks"), ("general.alignment", 32),
            ("tokenizer.huggingface.json", "{}"), ("nllb.vocab_size", VOCAB), ("nllb.embedding_length", c["d"]),
            ("nllb.encoder.block_count", c["layers"]), ("nllb.decoder.block_count", c["layers"]),
            ("nllb.encoder.attention.head_count", c["heads"]), ("nllb.decoder.attention.head_count", c["heads"]),
            ("nllb.encoder.feed_forward_length", c["ffn"]), ("nllb.decoder.feed_forward_length", c["ffn"]),
            ("nllb.context_length", 1024), ("nllb.scale_embedding", True), ("nllb.max_length", 200),
            ("tokenizer.ggml.bos_token_id", 0), ("tokenizer.ggml.padding_token_id", 1),
            ("tokenizer.ggml.eos_token_id", 2), ("tokenizer.ggml.decoder_start_token_id", 2)]
    ts = _tensors(model, preset)

    def text(s):
        return struct.pack("<Q", len(s.encode())) + s.encode()

    head = struct.pack("<IIQQ", 0x46554747, 3, len(ts), len(meta))
    for k, v in meta:
        head += text(k)
        if isinstance(v, bool):
            head += struct.pack("<I?", 7, v)
        elif isinstance(v, int):
            head += struct.pack("<II", 4, v)
        else:
            head += struct.pack("<I", 8) + text(v)
    off = 0
    for name, (shape, t) in ts.items():
        head += text(name) + struct.pack("<I", len(shape)) + b"".join(struct.pack("<Q", n) for n in reversed(shape))
        head += struct.pack("<IQ", t, off)
        n = int(np.prod(shape))
        size = 4 * n if t == F32 else n // BLOCK[t][0] * BLOCK[t][1]
        off += (size + 31) // 32 * 32
    tmp = path.with_suffix(".%d.tmp" % os.getpid())
    with open(tmp, "wb") as f:
        f.write(head + b"\0" * (-len(head) % 32))
        for name, (shape, t) in ts.items():
            b = (_vector(model, name, shape[0]) if t == F32 else _rows_bytes(t, _blocks(t, *shape, _key(model, name)))).tobytes()
            f.write(b + b"\0" * (-len(b) % 32))
    os.replace(tmp, path)
    return path


_LOADED: dict = {}


def _translator(model, preset):
    if (model, preset) not in _LOADED:
        _LOADED[model, preset] = M.Translator.load(_model_file(model, preset))
    return _LOADED[model, preset]


# --------------------------------------------------------------------- matrices

class _Matrix:
    def __init__(self, t, N, K, key):
        lib = _lib.load()
        if "ctx" not in _LOADED:
            h = ctypes.c_void_p()
            _lib.check(lib.mlg_ctx_create(0, ctypes.byref(h)))
            _LOADED["ctx"] = h
        raw = _rows_bytes(t, _blocks(t, N, K, key))
        self.lib, self.h = lib, ctypes.c_void_p()
        _lib.check(lib.mlg_matrix_upload(_LOADED["ctx"], t, N, K, raw.ctypes.data, ctypes.byref(self.h)))

    def __del__(self):
        if self.h:
            self.lib.mlg_matrix_free(self.h)
            self.h = None


def _matrix_key(case, seed):
    # a vocabulary-wide matrix is one model's head, kept; smaller ones follow the seed
    return _key(case["type"], case["N"], case["K"], 0 if case["N"] * case["K"] > 1 << 26 else seed)


def _matrix(case, seed):
    t, key = TYPES[case["type"]], _matrix_key(case, seed)
    if case["N"] * case["K"] <= 1 << 26:
        return _Matrix(t, case["N"], case["K"], key)
    if key not in _LOADED:
        _LOADED[key] = _Matrix(t, case["N"], case["K"], key)
    return _LOADED[key]


# ------------------------------------------------------------------ inputs, a pass

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _normal(shape, seed, std=1.0):
    return torch.randn(shape, generator=_gen(seed), device="cuda", dtype=torch.float32) * std


def _linear_inputs(case, seed):
    x = _normal((case["rows"], case["K"]), seed)
    if case["K"] > case["N"]:  # the FFN's activations
        x = x.clamp_(min=0)
    s = dict(x=x, bias=_normal((case["N"],), seed + 1, 0.05) if case["bias"] else None,
             r=_normal((case["rows"], case["N"]), seed + 2) if case["resid"] else None)
    return s


def _attention_inputs(case, seed):
    b, H, hd, L = case["rows"], case["heads"], case["hd"], case["L"]
    r = np.random.default_rng(seed)
    lens = torch.from_numpy(r.integers(max(1, L // 2), L + 1, b).astype(np.int32)).cuda()
    return dict(q=_normal((b, H * hd), seed, hd ** -0.5), k=_normal((b, H, L, hd), seed + 1).half(),
                v=_normal((b, H, L, hd), seed + 2).half(), lens=lens)


def _topk_inputs(case, seed):
    return dict(x=_normal((case["rows"], case["V"]), seed, 3.0))


def _sources(case, seed):
    r = np.random.default_rng(seed)
    mu = math.log(case["mean"]) - case["spread"] ** 2 / 2
    lens = np.clip(np.rint(r.lognormal(mu, case["spread"], case["batch"])) if case["spread"] else
                   np.full(case["batch"], case["mean"]), 3, 128).astype(int)
    return [r.integers(4, VOCAB - 206, n).tolist() for n in sorted(lens.tolist(), reverse=True)]


def prepare(case, seed):
    if case["kind"] == "translate":
        return dict(kind="translate", t=_translator(case["model"], case["preset"]), src=_sources(case, seed), new=case["new"])
    if case["kind"] == "linear":
        s = _linear_inputs(case, seed)
        w = _matrix(case, seed)
        few = not case["resid"] and case["rows"] <= _lib.load().mlg_gemv_max_batch(w.h)
        return dict(s, kind="linear", w=w, rows=case["rows"], relu=int(case["relu"]), few=few,
                    y=torch.empty((case["rows"], case["N"]), device="cuda"))
    if case["kind"] == "attention":
        s = _attention_inputs(case, seed)
        return dict(s, kind="attention", dims=(case["rows"], case["heads"], case["hd"], case["L"]), out=torch.empty_like(s["q"]))
    s = _topk_inputs(case, seed)
    rows, k = case["rows"], case["k"]
    work = _lib.load().mlg_logsoftmax_topk_scratch(rows, k)
    return dict(s, kind="topk", dims=(rows, case["V"], k), work=torch.empty(work, dtype=torch.uint8, device="cuda"),
                vals=torch.empty((rows, k), device="cuda"), idx=torch.empty((rows, k), dtype=torch.int32, device="cuda"))


def run(state):
    lib = _lib.load()
    kind = state["kind"]
    if kind == "translate":
        t = state["t"]
        batch = t.encode_cross(state["src"])
        toks, logits = t.greedy_top(batch, TGT_LANG, state["new"], eos_mask=True)
        batch.close()
        return dict(tokens=np.array(toks, np.int64), logits=np.array(logits, np.float32))
    st = torch.cuda.current_stream().cuda_stream
    if kind == "linear":
        bias = state["bias"].data_ptr() if state["bias"] is not None else None
        w, x, y = state["w"].h, state["x"].data_ptr(), state["y"].data_ptr()
        if state["r"] is not None:
            _lib.check(lib.mlg_gemm_resid(w, x, state["rows"], y, bias, state["relu"], state["r"].data_ptr(), st))
        elif state["few"]:
            _lib.check(lib.mlg_gemv(w, x, state["rows"], y, bias, state["relu"], st))
        else:
            _lib.check(lib.mlg_gemm(w, x, state["rows"], y, bias, state["relu"], st))
        return state["y"]
    if kind == "attention":
        b, H, hd, L = state["dims"]
        _lib.check(lib.mlg_attn_decode(state["q"].data_ptr(), state["k"].data_ptr(), state["v"].data_ptr(), b, H, hd, L,
                                       state["lens"].data_ptr(), None, state["out"].data_ptr(), st))
        return state["out"]
    rows, V, k = state["dims"]
    _lib.check(lib.mlg_logsoftmax_topk(state["x"].data_ptr(), rows, V, k, -1, state["work"].data_ptr(),
                                       state["vals"].data_ptr(), state["idx"].data_ptr(), st))
    return dict(vals=state["vals"], idx=state["idx"])


# ------------------------------------------------------------------- work, limits

def _weight_bytes(t, n):
    return n // BLOCK[t][0] * BLOCK[t][1]


def work(case):
    if case["kind"] == "linear":
        n, k, m = case["N"], case["K"], case["rows"]
        return dict(bytes=_weight_bytes(TYPES[case["type"]], n * k) + 4 * (m * k + m * n * (2 if case["resid"] else 1)),
                    flops=2.0 * m * n * k)
    if case["kind"] == "attention":
        kv = case["rows"] * case["heads"] * case["hd"] * case["L"] * 0.75  # keys a row has, on average
        return dict(bytes=4 * kv + 8 * case["rows"] * case["heads"] * case["hd"], flops=4 * kv)
    if case["kind"] == "topk":
        return dict(bytes=4.0 * case["rows"] * case["V"], flops=3.0 * case["rows"] * case["V"])
    c, (lin, down) = MODELS[case["model"]], PRESETS[case["preset"]]
    d, f, L = c["d"], c["ffn"], c["layers"]
    tokens, steps = case["batch"] * case["mean"], case["new"] + 1
    enc_l, dec_l, kv_l = 4 * d * d + f * d, 6 * d * d + f * d, 2 * d * d
    enc = L * (_weight_bytes(lin, enc_l + kv_l) + _weight_bytes(down, f * d))
    dec = L * (_weight_bytes(lin, dec_l) + _weight_bytes(down, f * d)) + _weight_bytes(down, VOCAB * d)
    kv = case["batch"] * L * 2 * d * 2 * (case["mean"] + steps / 2)
    return dict(bytes=float(enc + steps * (dec + kv)),
                flops=2.0 * (tokens * L * (enc_l + kv_l + f * d)
                             + steps * case["batch"] * (L * (dec_l + f * d) + VOCAB * d)))


def tolerance(case):
    # about four times the distance to exact() measured over these ranges: 1e-7 to 5e-7 (largest
    # value 3e-6) for the single blocks, whose sums are 32-bit; 2e-5 to 8.5e-5 (largest 2.6e-4)
    # for the logits of a whole call, which keeps its K/V in 16 bits
    if case["kind"] == "translate":
        return dict(rel=3e-4, max=1e-3, differ=0.0)
    if case["kind"] == "topk":
        return dict(rel=1e-6, max=1e-5, differ=0.0)
    return dict(rel=2e-6, max=1e-5)


# ----------------------------------------------------------------- in 64 bits

def exact(case, seed):
    if case["kind"] == "linear":
        s = _linear_inputs(case, seed)
        t = TYPES[case["type"]]
        w = _rows_exact(t, _blocks(t, case["N"], case["K"], _matrix_key(case, seed)), "cuda")
        y = s["x"].double() @ w.T.contiguous()
        if s["bias"] is not None:
            y += s["bias"].double()
        if s["r"] is not None:
            y += s["r"].double()
        return y.clamp(min=0) if case["relu"] else y
    if case["kind"] == "attention":
        s = _attention_inputs(case, seed)
        b, H, hd, L = case["rows"], case["heads"], case["hd"], case["L"]
        p = (s["k"].double() * s["q"].double().reshape(b, H, 1, hd)).sum(-1)
        gone = torch.arange(L, device="cuda")[None, :] >= s["lens"].long()[:, None]
        p = torch.softmax(p.masked_fill(gone[:, None, :], -math.inf), -1)
        return (p[..., None] * s["v"].double()).sum(2).reshape(b, H * hd)
    if case["kind"] == "topk":
        x = _topk_inputs(case, seed)["x"].double()
        v, i = torch.topk(torch.log_softmax(x, -1), case["k"], dim=-1)
        return dict(vals=v, idx=i)
    return _exact_translate(case, seed)


def _exact_translate(case, seed):
    name, c = case["model"], MODELS[case["model"]]
    d, H, L = c["d"], c["heads"], c["layers"]
    hd = d // H
    ts = _tensors(name, case["preset"])

    def load(n):
        shape, t = ts[n]
        if t == F32:
            return torch.from_numpy(_vector(name, n, shape[0])).cuda().double()
        return _rows_exact(t, _blocks(t, *shape, _key(name, n)), "cuda")

    def linear(x, n):
        return x @ load(n + ".weight").T.contiguous() + load(n + ".bias")

    def norm(x, n):
        return torch.nn.functional.layer_norm(x, (d,), load(n + ".weight"), load(n + ".bias"), 1e-5)

    def heads(x):
        return x.reshape(x.shape[0], x.shape[1], H, hd).transpose(1, 2).contiguous()

    def attend(q, k, v, gone):  # [b, H, t, hd]; gone: broadcast to [b, H, t, keys]
        s = q @ k.transpose(2, 3).contiguous()
        a = torch.softmax(s.masked_fill(gone, -math.inf), -1) @ v
        return a.transpose(1, 2).reshape(a.shape[0], a.shape[2], d)

    half = d // 2
    freq = np.exp(-np.arange(half) * (math.log(10000.0) / (half - 1)))
    ang = np.arange(1026)[:, None] * freq[None, :]
    pos = torch.from_numpy(np.concatenate([np.sin(ang), np.cos(ang)], 1)).cuda()
    emb = load("token_embd.weight")

    src = _sources(case, seed)
    b, s = len(src), max(map(len, src))
    ids = torch.full((b, s), 1, dtype=torch.long)
    for i, row in enumerate(src):
        ids[i, :len(row)] = torch.tensor(row)
    ids = ids.cuda()
    lens = torch.tensor([len(r) for r in src], device="cuda")
    gone = (torch.arange(s, device="cuda")[None, :] >= lens[:, None])[:, None, None, :]
    x = emb[ids] * math.sqrt(d) + pos[2:2 + s]
    for i in range(L):
        p = "enc.blk.%d." % i
        q, k, v = linear(norm(x, p + "attn_norm"), p + "attn_qkv").split(d, -1)
        x = x + linear(attend(heads(q), heads(k), heads(v), gone), p + "attn_out")
        x = x + linear(linear(norm(x, p + "ffn_norm"), p + "ffn_up").clamp(min=0), p + "ffn_down")
    x = norm(x, "enc.output_norm")
    cross = [[heads(y) for y in linear(x, "dec.blk.%d.cross_attn_kv" % i).split(d, -1)] for i in range(L)]
    kept = [[None, None] for _ in range(L)]
    dec = {n: load(n) for n in ts if n.startswith("dec.") and "cross_attn_kv" not in n}

    def load(n):  # noqa: F811 - the decoder's weights, laid out once for all steps
        return dec[n]

    nothing = torch.zeros((1, 1, 1, 1), dtype=torch.bool, device="cuda")
    feed, toks, tops = [2, TGT_LANG], [], []
    tok = None
    head = emb.T.contiguous()
    for step in range(case["new"] + 1):
        tok = torch.full((b,), feed[step], device="cuda") if step < 2 else tok
        x = (emb[tok] * math.sqrt(d) + pos[step + 2])[:, None, :]
        for i in range(L):
            p = "dec.blk.%d." % i
            q, k, v = linear(norm(x, p + "attn_norm"), p + "attn_qkv").split(d, -1)
            kept[i] = [heads(y) if o is None else torch.cat([o, heads(y)], 2) for o, y in zip(kept[i], (k, v))]
            x = x + linear(attend(heads(q), *kept[i], nothing), p + "attn_out")
            q = linear(norm(x, p + "cross_attn_norm"), p + "cross_attn_q")
            x = x + linear(attend(heads(q), *cross[i], gone), p + "cross_attn_out")
            x = x + linear(linear(norm(x, p + "ffn_norm"), p + "ffn_up").clamp(min=0), p + "ffn_down")
        if step == 0:
            continue
        z = norm(x[:, 0], "dec.output_norm") @ head
        z[:, 2] = -math.inf  # EOS is never chosen in these cases: every row has the same length
        top, tok = z.max(-1)
        toks.append(tok)
        tops.append(top)
    return dict(tokens=torch.stack(toks, 1), logits=torch.stack(tops, 1))
