"""Performance cases of the packed-weight framework: what its users call, over the sizes they call it with.

A case is a dict of plain values with a ``kind``:

* ``linear``: one ``GSQLinear`` on ``m`` activation rows: a decode projection (1 row), a few
  sequences or drafted tokens (2-16 rows), a prompt (17-2048 rows).
* ``embedding``: ``GSQEmbedding`` on ``m`` token ids.
* ``gdn`` / ``attn``: one mixer of the Qwen3.5-hybrid decoder (GatedDeltaNet / gated attention, with
  its packed projections) over a prompt of ``m`` tokens per sequence, from an empty cache.
* ``prefill`` / ``decode``: four layers of that decoder at the 27B widths (three GatedDeltaNet, one
  attention; a 16384-row vocabulary keeps the head's share of the work), over a prompt of ``m``
  tokens, or ``m`` graph-captured single-token steps from an empty cache.

Weights are random superblocks whose scales give them a standard deviation of about 1/sqrt(K), the
codebooks are seeded tables of the published shapes and value sets, and ``exact`` restates the
arithmetic in float64 torch.
"""
from __future__ import annotations

import math
import os
import sys
from functools import lru_cache

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "mlx-gsq-rco_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

from mlx_gsq_amd import tables  # noqa: E402
from mlx_gsq_amd.models import GraphDecoder, Qwen35Args, build_qwen35  # noqa: E402
from mlx_gsq_amd.models.qwen35 import FullAttention, GatedDeltaNet, Qwen35Cache  # noqa: E402
from mlx_gsq_amd.nn import GSQEmbedding, GSQFusedLinear, GSQLinear  # noqa: E402
from mlx_gsq_amd.runtime.store import PackedWeight  # noqa: E402

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
SIZES = {"fp16": 2, "bf16": 2, "fp32": 4}
TYPE_IDS = {"Q2_K": 10, "Q4_K": 12, "Q6_K": 14, "IQ2_XXS": 16, "IQ2_XS": 17, "IQ3_XXS": 18, "IQ1_S": 19,
            "IQ3_S": 21, "IQ2_S": 22, "IQ4_XS": 23, "IQ1_M": 29}
BLOCK_BYTES = {"IQ1_M": 56, "IQ1_S": 50, "IQ2_XXS": 66, "IQ2_XS": 74, "IQ2_S": 82, "IQ3_XXS": 98, "IQ3_S": 110,
               "IQ4_XS": 136, "Q2_K": 84, "Q4_K": 144, "Q6_K": 210}

LAYERS, VOCAB = 4, 16384
ARGS = Qwen35Args(num_hidden_layers=LAYERS, vocab_size=VOCAB)
# type of each projection: the mixed 27B checkpoint of the repository's benchmark
MODEL_TYPES = {"attn_qkv": "IQ2_XS", "attn_gate": "IQ2_XS", "ssm_out": "IQ3_S", "attn_q": "IQ2_XS",
               "attn_k": "IQ2_XS", "attn_v": "IQ4_XS", "attn_output": "IQ3_S", "ffn_gate": "IQ2_S",
               "ffn_up": "IQ2_S", "ffn_down": "Q4_K", "output": "Q6_K", "token_embd": "IQ2_S"}


# ---- the cases ---------------------------------------------------------------------------

def _linear(name, qtype, n, k, m, dtype="fp16"):
    case = {"kind": "linear", "qtype": qtype, "n": n, "k": k, "m": m, "dtype": dtype}
    return dict(case, name=name) if name else case


def listed():
    return [
        # single-token decode: the smallest projection (launch latency) and a large one
        _linear("k_proj_1row", "IQ2_XS", 1024, 5120, 1),
        _linear("down_1row", "Q4_K", 5120, 17408, 1),
        # a few drafted tokens verified together; a batch of sequences decoded together
        _linear("gate_4rows", "IQ2_S", 17408, 5120, 4),
        _linear("o_proj_16rows", "IQ3_S", 5120, 5120, 16),
        # prompts: short and ragged, medium in bfloat16 (a bf16 checkpoint), long
        _linear("up_182rows", "IQ2_S", 17408, 5120, 182),
        _linear("down_512rows_bf16", "Q4_K", 5120, 17408, 512, "bf16"),
        _linear("gate_2048rows", "IQ3_S", 17408, 5120, 2048),
        # the token embedding of a long prompt, bf16 rows as GSQEmbedding returns by default
        {"name": "embedding_4096ids", "kind": "embedding", "n": 248320, "k": 5120, "m": 4096, "dtype": "bf16"},
        # the two mixers of the hybrid decoder over a prompt
        {"name": "gdn_prompt_512", "kind": "gdn", "b": 1, "m": 512},
        {"name": "attn_prompt_1024", "kind": "attn", "b": 1, "m": 1024, "max_len": 4096},
        # whole calls: a prompt through the decoder, and token-by-token decoding
        {"name": "model_prompt_182", "kind": "prefill", "b": 1, "m": 182, "max_len": 1024},
        {"name": "model_decode_16steps", "kind": "decode", "b": 1, "m": 16, "max_len": 1024},
    ]


MAX_WORK = 2048 * 17408 * 5120      # largest listed product, multiply-adds
MAX_WORK_WIDE = 512 * 5120 * 17408  # and of the 16-bit-staged (bf16 / fp32) ones


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["linear", "embedding", "gdn", "attn", "prefill", "decode"], [14, 2, 2, 2, 1, 1])[0]
    if kind == "linear":
        qtype = rng.choice(sorted(BLOCK_BYTES))
        dtype = rng.choices(["fp16", "bf16", "fp32"], [7, 3, 1])[0]
        limit = MAX_WORK if dtype == "fp16" else MAX_WORK_WIDE
        while True:
            if rng.random() < 0.5:
                n, k = rng.choice([(1024, 5120), (5120, 5120), (17408, 5120), (5120, 17408)])
            else:  # any width of whole superblocks, any row count
                n, k = _log(rng, 257, 20000), 256 * _log(rng, 2, 68)
            m = _log(rng, 1, 2048)
            if m * n * k <= limit:
                return _linear(None, qtype, n, k, m, dtype)
    if kind == "embedding":
        return {"kind": kind, "n": rng.choice([32768, 100003, 248320]), "k": 256 * rng.choice([4, 9, 20, 21]),
                "m": _log(rng, 1, 4096), "dtype": rng.choice(["bf16", "fp16", "fp32"])}
    if kind == "gdn":
        return {"kind": kind, "b": rng.choice([1, 1, 2]), "m": _log(rng, 2, 768)}
    if kind == "attn":
        m = _log(rng, 2, 1024)
        return {"kind": kind, "b": rng.choice([1, 1, 2]) if m <= 512 else 1, "m": m,
                "max_len": rng.choice([1024, 2048, 4096])}
    if kind == "prefill":
        return {"kind": kind, "b": 1, "m": _log(rng, 9, 400), "max_len": 1024}
    return {"kind": kind, "b": rng.choice([1, 1, 2, 4, 8]), "m": rng.randint(3, 16), "max_len": 1024}


# ---- inputs ------------------------------------------------------------------------------

def _device():
    return torch.device("cuda", torch.cuda.current_device())


@lru_cache(None)
def _codebooks():
    """Codebooks of the published shapes and value sets: unique entries, sorted by code."""
    shapes = {"IQ1_S": (2048, 8, (-1, 0, 1)), "IQ2_XXS": (256, 8, (8, 25, 43)), "IQ2_XS": (512, 8, (8, 25, 43)),
              "IQ2_S": (1024, 8, (8, 25, 43, 62)), "IQ3_XXS": (256, 4, (4, 12, 20, 28, 36, 44, 52, 62)),
              "IQ3_S": (512, 4, (1, 3, 5, 7, 9, 11, 13, 15))}
    rng = np.random.default_rng(2024)
    books = {}
    for q, (n, c, vals) in shapes.items():
        code = np.sort(rng.choice(len(vals) ** c, size=n, replace=False))
        books[q] = np.array(vals, np.float32)[code[:, None] // len(vals) ** np.arange(c) % len(vals)]
    books["IQ1_M"] = books["IQ1_S"]
    tables.set_tables(books)
    return books


def _set_scale(raw, qtype, d):
    """Writes the fp16 scale d (blocks,) into its field; a K-quant's minimum scale balances it."""
    h = d.to(torch.float16)

    def put(off, v):
        raw[:, off:off + 2] = v.contiguous().view(torch.uint8).reshape(-1, 2)

    if qtype == "IQ1_M":  # the fp16 bits, a nibble on top of each of the four scale words
        bits = h.view(torch.int16).to(torch.int32) & 0xFFFF
        for i in range(4):
            raw[:, 49 + 2 * i] = ((raw[:, 49 + 2 * i].to(torch.int32) & 15) | (bits >> (4 * i) & 15) << 4).to(torch.uint8)
    elif qtype in ("Q2_K", "Q4_K"):
        off, ratio = (80, 1.5) if qtype == "Q2_K" else (0, 7.5)
        put(off, h)
        put(off + 2, (d * ratio).to(torch.float16))
    else:
        put(208 if qtype == "Q6_K" else 0, h)


def _blocks(qtype, count, gen, device, scale):
    raw = torch.randint(0, 256, (count, BLOCK_BYTES[qtype]), dtype=torch.uint8, device=device, generator=gen)
    _set_scale(raw, qtype, (0.5 + torch.rand(count, device=device, generator=gen)) * scale)
    return raw


@lru_cache(None)
def _rms(qtype):
    """Root mean square of a random matrix's weights at scale 1."""
    gen = torch.Generator("cpu").manual_seed(7)
    return float(_decode(qtype, _blocks(qtype, 2048, gen, "cpu", 1.0)).square().mean().sqrt())


def _weight(name, qtype, n, k, gen, std=None):
    """A random packed matrix with weights of the given standard deviation (default 1/sqrt(k))."""
    _codebooks()
    scale = (std or k ** -0.5) / _rms(qtype)
    data = _blocks(qtype, n * (k // 256), gen, gen.device, scale).reshape(-1)
    return PackedWeight(name=name, data=data, gguf_shape=(k, n), logical_shape=(n, k), quantization_type=qtype,
                        quantization_type_id=TYPE_IDS[qtype], num_elements=n * k, num_bytes=data.numel())


class Store:
    """The weights of a case's layers under their checkpoint names, as ``build_qwen35`` reads them."""

    def __init__(self, gen, kinds):
        self.packed, self.plain, self.gen = {}, {}, gen
        a, H = ARGS, ARGS.hidden_size
        hv, dv = a.linear_num_value_heads, a.linear_value_head_dim
        if "model" in kinds:
            self._add("token_embd", VOCAB, H, std=1.0)
            self._add("output", VOCAB, H)
            self._norm("output_norm.weight", H)
        for i in range(LAYERS):
            p = f"blk.{i}."
            if "model" in kinds:
                self._norm(p + "attn_norm.weight", H)
                self._norm(p + "post_attention_norm.weight", H)
                self._add("ffn_gate", a.intermediate_size, H, p)
                self._add("ffn_up", a.intermediate_size, H, p)
                self._add("ffn_down", H, a.intermediate_size, p)
            if a.is_linear(i) and ("model" in kinds or "gdn" in kinds and i == 0):
                self._add("attn_qkv", a.conv_dim, H, p)
                self._add("attn_gate", a.value_dim, H, p)
                self._add("ssm_out", H, a.value_dim, p)
                self.plain[p + "ssm_alpha.weight"] = self._randn(hv, H) * H ** -0.5
                self.plain[p + "ssm_beta.weight"] = self._randn(hv, H) * H ** -0.5
                self.plain[p + "ssm_conv1d.weight"] = 0.5 * self._randn(a.conv_dim, a.linear_conv_kernel_dim)
                # A in [1, 16] and softplus(dt_bias) in [0.001, 0.1]: the architecture's initial range
                self.plain[p + "ssm_a"] = -torch.exp(self._rand(hv) * math.log(16.0))
                dt = torch.exp(self._rand(hv) * math.log(100.0) + math.log(0.001))
                self.plain[p + "ssm_dt.bias"] = torch.log(torch.expm1(dt))
                self._norm(p + "ssm_norm.weight", dv)
            if not a.is_linear(i) and ("model" in kinds or "attn" in kinds):
                self._add("attn_q", a.num_attention_heads * a.head_dim * 2, H, p)
                self._add("attn_k", a.num_key_value_heads * a.head_dim, H, p)
                self._add("attn_v", a.num_key_value_heads * a.head_dim, H, p)
                self._add("attn_output", H, a.num_attention_heads * a.head_dim, p)
                self._norm(p + "attn_q_norm.weight", a.head_dim)
                self._norm(p + "attn_k_norm.weight", a.head_dim)

    def _randn(self, *shape):
        return torch.randn(*shape, device=self.gen.device, generator=self.gen)

    def _rand(self, *shape):
        return torch.rand(*shape, device=self.gen.device, generator=self.gen)

    def _norm(self, name, n):
        self.plain[name] = 1.0 + 0.1 * self._randn(n)

    def _add(self, kind, n, k, prefix="", std=None):
        name = f"{prefix}{kind}.weight"
        self.packed[name] = _weight(name, MODEL_TYPES[kind], n, k, self.gen, std)

    def weight(self, name):
        return self.packed[name]

    def materialize_plain(self, name):
        return self.plain[name]


def _gen(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed))


def _inputs(case, seed):
    """(the weights of the case, its activations or token ids)."""
    gen = _gen(seed)
    dev = gen.device
    kind = case["kind"]
    if kind == "linear":
        w = _weight("w", case["qtype"], case["n"], case["k"], gen)
        return w, torch.randn(case["m"], case["k"], device=dev, generator=gen).to(DTYPES[case["dtype"]])
    if kind == "embedding":
        w = _weight("token_embd.weight", "IQ2_S", case["n"], case["k"], gen, std=1.0)
        return w, torch.randint(0, case["n"], (case["m"],), device=dev, generator=gen)
    store = Store(gen, {"gdn": "gdn", "attn": "attn"}.get(kind, "model"))
    if kind in ("gdn", "attn"):
        return store, torch.randn(case["b"], case["m"], ARGS.hidden_size, device=dev, generator=gen).half()
    return store, torch.randint(0, VOCAB, (case["b"], case["m"]), device=dev, generator=gen)


def prepare(case, seed):
    w, x = _inputs(case, seed)
    kind = case["kind"]
    s = {"kind": kind, "x": x}
    if kind == "linear":
        s["mod"] = GSQLinear(w)
    elif kind == "embedding":
        s["mod"] = GSQEmbedding(w, dtype=DTYPES[case["dtype"]])
    elif kind == "gdn":
        s["mod"], s["layer"] = _gdn(w, 0), 0
        s["cache"] = Qwen35Cache(ARGS, case["b"], case["m"], x.device, torch.float16)
    elif kind == "attn":
        s["mod"], s["layer"] = _attn(w, LAYERS - 1), LAYERS - 1
        s["cache"] = Qwen35Cache(ARGS, case["b"], case["max_len"], x.device, torch.float16)
    else:
        model = build_qwen35(w, dtype=torch.float16, args=ARGS)
        s["mod"] = model
        s["cache"] = model.new_cache(batch=case["b"], max_len=case["max_len"])
        if kind == "decode":
            with torch.no_grad():
                s["decoder"] = GraphDecoder(model, s["cache"], batch=case["b"])
    return s


def _gdn(store, i):
    p = f"blk.{i}."
    half = {k: v.half() for k, v in store.plain.items()}
    return GatedDeltaNet(ARGS, i, GSQFusedLinear([store.weight(p + "attn_qkv.weight"), store.weight(p + "attn_gate.weight")],
                                                 concat=True),
                         GSQLinear(store.weight(p + "ssm_out.weight")), half[p + "ssm_alpha.weight"],
                         half[p + "ssm_beta.weight"], half[p + "ssm_conv1d.weight"], store.plain[p + "ssm_a"],
                         half[p + "ssm_dt.bias"], half[p + "ssm_norm.weight"])


def _attn(store, i):
    p = f"blk.{i}."
    half = {k: v.half() for k, v in store.plain.items()}
    return FullAttention(ARGS, i, GSQFusedLinear([store.weight(p + "attn_q.weight"), store.weight(p + "attn_k.weight")],
                                                 concat=True),
                         GSQLinear(store.weight(p + "attn_v.weight")), GSQLinear(store.weight(p + "attn_output.weight")),
                         half[p + "attn_q_norm.weight"], half[p + "attn_k_norm.weight"])


# ---- one pass ----------------------------------------------------------------------------

def run(state):
    kind, x, mod = state["kind"], state["x"], state["mod"]
    with torch.no_grad():
        if kind in ("linear", "embedding"):
            return mod(x)
        cache = state["cache"]
        cache.reset()  # a new sequence
        if kind == "gdn":
            i = state["layer"]
            return {"y": mod(x, cache), "conv": cache.conv[i], "rec": cache.rec[i]}
        if kind == "attn":
            i, S = state["layer"], x.shape[1]
            return {"y": mod(x, cache), "k": cache.k[i][:, :, :S], "v": cache.v[i][:, :, :S]}
        if kind == "prefill":
            return {"logits": mod(x, cache), "rec": [cache.rec[i] for i in sorted(cache.rec)]}
        dec = state["decoder"]
        logits = [dec.step(x[:, t:t + 1]).clone() for t in range(x.shape[1])]
        return {"logits": logits, "rec": [cache.rec[i] for i in sorted(cache.rec)]}


# ---- what a pass cannot do without -------------------------------------------------------

def _proj(kind, n, k, rows):
    return n * (k // 256) * BLOCK_BYTES[MODEL_TYPES[kind]], 2.0 * rows * n * k


def _mixer_work(kind, b, s):
    """(bytes of weights and states, flops) of one mixer over b sequences of s tokens."""
    a, H, rows = ARGS, ARGS.hidden_size, b * s
    if kind == "gdn":
        parts = [_proj("attn_qkv", a.conv_dim, H, rows), _proj("attn_gate", a.value_dim, H, rows),
                 _proj("ssm_out", H, a.value_dim, rows)]
        state = a.linear_num_value_heads * a.linear_key_head_dim * a.linear_value_head_dim
        nbytes, flops = 8 * b * state + 2 * 2 * a.linear_num_value_heads * H, 7.0 * rows * state
        flops += 2.0 * rows * 2 * a.linear_num_value_heads * H
    else:
        kv = a.num_key_value_heads * a.head_dim
        parts = [_proj("attn_q", a.num_attention_heads * a.head_dim * 2, H, rows), _proj("attn_k", kv, H, rows),
                 _proj("attn_v", kv, H, rows), _proj("attn_output", H, a.num_attention_heads * a.head_dim, rows)]
        nbytes, flops = 2 * 2 * rows * kv, 4.0 * b * (s * (s + 1) / 2) * a.num_attention_heads * a.head_dim
    return nbytes + sum(p[0] for p in parts), flops + sum(p[1] for p in parts)


def work(case):
    kind, m = case["kind"], case["m"]
    if kind == "linear":
        n, k, size = case["n"], case["k"], SIZES[case["dtype"]]
        return {"bytes": n * (k // 256) * BLOCK_BYTES[case["qtype"]] + (m * k + m * n) * size, "flops": 2.0 * m * n * k}
    if kind == "embedding":
        k = case["k"]
        return {"bytes": m * (8 + k // 256 * BLOCK_BYTES["IQ2_S"] + k * SIZES[case["dtype"]]), "flops": 0}
    b, H = case["b"], ARGS.hidden_size
    if kind in ("gdn", "attn"):
        nbytes, flops = _mixer_work(kind, b, m)
        return {"bytes": nbytes + 2 * 2 * b * m * H, "flops": flops}

    def call(s, ctx_flops=0.0):
        nbytes, flops = 0, ctx_flops
        for i in range(LAYERS):
            for n_, f in (_mixer_work("gdn" if ARGS.is_linear(i) else "attn", b, s),
                          _proj("ffn_gate", ARGS.intermediate_size, H, b * s),
                          _proj("ffn_up", ARGS.intermediate_size, H, b * s),
                          _proj("ffn_down", H, ARGS.intermediate_size, b * s), ):
                nbytes, flops = nbytes + n_, flops + f
        head, f = _proj("output", VOCAB, H, b * s)
        return nbytes + head + 2 * b * s * VOCAB, flops + f

    nbytes, flops = call(m) if kind == "prefill" else (m * v for v in call(1))
    return {"bytes": nbytes, "flops": flops}


# About four times the error against float64 that was measured: 16-bit outputs (fp16 2.1e-4, bf16
# 1.7e-3), with fp16 weights in the matrix products (2.9e-4); 6.5e-4 over a mixer's chain of 16-bit
# steps, 1.7e-3 over four layers of them. A gathered embedding row is rounded once: exact.
TOLERANCE = {"gdn": 2.6e-3, "attn": 2.6e-3, "prefill": 7e-3, "decode": 7e-3}


def tolerance(case):
    kind = case["kind"]
    if kind == "embedding":
        return "exact"
    if kind == "linear":
        return {"rel": 7e-3 if case["dtype"] == "bf16" else 1.2e-3}
    return {"rel": TOLERANCE[kind]}


# ---- float64 restatement -----------------------------------------------------------------

def _half_at(raw, off):
    return raw[:, off:off + 2].contiguous().view(torch.float16).double()


def _decode(qtype, raw):
    """float64 weights (blocks, 256) of superblocks (blocks, bytes): the published formats."""
    dev = raw.device
    e = torch.arange(256, device=dev)
    i = raw.to(torch.int32)

    def u16(off, count):
        return i[:, off:off + 2 * count:2] | i[:, off + 1:off + 2 * count:2] << 8

    def signs(bits, c):
        return 1.0 - 2.0 * (bits >> c & 1).double()

    def parity_signs(seven, c):  # seven stored sign bits; the eighth makes their number even
        p = seven ^ seven >> 4
        p = p ^ p >> 2
        p = (p ^ p >> 1) & 1
        return signs(seven | p << 7, c)

    book = None
    if qtype in _codebooks():
        book = torch.from_numpy(_codebooks()[qtype]).to(dev).double()
    g32, o8, c8 = e // 32, e // 8, e % 8
    if qtype == "Q2_K":
        q = i[:, 16 + e // 128 * 32 + e % 32] >> 2 * (e % 128 // 32) & 3
        s = i[:, e // 16]
        return _half_at(raw, 80) * (s & 15) * q - _half_at(raw, 82) * (s >> 4)
    if qtype == "Q4_K":
        q = i[:, 16 + e // 64 * 32 + e % 32] >> 4 * (g32 & 1) & 15
        a, m, x = i[:, 4:8], i[:, 8:12], i[:, 12:16]
        sc = torch.cat([a & 63, x & 15 | a >> 2 & 48], 1)[:, g32]
        mn = torch.cat([m & 63, x >> 4 | m >> 2 & 48], 1)[:, g32]
        return _half_at(raw, 0) * sc * q - _half_at(raw, 2) * mn
    if qtype == "Q6_K":
        lo = i[:, e // 128 * 64 + e % 64] >> 4 * (e % 128 // 64) & 15
        hi = i[:, 128 + e // 128 * 32 + e % 32] >> 2 * (e % 128 // 32) & 3
        sc = raw[:, 192:208].contiguous().view(torch.int8).double()[:, e // 16]
        return _half_at(raw, 208) * sc * ((lo | hi << 4) - 32)
    if qtype == "IQ4_XS":
        values = torch.tensor([-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113], device=dev).double()
        q = i[:, 8 + g32 * 16 + e % 16] >> 4 * (e % 32 // 16) & 15
        sc = (i[:, 4 + g32 // 2] >> 4 * (g32 & 1) & 15) | (u16(2, 1) >> 2 * g32 & 3) << 4
        return _half_at(raw, 0) * (sc - 32) * values[q.long()]
    if qtype == "IQ3_S":
        l4 = e // 4
        idx = i[:, 2 + l4] | (i[:, 66 + g32] >> l4 % 8 & 1) << 8
        sc = 2 * (i[:, 106 + g32 // 2] >> 4 * (g32 & 1) & 15) + 1
        return _half_at(raw, 0) * sc * book[idx.long(), e % 4] * signs(i[:, 74 + o8], c8)
    if qtype in ("IQ3_XXS", "IQ2_XXS"):
        aux = raw[:, 66:98] if qtype == "IQ3_XXS" else raw[:, 2:66].reshape(-1, 8, 8)[:, :, 4:].reshape(-1, 32)
        u = aux.contiguous().view(torch.int32).to(torch.int64)[:, g32] & 0xFFFFFFFF
        sg = parity_signs(u >> 7 * (o8 % 4) & 127, c8)
        if qtype == "IQ3_XXS":
            v, scale = book[i[:, 2 + e // 4].long(), e % 4], 0.5
        else:
            v, scale = book[i[:, 2 + g32 * 8 + o8 % 4].long(), c8], 0.25
        return _half_at(raw, 0) * (0.5 + (u >> 28).double()) * scale * v * sg
    if qtype == "IQ2_XS":
        q = u16(2, 32)[:, o8]
        sc = i[:, 66 + g32] >> 4 * (e // 16 & 1) & 15
        return _half_at(raw, 0) * (0.5 + sc.double()) * 0.25 * book[(q & 511).long(), c8] * parity_signs(q >> 9, c8)
    if qtype == "IQ2_S":
        q = i[:, 2 + o8] | (i[:, 66 + g32] >> 2 * (o8 % 4) & 3) << 8
        sc = i[:, 74 + g32] >> 4 * (e // 16 & 1) & 15
        return _half_at(raw, 0) * (0.5 + sc.double()) * 0.25 * book[q.long(), c8] * signs(i[:, 34 + o8], c8)
    if qtype == "IQ1_S":
        h = u16(34, 8)[:, g32]
        q = i[:, 2 + o8] | (h >> 3 * (o8 % 4) & 7) << 8
        delta = 0.125 - 0.25 * (h >> 15 & 1).double()
        return _half_at(raw, 0) * (2 * (h >> 12 & 7) + 1) * (book[q.long(), c8] + delta)
    assert qtype == "IQ1_M"
    w = u16(48, 4)
    bits = w[:, 0] >> 12 | (w[:, 1] >> 12) << 4 | (w[:, 2] >> 12) << 8 | (w[:, 3] >> 12) << 12
    d = bits.to(torch.int16).view(torch.float16).double()[:, None]
    h = i[:, 32 + e // 16] >> 4 * (o8 & 1) & 15
    q = i[:, o8] | (h & 7) << 8
    sc = w[:, e // 64] >> 3 * (e // 16 % 4) & 7
    return d * (2 * sc + 1) * (book[q.long(), c8] + 0.125 - 0.25 * (h >> 3).double())


def _matmul(x, w):
    """x @ W^T in float64, the packed matrix decoded a piece at a time."""
    n, k = w.logical_shape
    raw = w.data.reshape(n, -1)
    out = []
    for r in range(0, n, 1024):
        part = raw[r:r + 1024]
        dense = _decode(w.quantization_type, part.reshape(-1, BLOCK_BYTES[w.quantization_type])).reshape(-1, k)
        out.append(x.reshape(-1, k) @ dense.t().contiguous())
    return torch.cat(out, 1).reshape(*x.shape[:-1], n)


def _rms_norm(x, w, eps):
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _silu(x):
    return x * torch.sigmoid(x)


def _plain(store, name):
    t = store.plain[name]
    return (t if name.endswith("ssm_a") else t.half()).double()


def _gdn_exact(store, i, x):
    """One GatedDeltaNet over whole sequences: (y, last convolution inputs, final state)."""
    a, p = ARGS, f"blk.{i}."
    B, S, _ = x.shape
    hk, hv, dk, dv = (a.linear_num_key_heads, a.linear_num_value_heads, a.linear_key_head_dim,
                      a.linear_value_head_dim)
    kw = a.linear_conv_kernel_dim
    qkv = _matmul(x, store.weight(p + "attn_qkv.weight"))
    z = _matmul(x, store.weight(p + "attn_gate.weight"))
    cw = _plain(store, p + "ssm_conv1d.weight")
    padded = torch.cat([qkv.new_zeros(B, kw - 1, a.conv_dim), qkv], 1)
    conv = _silu(sum(padded[:, j:j + S] * cw[:, j] for j in range(kw)))
    q, k, v = conv.split([a.key_dim, a.key_dim, a.value_dim], -1)
    reps = hv // hk  # value head h reads query / key head h mod hk
    q = (_rms_norm(q.reshape(B, S, hk, dk), None, 1e-6) / dk).repeat(1, 1, reps, 1)
    k = (_rms_norm(k.reshape(B, S, hk, dk), None, 1e-6) * dk ** -0.5).repeat(1, 1, reps, 1)
    v = v.reshape(B, S, hv, dv)
    alpha = x @ _plain(store, p + "ssm_alpha.weight").t().contiguous()
    beta = torch.sigmoid(x @ _plain(store, p + "ssm_beta.weight").t().contiguous())
    decay = torch.exp(_plain(store, p + "ssm_a") * torch.nn.functional.softplus(alpha + _plain(store, p + "ssm_dt.bias")))
    st = x.new_zeros(B, hv, dk, dv)
    outs = []
    for t in range(S):
        st = st * decay[:, t, :, None, None]
        delta = (v[:, t] - (st * k[:, t, :, :, None]).sum(-2)) * beta[:, t, :, None]
        st = st + k[:, t, :, :, None] * delta[:, :, None, :]
        outs.append((st * q[:, t, :, :, None]).sum(-2))
    out = _rms_norm(torch.stack(outs, 1), _plain(store, p + "ssm_norm.weight"), a.rms_norm_eps)
    out = (out * _silu(z.reshape(B, S, hv, dv))).reshape(B, S, -1)
    return _matmul(out, store.weight(p + "ssm_out.weight")), padded[:, S:], st


def _attn_exact(store, i, x):
    """One gated attention layer over whole sequences: (y, rotated keys, values)."""
    a, p = ARGS, f"blk.{i}."
    B, S, _ = x.shape
    H, G, hd, rd = a.num_attention_heads, a.num_key_value_heads, a.head_dim, a.rotary_dim
    qg = _matmul(x, store.weight(p + "attn_q.weight")).reshape(B, S, H, 2 * hd)
    q, gate = qg[..., :hd], qg[..., hd:]
    k = _matmul(x, store.weight(p + "attn_k.weight")).reshape(B, S, G, hd)
    v = _matmul(x, store.weight(p + "attn_v.weight")).reshape(B, S, G, hd)
    q = _rms_norm(q, _plain(store, p + "attn_q_norm.weight"), a.rms_norm_eps)
    k = _rms_norm(k, _plain(store, p + "attn_k_norm.weight"), a.rms_norm_eps)
    freq = a.rope_theta ** (-torch.arange(0, rd, 2, device=x.device).double() / rd)
    ang = torch.arange(S, device=x.device).double()[:, None] * freq
    cos, sin = ang.cos()[None, :, None], ang.sin()[None, :, None]

    def rotate(t):
        lo, hi = t[..., :rd // 2], t[..., rd // 2:rd]
        return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin, t[..., rd:]], -1)

    q, k, v = rotate(q).transpose(1, 2), rotate(k).transpose(1, 2).contiguous(), v.transpose(1, 2).contiguous()
    later = torch.arange(S, device=x.device)[None, :] > torch.arange(S, device=x.device)[:, None]
    outs = []
    for h in range(H):
        keys, vals = k[:, h // (H // G)], v[:, h // (H // G)]
        sc = torch.matmul(q[:, h].contiguous(), keys.transpose(1, 2).contiguous()) * hd ** -0.5
        outs.append(torch.matmul(torch.softmax(sc.masked_fill(later, float("-inf")), -1), vals))
    out = torch.stack(outs, 2) * torch.sigmoid(gate)
    return _matmul(out.reshape(B, S, H * hd), store.weight(p + "attn_output.weight")), k, v


def _embed_exact(w, ids):
    raw = w.data.reshape(w.logical_shape[0], -1)[ids.reshape(-1)]
    return _decode("IQ2_S", raw.reshape(-1, 82)).reshape(*ids.shape, -1)


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        w, x = _inputs(case, seed)
        if kind == "linear":
            return _matmul(x.double(), w)
        if kind == "embedding":
            return _embed_exact(w, x)
        if kind == "gdn":
            y, conv, rec = _gdn_exact(w, 0, x.double())
            return {"y": y, "conv": conv, "rec": rec}
        if kind == "attn":
            y, k, v = _attn_exact(w, LAYERS - 1, x.double())
            return {"y": y, "k": k, "v": v}
        eps = ARGS.rms_norm_eps
        h, rec = _embed_exact(w.weight("token_embd.weight"), x), []
        for i in range(LAYERS):
            p = f"blk.{i}."
            hn = _rms_norm(h, _plain(w, p + "attn_norm.weight"), eps)
            if ARGS.is_linear(i):
                y, _, st = _gdn_exact(w, i, hn)
                rec.append(st)
            else:
                y = _attn_exact(w, i, hn)[0]
            h = h + y
            hn = _rms_norm(h, _plain(w, p + "post_attention_norm.weight"), eps)
            act = _silu(_matmul(hn, w.weight(p + "ffn_gate.weight"))) * _matmul(hn, w.weight(p + "ffn_up.weight"))
            h = h + _matmul(act, w.weight(p + "ffn_down.weight"))
        logits = _matmul(_rms_norm(h, _plain(w, "output_norm.weight"), eps), w.weight("output.weight"))
        if kind == "decode":
            logits = [logits[:, t:t + 1] for t in range(x.shape[1])]
        return {"logits": logits, "rec": rec}
