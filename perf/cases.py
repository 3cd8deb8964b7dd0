"""Cases for timing the framework's work through its public entry points, with their algorithmic work, a
tolerance and a float64 computation of the same outputs that uses none of the framework's code.

Kinds of case (the field `kind`):
  attn    one attention layer of an engine step on the paged pool: `HipBackend.forward_rotary`, the call that
          `LlamaAttention` makes once per layer, with the step's metadata and plan in hand (they are built once
          per step and shared by its layers).  Outputs: the attention output and both pools after the append.
  dense   contiguous causal attention: `HipBackend.prefill`, the layer of a forward pass without a KV cache
          (batch-1 generation by recomputation, scoring of padded batches, float32 correctness runs).
  layer   one `LlamaDecoderLayer` of Llama-3.1-8B's shape on a paged step: norms, projections, rotary
          embedding, attention, MLP.  Outputs: the hidden state and both pools.
  step    a whole engine step as `EngineCore` runs it: the metadata from the resident block tables, then
          `LlamaForCausalLM` (Llama-3.1-8B's shape, two layers) over the rows' new tokens.  Outputs: the
          metadata and the rows' logits.

Rows of the paged kinds are (cached tokens, new tokens): a decode row has one new token, a prompt chunk
several.  They come from a rule named by `rows` and from the seed of the case (`shape_seed`), so that every
preparation of a case has the same sizes, whatever its values.
"""

from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import torch

_ROOT = Path(__file__).resolve().parent.parent
if str(_ROOT / "mini-llm-inference-server_amd") not in sys.path:
    sys.path.insert(0, str(_ROOT / "mini-llm-inference-server_amd"))

DEV = "cuda:0"
BLOCK = 16
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
FP8 = torch.float8_e4m3fn
K_SCALE, V_SCALE = 0.015, 0.0125  # fp8 pools: N(0, 1) keys and values reach about +-6, e4m3 holds +-448

# Llama-3.1-8B's decoder layer (the framework's LLAMA_3_1_8B)
HIDDEN, FFN, VOCAB, HEADS, KV_HEADS, DH = 4096, 14336, 128256, 32, 8, 128
EPS, THETA = 1e-5, 500000.0
ROPE = {"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
        "original_max_position_embeddings": 8192}
STEP_LAYERS = 2


def listed() -> list[dict]:
    heads = {"h": HEADS, "hkv": KV_HEADS}
    return [
        # the smallest engine step: four chat requests early in their answers (latency and launches)
        {"name": "attn_decode_4", "kind": "attn", "rows": "decode_4", "shape_seed": 0, "kv": "bf16", "dtype": "bf16",
         **heads},
        # an ordinary decode step of a lightly loaded fp16 server, short and long contexts side by side
        {"name": "attn_decode_37_fp16", "kind": "attn", "rows": "decode", "n": 37, "lo": 16, "hi": 2048,
         "shape_seed": 1, "kv": "fp16", "dtype": "fp16", **heads},
        # a full decode step: 256 requests of 128-4096 tokens (the framework's headline workload)
        {"name": "attn_decode_256", "kind": "attn", "rows": "decode", "n": 256, "lo": 128, "hi": 4096,
         "shape_seed": 2, "kv": "bf16", "dtype": "bf16", **heads},
        # the same step on an fp8 pool
        {"name": "attn_decode_256_fp8", "kind": "attn", "rows": "decode", "n": 256, "lo": 128, "hi": 4096,
         "shape_seed": 2, "kv": "fp8", "dtype": "bf16", **heads},
        # continuous batching under load: prompt chunks admitted beside 120 long decode rows
        {"name": "attn_mixed_128", "kind": "attn", "rows": "mixed", "n": 120, "lo": 256, "hi": 8192, "chunks": 8,
         "new": 512, "past": 1024, "shape_seed": 3, "kv": "bf16", "dtype": "bf16", **heads},
        # 64 requests that share a 2048-token system prompt, each with its own 64-512 new tokens
        {"name": "attn_prefix_64", "kind": "attn", "rows": "prefix", "n": 64, "prefix": 2048, "lo": 64, "hi": 512,
         "shape_seed": 4, "kv": "bf16", "dtype": "bf16", **heads},
        # generation without a cache: the attention of one 512-token sequence
        {"name": "dense_1x512", "kind": "dense", "b": 1, "tq": 512, "tk": 512, "dh": DH, "dtype": "bf16",
         "valid": False, "shape_seed": 5, **heads},
        # scoring a left-padded batch of four prompts of up to 777 tokens (views as the model makes them)
        {"name": "dense_4x777_padded", "kind": "dense", "b": 4, "tq": 777, "tk": 777, "dh": DH, "dtype": "bf16",
         "valid": True, "shape_seed": 6, **heads},
        # a float32 correctness run on a small model: new tokens on top of earlier ones
        {"name": "dense_fp32_300_of_700", "kind": "dense", "b": 1, "tq": 300, "tk": 700, "dh": DH, "dtype": "fp32",
         "valid": False, "shape_seed": 7, "h": 8, "hkv": 2},
        # a decode step of a small batch: the weights are most of what is read
        {"name": "layer_decode_8", "kind": "layer", "rows": "decode", "n": 8, "lo": 200, "hi": 2000, "shape_seed": 8,
         "kv": "bf16", "dtype": "bf16"},
        # the prompts of three new requests
        {"name": "layer_prompt_3", "kind": "layer", "rows": "mixed", "n": 0, "lo": 16, "hi": 16, "chunks": 3,
         "new": 256, "past": 0, "shape_seed": 9, "kv": "bf16", "dtype": "bf16"},
        # a whole decode step of 32 requests, tables to logits
        {"name": "step_decode_32", "kind": "step", "rows": "decode", "n": 32, "lo": 64, "hi": 2048, "shape_seed": 10,
         "kv": "bf16", "dtype": "bf16"},
    ]


def draw(rng: random.Random) -> dict:
    """One more case of the listed ranges; odd sizes, other head counts (a tensor-parallel shard's) and types."""

    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    seed = rng.randrange(1 << 20)
    kind = rng.choice(["attn", "attn", "attn", "dense", "dense", "layer", "layer", "step"])
    if kind == "dense":
        h, hkv = rng.choice([(32, 8), (32, 8), (8, 2), (4, 4), (8, 1)])
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        b = rng.choice([1, 1, 2, 3, 4])
        tk = log(8, 1100 // (2 if dtype == "fp32" else 1))
        tq = tk if rng.random() < 0.7 else log(1, tk)
        return {"kind": "dense", "b": b, "tq": tq, "tk": tk, "dh": rng.choice([128, 128, 64]), "dtype": dtype,
                "valid": rng.random() < 0.4, "shape_seed": seed, "h": h, "hkv": hkv}
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    kv = rng.choice([dtype, dtype, "fp8"])
    rows = rng.choice(["decode", "decode", "mixed"] if kind != "attn" else ["decode", "decode", "mixed", "prefix"])
    if kind == "attn":
        h, hkv = rng.choice([(32, 8), (32, 8), (16, 4), (8, 2)])
        case = {"kind": kind, "rows": rows, "shape_seed": seed, "kv": kv, "dtype": dtype, "h": h, "hkv": hkv}
        most = 256
    else:
        case = {"kind": kind, "rows": rows, "shape_seed": seed, "kv": kv, "dtype": dtype}
        most = 96
    if rows == "decode":
        hi = log(64, 4096)
        case.update(n=log(1, most), lo=max(1, hi // 32), hi=hi)
    elif rows == "mixed":
        hi = log(256, 8192 if kind == "attn" else 2048)
        case.update(n=log(1, most // 3), lo=max(1, hi // 32), hi=hi, chunks=rng.randint(1, 8 if kind == "attn" else 3),
                    new=log(16, 512), past=rng.choice([0, 0, 1024]))
    else:
        case.update(n=log(2, 64), prefix=16 * log(16, 128), lo=8, hi=log(16, 512))
    return case


# ---------------------------------------------------------------- sizes


def _rows(case: dict) -> tuple[list[tuple[int, int]], int]:
    """The step's rows (cached, new), in row order, and the tokens of the prefix they all share."""
    rng = random.Random(case["shape_seed"])
    if case["rows"] == "decode_4":
        return [(c, 1) for c in (37, 128, 211, 500)], 0
    if case["rows"] == "decode":
        return [(rng.randint(case["lo"], case["hi"]), 1) for _ in range(case["n"])], 0
    if case["rows"] == "prefix":
        return [(case["prefix"], rng.randint(case["lo"], case["hi"])) for _ in range(case["n"])], case["prefix"]
    rows = [(rng.randint(case["lo"], case["hi"]), 1) for _ in range(case["n"])]
    for _ in range(case["chunks"]):
        new = min(2048, max(2, round(case["new"] * math.exp(rng.gauss(0.0, 0.5)))))
        rows.append((rng.randint(0, case["past"]), new))
    rng.shuffle(rows)
    return rows, 0


def _tables(case: dict) -> tuple[list[list[int]], int]:
    """Each row's block ids (shuffled pages of a pool half as large again as needed) and the pool's blocks."""
    rows, prefix = _rows(case)
    shared = prefix // BLOCK
    need = [-(-(c + n) // BLOCK) - shared for c, n in rows]
    pool = 3 * (shared + sum(need)) // 2 + 8
    ids = list(range(pool))
    random.Random(case["shape_seed"] + 1).shuffle(ids)
    out, at = [], shared
    for k in need:
        out.append(ids[:shared] + ids[at:at + k])
        at += k
    return out, pool


def _heads(case: dict) -> tuple[int, int]:
    return case.get("h", HEADS), case.get("hkv", KV_HEADS)


# ---------------------------------------------------------------- inputs


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, shape, dtype, std: float = 1.0, mean: float = 0.0) -> torch.Tensor:
    return torch.empty(shape, dtype=torch.float32, device=DEV).normal_(mean, std, generator=g).to(dtype)


def _pool(g, case: dict, blocks: int, hkv: int, scale: float) -> torch.Tensor:
    x = torch.empty((blocks, BLOCK, hkv, DH), dtype=torch.float32, device=DEV).normal_(0.0, 1.0, generator=g)
    return (x / scale).to(FP8) if case["kv"] == "fp8" else x.to(DTYPES[case["kv"]])


def _scales(case: dict) -> dict:
    return {"k_scale": K_SCALE, "v_scale": V_SCALE} if case["kv"] == "fp8" else {}


def _config(layers: int):
    from minillm.model.config import LlamaConfig

    return LlamaConfig(vocab_size=VOCAB, hidden_size=HIDDEN, intermediate_size=FFN, num_hidden_layers=layers,
                       num_attention_heads=HEADS, num_key_value_heads=KV_HEADS, head_dim=DH, rms_norm_eps=EPS,
                       rope_theta=THETA, rope_scaling=ROPE, max_position_embeddings=131072)


def _inv_freq() -> torch.Tensor:
    """Llama 3's scaled rotary frequencies, float64."""
    inv = THETA ** (-torch.arange(0, DH, 2, dtype=torch.float64) / DH)
    wave = 2 * math.pi / inv
    old, lo, hi, f = (ROPE["original_max_position_embeddings"], ROPE["low_freq_factor"], ROPE["high_freq_factor"],
                      ROPE["factor"])
    mix = ((old / wave - lo) / (hi - lo)).clamp(0.0, 1.0)  # 0: wavelengths past old / lo, 1: below old / hi
    return ((1 - mix) * inv / f + mix * inv).to(DEV)


def _angles(positions: torch.Tensor) -> torch.Tensor:
    a = positions.double()[:, None] * _inv_freq()
    return torch.cat([a, a], dim=-1)


def _positions(rows) -> torch.Tensor:
    return torch.cat([torch.arange(c, c + n) for c, n in rows]).to(DEV)


def _metadata(case: dict):
    from minillm.attention.metadata import AttentionMetadata, SeqStep

    rows, _ = _rows(case)
    tables, _ = _tables(case)
    return AttentionMetadata.build([SeqStep(c, n, t) for (c, n), t in zip(rows, tables)], BLOCK, DEV)


def _weights(g, module, dtype) -> None:
    """Seeded weights: matrices N(0, 0.02), norms around 1."""
    for name, p in module.named_parameters():
        mean, std = (1.0, 0.1) if "norm" in name else (0.0, 0.02)
        p.data.normal_(mean, std, generator=g)


def _build(make, dtype):
    """A module made directly on the GPU in `dtype` (its weights are filled afterwards)."""
    old = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    try:
        with torch.device("meta"):
            module = make()
    finally:
        torch.set_default_dtype(old)
    return module.to_empty(device=DEV)


def _attn_inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    dt = DTYPES[case["dtype"]]
    h, hkv = _heads(case)
    rows, _ = _rows(case)
    _, blocks = _tables(case)
    n = sum(new for _, new in rows)
    ang = _angles(_positions(rows))
    return {"q": _randn(g, (n, h, DH), dt), "k": _randn(g, (n, hkv, DH), dt), "v": _randn(g, (n, hkv, DH), dt),
            "cos": ang.cos().to(dt), "sin": ang.sin().to(dt), "kc": _pool(g, case, blocks, hkv, K_SCALE),
            "vc": _pool(g, case, blocks, hkv, V_SCALE)}


def _dense_inputs(case: dict, seed: int) -> dict:
    """q, k, v as [B, T, H, Dh] storage seen as [B, H, T, Dh] (what the model's view + transpose gives), and for
    padded batches the mask of real keys: left padding, one row unpadded."""
    g = _gen(seed)
    dt = DTYPES[case["dtype"]]
    b, tq, tk, dh = case["b"], case["tq"], case["tk"], case["dh"]
    q, k, v = (_randn(g, (b, t, heads, dh), dt).transpose(1, 2)
               for t, heads in ((tq, case["h"]), (tk, case["hkv"]), (tk, case["hkv"])))
    valid = None
    if case["valid"]:
        rng = random.Random(case["shape_seed"])
        pad = [0] + [rng.randint(0, tk // 2) for _ in range(b - 1)]
        valid = torch.arange(tk, device=DEV)[None, :] >= torch.tensor(pad, device=DEV)[:, None]
    return {"q": q, "k": k, "v": v, "key_valid": valid}


def _layer_inputs(case: dict, seed: int) -> dict:
    from minillm.attention.hip_backend import HipBackend
    from minillm.cache.paged import PagedKVCache
    from minillm.model.llama import LlamaDecoderLayer

    g = _gen(seed)
    dt = DTYPES[case["dtype"]]
    cfg = _config(1)
    rows, _ = _rows(case)
    _, blocks = _tables(case)
    n = sum(new for _, new in rows)
    layer = _build(lambda: LlamaDecoderLayer(cfg, HipBackend(), 0), dt)
    _weights(g, layer, dt)
    cache = PagedKVCache(cfg, 1, DEV, FP8 if case["kv"] == "fp8" else DTYPES[case["kv"]], **_scales(case))
    cache.num_blocks = blocks
    cache.k, cache.v = [_pool(g, case, blocks, KV_HEADS, K_SCALE)], [_pool(g, case, blocks, KV_HEADS, V_SCALE)]
    ang = _angles(_positions(rows))
    return {"layer": layer, "cache": cache, "x": _randn(g, (1, n, HIDDEN), dt), "cos": ang.cos().to(dt)[None],
            "sin": ang.sin().to(dt)[None]}


def _step_inputs(case: dict, seed: int) -> dict:
    from minillm.attention.hip_backend import HipBackend
    from minillm.attention.metadata import DeviceBlockTables, SeqStep
    from minillm.cache.paged import PagedKVCache
    from minillm.model.llama import LlamaForCausalLM

    g = _gen(seed)
    dt = DTYPES[case["dtype"]]
    cfg = _config(STEP_LAYERS)
    rows, _ = _rows(case)
    tables, blocks = _tables(case)
    n = sum(new for _, new in rows)
    model = _build(lambda: LlamaForCausalLM(cfg, HipBackend()), dt)
    _weights(g, model, dt)
    cache = PagedKVCache(cfg, 1, DEV, FP8 if case["kv"] == "fp8" else DTYPES[case["kv"]], **_scales(case))
    cache.num_blocks = blocks
    cache.k = [_pool(g, case, blocks, KV_HEADS, K_SCALE) for _ in range(STEP_LAYERS)]
    cache.v = [_pool(g, case, blocks, KV_HEADS, V_SCALE) for _ in range(STEP_LAYERS)]
    seqs = [SeqStep(c, new, t) for (c, new), t in zip(rows, tables)]
    return {"model": model, "cache": cache, "tables": DeviceBlockTables(len(rows), max(map(len, tables)), DEV),
            "keys": list(range(len(rows))), "seqs": seqs,
            "ids": torch.randint(0, VOCAB, (1, n), device=DEV, generator=g)}


def prepare(case: dict, seed: int) -> dict:
    from minillm.attention.hip_backend import HipBackend

    kind = case["kind"]
    if kind == "attn":
        s = _attn_inputs(case, seed)
        s.update(backend=HipBackend(), meta=_metadata(case), scales=_scales(case))
    elif kind == "dense":
        s = _dense_inputs(case, seed)
        s["backend"] = HipBackend()
    elif kind == "layer":
        s = _layer_inputs(case, seed)
        s["kv_cache"] = s["cache"].step(_metadata(case))
    else:
        s = _step_inputs(case, seed)
    s["kind"] = kind
    return s


def _bytes(pool: torch.Tensor) -> torch.Tensor:
    return pool.view(torch.uint8) if pool.dtype == FP8 else pool


@torch.inference_mode()
def run(s: dict):
    kind = s["kind"]
    if kind == "attn":
        out = s["backend"].forward_rotary(s["q"], s["k"], s["v"], s["cos"], s["sin"], s["kc"], s["vc"], s["meta"],
                                          **s["scales"])
        return {"out": out, "k_pool": _bytes(s["kc"]), "v_pool": _bytes(s["vc"])}
    if kind == "dense":
        return {"out": s["backend"].prefill(s["q"], s["k"], s["v"], key_valid=s["key_valid"])}
    if kind == "layer":
        out = s["layer"](s["x"], s["cos"], s["sin"], s["kv_cache"])
        return {"out": out, "k_pool": _bytes(s["cache"].k[0]), "v_pool": _bytes(s["cache"].v[0])}
    meta = s["tables"].build(s["keys"], s["seqs"], BLOCK)
    logits = s["model"](s["ids"], kv_cache=s["cache"].step(meta), last_index=meta.logits_index)[:, -1]
    return {"logits": logits, "positions": meta.positions, "slots": meta.slot_mapping, "tables": meta.block_tables,
            "qo_indptr": meta.qo_indptr, "kv_indptr": meta.kv_indptr, "kv_indices": meta.kv_indices,
            "seq_lens": meta.seq_lens_i32, "last_page": meta.kv_last_page_len, "last": meta.logits_index}


# ---------------------------------------------------------------- work and tolerance


def _attn_work(case: dict) -> tuple[int, int]:
    """(bytes, flops) of one paged attention layer with its append: every distinct context token's K and V once,
    q, k, v, cos and sin in, the output and the appended rows out."""
    rows, prefix = _rows(case)
    h, hkv = _heads(case)
    kv = 1 if case["kv"] == "fp8" else 2
    n = sum(new for _, new in rows)
    ctx = prefix + sum(c - prefix for c, _ in rows)  # cached tokens, the shared prefix once
    nbytes = 2 * ctx * hkv * DH * kv + n * (2 * 2 * h * DH + 2 * hkv * DH * (2 + kv) + 2 * 2 * DH)
    return nbytes, sum(4 * h * DH * (new * c + new * (new + 1) // 2) for c, new in rows)


def work(case: dict) -> dict:
    if case["kind"] == "dense":
        b, h, hkv, tq, tk, dh = (case[x] for x in ("b", "h", "hkv", "tq", "tk", "dh"))
        es = 4 if case["dtype"] == "fp32" else 2
        rng = random.Random(case["shape_seed"])
        pads = [0] + [rng.randint(0, tk // 2) for _ in range(b - 1)] if case["valid"] else [0] * b
        pairs = sum(max(tk - tq + i + 1 - pad, 1) for pad in pads for i in range(tq))
        return {"bytes": es * b * dh * (2 * h * tq + 2 * hkv * tk), "flops": 4 * h * dh * pairs}
    nbytes, flops = _attn_work(case)
    if case["kind"] == "attn":
        return {"bytes": nbytes, "flops": flops}
    n = sum(new for _, new in _rows(case)[0])
    # the layer's own q, k, v and output are intermediates: only the context and the appended rows count
    kv = 1 if case["kv"] == "fp8" else 2
    nbytes -= n * (2 * 2 * HEADS * DH + 2 * KV_HEADS * DH * 2 + 2 * 2 * DH)
    params = HIDDEN * DH * (2 * HEADS + 2 * KV_HEADS) + 3 * HIDDEN * FFN
    layers = 1 if case["kind"] == "layer" else STEP_LAYERS
    nbytes, flops = layers * (nbytes + 2 * params + 4 * HIDDEN), layers * (flops + 2 * n * params)
    if case["kind"] == "layer":
        return {"bytes": nbytes + 2 * 2 * n * HIDDEN + 2 * 2 * n * DH, "flops": flops}
    s = len(_rows(case)[0])
    return {"bytes": nbytes + 2 * n * HIDDEN + 2 * VOCAB * HIDDEN + 2 * s * VOCAB,
            "flops": flops + 2 * s * HIDDEN * VOCAB}


def tolerance(case: dict) -> dict:
    """Relative 2-norm errors, about four times what the path shows against float64 (dense: 1.6e-3 bf16, 2e-4 fp16,
    5e-7 fp32; paged attention: 3.5e-3 bf16, 4e-4 fp16; a layer 6e-3 to 7e-3 and a two-layer step 1.3e-2 in bf16)."""
    if case["kind"] == "dense":
        return {"rel": {"bf16": 7e-3, "fp16": 9e-4, "fp32": 2e-6}[case["dtype"]]}
    if case["kind"] == "attn":
        return {"rel": 1.4e-2 if case["dtype"] == "bf16" else 2e-3}
    # a rounding changed in one product travels through the norms and layers after it
    rel = 2.5e-2 if case["kind"] == "layer" else 3e-2
    return {"rel": rel if case["dtype"] == "bf16" else rel / 6}


# ---------------------------------------------------------------- the same in float64


def _softmax_v(s: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    p = torch.exp(s - s.amax(dim=-1, keepdim=True))
    return torch.matmul(p / p.sum(dim=-1, keepdim=True), v.contiguous())


def _rotate(x: torch.Tensor, ang: torch.Tensor) -> torch.Tensor:
    half = x.shape[-1] // 2
    turned = torch.cat([-x[..., half:], x[..., :half]], dim=-1)
    return x * ang.cos()[:, None] + turned * ang.sin()[:, None]


def _paged(case: dict, q, k, v, kc, vc) -> torch.Tensor:
    """Attention of new tokens q [N, H, Dh] (rotated) over their rows' contexts: the pool's cached tokens, then
    the step's own k and v."""
    rows, _ = _rows(case)
    tables, _ = _tables(case)
    h, hkv = _heads(case)
    ks, vs = (K_SCALE, V_SCALE) if case["kv"] == "fp8" else (1.0, 1.0)
    if case["kv"] == "fp8":  # the step's own rows are stored in the pool, too
        dt = DTYPES[case["dtype"]]
        k, v = ((x.to(dt).float() * (1.0 / sc)).to(FP8).double() * sc for x, sc in ((k, ks), (v, vs)))
    out, at = [], 0
    for (c, n), t in zip(rows, tables):
        blocks = torch.tensor(t, device=DEV)
        ctx = [torch.cat([(p[blocks].reshape(-1, hkv, DH)[:c].double() * sc), x[at:at + n]]).transpose(0, 1)
               for p, x, sc in ((kc, k, ks), (vc, v, vs))]
        qg = q[at:at + n].reshape(n, hkv, h // hkv, DH).permute(1, 2, 0, 3).reshape(hkv, -1, DH)
        s = torch.matmul(qg.contiguous(), ctx[0].transpose(1, 2).contiguous()) * DH ** -0.5
        if n > 1:
            pos = c + torch.arange(n, device=DEV)
            seen = torch.arange(c + n, device=DEV)[None, :] <= pos[:, None]
            s = s.masked_fill(~seen.repeat(h // hkv, 1)[None], -math.inf)
        o = _softmax_v(s, ctx[1])
        out.append(o.reshape(hkv, h // hkv, n, DH).permute(2, 0, 1, 3).reshape(n, h, DH))
        at += n
    return torch.cat(out)


def _norm(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return w.double() * (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS))


def _mm(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return torch.matmul(x, w.double().t().contiguous())


def _layer(case: dict, layer, x, kc, vc) -> torch.Tensor:
    rows, _ = _rows(case)
    n = x.shape[0]
    ang = _angles(_positions(rows))
    at, mlp = layer.self_attn, layer.mlp
    hid = _norm(x, layer.input_layernorm.weight)
    q, k, v = (_mm(hid, w.weight).view(n, -1, DH) for w in (at.q_proj, at.k_proj, at.v_proj))
    o = _paged(case, _rotate(q, ang), _rotate(k, ang), v, kc, vc)
    x = x + _mm(o.reshape(n, -1), at.o_proj.weight)
    hid = _norm(x, layer.post_attention_layernorm.weight)
    gate = _mm(hid, mlp.gate_proj.weight)
    return x + _mm(gate / (1 + torch.exp(-gate)) * _mm(hid, mlp.up_proj.weight), mlp.down_proj.weight)


@torch.inference_mode()
def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "attn":
        s = _attn_inputs(case, seed)
        ang = _angles(_positions(_rows(case)[0]))
        out = _paged(case, _rotate(s["q"].double(), ang), _rotate(s["k"].double(), ang), s["v"].double(), s["kc"],
                     s["vc"])
        return {"out": out, "k_pool": None, "v_pool": None}
    if kind == "dense":
        s = _dense_inputs(case, seed)
        b, h, hkv, tq, tk = (case[x] for x in ("b", "h", "hkv", "tq", "tk"))
        out = torch.empty((b, h, tq, case["dh"]), dtype=torch.float64, device=DEV)
        pos = tk - tq + torch.arange(tq, device=DEV)
        keys = torch.arange(tk, device=DEV)
        for i in range(b):
            seen = keys[None, :] <= pos[:, None]
            if s["key_valid"] is not None:
                seen = seen & s["key_valid"][i][None, :]
                alone = ~seen.any(dim=-1, keepdim=True)  # a query without a real key sees its own position
                seen = seen | (alone & (keys[None, :] == pos[:, None]))
            for j in range(h):
                k, v = (s[x][i, j // (h // hkv)].double() for x in ("k", "v"))
                sc = torch.matmul(s["q"][i, j].double(), k.t().contiguous()) * case["dh"] ** -0.5
                out[i, j] = _softmax_v(sc.masked_fill(~seen, -math.inf), v)
        return {"out": out}
    if kind == "layer":
        s = _layer_inputs(case, seed)
        return {"out": _layer(case, s["layer"], s["x"][0].double(), s["cache"].k[0], s["cache"].v[0])[None],
                "k_pool": None, "v_pool": None}
    s = _step_inputs(case, seed)
    model = s["model"]
    x = model.model.embed_tokens.weight[s["ids"][0]].double()
    for i, layer in enumerate(model.model.layers):
        x = _layer(case, layer, x, s["cache"].k[i], s["cache"].v[i])
    last = torch.tensor([new for _, new in _rows(case)[0]]).cumsum(0).to(DEV) - 1
    logits = _mm(_norm(x[last], model.model.norm.weight), model.lm_head.weight)
    return {"logits": logits, **{k: None for k in ("positions", "slots", "tables", "qo_indptr", "kv_indptr",
                                                   "kv_indices", "seq_lens", "last_page", "last")}}
