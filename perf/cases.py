"""Workloads of the KV-cache movement API, each one pass through the public entry points.

A case is a dict of plain values: the path it takes (``path``), the sizes of the caches and of the
call, the element type and the options.  ``listed()`` names the cases that are measured by default,
``draw()`` makes further ones over the same ranges, and ``prepare()`` / ``run()`` build a case's
inputs on the GPU and make the call the way a serving engine makes it.

Block tables are random permutations of the cache's blocks: every sequence owns whole blocks and
fills them in order, as a paged allocator hands them out.  A decode step instead touches one slot at
a random offset of each sequence's last block.  ``skip`` is the share of tokens whose slot is -1
(padding of a fixed-size batch).
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "musa-aiter_amd"))

import musa_aiter  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed() -> list[dict]:
    return [
        # One decode step of 64 sequences: each appends one token to one layer's cache (Llama-3-8B heads).
        {"name": "decode_store", "path": "store", "layers": 1, "tokens": 64, "seq_lo": 1, "seq_hi": 1, "decode": True,
         "blocks": 8192, "heads": 8, "head_dim": 128, "page": 16, "dtype": "bf16", "skip": 0.0},
        # The same step into an FP8 cache, with per-head scales.
        {"name": "decode_quant", "path": "quant", "layers": 1, "tokens": 48, "seq_lo": 1, "seq_hi": 1, "decode": True,
         "blocks": 8192, "heads": 8, "head_dim": 128, "page": 16, "dtype": "bf16", "format": "e4m3",
         "scale": "head", "skip": 0.0},
        # A small batch's whole context read from one layer (32 sequences of up to 512 tokens).
        {"name": "load_layer_fp16", "path": "load", "layers": 1, "tokens": 7456, "seq_lo": 1, "seq_hi": 512,
         "decode": False, "blocks": 1024, "heads": 8, "head_dim": 128, "page": 16, "dtype": "fp16", "skip": 0.0},
        # Prefilled sequences stored into all 32 layers at once (the largest call).
        {"name": "prefill_store", "path": "store", "layers": 32, "tokens": 15851, "seq_lo": 128, "seq_hi": 4096,
         "decode": False, "blocks": 1152, "heads": 8, "head_dim": 128, "page": 16, "dtype": "bf16", "skip": 0.0},
        # Cached prefixes read back from all layers of a cache with 64-token pages, some tokens padded.
        {"name": "prefix_load_page64", "path": "load", "layers": 16, "tokens": 9001, "seq_lo": 64, "seq_hi": 2048,
         "decode": False, "blocks": 512, "heads": 8, "head_dim": 128, "page": 64, "dtype": "bf16", "skip": 0.01},
        # Prefilled sequences quantised into one layer's FP8 cache.
        {"name": "prefill_quant", "path": "quant", "layers": 1, "tokens": 30977, "seq_lo": 128, "seq_hi": 4096,
         "decode": False, "blocks": 2560, "heads": 8, "head_dim": 128, "page": 16, "dtype": "bf16",
         "format": "e4m3", "scale": "head", "skip": 0.0},
        # Contexts dequantised from the FP8 caches of 8 layers with 32-token pages, one scale per layer and head.
        {"name": "dequant_load_page32", "path": "dequant", "layers": 8, "tokens": 6007, "seq_lo": 16, "seq_hi": 2048,
         "decode": False, "blocks": 512, "heads": 8, "head_dim": 128, "page": 32, "dtype": "bf16",
         "format": "e4m3", "scale": "layer", "skip": 0.0},
        # Dense [batch, length] preload of one layer for an attention kernel.
        {"name": "dense_preload", "path": "dense", "batch": 16, "seq_lo": 128, "seq_hi": 2048, "blocks": 2304,
         "heads": 8, "head_dim": 128, "page": 16, "dtype": "bf16"},
        # One 256-token LMCache chunk read from the 2 x 32 caches of an SGLang-MP pool.
        {"name": "lmcache_chunk_load", "path": "chunk", "store": False, "layers": 32, "tokens": 256, "blocks": 512,
         "heads": 8, "head_dim": 128, "page": 16, "dtype": "bf16"},
        # DeepSeek latent rows (512 + 64 values) of prefilled sequences stored into 61 layers, 64-token pages.
        {"name": "mla_store", "path": "mla", "store": True, "layers": 61, "tokens": 12345, "seq_lo": 256,
         "seq_hi": 8192, "blocks": 320, "hidden": 576, "page": 64, "dtype": "bf16"},
        # SGLang HiCache: items of all layers backed up from the layer-first to the page-first pool.
        {"name": "hicache_backup", "path": "hicache", "layers": 32, "items": 4096, "pages": 6144, "row": 1024,
         "dtype": "bf16"},
        # CacheGen-style encoding of one 256-token, 32-layer chunk.
        {"name": "cachegen_encode", "path": "cachegen", "encode": True, "layers": 32, "tokens": 256, "heads": 8,
         "head_dim": 128, "bins": 256, "dtype": "bf16"},
    ]


# A drawn case moves at most this many payload bytes (the largest listed case's).
MAX_BYTES = 4.1e9


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _paged(rng, path: str) -> dict:
    """A store or load on paged caches: a decode step, or whole sequences."""
    fp8 = path in ("quant", "dequant")
    heads, head_dim = rng.choice([1, 2, 4, 8, 8]), rng.choice([64, 96, 128, 128])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    page = rng.choice([16, 16, 32, 64] if fp8 else [8, 16, 16, 32, 64])
    decode = path in ("store", "quant") and rng.random() < 0.4
    layers = 1 if decode else rng.choice([1, 1, 4, 16, 32])
    if decode:
        tokens, lo, hi = _log_int(rng, 4, 512), 1, 1
        blocks = tokens + rng.randrange(64, 4096)
    else:
        most = int(MAX_BYTES / (layers * 2 * heads * head_dim * 8))
        tokens = _log_int(rng, 200, min(most, 60000))
        hi = max(64, min(4096, tokens // 2))
        lo = max(16, hi // 16)
        blocks = tokens // page + tokens // lo + 2 + rng.randrange(1, 1 + tokens // page)
    case = {"path": path, "layers": layers, "tokens": tokens, "seq_lo": lo, "seq_hi": hi, "decode": decode,
            "blocks": blocks, "heads": heads, "head_dim": head_dim, "page": page, "dtype": dtype,
            "skip": rng.choice([0.0, 0.0, 0.02])}
    if fp8:
        case["format"] = rng.choice(["e4m3", "e4m3", "e5m2"])
        case["scale"] = rng.choice(["scalar", "head", "layer" if layers > 1 else "head"])
    return case


def draw(rng) -> dict:
    path = rng.choice(["store", "load", "quant", "dequant", "store", "load", "dense", "chunk", "mla", "hicache",
                       "cachegen"])
    if path in ("store", "load", "quant", "dequant"):
        return _paged(rng, path)
    if path == "dense":
        page, hi = rng.choice([8, 16, 16, 32, 64]), _log_int(rng, 128, 4096)
        batch = rng.randrange(1, 33)
        return {"path": path, "batch": batch, "seq_lo": max(1, hi // 16), "seq_hi": hi,
                "blocks": batch * (hi // page + 1) + rng.randrange(1, 512), "heads": rng.choice([1, 2, 4, 8, 8]),
                "head_dim": rng.choice([64, 96, 128, 128]), "page": page, "dtype": rng.choice(["bf16", "fp16", "fp32"])}
    if path == "chunk":
        tokens = rng.choice([64, 256, 256, 1000])
        page = rng.choice([16, 16, 64])
        return {"path": path, "store": rng.random() < 0.5, "layers": rng.choice([16, 32, 32, 40]), "tokens": tokens,
                "blocks": tokens // page + rng.randrange(64, 512), "heads": rng.choice([2, 4, 8, 8]),
                "head_dim": rng.choice([64, 96, 128, 128]), "page": page, "dtype": rng.choice(["bf16", "fp16"])}
    if path == "mla":
        tokens, layers = _log_int(rng, 64, 20000), rng.choice([1, 27, 61])
        hi = max(64, tokens // 2)
        lo = max(32, hi // 32)
        return {"path": path, "store": rng.random() < 0.5, "layers": layers, "tokens": tokens, "seq_lo": lo,
                "seq_hi": hi, "blocks": tokens // 64 + tokens // lo + 2 + rng.randrange(1, 64), "hidden": 576,
                "page": 64, "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    if path == "hicache":
        items = _log_int(rng, 64, 8192)
        return {"path": path, "layers": rng.choice([16, 32, 32]), "items": items, "pages": items + rng.randrange(64, 4096),
                "row": rng.choice([256, 512, 1024, 1024]), "dtype": rng.choice(["bf16", "fp16"])}
    return {"path": path, "encode": rng.random() < 0.5, "layers": rng.choice([16, 32, 32]),
            "tokens": _log_int(rng, 64, 4096), "heads": rng.choice([2, 4, 8]), "head_dim": rng.choice([64, 128]),
            "bins": rng.choice([16, 255, 256, 256]), "dtype": rng.choice(["bf16", "fp16", "fp32"])}


# ----- inputs -----------------------------------------------------------------------------------


def _lengths(rng: np.random.Generator, tokens: int, lo: int, hi: int) -> np.ndarray:
    """Sequence lengths uniform in [lo, hi] that add up to ``tokens`` (the last one cut short)."""
    ends = np.cumsum(rng.integers(lo, hi + 1, size=tokens // lo + 1))
    ends = np.append(ends[ends < tokens], tokens)
    return np.diff(ends, prepend=0)


def _slots(rng: np.random.Generator, case: dict, device: torch.device) -> torch.Tensor:
    """int64 slot of every token of the call."""
    page, tokens = case["page"], case["tokens"]
    order = rng.permutation(case["blocks"])
    if case.get("decode"):
        slots = order[:tokens] * page + rng.integers(0, page, size=tokens)
    else:
        parts, used = [], 0
        for n in _lengths(rng, tokens, case.get("seq_lo", tokens), case.get("seq_hi", tokens)):
            j = np.arange(n)
            parts.append(order[used + j // page] * page + j % page)
            used += -(-int(n) // page)
        slots = np.concatenate(parts)
    if case.get("skip"):
        slots[rng.random(tokens) < case["skip"]] = -1
    return torch.from_numpy(slots.astype(np.int64)).to(device)


def _normal(gen: torch.Generator, shape, dtype: torch.dtype) -> torch.Tensor:
    return torch.randn(shape, generator=gen, device=gen.device, dtype=dtype)


def _fp8_values(gen: torch.Generator, shape, dtype: torch.dtype) -> torch.Tensor:
    """N(0, 2) with 1 % of the entries scaled by 50: activations with outliers that saturate."""
    x = _normal(gen, shape, torch.float32).mul_(math.sqrt(2.0))
    x.mul_(torch.where(torch.rand(shape, generator=gen, device=gen.device) < 0.01, 50.0, 1.0))
    return x.to(dtype)


def _scale(gen: torch.Generator, case: dict) -> torch.Tensor:
    shape = {"scalar": (), "head": (case["heads"],), "layer": (case["layers"], case["heads"])}[case["scale"]]
    return torch.rand(shape, generator=gen, device=gen.device) * 0.2 + 0.1


def prepare(case: dict, seed: int) -> dict:
    device = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=device).manual_seed(seed)
    rng = np.random.default_rng(seed)
    path, dtype = case["path"], DTYPES[case["dtype"]]
    state = {"case": case}
    if path in ("store", "load", "quant", "dequant"):
        nl, heads, hd, page, tokens = case["layers"], case["heads"], case["head_dim"], case["page"], case["tokens"]
        lead = (nl,) if nl > 1 else ()
        shape = lead + (case["blocks"], heads, hd, page)
        state["slots"] = _slots(rng, case, device)
        if path in ("store", "load"):
            state["caches"] = [_normal(gen, shape, dtype) for _ in range(2)]
        else:
            # Codes with a cleared top exponent bit: finite values of ordinary size in both formats.
            state["caches"] = [torch.randint(0, 256, shape, generator=gen, device=device, dtype=torch.uint8)
                               .bitwise_and_(0xBF) for _ in range(2)]
            state["scales"] = [_scale(gen, case) for _ in range(2)]
        if path in ("store", "quant"):
            make = _normal if path == "store" else _fp8_values
            state["linear"] = [make(gen, lead + (tokens, heads, hd), dtype) for _ in range(2)]
    elif path == "dense":
        page, batch = case["page"], case["batch"]
        lengths = rng.integers(case["seq_lo"], case["seq_hi"] + 1, size=batch)
        lengths[0] = case["seq_hi"]
        order = rng.permutation(case["blocks"])
        tables = np.zeros((batch, -(-case["seq_hi"] // page)), dtype=np.int64)
        used = 0
        for b, n in enumerate(lengths):
            k = -(-int(n) // page)
            tables[b, :k] = order[used:used + k]
            used += k
        shape = (case["blocks"], case["heads"], case["head_dim"], page)
        state["caches"] = [_normal(gen, shape, dtype) for _ in range(2)]
        state["tables"] = torch.from_numpy(tables).to(device)
        state["lengths"] = torch.from_numpy(lengths.astype(np.int64)).to(device)
    elif path == "chunk":
        nl, heads, hd, page = case["layers"], case["heads"], case["head_dim"], case["page"]
        pool = _normal(gen, (2, nl, case["blocks"], page, heads, hd), dtype)
        state["pool"] = pool
        state["caches"] = [[pool[kv, layer] for layer in range(nl)] for kv in range(2)]
        state["buffer"] = _normal(gen, (2, nl, case["tokens"], heads * hd), dtype)
        state["slots"] = _slots(rng, case, device)
    elif path == "mla":
        state["cache"] = _normal(gen, (case["layers"], case["blocks"], case["page"], case["hidden"]), dtype)
        state["buffer"] = _normal(gen, (case["layers"], case["tokens"], case["hidden"]), dtype)
        state["slots"] = _slots(rng, case, device)
    elif path == "hicache":
        nl, pages, row, items = case["layers"], case["pages"], case["row"], case["items"]
        state["device_pool"] = [_normal(gen, (nl, pages, row), dtype) for _ in range(2)]
        state["page_pool"] = [torch.zeros((pages, nl, row), dtype=dtype, device=device) for _ in range(2)]
        state["src"], state["dst"] = (torch.from_numpy(rng.permutation(pages)[:items].astype(np.int64)).to(device)
                                      for _ in range(2))
    else:
        shape = (case["layers"], 2, case["tokens"], case["heads"], case["head_dim"])
        if case["encode"]:
            state["kv"] = _normal(gen, shape, dtype)
        else:
            state["codes"] = torch.randint(0, case["bins"], shape, generator=gen, device=device, dtype=torch.uint8)
            state["codebook"] = torch.linspace(-4.5 - seed % 7, 4.25, case["bins"], device=device)
    return state


# ----- one pass ---------------------------------------------------------------------------------


def run(state: dict):
    case = state["case"]
    path = case["path"]
    many = case.get("layers", 1) > 1
    if path == "store":
        call = musa_aiter.kv_linear_to_paged_multi_layer if many else musa_aiter.kv_linear_to_paged
        call(*state["linear"], *state["caches"], state["slots"])
        return state["caches"]
    if path == "load":
        call = musa_aiter.kv_paged_to_linear_multi_layer if many else musa_aiter.kv_paged_to_linear
        return call(*state["caches"], state["slots"])
    if path == "quant":
        call = musa_aiter.kv_linear_to_paged_fp8_multi_layer if many else musa_aiter.kv_linear_to_paged_fp8
        call(*state["linear"], *state["caches"], state["slots"], *state["scales"], fp8_format=case["format"])
        return state["caches"]
    if path == "dequant":
        call = musa_aiter.kv_paged_fp8_to_linear_multi_layer if many else musa_aiter.kv_paged_fp8_to_linear
        return call(*state["caches"], state["slots"], *state["scales"], out_dtype=DTYPES[case["dtype"]],
                    fp8_format=case["format"])
    if path == "dense":
        return musa_aiter.kv_load_and_reshape_flash(*state["caches"], state["tables"], state["lengths"])
    if path == "chunk":
        sizes = (case["page"], case["heads"], case["head_dim"])
        if case["store"]:
            musa_aiter.lmcache_kv_buffer_to_paged_two_x_nl(state["buffer"], state["caches"], state["slots"], 0, *sizes)
            return state["pool"]
        musa_aiter.lmcache_kv_paged_to_buffer_two_x_nl(state["caches"], state["buffer"], state["slots"], *sizes)
        return state["buffer"]
    if path == "mla":
        if case["store"]:
            musa_aiter.lmcache_kv_buffer_to_paged_mla(state["buffer"], state["cache"], state["slots"])
            return state["cache"]
        musa_aiter.lmcache_paged_to_kv_buffer_mla(state["cache"], state["buffer"], state["slots"])
        return state["buffer"]
    if path == "hicache":
        k, v = state["device_pool"]
        dst_k, dst_v = state["page_pool"]
        musa_aiter.hicache_transfer_kv_all_layer_lf_pf(k, dst_k, v, dst_v, state["src"], state["dst"])
        return state["page_pool"]
    if case["encode"]:
        return musa_aiter.kv_cachegen_encode(state["kv"], num_bins=case["bins"])
    return musa_aiter.kv_cachegen_decode(state["codes"], state["codebook"], dtype=DTYPES[case["dtype"]])


# ----- what a pass cannot do without ------------------------------------------------------------


def work(case: dict) -> dict:
    path, elt = case["path"], DTYPES[case["dtype"]].itemsize
    if path in ("store", "load", "quant", "dequant"):
        values = 2 * case["layers"] * case["tokens"] * case["heads"] * case["head_dim"]
        paged = 1 if path in ("quant", "dequant") else elt
        total = values * (elt + paged) + 8 * case["tokens"]
    elif path == "dense":
        # Rows past a sequence's length are written as zeros, not read; lengths are uniform in [lo, hi], the first hi.
        row = 2 * case["heads"] * case["head_dim"] * elt
        rows = case["seq_hi"] + (case["batch"] - 1) * (case["seq_lo"] + case["seq_hi"]) / 2
        total = row * (rows + case["batch"] * case["seq_hi"]) + 8 * rows / case["page"]
    elif path == "chunk":
        total = 4 * case["layers"] * case["tokens"] * case["heads"] * case["head_dim"] * elt + 8 * case["tokens"]
    elif path == "mla":
        total = 2 * case["layers"] * case["tokens"] * case["hidden"] * elt + 8 * case["tokens"]
    elif path == "hicache":
        total = 4 * case["layers"] * case["items"] * case["row"] * elt + 16 * case["items"]
    else:
        total = 2 * case["layers"] * case["tokens"] * case["heads"] * case["head_dim"] * (elt + 1) + 4 * case["bins"]
    return {"bytes": total, "flops": 0}


def tolerance(case: dict):
    """Copies, FP8 codes and decoded values are exact: the API promises the bits.  The CacheGen codebook and CDF
    are float32 arithmetic (one rounding per entry); the bins themselves are whole numbers and stay the same."""
    if case["path"] == "cachegen" and case["encode"]:
        return {"rel": 5e-7, "max": 5e-6, "differ": 0.0}
    return "exact"


# ----- the computed outputs in 64 bits ------------------------------------------------------------


def _decode_fp8(codes: torch.Tensor, fmt: str) -> torch.Tensor:
    """float64 values of FP8 codes: exponent field 0 is a signed zero, every other code a normal number."""
    mantissa, bias = (3, 7) if fmt == "e4m3" else (2, 15)
    c = codes.to(torch.int64)
    exponent, fraction = (c & 0x7F) >> mantissa, c & ((1 << mantissa) - 1)
    value = torch.ldexp(1.0 + fraction.double() / (1 << mantissa), (exponent - bias).double())
    return torch.where(exponent == 0, 0.0, value) * torch.where(c >= 128, -1.0, 1.0)


def exact(case: dict, seed: int):
    path = case["path"]
    if path == "dequant":
        state = prepare(case, seed)
        many = case["layers"] > 1
        out = []
        for cache, scale in zip(state["caches"], state["scales"]):
            cache = cache if many else cache.unsqueeze(0)
            rows = cache.permute(0, 1, 4, 2, 3).reshape(cache.shape[0], -1, case["heads"], case["head_dim"])
            value = _decode_fp8(rows[:, state["slots"].clamp(min=0)], case["format"])
            factor = scale.double()
            factor = factor[:, None, :, None] if factor.dim() == 2 else factor[:, None] if factor.dim() == 1 else factor
            value = value * factor * (state["slots"] >= 0)[None, :, None, None]
            out.append(value if many else value[0])
        return tuple(out)
    if path == "cachegen" and case["encode"]:
        x = prepare(case, seed)["kv"].double()
        lo, hi, bins = x.min(), x.max(), case["bins"]
        index = ((x - lo) * ((bins - 1) / (hi - lo))).round().clamp(0, bins - 1).to(torch.int64)
        counts = torch.bincount(index.reshape(-1), minlength=bins).double()
        steps = torch.arange(bins, device=x.device, dtype=torch.float64) / (bins - 1)
        cdf = torch.cat([torch.zeros(1, device=x.device, dtype=torch.float64), counts.cumsum(0) / x.numel()])
        return None, lo + (hi - lo) * steps, cdf
    if path == "cachegen":
        state = prepare(case, seed)
        return state["codebook"].double()[state["codes"].to(torch.int64)]
    return None
