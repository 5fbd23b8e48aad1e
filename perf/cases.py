"""The timed cases of the compressed-KV decode path: what a serving program asks of this package, layer by layer.

A case is one call (or the few calls that belong together) of one layer, at the sizes of a model in use: the prompt
pass that fills a compressed cache (fp8 append, dense fp8 encode, KIVI quantization with its ring, Quest page bounds)
and the decode pass that attends over it (paged fp8, KIVI, Quest, dense buffers, vLLM's KIVI cells), from one short
request to a full batch. ``listed()`` gives the fixed cases, ``draw(rng)`` more of the same ranges, ``prepare`` what a
program holds before the call, ``run`` the call, ``work`` the bytes and operations no implementation can avoid,
``exact`` the same outputs in 64 bits from plain torch, ``tolerance`` how far a correct implementation may be from
another.

K and V are N(0, 1) (KIVI's with 4 outlier key channels ten times larger, Quest's with planted pages near the query),
in the page order of a shuffled pool. Row lengths spread evenly over [len_lo, len_hi].
"""

from __future__ import annotations

import math

import torch

from economize_amd.decode import decode_attention
from economize_amd.fp8 import fp8_encode
from economize_amd.kivi import KIVI_PAGE, PagedKIVICache, kivi_append, kivi_decode_attention, kivi_quantize
from economize_amd.paged import PAGE, PagedKVCache, head_scales, paged_append, paged_decode_attention
from economize_amd.quest import QuestState, paged_quest_decode_attention
from economize_amd.vllm_kivi import cell_layout, paged_kivi_attention, quantize_committed

DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32, "e4m3": torch.float8_e4m3fn,
          "e5m2": torch.float8_e5m2}
RESIDUAL, HEADROOM, GROUP = 128, 256, 32  # KIVI's defaults here
CELL_PAGE = 32  # tokens per page of vLLM's cache


def _case(kind: str, batch: int, len_lo: int, len_hi: int, heads: tuple[int, int], dim: int, **more) -> dict:
    return {"kind": kind, "batch": batch, "len_lo": len_lo, "len_hi": len_hi, "q_heads": heads[0],
            "kv_heads": heads[1], "dim": dim, "queries": 1, **more}


def listed() -> list[dict]:
    gqa = (32, 8)
    cases = [
        # the first tokens of one short request on a small model: launch and host time
        ("fp8_decode_one", _case("fp8_decode", 1, 512, 512, (8, 2), 64, kv="e4m3", q="bf16")),
        # a full decoding batch at equal lengths: the headline shape
        ("fp8_decode_batch", _case("fp8_decode", 32, 4096, 4096, gqa, 128, kv="e4m3", q="bf16")),
        # a serving batch whose requests are at all stages
        ("fp8_decode_ragged", _case("fp8_decode", 32, 1024, 8192, gqa, 128, kv="e4m3", q="bf16")),
        # a prompt pass written to the paged fp8 cache
        ("fp8_prompt_append", _case("fp8_append", 8, 4096, 4096, gqa, 128, kv="e4m3", q="bf16")),
        # a prompt pass into dense fp8 buffers with a scale per token (FP8KVConfig(scale="token"))
        ("fp8_prompt_encode", _case("fp8_encode", 8, 4096, 4096, gqa, 128, kv="e4m3", q="bf16")),
        # long-context decode over 2-bit codes
        ("kivi2_decode_batch", _case("kivi_decode", 16, 8192, 8192, gqa, 128, bits=2)),
        # speculative decoding: 8 draft tokens verified at once over 4-bit codes
        ("kivi4_verify", {**_case("kivi_decode", 64, 1024, 4096, (64, 8), 128, bits=4), "queries": 8}),
        # a prompt pass quantized to 4-bit codes, its newest tokens in the rings
        ("kivi4_prompt", _case("kivi_prompt", 8, 4096, 4096, gqa, 128, bits=4)),
        # one page-sparse decode step: append, selection, attention over the selected pages
        ("quest_step", _case("quest_step", 8, 32768, 32768, gqa, 128, pages=63)),
        # the page bounds of a long prompt, computed when its decoding begins
        ("quest_prompt_bounds", _case("quest_bounds", 8, 32768, 32768, gqa, 128, pages=63)),
        # decode over a model's own dense cache
        ("dense_decode_bf16", _case("dense_decode", 32, 4096, 4096, gqa, 128, kv="bf16", q="bf16", padded=False)),
        # decode over vLLM's KIVI cells
        ("cells2_decode", _case("cells_decode", 16, 8192, 8192, gqa, 128, bits=2)),
    ]
    return [{"name": name, **case} for name, case in cases]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    """A case of one of the listed kinds: batch and length over the logarithm of their range, the tokens at most the
    listed case's."""
    kind = rng.choice(("fp8_decode", "fp8_append", "fp8_encode", "kivi_decode", "kivi_prompt", "quest_step",
                       "quest_bounds", "dense_decode", "cells_decode"))
    most_batch, longest, tokens = {
        "fp8_decode": (64, 32768, 1 << 17), "fp8_append": (32, 8192, 1 << 15), "fp8_encode": (32, 8192, 1 << 15),
        "kivi_decode": (64, 32768, 1 << 17), "kivi_prompt": (16, 8192, 1 << 15), "quest_step": (16, 65536, 1 << 18),
        "quest_bounds": (16, 65536, 1 << 18), "dense_decode": (64, 32768, 1 << 17),
        "cells_decode": (32, 32768, 1 << 17)}[kind]
    shortest = {"fp8_append": 1, "fp8_encode": 1, "quest_step": 2048, "quest_bounds": 1024, "kivi_prompt": 257}
    batch = _log_int(rng, 1, most_batch)
    hi = _log_int(rng, shortest.get(kind, 64), max(shortest.get(kind, 64) + 1, min(longest, tokens // batch)))
    lo = hi
    if kind in ("fp8_decode", "kivi_decode", "cells_decode") and rng.random() < 0.5:
        lo = max(1, hi // rng.choice((2, 4, 8)))
    heads = rng.choice(((32, 8), (28, 4), (64, 8), (16, 8)))
    case = _case(kind, batch, lo, hi, heads, 128)
    if heads[0] > 32 and hi * batch > tokens // 2:
        case["q_heads"] = 32
    if kind in ("fp8_decode", "fp8_append", "fp8_encode"):
        case.update(dim=rng.choice((64, 128)), kv=rng.choice(("e4m3", "e4m3", "e5m2")),
                    q=rng.choice(("bf16", "bf16", "fp16")))
    elif kind == "kivi_decode":
        queries = rng.choice((1, 1, 2, 5, 8))
        case.update(dim=rng.choice((64, 128, 128)), bits=rng.choice((2, 4)), queries=queries,
                    len_lo=max(lo, queries))
    elif kind == "kivi_prompt":
        case.update(dim=rng.choice((64, 128, 128)), bits=rng.choice((2, 4)))
    elif kind in ("quest_step", "quest_bounds"):
        case.update(pages=rng.choice((31, 63, 127)))
    elif kind == "dense_decode":
        q = rng.choice(("bf16", "bf16", "fp16"))
        case.update(dim=rng.choice((64, 128)), q=q, kv=rng.choice((q, q, "e4m3")), padded=rng.random() < 0.25)
    else:
        case.update(bits=rng.choice((2, 4)))
    return case


# ---- inputs ---------------------------------------------------------------------------------------------------


def _lens(case: dict) -> list[int]:
    """Row lengths spread evenly over [len_lo, len_hi], in an order that puts neighbours far apart."""
    lo, hi, batch = case["len_lo"], case["len_hi"], case["batch"]
    golden = (math.sqrt(5) - 1) / 2
    return [lo + round((hi - lo) * ((i + 1) * golden % 1.0)) for i in range(batch - 1)] + [hi]


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _int32(values) -> torch.Tensor:
    return torch.tensor(values, dtype=torch.int32, device=DEVICE)


def _query(case: dict, gen, dtype: torch.dtype) -> torch.Tensor:
    """The query states ``[B, Q, Hq, D]``, as a projection leaves them."""
    return torch.randn(case["batch"], case["queries"], case["q_heads"], case["dim"], generator=gen,
                       device=DEVICE).to(dtype)


def _kv(case: dict, gen, dtype: torch.dtype, outliers: bool = False) -> tuple[torch.Tensor, torch.Tensor]:
    """Key and value states ``[B, Hkv, S, D]``."""
    shape = (case["batch"], case["kv_heads"], max(_lens(case)), case["dim"])
    k = torch.randn(shape, generator=gen, device=DEVICE)
    if outliers:
        k[..., torch.randperm(case["dim"], generator=gen, device=DEVICE)[:4]] *= 10.0
    v = torch.randn(shape, generator=gen, device=DEVICE)
    return k.to(dtype), v.to(dtype)


def _table(case: dict, gen, page: int) -> tuple[torch.Tensor, int]:
    """Block table ``[B, pages per row]`` over a shuffled pool, and the pool's pages."""
    per_row = [-(-n // page) for n in _lens(case)]
    order = torch.randperm(sum(per_row) + 3, generator=gen, device=DEVICE).to(torch.int32)
    table = torch.full((case["batch"], max(per_row)), -1, dtype=torch.int32, device=DEVICE)
    at = 0
    for b, n in enumerate(per_row):
        table[b, :n] = order[at: at + n]
        at += n
    return table, sum(per_row) + 3


def _slots(table: torch.Tensor, lens: list[int], page: int) -> torch.Tensor:
    """``[B * S]`` cache slots of every row's tokens, -1 past its length."""
    t = torch.arange(max(lens), device=DEVICE)
    slots = table[:, t // page] * page + (t % page).to(torch.int32)
    return torch.where(t[None, :] < _int32(lens)[:, None], slots, -1).to(torch.int32).reshape(-1)


def _token_major(x: torch.Tensor) -> torch.Tensor:
    """``[B, H, S, D]`` states as ``[B * S, H, D]`` tokens."""
    return x.transpose(1, 2).reshape(-1, x.shape[1], x.shape[3])


def _kivi_counts(lens: list[int], queries: int) -> tuple[list[int], list[int]]:
    """Quantized keys and values of rows whose last ``queries`` tokens are this pass's."""
    committed = [n - queries for n in lens]
    return [c // RESIDUAL * RESIDUAL for c in committed], [max(0, c - RESIDUAL) for c in committed]


# ---- prepare --------------------------------------------------------------------------------------------------


def _prepare_fp8_decode(case: dict, gen) -> dict:
    lens = _lens(case)
    q = _query(case, gen, DTYPES[case["q"]])
    k, v = _kv(case, gen, DTYPES[case["q"]])
    table, pages = _table(case, gen, PAGE)
    cache = PagedKVCache.empty(pages, case["kv_heads"], case["dim"], DTYPES[case["kv"]], DEVICE,
                               head_scales(k, DTYPES[case["kv"]]), head_scales(v, DTYPES[case["kv"]]))
    paged_append(cache, _token_major(k), _token_major(v), _slots(table, lens, PAGE))
    return {"q": q, "cache": cache, "table": table, "lens": _int32(lens), "longest": max(lens)}


def _prepare_fp8_append(case: dict, gen) -> dict:
    k, v = _kv(case, gen, DTYPES[case["q"]])
    table, pages = _table(case, gen, PAGE)
    cache = PagedKVCache.empty(pages, case["kv_heads"], case["dim"], DTYPES[case["kv"]], DEVICE,
                               head_scales(k, DTYPES[case["kv"]]), head_scales(v, DTYPES[case["kv"]]))
    return {"k": _token_major(k), "v": _token_major(v), "slots": _slots(table, _lens(case), PAGE), "cache": cache}


def _prepare_fp8_encode(case: dict, gen) -> dict:
    k, v = _kv(case, gen, DTYPES[case["q"]])
    dtype = DTYPES[case["kv"]]
    return {"k": k, "v": v, "dtype": dtype, "codes": (torch.zeros(k.shape, dtype=dtype, device=DEVICE),
                                                       torch.zeros(v.shape, dtype=dtype, device=DEVICE)),
            "scales": (torch.zeros(k.shape[:3], device=DEVICE), torch.zeros(v.shape[:3], device=DEVICE))}


def _kivi_state(case: dict, gen) -> dict:
    lens = _lens(case)
    k, v = _kv(case, gen, torch.bfloat16, outliers=True)
    table, pages = _table(case, gen, KIVI_PAGE)
    cache = PagedKIVICache.empty(pages, case["batch"], case["kv_heads"], case["dim"], case["bits"], DEVICE,
                                 residual=RESIDUAL, headroom=HEADROOM)
    kq, vq = _kivi_counts(lens, 0 if case["kind"] == "kivi_prompt" else case["queries"])
    ring = cache.ring
    rows = torch.cat([torch.full((min(n, ring),), b) for b, n in enumerate(lens)]).to(DEVICE)
    at = torch.cat([torch.arange(max(0, n - ring), n) for n in lens]).to(DEVICE)
    return {"cache": cache, "table": table, "k": k, "v": v, "zero": _int32([0] * len(lens)), "kq": _int32(kq),
            "vq": _int32(vq), "most": (max(kq), max(vq)), "k_new": k[rows, :, at], "v_new": v[rows, :, at],
            "rows": rows.to(torch.int32), "at": at.to(torch.int32)}


def _kivi_fill(s: dict) -> None:
    """A prompt pass of the KIVI cache: the committed tokens quantized, the newest into the rings."""
    kivi_quantize(s["cache"], s["table"], s["k"], "k", s["zero"], s["kq"], s["most"][0])
    kivi_quantize(s["cache"], s["table"], s["v"], "v", s["zero"], s["vq"], s["most"][1])
    kivi_append(s["cache"], s["k_new"], s["v_new"], s["rows"], s["at"])


def _prepare_kivi_decode(case: dict, gen) -> dict:
    q = _query(case, gen, torch.bfloat16)
    s = _kivi_state(case, gen)
    _kivi_fill(s)
    s["cache"].keys_quantized.copy_(s["kq"])
    s["cache"].values_quantized.copy_(s["vq"])
    return {"q": q, "cache": s["cache"], "table": s["table"], "lens": _int32(_lens(case)),
            "longest": case["len_hi"]}


def _quest_inputs(case: dict, gen) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Query, keys and values; half of the budget's pages per KV head hold keys near its group's first query."""
    q = _query(case, gen, torch.bfloat16)
    batch, heads, dim, length = case["batch"], case["kv_heads"], case["dim"], case["len_hi"]
    k, v = _kv(case, gen, torch.bfloat16)
    whole = length // PAGE
    planted = min(case["pages"] // 2, whole - 1)
    picks = torch.rand(batch, heads, whole, generator=gen, device=DEVICE).topk(planted, dim=2).indices
    at = (picks[..., None] * PAGE + torch.arange(PAGE, device=DEVICE)).flatten(2)
    near = q[:, 0, :: case["q_heads"] // heads].float()[:, :, None, :]
    noise = 0.1 * torch.randn(batch, heads, planted * PAGE, dim, generator=gen, device=DEVICE)
    k.scatter_(2, at[..., None].expand(-1, -1, -1, dim), (near + noise).to(torch.bfloat16))
    return q, k, v


def _prepare_quest(case: dict, gen) -> dict:
    q, k, v = _quest_inputs(case, gen)
    lens = _lens(case)
    table, pages = _table(case, gen, PAGE)
    cache = PagedKVCache.empty(pages, case["kv_heads"], case["dim"], torch.bfloat16, DEVICE)
    paged_append(cache, _token_major(k), _token_major(v), _slots(table, lens, PAGE))
    committed = _int32([n - 1 for n in lens])  # the last token is the step's own
    state = QuestState(case["batch"], case["kv_heads"], case["dim"], table.shape[1], PAGE, case["pages"], DEVICE)
    state.refresh(cache, table, committed)
    last = case["len_hi"] - 1
    return {"q": q.transpose(1, 2), "cache": cache, "table": table, "lens": _int32(lens), "longest": max(lens),
            "committed": committed, "state": state, "k_new": k[:, :, last].contiguous(),
            "v_new": v[:, :, last].contiguous(),
            "slots": (table[:, last // PAGE] * PAGE + last % PAGE).contiguous()}


def _dense_mask(case: dict) -> torch.Tensor | None:
    """Left padding of a batch of prompts: row ``b`` hides its first ``b * S / (2 B)`` slots."""
    if not case["padded"]:
        return None
    hidden = torch.arange(case["batch"], device=DEVICE) * case["len_hi"] // (2 * case["batch"])
    return (torch.arange(case["len_hi"], device=DEVICE)[None, :] >= hidden[:, None])[:, None, None, :]


def _prepare_dense_decode(case: dict, gen) -> dict:
    q = _query(case, gen, DTYPES[case["q"]])
    k, v = _kv(case, gen, DTYPES[case["q"]])
    return {"q": q.transpose(1, 2), "k": k.to(DTYPES[case["kv"]]), "v": v.to(DTYPES[case["kv"]]),
            "mask": _dense_mask(case), "scale": case["dim"] ** -0.5}


def _prepare_cells_decode(case: dict, gen) -> dict:
    lens = _lens(case)
    q = _query(case, gen, torch.bfloat16)
    k, v = _kv(case, gen, torch.bfloat16)
    table, pages = _table(case, gen, CELL_PAGE)
    layout = cell_layout(case["dim"], torch.bfloat16, case["bits"], GROUP)
    cells = torch.zeros(pages, case["kv_heads"], CELL_PAGE, layout.size // 2, dtype=torch.bfloat16, device=DEVICE)
    kv = torch.cat([k, v], dim=3)
    t = torch.arange(max(lens), device=DEVICE)
    for b, n in enumerate(lens):
        cells[table[b, t[:n] // CELL_PAGE].long(), :, t[:n] % CELL_PAGE, : 2 * case["dim"]] = kv[b, :, :n].transpose(0, 1)
    starts = torch.arange(case["batch"] + 1, dtype=torch.int32, device=DEVICE)
    quantize_committed(cells, layout, RESIDUAL, table, starts, _int32(lens), _int32([0] * len(lens)))
    return {"q": q[:, 0].contiguous(), "cells": cells, "layout": layout, "table": table, "starts": starts,
            "lens": _int32(lens), "longest": max(lens)}


# ---- run ------------------------------------------------------------------------------------------------------


def _run_fp8_decode(s: dict):
    return paged_decode_attention(s["q"], s["cache"], s["table"], s["lens"], s["longest"])


def _run_fp8_append(s: dict):
    cache = s["cache"]
    paged_append(cache, s["k"], s["v"], s["slots"])
    return {"keys": cache.keys.view(torch.uint8), "values": cache.values.view(torch.uint8)}


def _run_fp8_encode(s: dict):
    codes = []
    for x, out, scale in zip((s["k"], s["v"]), s["codes"], s["scales"]):
        codes.append(fp8_encode(x, s["dtype"], out=out, token_scale=scale).view(torch.uint8))
    return {"codes": codes, "scales": list(s["scales"])}


def _run_kivi_decode(s: dict):
    return kivi_decode_attention(s["q"], s["cache"], s["table"], s["lens"], s["longest"])


def _run_kivi_prompt(s: dict):
    _kivi_fill(s)
    cache = s["cache"]
    return {"blocks": cache.blocks, "k_ring": cache.k_ring, "v_ring": cache.v_ring}


def _run_quest_step(s: dict):
    s["state"].append(s["cache"], s["k_new"], s["v_new"], s["slots"], s["table"], s["committed"])
    handle = s["state"].pages_handle()
    index = handle.select(s["q"])
    out = paged_quest_decode_attention(s["q"], s["cache"], s["table"], s["lens"], s["longest"], handle, index=index)
    return {"out": out, "index": index}


def _run_quest_bounds(s: dict):
    state = s["state"]
    state.reset()
    state.refresh(s["cache"], s["table"], s["committed"])
    return {"kmin": state.kmin, "kmax": state.kmax, "done": state.done}


def _run_dense_decode(s: dict):
    return decode_attention(s["q"], s["k"], s["v"], s["mask"], s["scale"])


def _run_cells_decode(s: dict):
    return paged_kivi_attention(s["q"], s["cells"], s["layout"], s["table"], s["starts"], s["lens"], 1, s["longest"])


_PREPARE = {"fp8_decode": _prepare_fp8_decode, "fp8_append": _prepare_fp8_append, "fp8_encode": _prepare_fp8_encode,
            "kivi_decode": _prepare_kivi_decode, "kivi_prompt": _kivi_state, "quest_step": _prepare_quest,
            "quest_bounds": _prepare_quest, "dense_decode": _prepare_dense_decode,
            "cells_decode": _prepare_cells_decode}
_RUN = {"fp8_decode": _run_fp8_decode, "fp8_append": _run_fp8_append, "fp8_encode": _run_fp8_encode,
        "kivi_decode": _run_kivi_decode, "kivi_prompt": _run_kivi_prompt, "quest_step": _run_quest_step,
        "quest_bounds": _run_quest_bounds, "dense_decode": _run_dense_decode, "cells_decode": _run_cells_decode}


def prepare(case: dict, seed: int) -> dict:
    return {**_PREPARE[case["kind"]](case, _gen(seed)), "kind": case["kind"]}


def run(state: dict):
    return _RUN[state["kind"]](state)


# ---- work -----------------------------------------------------------------------------------------------------


def work(case: dict) -> dict:
    kind, d, hkv, lens = case["kind"], case["dim"], case["kv_heads"], _lens(case)
    tokens = sum(lens)
    vectors = tokens * hkv * d  # elements of K (as many of V)
    attend = 2 * 2 * case["q_heads"] * case["queries"] * d  # flops per key
    qo = 2 * case["batch"] * case["queries"] * case["q_heads"] * d * 2
    kq, vq = _kivi_counts(lens, 0 if kind == "kivi_prompt" else case["queries"])
    codes = d * case.get("bits", 0) // 8 + 4 * d // GROUP  # codes, scale and zero-point share of a quantized token
    if kind == "fp8_decode":
        return {"bytes": 2 * vectors + qo + 4 * (tokens // PAGE), "flops": attend * tokens}
    if kind in ("fp8_append", "fp8_encode"):
        scales = 2 * 4 * tokens * hkv if kind == "fp8_encode" else 4 * tokens
        return {"bytes": 2 * vectors * (2 + 1) + scales, "flops": 2 * vectors}
    if kind in ("kivi_decode", "cells_decode"):
        kept = sum(2 * n - a - b for n, a, b in zip(lens, kq, vq))
        return {"bytes": hkv * (codes * (sum(kq) + sum(vq)) + 2 * d * kept) + qo, "flops": attend * tokens}
    if kind == "kivi_prompt":
        ring = sum(min(n, RESIDUAL + HEADROOM) for n in lens)
        moved = 2 * d * (sum(kq) + sum(vq)) + codes * (sum(kq) + sum(vq)) + 2 * ring * 2 * 2 * d
        return {"bytes": hkv * moved, "flops": 4 * vectors}
    done = sum((n - 1) // PAGE for n in lens)
    bounds = done * hkv * 2 * d * 2
    if kind == "quest_bounds":
        return {"bytes": done * PAGE * hkv * d * 2 + bounds, "flops": 2 * done * PAGE * hkv * d}
    if kind == "quest_step":
        read = sum(min(case["pages"], (n - 1) // PAGE) * PAGE + n - (n - 1) // PAGE * PAGE for n in lens)
        return {"bytes": bounds + read * hkv * 2 * d * 2 + qo, "flops": attend * read + 4 * done * hkv * d}
    size = 1 if case["kv"] in ("e4m3", "e5m2") else 2
    return {"bytes": 2 * vectors * size + qo, "flops": attend * tokens}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------


def _fp8_scale(x: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    """fp32 ``[1, H, 1, 1]``: absmax over the format's maximum."""
    return (x.float().abs().amax(dim=(0, 2, 3)) / torch.full((), torch.finfo(dtype).max, device=DEVICE))[None, :, None,
                                                                                                          None]


def _fp8_round_trip(x: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    scale = _fp8_scale(x, dtype)
    top = torch.finfo(dtype).max
    return (x.float() / scale).clamp(-top, top).to(dtype).double() * scale.double()


def _kivi_round_trip(x: torch.Tensor, bits: int, axis: int) -> torch.Tensor:
    """``x`` ``[H, T, D]`` quantized in groups of 32 along ``axis`` (1: tokens, 2: channels) and dequantized to the
    model's dtype: fp32 minimum and maximum, scale and zero point rounded to fp16, codes rounded half to even."""
    levels = torch.full((), float(2 ** bits - 1), device=DEVICE)
    g = x.float().unflatten(axis, (-1, GROUP))
    low, high = g.amin(dim=axis + 1, keepdim=True), g.amax(dim=axis + 1, keepdim=True)
    scale = ((high - low) / levels).half().float()
    zero = low.half().float()
    code = ((g - zero) / torch.where(scale > 0, scale, 1.0)).round().clamp(0, 2 ** bits - 1)
    return (code * scale + zero).flatten(axis, axis + 1).to(x.dtype)


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, hide: torch.Tensor | None) -> torch.Tensor:
    """``[Q, Hq, D]`` in 64 bits: q ``[Q, Hq, D]`` over k, v ``[Hkv, S, D]``; ``hide`` ``[Hkv or 1, Q or 1, S]``."""
    queries, q_heads, dim = q.shape
    kv_heads = k.shape[0]
    qg = q.double().view(queries, kv_heads, q_heads // kv_heads, dim).permute(1, 2, 0, 3)  # [Hkv, G, Q, D]
    scores = torch.matmul(qg.reshape(kv_heads, -1, dim), k.double().transpose(1, 2).contiguous()) / math.sqrt(dim)
    scores = scores.view(kv_heads, -1, queries, k.shape[1])
    if hide is not None:
        scores = scores.masked_fill(hide[:, None], -math.inf)
    p = scores.softmax(dim=3).reshape(kv_heads, -1, k.shape[1])
    out = torch.matmul(p, v.double().contiguous()).view(kv_heads, -1, queries, dim)
    return out.permute(2, 0, 1, 3).reshape(queries, q_heads, dim)


def _causal(queries: int, keys: int) -> torch.Tensor | None:
    if queries == 1:
        return None
    at = torch.arange(keys, device=DEVICE)
    return (at[None, :] > keys - queries + torch.arange(queries, device=DEVICE)[:, None])[None]


def exact(case: dict, seed: int):
    gen, kind, lens = _gen(seed), case["kind"], _lens(case)
    if kind in ("fp8_append", "kivi_prompt"):
        return None  # codes and copies: whole values
    if kind == "fp8_encode":
        top = torch.finfo(DTYPES[case["kv"]]).max
        scales = [(x.double().abs().amax(dim=3) / top).clamp(min=1e-12) for x in _kv(case, gen, DTYPES[case["q"]])]
        return {"codes": [None, None], "scales": scales}
    if kind in ("fp8_decode", "dense_decode"):
        q = _query(case, gen, DTYPES[case["q"]])
        k, v = _kv(case, gen, DTYPES[case["q"]])
        kv = DTYPES[case["kv"]]
        if kind == "dense_decode":
            k, v, mask = k.to(kv), v.to(kv), _dense_mask(case)
            rows = [_attend(q[b], k[b], v[b], None if mask is None else ~mask[b]) for b in range(len(lens))]
        else:
            k, v = _fp8_round_trip(k, kv), _fp8_round_trip(v, kv)
            rows = [_attend(q[b], k[b, :, :n], v[b, :, :n], None) for b, n in enumerate(lens)]
        return torch.stack(rows)
    if kind in ("kivi_decode", "cells_decode"):
        q = _query(case, gen, torch.bfloat16)
        k, v = _kv(case, gen, torch.bfloat16, outliers=kind == "kivi_decode")
        rows = []
        for b, (n, kq, vq) in enumerate(zip(lens, *_kivi_counts(lens, case["queries"]))):
            kb, vb = k[b, :, :n].clone(), v[b, :, :n].clone()
            if kq:
                kb[:, :kq] = _kivi_round_trip(kb[:, :kq], case["bits"], 1)
            if vq:
                vb[:, :vq] = _kivi_round_trip(vb[:, :vq], case["bits"], 2)
            rows.append(_attend(q[b], kb, vb, _causal(case["queries"], n)))
        out = torch.stack(rows)
        return out[:, 0] if kind == "cells_decode" else out
    q, k, v = _quest_inputs(case, gen)
    done = (case["len_hi"] - 1) // PAGE
    pages = k[:, :, : done * PAGE].unflatten(2, (done, PAGE))
    low, high = pages.amin(dim=3), pages.amax(dim=3)
    if kind == "quest_bounds":
        pad = (0, 0, 0, -(-case["len_hi"] // PAGE) - done)
        return {"kmin": torch.nn.functional.pad(low.double(), pad), "kmax": torch.nn.functional.pad(high.double(), pad),
                "done": None}
    rows = []
    for b in range(len(lens)):
        qg = q[b, 0].double().view(case["kv_heads"], -1, case["dim"])
        score = torch.matmul((low[b].double() + high[b].double()) / 2, qg.sum(dim=1)[:, :, None]) + \
            torch.matmul((high[b].double() - low[b].double()) / 2, qg.abs().sum(dim=1)[:, :, None])
        index = score[..., 0].topk(min(case["pages"], done), dim=1).indices
        hide = torch.ones(case["kv_heads"], done, dtype=torch.bool, device=DEVICE).scatter_(1, index, False)
        hide = hide.repeat_interleave(PAGE, dim=1)
        hide = torch.nn.functional.pad(hide, (0, case["len_hi"] - done * PAGE))
        rows.append(_attend(q[b], k[b], v[b], hide[:, None, :]))
    return {"out": torch.stack(rows), "index": None}


def tolerance(case: dict):
    if case["kind"] in ("fp8_append", "fp8_encode", "kivi_prompt", "quest_bounds"):
        return "exact"  # codes, scales and bounds
    # one rounding of the output to 16 bits and softmax weights of at least 11: bf16 outputs lie 1.7e-3 from the 64-bit
    # result, fp16 ones an eighth of that plus the weights' share
    return {"rel": 1.5e-3, "max": 1e-2} if case.get("q") == "fp16" else {"rel": 6e-3, "max": 3e-2}
