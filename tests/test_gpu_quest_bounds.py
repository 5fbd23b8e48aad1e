"""Quest page bounds over a prompt's pages (``paged_page_bounds``, ``QuestState.refresh``) where the packed reduction
can go wrong: every head dim it has an instance for and ones it has not, pages of several cache pages, more cache pages
than one window of the block table, rows of different lengths, signed zeros (-0 below +0), infinities and NaN (which the
minimum and maximum skip), missing pages (left untouched) and bounds at an odd element offset. Exact: the bounds' bits."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

B, HKV = 2, 3


def _cache(dtype, dim: int, pages: int, seed: int):
    """A cache of special and random keys, its block table (one missing page) and the keys ``[B, H, S, D]``."""
    from economize_amd.paged import PagedKVCache

    gen = torch.Generator().manual_seed(seed)
    x = 16 // torch.empty((), dtype=dtype).element_size()
    total = B * pages + 3
    keys = torch.randn(total, HKV, dim // x, 16, x, generator=gen)
    at = torch.rand(keys.shape, generator=gen)
    for k, special in enumerate((0.0, -0.0, 448.0, -448.0, 1e-3, -1e-3)):
        keys = torch.where((at > 0.01 * k) & (at < 0.01 * (k + 1)), torch.tensor(special), keys)
    # every fourth page has a zero of some sign for its minimum in most channels, the next one for its maximum
    zeros = torch.where(torch.rand(keys.shape, generator=gen) < 0.5, 0.0, -0.0)
    halves = torch.where(torch.rand(keys.shape, generator=gen) < 0.3, zeros, keys.abs())
    kind = (torch.arange(total) % 4).view(-1, 1, 1, 1, 1)
    keys = torch.where(kind == 1, halves, torch.where(kind == 2, -halves, keys))
    # pages 0 .. total / 2 carry NaN of both signs, the others none
    nan = (at > 0.995) & (torch.arange(total) < total // 2).view(-1, 1, 1, 1, 1)
    stored = keys.to(dtype)
    raw = stored.view(torch.int16 if dtype == torch.bfloat16 else torch.uint8)
    pos, neg = {torch.bfloat16: (0x7FC0, -0x40), torch.float8_e4m3fn: (0x7F, 0xFF), torch.float8_e5m2: (0x7E, 0xFE)}[dtype]
    raw[nan & (keys > 0)] = pos
    raw[nan & (keys <= 0)] = neg
    if dtype != torch.float8_e4m3fn:  # a whole channel of NaN and infinities of both signs
        raw[0, :, 0, :, 0] = pos
        stored[1, :, 0, 3, 1], stored[1, :, 0, 5, 1] = float("inf"), float("-inf")
    table = torch.randperm(total, generator=gen)[: B * pages].view(B, pages).to(torch.int32)
    dense = stored.float()[table.long()]  # [B, pages, H, runs, 16, X]
    dense = dense.permute(0, 2, 1, 4, 3, 5).reshape(B, HKV, pages * 16, dim)
    table[1, pages // 2] = -1
    cache = PagedKVCache.empty(total, HKV, dim, dtype, "cuda")
    cache.keys.copy_(stored)
    return cache, table.cuda(), dense.numpy()


def _ordered(bits: np.ndarray) -> np.ndarray:
    return bits ^ ((bits >> 15) & np.int16(0x7FFF))


def _expected(dense: np.ndarray, table: np.ndarray, quest_page: int, q0: int, q1: int):
    """bf16 bits of the bounds of Quest pages [q0, q1), the infinities of no key where all are NaN, and which pages are
    held. The minimum and maximum are those of the bits as int16 in the order of the floats (the map is its inverse)."""
    span = quest_page // 16
    x = dense[:, :, q0 * quest_page: q1 * quest_page].reshape(B, HKV, q1 - q0, quest_page, -1)
    held = (table[:, q0 * span: q1 * span].reshape(B, q1 - q0, span) >= 0).all(axis=2)
    bits = (x.view(np.uint32) >> 16).astype(np.uint16).view(np.int16)  # the keys are bf16 values
    ordered = _ordered(bits)
    top = np.int16(0x7F80)  # infinity; its negative's place is ~top
    lo = np.where(np.isnan(x), top, ordered).min(axis=3)
    hi = np.where(np.isnan(x), ~top, ordered).max(axis=3)
    return _ordered(lo), _ordered(hi), held[:, None, :, None]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize(("dim", "quest_page", "quest_pages"), [(128, 16, 150), (128, 64, 37), (64, 16, 65),
                                                                (64, 32, 40), (256, 16, 9), (192, 16, 33),
                                                                (128, 1024, 2), (128, 2048, 1), (128, 16, 1)])
def test_bounds_of_a_prompt(dtype, dim, quest_page, quest_pages) -> None:
    from economize_amd.quest import QuestState, paged_page_bounds

    pages = quest_pages * quest_page // 16
    cache, table, dense = _cache(dtype, dim, pages, seed=dim + quest_page + quest_pages)
    want = _expected(dense, table.cpu().numpy(), quest_page, 0, quest_pages)

    def check(kmin, kmax, limit=(quest_pages, quest_pages)):
        lo, hi, held = want
        for b, n in enumerate(limit):
            for got, ref in ((kmin, lo), (kmax, hi)):
                ref = np.where(held[b], ref[b], np.int16(0))[:, :n]
                np.testing.assert_array_equal(got[b, :, :n].view(torch.int16).cpu().numpy(), ref)

    check(*paged_page_bounds(cache, table, 0, quest_pages, quest_page))
    # into bounds that start at an odd element: 2-byte stores only
    flat = torch.zeros(2, B * HKV * quest_pages * dim + 1, dtype=torch.bfloat16, device="cuda")
    out = tuple(f[1:].view(B, HKV, quest_pages, dim) for f in flat)
    paged_page_bounds(cache, table, 0, quest_pages, quest_page, out=out)
    check(*out)
    # kept on the device: rows of different lengths, a first step and the rest of the prompt
    state = QuestState(B, HKV, dim, quest_pages, quest_page, 4, "cuda")
    for committed in ([quest_page * quest_pages // 3, quest_page - 1], [quest_page * quest_pages - 1, 10 ** 6]):
        state.refresh(cache, table, torch.tensor(committed, dtype=torch.int32, device="cuda"))
        done = [min(c // quest_page, quest_pages) for c in committed]
        assert state.done.tolist() == done
        check(state.kmin, state.kmax, done)
        for b, n in enumerate(done):
            assert not state.kmin[b, :, n:].any() and not state.kmax[b, :, n:].any()
