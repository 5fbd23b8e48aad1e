"""Appends by windows of 16 tokens (the paged fp8 / bf16 cache and the KIVI rings, 16-bit states with aligned channels)
against the kernels that take any states one token per workgroup: aligned prompts, prompts that start or end within a
page, pages in any order, padding, single tokens, reversed and gapped slots, several rows, NaN and values beyond the
corrected quotient's limits; calls of one wave per workgroup, keys and values apart, and of four waves. Exact: whole bytes."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

PAGES = 12


def _slots(kind: str) -> list[int]:
    gen = torch.Generator().manual_seed(len(kind))
    pages = torch.randperm(PAGES, generator=gen).tolist()
    at = [pages[t // 16] * 16 + t % 16 for t in range(16 * PAGES)]
    if kind == "one":
        return at[37:38]
    if kind == "decode":
        return at[3::16]
    if kind == "aligned":
        return at[:128]
    if kind == "ragged":  # two rows, both from within a page, padding between and after
        return at[5:75] + [-1] * 7 + at[85:150] + [-1]
    if kind == "padded":
        return [-1] * 3 + at[:33] + [-1, 10 ** 6] + at[48:64] + [-16] + at[64:80]
    if kind == "gaps":
        return [s for s in at if s % 7]
    if kind == "reversed":
        return at[:64][::-1]
    raise AssertionError(kind)


KINDS = ["one", "decode", "aligned", "ragged", "padded", "gaps", "reversed"]


# requests of these lengths, each from this place of a page, and padding after every third: a window may hold the end of
# one run, single tokens, padding and the start of another, and windows of one workgroup share runs
LENGTHS = (70, 9, 133, 16, 1, 250, 31, 47)
STARTS = (5, 0, 11, 3, 15, 7)


def _many_slots(windows: int) -> tuple[list[int], int]:
    """More than ``windows`` windows of 16 tokens, and the pages they are spread over."""
    at, page, i = [], 0, 0
    while len(at) <= 16 * windows:
        n, start = LENGTHS[i % len(LENGTHS)], STARTS[i % len(STARTS)]
        at += [page * 16 + start + t for t in range(n)] + [-1] * (i % 3 == 2) * (1 + i % 5)
        page += -(-(start + n) // 16)
        i += 1
    order = torch.randperm(page, generator=torch.Generator().manual_seed(page)).tolist()
    return [s if s < 0 else order[s // 16] * 16 + s % 16 for s in at], page


def _states(tokens: int, heads: int, dim: int, dtype, special: bool, seed: int) -> tuple[torch.Tensor, torch.Tensor]:
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(2, tokens, heads, dim, generator=gen) * torch.exp2(torch.randint(-9, 9, (2, tokens, heads, dim),
                                                                                   generator=gen).float())
    x = x.to(dtype)
    if special:
        at = torch.rand(x.shape, generator=gen)
        raw = x.view(torch.int16)
        patterns = (0x7F81, 0x7FC0, -0x7F, 0x7F80, -0x80, -0x8000, 0x7F00) if dtype == torch.bfloat16 else \
            (0x7C01, 0x7E00, -0x3FF, 0x7C00, -0x400, -0x8000, 0x0001)
        for k, v in enumerate(patterns):
            raw[(at > 1e-3 * k) & (at < 1e-3 * (k + 1))] = v
    return x[0].cuda(), x[1].cuda()


def _misaligned(x: torch.Tensor) -> torch.Tensor:
    return torch.empty(x.numel() + 1, dtype=x.dtype, device="cuda")[1:].view(x.shape).copy_(x)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize("source", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("heads", "dim"), [(1, 16), (3, 48), (2, 64), (8, 128)])
@pytest.mark.parametrize("kind", KINDS)
def test_paged_append(dtype, source, heads, dim, kind) -> None:
    _append_and_compare(dtype, source, heads, dim, _slots(kind), PAGES)


def _append_and_compare(dtype, source, heads, dim, slots, pages) -> None:
    from economize_amd.paged import PagedKVCache, paged_append

    slots = torch.tensor(slots, dtype=torch.int32, device="cuda")
    scales = [None, None] if dtype == torch.bfloat16 else [torch.full((heads,), 0.013), torch.full((heads,), 3.7e-3)]
    for special in (False, True):
        k, v = _states(slots.numel(), heads, dim, source, special, seed=dim + slots.numel())
        if special and scales[0] is not None:
            scales = [torch.tensor(([1.0, 2.0 ** -41, float("nan")] * heads)[:heads]), None]
        caches = []
        strided = torch.stack([k, v], dim=1)  # K and V of a token side by side
        for ks, vs in ((k, v), (strided[:, 0], strided[:, 1]), (_misaligned(k), _misaligned(v))):
            cache = PagedKVCache.empty(pages, heads, dim, dtype, "cuda", *(s if s is None else s.cuda() for s in scales))
            cache.keys.view(torch.uint8).fill_(0x5A)
            cache.values.view(torch.uint8).fill_(0x5A)
            paged_append(cache, ks, vs, slots)
            caches.append((cache.keys.view(torch.uint8), cache.values.view(torch.uint8)))
        for got in caches[:2]:
            assert torch.equal(got[0], caches[2][0]) and torch.equal(got[1], caches[2][1])


@pytest.mark.parametrize(("heads", "dim"), [(3, 64), (8, 128)])
@pytest.mark.parametrize("kind", KINDS)
def test_kivi_rings(heads, dim, kind) -> None:
    _ring_and_compare(heads, dim, _slots(kind), 3)


def _ring_and_compare(heads, dim, slots, batch) -> None:
    from economize_amd.kivi import PagedKIVICache, kivi_append

    # rings of 64 slots: slot s of the list is place s % 64, two laps on, of row s / 64
    slots = torch.tensor(slots)
    rows = torch.where(slots < 0, 0, slots // 64).to(torch.int32).cuda()
    positions = torch.where(slots < 0, -1, 128 + slots % 64).to(torch.int32).cuda()
    for special in (False, True):
        k, v = _states(slots.numel(), heads, dim, torch.bfloat16, special, seed=dim)
        rings = []
        for ks, vs in ((k, v), (_misaligned(k), _misaligned(v))):
            cache = PagedKIVICache.empty(4, batch, heads, dim, 4, "cuda", residual=32, headroom=32)
            kivi_append(cache, ks, vs, rows, positions)
            rings.append((cache.k_ring.view(torch.int16), cache.v_ring.view(torch.int16)))
        assert torch.equal(rings[0][0], rings[1][0]) and torch.equal(rings[0][1], rings[1][1])


# calls of more than 1024 waves (windows times units of 128 channels): four waves per workgroup
MANY = [(8, 128, 8), (5, 112, 5)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float8_e4m3fn, torch.float8_e5m2])
@pytest.mark.parametrize(("heads", "dim", "units"), MANY)
def test_paged_append_of_many_waves(dtype, heads, dim, units) -> None:
    slots, pages = _many_slots(1024 // units)
    for source in (torch.bfloat16, torch.float16):
        _append_and_compare(dtype, source, heads, dim, slots, pages)


@pytest.mark.parametrize(("heads", "dim", "units"), MANY[:1] + [(9, 64, 5)])
def test_kivi_rings_of_many_waves(heads, dim, units) -> None:
    slots, pages = _many_slots(1024 // units)
    _ring_and_compare(heads, dim, slots, -(-pages // 4))
