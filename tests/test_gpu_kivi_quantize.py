"""KIVI pages quantized by one wave each (bf16 and fp16 sources with contiguous channels) against the workgroup-per-page
kernels, which take the same values as fp32: whole pages, rows of different lengths, partial value pages that keep their
other tokens' codes, strided and ring sources, missing pages, NaN, infinities, constant groups and scales beyond fp16.
Exact: whole bytes."""

from __future__ import annotations

import dataclasses

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

B, H, PAGES = 3, 2, 9
S = 32 * PAGES


def _source(dtype, dim: int, kind: str, seed: int) -> torch.Tensor:
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(B, H, S, dim, generator=gen) * torch.exp2(torch.randint(-3, 4, (B, H, 1, dim), generator=gen).float())
    if kind == "grid":  # quotients on and next to half integers
        x = torch.randint(-31, 32, x.shape, generator=gen) * 0.5
        x[2] = x[2].abs() * (x[2].abs() < 3)  # groups whose minimum is a zero, of either sign
        x[2][(x[2] == 0) & (torch.rand(x[2].shape, generator=gen) < 0.5)] = -0.0
    elif kind == "special":
        at = torch.rand(x.shape, generator=gen)
        for k, v in enumerate((float("nan"), float("inf"), -float("inf"), 6e4, -6e4, 1e-7)):
            x = torch.where((at > 0.002 * k) & (at < 0.002 * (k + 1)), torch.tensor(v), x)
        x[0, 0, 32:64] = float("nan")
        x[0, 1, 32:64] = 1.25
        x[1, 0, 64:96] *= 1e-6
    elif kind == "huge":
        x = x * (1e5 if dtype == torch.bfloat16 else 1.5e4)
    return x.to(dtype)


def _run(source, bits: int, kind: str, start, stop, table, start_blocks, source_start: int = 0):
    from economize_amd.kivi import PagedKIVICache, kivi_quantize

    dim = source.shape[3]
    cache = PagedKIVICache.empty(B * PAGES + 1, B, H, dim, bits, "cuda", residual=32, headroom=32)
    cache.blocks.copy_(start_blocks.expand_as(cache.blocks))
    as_int = [torch.tensor(x, dtype=torch.int32, device="cuda") for x in (start, stop)]
    most = max(b - a for a, b in zip(start, stop))
    kivi_quantize(cache, table, source, kind, *as_int, most, source_start)
    return cache.blocks.cpu(), int(cache.overflow.item())


def _overflows(x: np.ndarray, bits: int, side: str, start, stop, table) -> int:
    """1 if a group quantized has a scale or minimum beyond fp16 (a group of NaN alone: the infinities of no value)."""
    for b, page in np.argwhere(table >= 0):
        lo_t, hi_t = max(32 * page, start[b]), min(32 * page + 32, stop[b])
        if hi_t - lo_t < (32 if side == "k" else 1):
            continue
        g = x[b, :, lo_t:hi_t]
        g = g[:, None] if side == "k" else g.reshape(H, hi_t - lo_t, -1, 32).swapaxes(2, 3)  # groups along axis 2
        low = np.where(np.isnan(g), np.inf, g).min(axis=2)
        high = np.where(np.isnan(g), -np.inf, g).max(axis=2)
        with np.errstate(invalid="ignore"):
            scale = (high - low) / np.float32(2 ** bits - 1)
        if ((np.abs(scale) > 65504) | (np.abs(low) > 65504)).any():
            return 1
    return 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("kind", ["normal", "grid", "special", "huge"])
def test_wave_pages_equal_the_general_kernels(dtype, dim, bits, kind) -> None:
    x = _source(dtype, dim, kind, seed=dim + bits).cuda()
    table = torch.randperm(B * PAGES + 1, generator=torch.Generator().manual_seed(1))[: B * PAGES].view(B, PAGES)
    table = table.to(torch.int32)
    table[1, 3] = -1
    table = table.cuda()
    before = torch.full((1, 1, 1), 0xA5, dtype=torch.uint8, device="cuda")
    token_major = x.transpose(1, 2).contiguous().transpose(1, 2)
    ranges = {"k": (([0, 32, 64], [S, 160, 64]),),
              "v": (([0, 0, 0], [S, 161, 1]), ([5, 31, 64], [6, 33, 127]), ([17, 250, 0], [150, S, 0]))}
    numbers, pages = x.float().cpu().numpy(), table.cpu().numpy()
    for side, many in ranges.items():
        for start, stop in many:
            want, flag = _run(x.float(), bits, side, start, stop, table, before)
            assert flag == _overflows(numbers, bits, side, start, stop, pages), (side, start, stop)
            for source in (x, token_major):
                got, got_flag = _run(source, bits, side, start, stop, table, before)
                assert torch.equal(got, want), (side, start, stop)
                assert got_flag == flag


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("bits", [2, 4])
def test_ring_sources(dim, bits) -> None:
    """Commits from rings of 96 slots, several laps: keys from an aligned ring against the same ring at an odd element
    (the general kernel); the values' ring is token-contiguous, the general kernel's either way."""
    from economize_amd.kivi import PagedKIVICache, kivi_commit

    table = torch.arange(B * PAGES, dtype=torch.int32, device="cuda").view(B, PAGES)
    cache = PagedKIVICache.empty(B * PAGES, B, H, dim, bits, "cuda", residual=32, headroom=64)
    ring = cache.k_ring
    odd = torch.empty(ring.numel() + 1, dtype=ring.dtype, device="cuda")[1:].view(ring.shape)
    other = dataclasses.replace(cache, blocks=torch.zeros_like(cache.blocks), k_ring=odd,
                                keys_quantized=torch.zeros_like(cache.keys_quantized),
                                values_quantized=torch.zeros_like(cache.values_quantized))
    gen = torch.Generator(device="cuda").manual_seed(dim + bits)
    committed = [0, 0, 0]
    for step in ([64, 40, 3], [64, 61, 33], [50, 64, 0], [64, 31, 64], [33, 64, 64]):
        committed = [c + s for c, s in zip(committed, step)]
        for x in (cache.k_ring, cache.v_ring):
            x.copy_(torch.randn(x.shape, generator=gen, device="cuda"))
        odd.copy_(cache.k_ring)
        for c in (cache, other):
            kivi_commit(c, table, torch.tensor(committed, dtype=torch.int32, device="cuda"), 64)
        assert torch.equal(cache.blocks, other.blocks), committed
    assert cache.keys_quantized.tolist() == [c // 32 * 32 for c in committed] and cache.blocks[:2].any()


@pytest.mark.parametrize("bits", [2, 4])
def test_source_offsets_and_misaligned_sources(bits) -> None:
    x = _source(torch.bfloat16, 64, "normal", seed=bits).cuda()
    table = torch.arange(B * PAGES, dtype=torch.int32, device="cuda").view(B, PAGES)
    before = torch.zeros(1, 1, 1, dtype=torch.uint8, device="cuda")
    start, stop = [96, 96, 128], [S, 160, 192]
    odd = torch.empty(x.numel() + 1, dtype=x.dtype, device="cuda")[1:].view(x.shape).copy_(x)
    for side in ("k", "v"):
        want, _ = _run(x.float(), bits, side, start, stop, table, before)
        for source, at in ((x, 0), (x[:, :, 96:], 96), (x[:, :, 93:], 93), (odd, 0)):
            assert torch.equal(_run(source, bits, side, start, stop, table, before, at)[0], want), (side, at)
