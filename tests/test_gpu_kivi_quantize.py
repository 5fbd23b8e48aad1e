"""KIVI pages quantized by one wave each (bf16 and fp16 sources with contiguous channels) against the workgroup-per-page
kernels, which take the same values as fp32: whole pages, rows of different lengths, partial value pages that keep their
other tokens' codes, strided and ring sources, missing pages, NaN, infinities, constant groups and scales beyond fp16.
Exact: whole bytes."""

from __future__ import annotations

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
    flags = set()
    for side, many in ranges.items():
        for start, stop in many:
            want, flag = _run(x.float(), bits, side, start, stop, table, before)
            flags.add(flag)
            for source in (x, token_major):
                got, got_flag = _run(source, bits, side, start, stop, table, before)
                assert torch.equal(got, want), (side, start, stop)
                assert got_flag == flag
    assert flags == ({0} if kind in ("normal", "grid") else {1} if kind == "huge" else flags)


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
