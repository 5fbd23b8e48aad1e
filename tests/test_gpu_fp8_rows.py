"""The fp8 encode of bf16 and fp16 rows by 16-byte loads against the same values encoded as fp32 (the kernel that takes
any row), bit for bit: head dims that leave lanes idle, token counts around a workgroup's rows, every scale mode, every
16-bit pattern, scales outside the corrected quotient's limits, misaligned sources, and destinations whose row stride the
kernel takes (a multiple of 8 bytes) or leaves to the other one."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

FORMATS = (torch.float8_e4m3fn, torch.float8_e5m2)


def _encode(x, dtype, **more):
    from economize_amd.fp8 import fp8_encode

    return fp8_encode(x, dtype, **more).view(torch.uint8)


def _compare(x: torch.Tensor, dtype, head_scale: torch.Tensor) -> None:
    wide = x.float()
    assert torch.equal(_encode(x, dtype), _encode(wide, dtype))
    assert torch.equal(_encode(x, dtype, head_scale=head_scale), _encode(wide, dtype, head_scale=head_scale))
    scales = [torch.full(x.shape[:3], -1.0, device="cuda") for _ in range(2)]
    got, want = (_encode(y, dtype, token_scale=s) for y, s in zip((x, wide), scales))
    assert torch.equal(got, want)
    assert torch.equal(scales[0].view(torch.int32), scales[1].view(torch.int32))


@pytest.mark.parametrize("dtype", FORMATS)
@pytest.mark.parametrize("source", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("dim", "tokens"), [(8, 129), (64, 127), (72, 1), (128, 64), (128, 65), (200, 33), (256, 31),
                                             (264, 17), (512, 16), (512, 1)])
def test_rows(dtype, source, dim, tokens) -> None:
    gen = torch.Generator().manual_seed(dim + tokens)
    x = torch.randn(2, 3, tokens, dim, generator=gen) * torch.exp2(torch.randint(-9, 9, (2, 3, tokens, dim),
                                                                                 generator=gen).float())
    x = x.to(source).cuda()
    _compare(x, dtype, torch.tensor([0.013, 3.0, 1.0], device="cuda"))
    # tokens before heads, and a copy at an odd element offset
    _compare(x.transpose(1, 2).contiguous().transpose(1, 2), dtype, torch.tensor([0.5, 7e-4, 1.7], device="cuda"))
    odd = torch.empty(x.numel() + 1, dtype=source, device="cuda")[1:].view(x.shape).copy_(x)
    _compare(odd, dtype, torch.tensor([0.5, 7e-4, 1.7], device="cuda"))
    for extra in (4, 8):
        buffer = torch.full((2, 3, tokens + 3, dim + extra), 0x5A, dtype=torch.uint8, device="cuda")
        _encode(x, dtype, out=buffer[:, :, 2: 2 + tokens, :dim].view(dtype))
        want = torch.full_like(buffer, 0x5A)
        want[:, :, 2: 2 + tokens, :dim] = _encode(x.float(), dtype)
        assert torch.equal(buffer, want)


@pytest.mark.parametrize("dtype", FORMATS)
@pytest.mark.parametrize("source", [torch.bfloat16, torch.float16])
def test_every_pattern_and_scales_at_the_limits(dtype, source) -> None:
    bits = torch.arange(65536, dtype=torch.int32).to(torch.int16)
    x = bits.view(source).view(1, 1, 512, 128).expand(1, 12, 512, 128).contiguous().cuda()
    scale = torch.tensor([1.0, 3e-5, 0.37, 2.0 ** -40, 2.0 ** -41, 2.0 ** 60, 2.0 ** 61, 0.0, -2.0, float("inf"),
                          float("nan"), 1e-38], device="cuda")
    _compare(x, dtype, scale)
    # finite rows without the infinities and NaN of their neighbours: the corrected quotient over the whole range
    finite = torch.where(x[:, :3].isfinite() & (x[:, :3].abs() < 1e18), x[:, :3], torch.zeros_like(x[:, :3]))
    _compare(finite, dtype, torch.tensor([1.0, 3e-5, 1e12], device="cuda"))
