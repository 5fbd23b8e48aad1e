"""The order of the dense kernel's sums, which its variants share: decode over vLLM's cells through their codes gives the
bits of dense decode over the numbers the codes stand for, and a block of few query rows weighs its keys against the
largest score so far."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("length", [33, 200, 2079])
def test_cells_equal_dense_buffers_bit_for_bit(bits, length) -> None:
    from economize_amd.decode import decode_attention
    from economize_amd.vllm_kivi import cell_layout, paged_kivi_attention, quantize_committed

    batch, kv_heads, q_heads, head, page = 3, 2, 8, 128, 32
    layout = cell_layout(head, torch.bfloat16, bits, 32)
    per_row = -(-length // page)
    gen = torch.Generator().manual_seed(bits + length)
    table = torch.randperm(batch * per_row + 2, generator=gen)[: batch * per_row].view(batch, per_row)
    cells = torch.randn(batch * per_row + 2, kv_heads, page, layout.size // 2, generator=gen).to(torch.bfloat16).cuda()
    cells.view(torch.uint8)[..., layout.off_flag: layout.off_flag + 2] = 0
    starts = torch.arange(batch + 1, dtype=torch.int32, device="cuda")
    lens = torch.full((batch,), length, dtype=torch.int32, device="cuda")
    on_gpu = table.to(torch.int32).cuda()
    quantize_committed(cells, layout, 32, on_gpu, starts, lens, torch.zeros_like(lens))
    # the dense entries of quantized cells hold the dequantized numbers
    t = torch.arange(length)
    entries = cells[table[:, t // page].cuda(), :, (t % page).cuda(), : 2 * head].transpose(1, 2)
    k, v = entries[..., :head].contiguous(), entries[..., head:].contiguous()
    q = torch.randn(batch, q_heads, head, generator=gen).to(torch.bfloat16).cuda()
    got = paged_kivi_attention(q, cells, layout, on_gpu, starts, lens, 1, length, scale=0.2)
    want = decode_attention(q[:, :, None], k, v, None, 0.2)
    assert torch.equal(got.view(torch.int16), want.reshape(got.shape).view(torch.int16))


def test_few_rows_weigh_keys_against_the_largest_score() -> None:
    """Two tiles of keys, one key of weight in each, the second's score s (log2 units) above the first's: relative to the
    largest score the second key's weight is 1, exact in the product's 16-bit operands, and out = 1 / (1 + 2^-s) to fp32
    rounding: 4 2^-24 for the score and its power, their sum and the division. Relative to the first key's score it
    would be 2^s, off by up to 2^-17 in the two bf16 terms."""
    from economize_amd.decode import decode_attention

    batch, dim = 2048, 64  # (as many blocks as leave every one a single split)
    q = torch.zeros(batch, 1, 1, dim)
    q[..., 0] = 1.0
    k = torch.zeros(batch, 1, 64, dim)
    k[..., 0] = -300.0
    k[:, :, 0, 0] = 0.0
    score = torch.linspace(0.1, 5.5, batch).to(torch.bfloat16).float()  # (below 8: the maximum could have stayed)
    k[:, 0, 32, 0] = score
    v = torch.zeros(batch, 1, 64, dim)
    v[:, :, 32] = 1.0
    out = decode_attention(q.cuda(), k.cuda(), v.cuda(), None, 1.0).cpu().numpy().reshape(batch, dim)
    want = 1.0 / (1.0 + np.exp(-score.double().numpy()))
    # the score's own rounding moves 2^-s by s ln 2 2^-24 of it
    assert np.abs(out / want[:, None] - 1.0).max() < 8 * 2.0 ** -24
