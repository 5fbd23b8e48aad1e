"""Cells between a request's last key and the end of its 32-key tile: whatever they hold (stale flags, NaN in their dense
entries, scales, zero points and codes of an earlier request), attention over vLLM's cells does not see it."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("page", [32, 64])
def test_cells_past_the_last_key_are_not_seen(bits, page) -> None:
    from economize_amd.vllm_kivi import cell_layout, paged_kivi_attention, quantize_committed

    kv_heads, q_heads, head = 2, 8, 128
    lens, qlens = [1, 31, 33, 95, 300, 64, 1000], [1, 2, 1, 5, 1, 1, 3]
    layout = cell_layout(head, torch.bfloat16, bits, 32)
    per_row = -(-max(lens) // page)
    pages = len(lens) * per_row
    gen = torch.Generator().manual_seed(bits + page)
    table = torch.randperm(pages, generator=gen).view(len(lens), per_row).to(torch.int32).cuda()
    cells = torch.randn(pages, kv_heads, page, layout.size // 2, generator=gen).to(torch.bfloat16).cuda()
    cells.view(torch.uint8)[..., layout.off_flag: layout.off_flag + 2] = 0
    starts = torch.tensor(np.concatenate([[0], np.cumsum(qlens)]), dtype=torch.int32).cuda()
    seq = torch.tensor(lens, dtype=torch.int32).cuda()
    quantize_committed(cells, layout, 32, table, starts, seq, torch.zeros_like(seq))
    q = torch.randn(sum(qlens), q_heads, head, generator=gen).to(torch.bfloat16).cuda()

    def attend():
        return paged_kivi_attention(q, cells, layout, table, starts, seq, max(qlens), max(lens), scale=0.1)

    want = attend()
    assert torch.isfinite(want.float()).all()
    past = torch.ones(pages, page, dtype=torch.bool)  # cells that no key of a request takes
    for b, n in enumerate(lens):
        t = torch.arange(n)
        past[table[b].cpu()[t // page].long(), t % page] = False
    past = past[:, None, :, None].cuda()
    u8 = cells.view(torch.uint8)
    stale = torch.randint(0, 256, u8.shape, generator=gen, dtype=torch.uint8)
    stale[..., layout.off_flag: layout.off_flag + 2] = 1
    for garbage in (torch.full_like(stale, 0xFF), stale):
        u8.copy_(torch.where(past, garbage.cuda(), u8))
        assert torch.equal(attend().view(torch.int16), want.view(torch.int16))
