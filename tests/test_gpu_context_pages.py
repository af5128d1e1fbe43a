"""Context attention's page lookup against the oracle where it changes from one 64 entries of the block table to
the next: for every page size that reads the table that way, in rows that cross the change unsplit, and in
two split ranges whose second one starts at the change, one tile and two tiles before it."""
from __future__ import annotations

import pytest
import torch

from conftest import bits
from oracle import ops
from test_gpu_context_attention import _case, _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,hq", [(128, 4), (128, 12), (64, 4)])  # four and eight wavefronts
@pytest.mark.parametrize("before", [0, 1, 2])                       # tiles from the second range's start to the change
@pytest.mark.parametrize("page_size", [8, 16, 32, 64, 256])
def test_the_next_64_table_entries(mas, dev, page_size, before, dim, hq):
    tiles = 2 * (page_size - before)      # entry 64 is key tile `page_size`
    q_len = 5
    kv_lens = {64 * tiles, 64 * tiles - 31, 64 * page_size - 1, 64 * page_size, 64 * page_size + 1, 64 * page_size + 64}
    row_bytes = (32 if hq == 4 else 64) * hq * (dim + 2) * 4  # one split's partials
    for kv_len in sorted(kv_lens):
        q, kc, vc, tables, seq, cu = _case(kv_len + hq, [q_len], [kv_len], hq, 1, dim, page_size)
        want = ops.paged_context_attention(bits(q), bits(kc), bits(vc), tables.numpy(), seq.numpy(), cu.numpy(), dim ** -0.5)
        args = q.to(dev), (kc.to(dev), vc.to(dev))
        for ws_bytes in (16, 2 * row_bytes + row_bytes // 2):
            ws = torch.full((ws_bytes,), 255, dtype=torch.uint8, device=dev)
            flags = torch.zeros(1, dtype=torch.int32, device=dev)
            got = mas.attention.trtllm_batch_context_with_kv_cache(
                *args, ws, tables.to(dev), seq.to(dev), q_len, kv_len, dim ** -0.5, 1.0, 1, cu.to(dev), error_flags=flags)
            assert int(flags.item()) == 0
            # rows of 10 key tiles and more are split in two where the workspace holds two splits' partials
            if ws_bytes == 16 or kv_len > 10 * 64:
                assert torch.all(ws == 255) == (ws_bytes == 16)
            _check(bits(got), want, min_exact=0.5)
