"""Decode attention's grid against the oracle: one and two kv heads per workgroup, and the rotation of a
row's splits, at even and odd split counts under tables that reach further than the rows."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import ATOL, RTOL, bits
from oracle import numerics as on
from oracle import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,hq,hk,dim,page_size,reach,longest", [
    (64, 8, 2, 128, 16, 8192, 700),    # 64 x 2 x 32 = 4096 work items: pairs of kv heads
    (63, 8, 2, 128, 16, 8192, 700),    # one row fewer: one kv head per workgroup
    (70, 24, 2, 128, 256, 7936, 600),  # 31 splits (odd), pairs, 256-slot pages
    (43, 12, 3, 64, 16, 8192, 500),    # an odd kv head count: never pairs
    (130, 4, 4, 64, 16, 2048, 300),    # pairs, head_dim 64, 8 splits
    (9, 8, 2, 256, 16, 65536, 600),    # head_dim 256: one kv head per workgroup
    (5, 8, 4, 128, 16, 512, 512),      # a small grid's short splits
])
def test_decode_grid_matches_oracle(mas, dev, batch, hq, hk, dim, page_size, reach, longest):
    g = torch.Generator().manual_seed(batch + reach)
    lens = torch.randint(1, longest + 1, (batch,), generator=g, dtype=torch.int32)
    lens[: min(4, batch)] = torch.tensor([1, longest, 256, 257], dtype=torch.int32)[: min(4, batch)]
    width, need = reach // page_size, -(-longest // page_size)
    pages = batch * need + 1
    tables = torch.full((batch, width), pages - 1, dtype=torch.int32)
    tables[:, :need] = torch.randperm(pages - 1, generator=g).reshape(batch, need).to(torch.int32)
    q = torch.randn(batch, hq, dim, generator=g).bfloat16()
    kc = torch.randn(pages, page_size, hk, dim, generator=g).bfloat16()
    vc = torch.randn(pages, page_size, hk, dim, generator=g).bfloat16()
    ws = torch.full((128 << 20,), 255, dtype=torch.uint8, device=dev)  # NaN partials on entry
    want = on.bf16_to_f32(ops.paged_decode_attention(bits(q), bits(kc), bits(vc), tables.numpy(), lens.numpy(), 0.1))
    args = q.to(dev), (kc.to(dev), vc.to(dev)), ws, tables.to(dev), lens.to(dev)
    for _ in range(2):
        got = mas.attention.trtllm_batch_decode_with_kv_cache(*args, reach, 0.1, 1.0)
        np.testing.assert_allclose(on.bf16_to_f32(bits(got)), want, rtol=RTOL, atol=ATOL)
