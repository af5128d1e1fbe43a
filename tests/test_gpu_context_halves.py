"""Context attention's 32-position half steps at their edges, against the oracle: lengths around whole
halves and tiles, for every workgroup shape and page mode, with scores whose running reference has to
move in a first half, a second half and not at all."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import ATOL, RTOL, bits
from oracle import ops
from test_gpu_context_attention import SPLIT_WS, _case, _check, _run

pytestmark = pytest.mark.gpu

LENGTHS = [(1, 1), (31, 31), (32, 32), (33, 33), (2, 34), (64, 64), (65, 65), (1, 96), (30, 97), (64, 128), (5, 129)]


@pytest.mark.parametrize("dim", [64, 128])
# four and eight wavefronts, one head per workgroup, and groups that leave wavefronts without a head
@pytest.mark.parametrize("hq,hk", [(8, 2), (24, 2), (3, 1), (5, 1), (7, 1), (9, 1), (11, 1)])
@pytest.mark.parametrize("page_size", [4, 8, 16, 32, 64])
def test_half_step_edges(mas, dev, dim, hq, hk, page_size):
    q_lens, kv_lens = [n for n, _ in LENGTHS], [n for _, n in LENGTHS]
    q, kc, vc, tables, seq, cu = _case(dim + hq + page_size, q_lens, kv_lens, hq, hk, dim, page_size)
    # Row r's keys grow (r % 3 == 1: 24-fold from position 32 on; 2: sixfold from 64 on): the reference
    # moves in a second half, or in a later tile's first half.
    for r, n in enumerate(kv_lens):
        for p in range(n):
            factor = 24.0 if r % 3 == 1 and p >= 32 else (6.0 if r % 3 == 2 and p >= 64 else 1.0)
            kc[int(tables[r, p // page_size]), p % page_size] *= factor
    want = ops.paged_context_attention(bits(q), bits(kc), bits(vc), tables.numpy(), seq.numpy(), cu.numpy(), 0.1)
    for ws_bytes in (16, SPLIT_WS):  # rows this short are not split, whatever the workspace holds
        got = _run(mas, dev, q, kc, vc, tables, seq, cu, 0.1, ws_bytes=ws_bytes, max_kv=max(kv_lens))
        _check(bits(got), want, min_exact=0.5)


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("hq,hk", [(8, 2), (24, 2)])
def test_output_rows_of_ragged_tiles(mas, dev, dim, hq, hk):
    """The last tile's tokens end inside a 32-token block: only a row's own tokens are written, in bf16
    and fp8, into a strided view."""
    q_lens, kv_lens = [37, 1, 70], [37, 80, 200]
    q, kc, vc, tables, seq, cu = _case(7, q_lens, kv_lens, hq, hk, dim, 16)
    want = ops.paged_context_attention(bits(q), bits(kc), bits(vc), tables.numpy(), seq.numpy(), cu.numpy(), 0.1)
    tokens = sum(q_lens)
    base = torch.full((tokens + 3, hq + 1, dim), 5.0, dtype=torch.bfloat16, device=dev)
    _run(mas, dev, q, kc, vc, tables, seq, cu, 0.1, out=base[:tokens, 1:])
    _check(bits(base[:tokens, 1:].contiguous()), want)
    assert torch.all(base[tokens:] == 5.0) and torch.all(base[:, 0] == 5.0)
    codes = torch.full((tokens + 3, hq + 1, dim), 1.0, device=dev).to(torch.float8_e4m3fn)
    _run(mas, dev, q, kc, vc, tables, seq, cu, 0.1, out=codes[:tokens, 1:], quant=0.05)
    y = base[:tokens, 1:].float() / 0.05
    assert torch.equal(codes[:tokens, 1:].float(), y.clamp(-448, 448).to(torch.float8_e4m3fn).float())
    assert torch.all(codes[tokens:].float() == 1.0) and torch.all(codes[:, 0].float() == 1.0)


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("tiles", [1, 2, 3, 4])
@pytest.mark.parametrize("page_size", [4, 16, 64])
def test_a_tiles_weights_add_in_one_chain(mas, dev, dim, tiles, page_size):
    """A lane adds its 32 weights of a 64-position tile one after the other, over both halves. Every tile has
    one weight of 1 (value 1) in a lane's first half and 16 of 2^-25 (value 0) in its second: each vanishes
    beside the 1, so the row's sum is the number of tiles, and an output scaled to 2^-22 above the middle of
    two bf16 values rounds up. The 16 added by themselves would make 2^-21 of each tile, and it would round
    down (the key's bf16 rounding moves 2^-25 by at most 2^0.15)."""
    scale, n = 0.1, 64 * tiles
    small = -25 / (scale * 1.4426950408889634)
    q, kc, vc, tables, seq, cu = _case(1, [1], [n], 4, 1, dim, page_size)
    q.zero_()
    q[..., 0] = 1
    kc.zero_()
    vc.zero_()
    for p in range(n):
        at = int(tables[0, p // page_size]), p % page_size, 0
        kc[at][0] = 0.0 if p % 64 == 0 else (small if p % 64 >= 32 and p % 8 < 4 else -20000.0)
        vc[at] = 1.0 if p % 64 == 0 else 0.0
    got = _run(mas, dev, q, kc, vc, tables, seq, cu, scale, scale2=1 + 2 ** -8 + 2 ** -22)
    assert torch.all(got == 1 + 2 ** -7), got.unique()


@pytest.mark.parametrize("page_size,kv_len,ws_bytes", [(4, 320, 16), (16, 320, 16), (64, 320, 16), (16, 1600, SPLIT_WS)])
@pytest.mark.parametrize("dim,hq,hk", [(64, 8, 2), (128, 8, 2), (128, 24, 2)])
def test_outputs_do_not_depend_on_the_tiles_other_tokens(mas, dev, dim, hq, hk, page_size, kv_len, ws_bytes):
    """Odd tokens' scores grow so that their softmax reference moves in every tile, or are nearly flat so that
    it never does: the even tokens between them, whose own scores rise a little, get the same bits."""
    q_len = 60
    q, kc, vc, tables, seq, cu = _case(dim + hq + kv_len, [q_len], [kv_len], hq, hk, dim, page_size)
    for p in range(64, kv_len):
        kc[int(tables[0, p // page_size]), p % page_size] *= 1 + p / kv_len
    got = []
    for factor in (30.0, 0.01):
        mixed = q.clone()
        mixed[1::2] *= factor
        got.append(_run(mas, dev, mixed, kc, vc, tables, seq, cu, 0.1, ws_bytes=ws_bytes, max_kv=kv_len))
    assert torch.equal(got[0][0::2], got[1][0::2])
    want = ops.paged_context_attention(bits(mixed), bits(kc), bits(vc), tables.numpy(), seq.numpy(), cu.numpy(), 0.1)
    _check(bits(got[1]), want, min_exact=0.5)


@pytest.mark.parametrize("dim,hq,hk", [(64, 4, 1), (128, 4, 1), (128, 5, 1), (128, 12, 1)])  # four, then eight wavefronts
@pytest.mark.parametrize("page_size", [4, 8, 16, 32, 64, 256])
def test_split_ranges_end_at_every_half(mas, dev, dim, hq, hk, page_size):
    """Rows of 17 and 18 key tiles under a table of 64, which gives ranges of 4: the last range is one or two
    tiles long and ends at, before and after a tile's middle. The workspace tells that the launch was split."""
    q_lens = [1, 31, 32, 33, 2, 30, 32, 5]
    kv_lens = [1024 + n for n in (1, 31, 32, 33, 64, 65, 96, 97)]
    q, kc, vc, tables, seq, cu = _case(hq + dim + page_size, q_lens, kv_lens, hq, hk, dim, page_size)
    tables = torch.nn.functional.pad(tables, (0, 4096 // page_size - tables.shape[1]))
    ws = torch.full((SPLIT_WS,), 255, dtype=torch.uint8, device=dev)
    got = mas.attention.trtllm_batch_context_with_kv_cache(
        q.to(dev), (kc.to(dev), vc.to(dev)), ws, tables.to(dev), seq.to(dev), 33, 4096, dim ** -0.5, 1.0, len(q_lens),
        cu.to(dev))
    assert not torch.all(ws == 255)
    want = ops.paged_context_attention(bits(q), bits(kc), bits(vc), tables.numpy(), seq.numpy(), cu.numpy(), dim ** -0.5)
    _check(bits(got), want, min_exact=0.5)


def _softmax64(q, kc, vc, table, kv_len, scale):
    """float64 causal attention of the last len(q) of kv_len positions, one kv head: IEEE's NaN and infinities."""
    rows = [c[table.long()].flatten(0, 1)[:kv_len, 0].double() for c in (kc, vc)]
    scores = torch.einsum("thd,pd->htp", q.double(), rows[0]) * scale
    at = torch.arange(kv_len)[None, :] > torch.arange(kv_len - len(q), kv_len)[:, None]
    p = torch.softmax(scores.masked_fill(at, -float("inf")), -1)
    return torch.stack([torch.stack([(row[:n, None] * rows[1][:n]).sum(0) for row, n in zip(
        head, range(kv_len - len(q) + 1, kv_len + 1))]) for head in p]).transpose(0, 1)


SPECIALS = ["inf key", "nan key", "inf value", "nan value"]


@pytest.mark.parametrize("what,kv_len,ws_bytes", [("nan query", 200, 16), *((w, 200, 16) for w in SPECIALS),
                                                  *((w, 1500, SPLIT_WS) for w in SPECIALS)])
@pytest.mark.parametrize("at", [3, 40, 70, 170])  # a first and a second half of the first tile and of later ones
@pytest.mark.parametrize("page_size,hq", [(4, 4), (16, 4), (64, 12)])
def test_nan_and_infinity(mas, dev, what, at, kv_len, ws_bytes, page_size, hq):
    """A query that is not a number gets NaN and no other token does; a key's infinite element makes scores
    of +inf (NaN outputs) and -inf (weight 0) by the query's sign; values pass into their column alone."""
    n, dim = 20, 64
    q, kc, vc, tables, seq, cu = _case(at, [n], [kv_len], hq, 1, dim, page_size)
    where, special = (int(tables[0, at // page_size]), at % page_size, 0), float(what[:3])
    if what == "nan query":
        q[7, 1, 5] = special
    else:
        (kc if "key" in what else vc)[where][5] = special
    want = _softmax64(q, kc, vc, tables[0], kv_len, 0.125)
    got = _run(mas, dev, q, kc, vc, tables, seq, cu, 0.125, ws_bytes=ws_bytes, max_kv=kv_len).double().cpu()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    finite = want.isfinite()
    assert finite.any() == (what != "nan key")
    np.testing.assert_allclose(got[finite], want[finite], rtol=RTOL, atol=ATOL)
