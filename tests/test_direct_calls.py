"""The direct calls (binding/direct_calls.cpp) against the wrappers' general way: the same bits for every
form they take, and None, with nothing done, for every form they leave to the wrappers."""
from __future__ import annotations

import ctypes
import timeit

import pytest
import torch

FP8 = torch.float8_e4m3fn


def _norm_args(dev="cpu", rows=3, hidden=64):
    return [torch.randn(rows, hidden, device=dev).bfloat16(), torch.randn(rows, hidden, device=dev).bfloat16(),
            torch.ones(hidden, device=dev).bfloat16(), 1e-5]


def test_direct_calls_leave_other_forms_to_the_wrappers(mas):
    """On the CPU: no form is taken, whatever the arguments are."""
    mas.load_library()
    d = mas._lib.direct
    assert d.fused_add_rmsnorm(*_norm_args()) is None
    assert d.fused_add_rmsnorm(None, 1, "x", ()) is None
    assert d.fused_add_rmsnorm() is None
    assert d.silu_and_mul(torch.ones(2, 4), torch.ones(2, 2)) is None
    assert d.decode_attention(*[None] * 11) is None
    assert d.context_attention(*[None] * 14) is None
    assert d.rope_append(*[None] * 15) is None
    with pytest.raises(ValueError, match="must be on a GPU device"):
        mas.norm.fused_add_rmsnorm(*_norm_args())
    with pytest.raises(TypeError):
        d.bind(None, None)
    with pytest.raises(KeyError):
        d.bind(None, {})
    d.bind(mas._lib._raw_stream, {n: mas._lib.ctypes.cast(getattr(mas._lib.load(), n), mas._lib.ctypes.c_void_p).value
                                  for n in mas._lib.exported_symbols()})


def test_a_form_left_to_the_wrappers_costs_little(mas):
    """A refusal is a comparison and a return (0.1-0.2 us); as a C++ exception it took 3-4 us of the call."""
    mas.load_library()
    d, norm = mas._lib.direct, _norm_args()
    for call in (lambda: d.fused_add_rmsnorm(*norm), lambda: d.silu_and_mul_quant(*norm[:2], 1.0),
                 lambda: d.decode_attention(*[None] * 11), lambda: d.context_attention(*[None] * 14),
                 lambda: d.rope_append(*norm, 64, *[None] * 10)):
        assert call() is None
        assert min(timeit.repeat(call, number=1000, repeat=20)) / 1000 < 1.5e-6


def _addresses(mas):
    lib = mas._lib.load()
    return {n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in mas._lib.exported_symbols()}


def test_the_library_loads_without_the_extension(mas, monkeypatch, tmp_path):
    """No extension, one that is none, or one built for another torch: a warning, and the wrappers serve."""
    lib = mas._lib.load()
    other = tmp_path / "direct_calls.so"
    other.write_text("not a library")
    for path in (tmp_path / "absent.so", other):
        monkeypatch.setattr(mas._lib._build, "DIRECT_CALLS_PATH", path)
        with pytest.warns(RuntimeWarning, match="is not used"):
            assert mas._lib._load_direct(lib) is None
    monkeypatch.undo()
    monkeypatch.setattr(torch, "__version__", "0.0.1+other")
    with pytest.warns(RuntimeWarning, match="built for torch"):
        assert mas._lib._load_direct(lib) is None
    monkeypatch.undo()
    assert mas._lib._load_direct(lib) is not None


def test_the_extension_is_bound_to_its_own_library_version_only(mas):
    mas.load_library()
    other = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: 1 << 24)
    with pytest.raises(ValueError, match="version"):
        mas._lib.direct.bind(mas._lib._raw_stream,
                             _addresses(mas) | {"mas_version": ctypes.cast(other, ctypes.c_void_p).value})


def test_a_build_without_a_compiler_goes_on_without_the_extension(mas, monkeypatch, tmp_path):
    monkeypatch.setattr(mas._lib._build, "DIRECT_CALLS_PATH", tmp_path / "direct_calls.so")
    monkeypatch.setenv("CXX", str(tmp_path / "no-compiler"))
    with pytest.warns(RuntimeWarning, match="failed"):
        assert mas._lib._build.build_direct_calls() is None


@pytest.mark.gpu
def test_a_failed_bind_leaves_the_calls_bound(mas, dev):
    mas.load_library()
    d = mas._lib.direct
    some = dict(list(_addresses(mas).items())[:3])
    for names in ({}, some, _addresses(mas) | {"mas_silu_and_mul_bf16": None}):
        with pytest.raises((KeyError, TypeError)):
            d.bind(None, names)
    assert d.silu_and_mul(torch.ones(2, 64, device=dev).bfloat16(), torch.empty(2, 32, device=dev).bfloat16()) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 5])
@pytest.mark.parametrize("view", [False, True])
def test_norm_and_activation_match_the_general_way(mas, dev, rows, view):
    mas.load_library()
    d, hidden = mas._lib.direct, 64
    wide = torch.randn(rows, 4 * hidden, device=dev).bfloat16()
    x = wide[:, hidden:2 * hidden] if view else wide[:, :hidden].contiguous()
    r, w = torch.randn(rows, hidden, device=dev).bfloat16(), torch.randn(hidden, device=dev).bfloat16()
    gate_up = wide[:, 2 * hidden:] if view else wide[:, 2 * hidden:].contiguous()
    for scale in (torch.tensor(0.1, device=dev), 0.1):
        outs, resids = [torch.zeros(rows, hidden, device=dev).to(FP8) for _ in range(2)], [r.clone(), r.clone()]
        assert d.fused_add_rmsnorm_quant(outs[0], x, resids[0], w, scale, 1e-5) == 0
        mas.norm._fused_add_rmsnorm_quant(outs[1], x, resids[1], w, scale, 1e-5)
        assert torch.equal(outs[0].view(torch.uint8), outs[1].view(torch.uint8)) and torch.equal(*resids)
        assert d.silu_and_mul_quant(gate_up, outs[0], scale) == 0
        mas.activation._silu_and_mul_quant(gate_up, outs[1], scale)
        assert torch.equal(outs[0].view(torch.uint8), outs[1].view(torch.uint8))
    outs = [torch.zeros(rows, hidden, device=dev).bfloat16() for _ in range(2)]
    assert d.silu_and_mul(gate_up, outs[0]) == 0
    mas.activation._silu_and_mul(gate_up, outs[1])
    assert torch.equal(*outs)
    xs, resids = [x.clone(), x.clone()], [r.clone(), r.clone()]
    assert d.fused_add_rmsnorm(xs[0], resids[0], w, 1e-5) == 0
    mas.norm._fused_add_rmsnorm(xs[1], resids[1], w, 1e-5)
    assert torch.equal(*xs) and torch.equal(*resids)
    # left to the wrappers: other ranks, types, strides, empty tensors, sizes that do not fit
    assert d.fused_add_rmsnorm(x[0], r[0], w, 1e-5) is None
    assert d.fused_add_rmsnorm(x.float(), r, w, 1e-5) is None
    assert d.fused_add_rmsnorm(x, r, w[:-1], 1e-5) is None
    assert d.fused_add_rmsnorm(x, r, w, -1.0) is None
    assert d.fused_add_rmsnorm(x.t(), r.t(), w[:rows], 1e-5) is None or rows == 1
    assert d.fused_add_rmsnorm(x[:0], r[:0], w, 1e-5) is None
    assert d.fused_add_rmsnorm(x, r.cpu(), w, 1e-5) is None
    assert d.silu_and_mul_quant(gate_up, outs[0].to(FP8), 0.0) is None


def _attention(dev, layout, hq=8, hk=2, dim=64, ps=16):
    g = torch.Generator().manual_seed(3)
    kv = (9, ps, hk, dim) if layout == "NHD" else (9, hk, ps, dim)
    k, v = (torch.randn(kv, generator=g).bfloat16().to(dev) for _ in range(2))
    tables = torch.randperm(8, generator=g)[:6].reshape(2, 3).to(torch.int32).to(dev)
    lens = torch.tensor([40, 17], dtype=torch.int32, device=dev)
    return (k, v), tables, lens, torch.full((1 << 20,), 255, dtype=torch.uint8, device=dev)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["NHD", "HND"])
@pytest.mark.parametrize("quant", [None, 0.05, "tensor"])
def test_attention_matches_the_general_way(mas, dev, layout, quant):
    mas.load_library()
    d = mas._lib.direct
    kv, tables, lens, ws = _attention(dev, layout)
    quant = torch.tensor([0.05], device=dev) if quant == "tensor" else quant
    qkv = torch.randn(11, 12 * 64, device=dev).bfloat16()
    cu = torch.tensor([0, 8, 11], dtype=torch.int32, device=dev)
    flags = torch.zeros(1, dtype=torch.int32, device=dev)

    def out_of(q):
        return torch.zeros(q.shape, device=dev).to(torch.bfloat16 if quant is None else FP8)

    q = qkv[:, : 8 * 64].view(11, 8, 64)
    a, b = out_of(q), out_of(q)
    for w in (ws, None):
        a.view(torch.uint8).fill_(17)
        b.view(torch.uint8).fill_(34)
        assert d.context_attention(q, kv, w, tables, lens, cu, 8, 40, 0.1, 1.0, a, layout, flags, quant) == 0
        mas.attention._context(q, kv, tables, lens, cu, 8, 0.1, 1.0, b, layout, flags, quant, w, 40)
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    q = q[:2]
    a, b = out_of(q), out_of(q)
    assert d.decode_attention(q, kv, ws, tables, lens, 0.1, 1.0, a, layout, flags, quant) == 0
    mas.attention._decode(q, kv, ws, tables, lens, 0.1, 1.0, b, layout, flags, quant)
    assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)) and int(flags.item()) == 0
    call = [q, kv, ws, tables, lens, 0.1, 1.0, a, layout, flags, quant]
    for at, other in ((0, q[:, :3]), (1, list(kv)), (2, None), (3, tables.long()), (4, lens[:1]), (5, 1), (7, a[:1]),
                      (8, "DNH"), (9, flags.long())):
        assert d.decode_attention(*call[:at], other, *call[at + 1:]) is None


@pytest.mark.gpu
@pytest.mark.parametrize("beta", [0.0, 0.1])
@pytest.mark.parametrize("layout", ["NHD", "HND"])
@pytest.mark.parametrize("neox", [True, False])
def test_rope_append_matches_the_general_way(mas, dev, beta, layout, neox):
    kv, tables, _, _ = _attention(dev, layout)
    qkv = torch.randn(5, 12 * 64, device=dev).bfloat16()
    pos = torch.tensor([0, 39, 3, 4, 16], dtype=torch.int32, device=dev)
    batch = torch.tensor([0, 0, 1, 1, 1], dtype=torch.int32, device=dev)
    indptr = torch.tensor([0, 3, 6], dtype=torch.int32, device=dev)
    table = mas.rope.cos_sin_cache(64, 64, 1e6).to(dev)
    got = []
    for public in (True, True, False):  # the public call's first run makes the query scale table
        x, cache = qkv.clone(), (kv[0].clone(), kv[1].clone())
        q, k, v = x[:, :512], x[:, 512:640], x[:, 640:].unflatten(-1, (2, 64))
        args = pos, q, k, v, 64, table, neox, batch, cache, tables.flatten(), indptr
        if public:
            mas.fused.apply_rope_and_append_paged_kv_cache(*args, None, layout, llama_4_scaling_beta=beta,
                                                           original_max_position_embeddings=16)
        else:
            mas.fused._fused(*args, layout, None, beta, 16)
        got.append((x, *cache))
    for other in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got[0], other))
    with pytest.raises(ValueError, match="same number of rows"):
        mas.fused.apply_rope_and_append_paged_kv_cache(pos[:4], *args[1:], None, layout)
    with pytest.raises(ValueError, match="head_dim"):
        mas.fused.apply_rope_and_append_paged_kv_cache(pos, q, k, v, 32, *args[5:], None, layout)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["NHD", "HND"])
@pytest.mark.parametrize("scaled", [False, True])
def test_rope_append_takes_the_layers_forms(mas, dev, layout, scaled):
    """The native call itself, of which the public one would hide a refusal."""
    mas.load_library()
    d = mas._lib.direct
    kv, tables, _, _ = _attention(dev, layout)
    pos = torch.tensor([0, 39, 3, 4, 16], dtype=torch.int32, device=dev)
    batch = torch.tensor([0, 0, 1, 1, 1], dtype=torch.int32, device=dev)
    indptr = torch.tensor([0, 3, 6], dtype=torch.int32, device=dev)
    table = mas.rope.cos_sin_cache(64, 64, 1e6).to(dev)
    flags = torch.zeros(1, dtype=torch.int32, device=dev)
    scale = (mas.fused.llama_4_q_scale_table(0.1, 16, 4, dev), 16) if scaled else (None, 0)
    qkv = torch.randn(5, 12 * 64, device=dev).bfloat16()
    got = []
    for native in (True, False):
        x, cache = qkv.clone(), (kv[0].clone(), kv[1].clone())
        q, k, v = x[:, :512], x[:, 512:640], x[:, 640:].unflatten(-1, (2, 64))
        args = [pos, q, k, v, 64, table, True, batch, cache, tables.flatten(), indptr, layout, flags]
        if native:
            assert d.rope_append(*args, *scale) == 0
        else:
            mas.fused._fused(*args, *((0.1, 16) if scaled else ()))
        got.append((x, *cache))
    assert all(torch.equal(a, b) for a, b in zip(*got)) and int(flags.item()) == 0
    assert not torch.equal(got[0][0], qkv) and not torch.equal(got[0][1], kv[0])
    call, before = [*args, *scale], x.clone()
    for at, other in ((0, pos[:4]), (0, pos.long()), (1, q[:, :500]), (1, q.float()), (2, k[:, :64]), (3, v[:4]), (4, 32),
                      (5, table[:, :32]), (5, table.double()), (6, 1), (7, batch.cpu()), (8, list(cache)),
                      (9, tables), (10, indptr.long()), (11, "DNH"), (12, flags.float()), (13, table[0])):
        assert d.rope_append(*call[:at], other, *call[at + 1:]) is None
    assert torch.equal(x, before)
