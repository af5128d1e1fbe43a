"""Timed cases of the layer kernels: what a serving engine on this package runs, each through a public entry point.

The sizes are those of ``workloads.SHAPES`` / ``ATTENTION_SHAPES`` / ``CONTEXT_SHAPES`` / ``STEP_SHAPES``
(Devstral-Small-2 24B: 32 query heads over 8 kv heads, hidden 5120, intermediate 32768; Devstral-2 123B: 96 over 8,
12288, 28672; 16-slot pages by default, 256-slot pages in the large configurations), plus ragged ones around them.
Sequence lengths come from the case alone (its ``lens`` seed), so that a pass's work does not depend on the values'
seed; the seed orders them over the rows and draws the values, pages and tables.
"""
from __future__ import annotations

import math
import random

import torch

from __graft_entry__ import load_package

mas = load_package()
workloads = mas.workloads

HEAD_DIM = 128
SCALE = HEAD_DIM ** -0.5
ACT_SCALE = 0.05           # the fp8 activation scale of the benchmark's fp8 dataflow
EPS = 1e-5
WORKSPACE = 128 << 20      # the engine's attention workspace
FP8 = torch.float8_e4m3fn
MAX_POSITION = 32768


def listed():
    return [
        # One RMSNorm + residual on [256, 5120]: the single-op configuration, and what a decode batch of 256 calls
        # twice per layer. Latency counts.
        {"name": "norm_256x5120", "op": "norm", "rows": 256, "hidden": 5120, "fp8": False},
        # The in-layer norm of an 8192-token prefill step, fp8 out (the qkv / gate_up GEMM's input).
        {"name": "norm_quant_8192x5120", "op": "norm", "rows": 8192, "hidden": 5120, "fp8": True},
        # SiluAndMul fused with the down_proj input's quantize in the same step: its largest memory stream.
        {"name": "silu_quant_8192x32768", "op": "silu", "rows": 8192, "inter": 32768, "fp8": True},
        # RoPE + llama-4 query scale + KV append of 4 prompts of 2048 tokens, 16-slot pages.
        {"name": "rope_append_8192", "op": "rope", "seqs": 4, "new": 2048, "cached": 0, "q_heads": 32, "kv_heads": 8,
         "page_size": 16, "q_scale": True},
        # One conversation being decoded: the smallest attention call, all latency.
        {"name": "decode_1x4096_24b", "op": "decode", "rows": 1, "max_len": 4096, "reach": 8192, "q_heads": 32,
         "kv_heads": 8, "page_size": 16, "fp8": False, "lens": 9},
        # A full decode batch: 64 rows of 1..8192 positions. Most of a decode step's time.
        {"name": "decode_64x8192_24b", "op": "decode", "rows": 64, "max_len": 8192, "reach": 8192, "q_heads": 32,
         "kv_heads": 8, "page_size": 16, "fp8": False, "lens": 0},
        # A middling batch of the larger model's heads, fp8 out (the o_proj input), 256-slot pages, odd lengths
        # under a table that reaches further.
        {"name": "decode_24x3000_123b", "op": "decode", "rows": 24, "max_len": 3000, "reach": 8192, "q_heads": 96,
         "kv_heads": 8, "page_size": 256, "fp8": True, "lens": 2},
        # Fresh prompts, 24B heads: the attention of an 8192-token prefill step.
        {"name": "context_4x2048_24b", "op": "context", "rows": 4, "new": 2048, "cached": 0, "ragged": False,
         "q_heads": 32, "kv_heads": 8, "page_size": 16, "fp8": False, "lens": 0},
        # Fresh prompts, 123B heads: the largest call.
        {"name": "context_4x4096_123b", "op": "context", "rows": 4, "new": 4096, "cached": 0, "ragged": False,
         "q_heads": 96, "kv_heads": 8, "page_size": 256, "fp8": False, "lens": 0},
        # An agent's turn: a few new tokens after a long cached prefix.
        {"name": "context_turn_128_after4096", "op": "context", "rows": 1, "new": 128, "cached": 4096, "ragged": False,
         "q_heads": 32, "kv_heads": 8, "page_size": 16, "fp8": False, "lens": 0},
        # Chunked prefill as it arrives: prompts of odd lengths after odd cached prefixes, fp8 out.
        {"name": "context_ragged_6x1500", "op": "context", "rows": 6, "new": 1500, "cached": 3000, "ragged": True,
         "q_heads": 32, "kv_heads": 8, "page_size": 16, "fp8": True, "lens": 3},
        # A whole captured step of 4 layers, as the engine replays it: 28 decode rows and a 100-token turn after
        # 4000 cached positions in the runner's 17 prompt rows.
        {"name": "step_28x8192_turn_4layers", "op": "step", "rows": 28, "max_len": 8192, "layers": 4, "new": 100,
         "cached": 4000, "lens": 0},
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


#: No drawn case costs more than the largest listed one (floating-point operations; bytes of the streams).
_MOST_FLOPS, _MOST_BYTES = 1.2e12, 3.0e9


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] <= _MOST_FLOPS and w["bytes"] <= _MOST_BYTES:
            return case


def _draw(rng):
    op = rng.choice(("norm", "silu", "rope", "decode", "decode", "decode", "context", "context", "context", "step"))
    if op == "norm":
        return {"op": op, "rows": _spread(rng, 1, 16384), "hidden": rng.choice((5120, 12288)),
                "fp8": rng.random() < 0.5}
    if op == "silu":
        return {"op": op, "rows": _spread(rng, 1, 16384), "inter": rng.choice((32768, 28672)),
                "fp8": rng.random() < 0.5}
    if op == "step":
        rows = rng.randint(1, 63)
        turn = rng.random() < 0.5
        return {"op": op, "rows": rows, "max_len": _spread(rng, 64, 8192), "layers": rng.randint(2, 4),
                "new": 64 * rng.randint(1, 3) - rows if turn else 0, "cached": rng.randint(1, 5000) if turn else 0,
                "lens": rng.randint(0, 999)}
    kv = rng.choice((8, 8, 8, 4, 1))                      # whole, or a shard's kv heads
    heads = {"q_heads": kv * rng.choice((4, 12)), "kv_heads": kv, "page_size": rng.choice((16, 16, 64, 256))}
    if op == "rope":
        return {"op": op, "seqs": rng.randint(1, 8), "new": _spread(rng, 1, 3000), "cached": rng.randint(0, 4000),
                **heads, "q_scale": rng.random() < 0.5}
    if op == "decode":
        most = _spread(rng, 32, 20000)
        return {"op": op, "rows": _spread(rng, 1, 200), "max_len": most,
                "reach": most if rng.random() < 0.5 else max(8192, most), **heads, "fp8": rng.random() < 0.5,
                "lens": rng.randint(0, 999)}
    return {"op": op, "rows": _spread(rng, 1, 12), "new": _spread(rng, 8, 5000),
            "cached": 0 if rng.random() < 0.4 else _spread(rng, 1, 9000), "ragged": rng.random() < 0.6, **heads,
            "fp8": rng.random() < 0.5, "lens": rng.randint(0, 999)}


# ---- lengths -----------------------------------------------------------------------------------------

def _decode_lens(case):
    r = random.Random(case["lens"])
    return [r.randint(1, case["max_len"]) for _ in range(case["rows"])]


def _context_lens(case):
    """(new tokens, cached positions) of each row."""
    if not case["ragged"]:
        return [(case["new"], case["cached"])] * case["rows"]
    r = random.Random(case["lens"])
    return [(r.randint(1, case["new"]), r.randint(0, case["cached"])) for _ in range(case["rows"])]


def _step_shape(case):
    prompts = ((case["new"], case["cached"]),) if case["new"] else ()
    return workloads.StepShape("step", case["rows"], case["max_len"], prompts=prompts, layers=case["layers"])


# ---- what a pass cannot do without ---------------------------------------------------------------------

def _attended(n, c):
    """(query, key) pairs of n new tokens after c cached positions, causal."""
    return n * c + n * (n + 1) // 2


def work(case):
    op = case["op"]
    if op == "norm":
        n, h = case["rows"], case["hidden"]
        return {"bytes": (7 if case["fp8"] else 8) * n * h + 2 * h, "flops": 5 * n * h}
    if op == "silu":
        n, i = case["rows"], case["inter"]
        return {"bytes": (5 if case["fp8"] else 6) * n * i, "flops": 6 * n * i}
    if op == "rope":
        n, hq, hk = case["seqs"] * case["new"], case["q_heads"], case["kv_heads"]
        return {"bytes": n * (4 * (hq + hk) * HEAD_DIM + 6 * hk * HEAD_DIM + 8), "flops": 3 * n * (hq + hk) * HEAD_DIM}
    if op == "decode":
        lens, hq, hk = _decode_lens(case), case["q_heads"], case["kv_heads"]
        out = 1 if case["fp8"] else 2
        pages = sum(-(-n // case["page_size"]) for n in lens)
        return {"bytes": sum(lens) * hk * HEAD_DIM * 4 + len(lens) * (hq * HEAD_DIM * (2 + out) + 4) + 4 * pages,
                "flops": 4 * sum(lens) * hq * HEAD_DIM}
    if op == "context":
        lens, hq, hk = _context_lens(case), case["q_heads"], case["kv_heads"]
        tokens, out = sum(n for n, _ in lens), 1 if case["fp8"] else 2
        return {"bytes": sum(n + c for n, c in lens) * hk * HEAD_DIM * 4 + tokens * hq * HEAD_DIM * (2 + out),
                "flops": 4 * sum(_attended(n, c) for n, c in lens) * hq * HEAD_DIM}
    ls = _step_shape(case).layer
    d, new, cached = case["rows"], case["new"], case["cached"]
    n, decoded = d + new, workloads.make_step_layout(_step_shape(case), case["lens"]).decode_positions
    hq, hk = ls.q_heads, ls.kv_heads
    layer = (14 * n * ls.hidden + 5 * n * ls.inter + n * (4 * (hq + hk) + 6 * hk) * HEAD_DIM
             + (decoded + (new + cached if new else 0)) * hk * HEAD_DIM * 4 + 3 * n * hq * HEAD_DIM)
    attn = 4 * hq * HEAD_DIM * (decoded + _attended(new, cached))
    return {"bytes": case["layers"] * layer + 12 * n * ls.hidden, "flops": case["layers"] * attn}


def tolerance(case):
    """About four times what two orders of the fp32 sums, or the fp32 result and the 64-bit one, differ by once
    rounded: bf16 outputs (2^-9 per value) and fp8 e4m3 outputs (2^-4), the latter only where a sum in another order
    moves a value over a rounding boundary."""
    if case["op"] == "rope":
        return "exact"                       # the table's values times bf16 pairs: one product order, one rounding
    if case["op"] in ("norm", "silu"):
        return {"rel": 0.01, "max": 0.15} if case["fp8"] else {"rel": 0.007, "max": 0.02}
    if case["op"] == "step" or case["fp8"]:
        return {"rel": 0.02, "max": 0.25}
    return {"rel": 0.008, "max": 0.05}


# ---- inputs --------------------------------------------------------------------------------------------

class _Values:
    """Seeded N(0, 1) tensors drawn on the GPU, and seeded choices on the host."""

    def __init__(self, seed):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)
        self.rng = random.Random(seed)
        self.host = torch.Generator().manual_seed(seed)

    def normal(self, *size):
        return torch.randn(*size, generator=self.gen, device=self.dev, dtype=torch.bfloat16)

    def weight(self, n):
        return (1 + 0.1 * torch.randn(n, generator=self.gen, device=self.dev)).to(torch.bfloat16)

    def ints(self, values, dtype=torch.int32):
        return torch.tensor(values, dtype=dtype, device=self.dev)

    def tables(self, lens, page_size, reach):
        """Block tables of rows of `lens` positions over a pool that just holds them, pages in random order;
        columns past a row's pages point at the pool's last page."""
        need = [-(-n // page_size) for n in lens]
        pages = sum(need) + 1
        width = max(max(need), -(-reach // page_size))
        perm = torch.randperm(pages - 1, generator=self.host).to(torch.int32)
        tables = torch.full((len(lens), width), pages - 1, dtype=torch.int32)
        at = 0
        for row, k in enumerate(need):
            tables[row, :k] = perm[at:at + k]
            at += k
        return tables.to(self.dev), pages


def _step(case, values):
    """The step of the case's lengths, its stand-ins, caches and embedding table drawn from the seed."""
    step = mas.layer_pass.ForwardStep(_step_shape(case), values.dev, seed=case["lens"], act_scale=ACT_SCALE)
    drawn = [step.final_in, step.embed_table]
    for layer in step.layers:
        drawn += [layer[k] for k in ("hidden", "qkv", "o_proj", "gate_up", "k_cache", "v_cache")]
    for t in drawn:
        t.normal_(generator=values.gen)
    return step


def prepare(case, seed):
    v, op = _Values(seed), case["op"]
    s = {"case": case, "act": torch.tensor(ACT_SCALE, device=v.dev)}
    if op == "norm":
        n, h = case["rows"], case["hidden"]
        s.update(x=v.normal(n, h), residual=v.normal(n, h), weight=v.weight(h))
        if case["fp8"]:
            s["out"] = torch.empty(n, h, dtype=FP8, device=v.dev)
    elif op == "silu":
        n, i = case["rows"], case["inter"]
        s.update(x=v.normal(n, 2 * i), out=torch.empty(n, i, dtype=FP8 if case["fp8"] else torch.bfloat16, device=v.dev))
    elif op == "rope":
        hq, hk, new, cached = case["q_heads"], case["kv_heads"], case["new"], case["cached"]
        n = case["seqs"] * new
        tables, pages = v.tables([cached + new] * case["seqs"], case["page_size"], 0)
        kv = (pages, case["page_size"], hk, HEAD_DIM)
        s.update(qkv=v.normal(n, (hq + 2 * hk) * HEAD_DIM), k_cache=torch.zeros(kv, dtype=torch.bfloat16, device=v.dev),
                 v_cache=torch.zeros(kv, dtype=torch.bfloat16, device=v.dev),
                 positions=torch.arange(cached, cached + new, dtype=torch.int32, device=v.dev).repeat(case["seqs"]),
                 batch=torch.arange(case["seqs"], dtype=torch.int32, device=v.dev).repeat_interleave(new),
                 tables=tables, kv_indices=tables.flatten(),
                 kv_indptr=v.ints([r * tables.shape[1] for r in range(case["seqs"] + 1)]),
                 table=mas.rope.cos_sin_cache(MAX_POSITION, HEAD_DIM, 1e6).to(v.dev))
    elif op in ("decode", "context"):
        hq, hk = case["q_heads"], case["kv_heads"]
        if op == "decode":
            kv_lens = _decode_lens(case)
            v.rng.shuffle(kv_lens)
            tokens, reach = len(kv_lens), case["reach"]
        else:
            lens = _context_lens(case)
            v.rng.shuffle(lens)
            kv_lens, tokens, reach = [n + c for n, c in lens], sum(n for n, _ in lens), 0
            cu = [0]
            for n, _ in lens:
                cu.append(cu[-1] + n)
            s.update(cu=v.ints(cu), max_q=max(n for n, _ in lens), max_kv=max(kv_lens), cu_host=cu)
        tables, pages = v.tables(kv_lens, case["page_size"], reach)
        kv = (pages, case["page_size"], hk, HEAD_DIM)
        s.update(q=v.normal(tokens, hq, HEAD_DIM), k_cache=v.normal(*kv), v_cache=v.normal(*kv), tables=tables,
                 seq_lens=v.ints(kv_lens), lens_host=kv_lens,
                 workspace=torch.zeros(WORKSPACE, dtype=torch.uint8, device=v.dev),
                 out=torch.empty(tokens, hq, HEAD_DIM, dtype=FP8 if case["fp8"] else torch.bfloat16, device=v.dev))
    else:
        s["step"] = step = _step(case, v)
        changed = [step.residual, step.final_in, step.layers[0]["hidden"]] + [x["qkv"] for x in step.layers]
        kept = [t.clone() for t in changed]
        step.run()                            # outside capture once, as the runner warms its graphs up
        for t, k in zip(changed, kept):
            t.copy_(k)
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            step.run()
    return s


# ---- a pass --------------------------------------------------------------------------------------------

def run(s):
    case = s["case"]
    op = case["op"]
    if op == "norm":
        if case["fp8"]:
            mas.norm.fused_add_rmsnorm_quant(s["out"], s["x"], s["residual"], s["weight"], s["act"], EPS)
            return {"out": s["out"], "residual": s["residual"]}
        mas.norm.fused_add_rmsnorm(s["x"], s["residual"], s["weight"], EPS)
        return {"out": s["x"], "residual": s["residual"]}
    if op == "silu":
        if case["fp8"]:
            return {"out": mas.activation.silu_and_mul_quant(s["x"], s["act"], out=s["out"])}
        return {"out": mas.activation.silu_and_mul(s["x"], out=s["out"])}
    if op == "rope":
        q, k, v = _qkv(s["qkv"], case["q_heads"], case["kv_heads"])
        mas.fused.apply_rope_and_append_paged_kv_cache(
            s["positions"], q, k, v.unflatten(-1, (case["kv_heads"], HEAD_DIM)), HEAD_DIM, s["table"], True, s["batch"],
            (s["k_cache"], s["v_cache"]), s["kv_indices"], s["kv_indptr"], None, "NHD",
            llama_4_scaling_beta=0.1 if case["q_scale"] else 0.0,
            original_max_position_embeddings=8192 if case["q_scale"] else 0)
        return {"qkv": s["qkv"], "k_cache": s["k_cache"], "v_cache": s["v_cache"]}
    if op == "decode":
        return {"out": mas.attention.trtllm_batch_decode_with_kv_cache(
            s["q"], (s["k_cache"], s["v_cache"]), s["workspace"], s["tables"], s["seq_lens"], case["reach"], SCALE, 1.0,
            out=s["out"], out_quant_scale=s["act"] if case["fp8"] else None)}
    if op == "context":
        return {"out": mas.attention.trtllm_batch_context_with_kv_cache(
            s["q"], (s["k_cache"], s["v_cache"]), s["workspace"], s["tables"], s["seq_lens"], s["max_q"], s["max_kv"],
            SCALE, 1.0, case["rows"], s["cu"], None, out=s["out"], out_quant_scale=s["act"] if case["fp8"] else None)}
    s["graph"].replay()
    step = s["step"]
    return {"residual": step.residual, "final": step.final_in, "norm": step.norm_out, "attn": step.attn_out,
            "silu": step.silu_out, "qkv": [x["qkv"] for x in step.layers],
            "caches": [(x["k_cache"], x["v_cache"]) for x in step.layers]}


def _qkv(qkv, hq, hk):
    a, b = hq * HEAD_DIM, (hq + hk) * HEAD_DIM
    return qkv[:, :a], qkv[:, a:b], qkv[:, b:]


# ---- the same in 64 bits -------------------------------------------------------------------------------

def _norm64(x, residual, weight):
    s = x.double() + residual.double()
    return s * torch.rsqrt(s.square().mean(-1, keepdim=True) + EPS) * weight.double(), s


def _quant64(y):
    return (y / float(torch.tensor(ACT_SCALE))).clamp(-448, 448)


def _silu64(x):
    gate, up = x.double().chunk(2, -1)
    return gate / (1 + torch.exp(-gate)) * up


def _rope64(x, positions, table):
    """Rotated heads of x [tokens, heads, HEAD_DIM], halves paired."""
    rows = table[positions.long()].double()[:, None, :]
    c, s = rows.chunk(2, -1)
    a, b = x.double().chunk(2, -1)
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _attend64(q, k, v, cached):
    """Causal attention of q [n, Hq, D] at positions cached .. over k, v [cached + n, Hk, D]."""
    n, hq, d = q.shape
    hk = k.shape[1]
    g = hq // hk
    out = torch.empty(n, hq, d, dtype=torch.float64, device=q.device)
    at = torch.arange(k.shape[0], device=q.device)[None, :] > torch.arange(cached, cached + n, device=q.device)[:, None]
    for h in range(hk):
        kt, vh = k[:, h].double().t().contiguous(), v[:, h].double().contiguous()
        for e in range(h * g, (h + 1) * g):
            scores = torch.mm(q[:, e].double().contiguous(), kt) * SCALE
            if n > 1:
                scores.masked_fill_(at, -math.inf)
            out[:, e] = torch.mm(torch.softmax(scores, -1), vh)
    return out


def _rows64(cache, table, length):
    page_size = cache.shape[1]
    pages = table[: -(-length // page_size)].long()
    return cache[pages].flatten(0, 1)[:length]


def exact(case, seed):
    op = case["op"]
    if op == "step":
        return _exact_step(case, seed)
    s = prepare(case, seed)
    if op == "norm":
        y, residual = _norm64(s["x"], s["residual"], s["weight"])
        return {"out": _quant64(y) if case["fp8"] else y, "residual": residual}
    if op == "silu":
        y = torch.cat([_silu64(x) for x in s["x"].split(1024)])
        return {"out": _quant64(y) if case["fp8"] else y}
    if op == "rope":
        hq, hk = case["q_heads"], case["kv_heads"]
        q, k, v = (t.unflatten(-1, (-1, HEAD_DIM)) for t in _qkv(s["qkv"], hq, hk))
        pos = s["positions"].long()
        q, k, v = _rope64(q, pos, s["table"]), _rope64(k, pos, s["table"]), v.double()
        if case["q_scale"]:
            q = q * (1 + 0.1 * torch.log1p(torch.floor(pos.double() / 8192)))[:, None, None]
        page = s["tables"][s["batch"].long(), pos // case["page_size"]].long()
        caches = []
        for x in (k, v):
            c = torch.zeros(s["k_cache"].shape, dtype=torch.float64, device=x.device)
            c[page, pos % case["page_size"]] = x
            caches.append(c)
        return {"qkv": torch.cat([t.flatten(1) for t in (q, k, v)], -1), "k_cache": caches[0], "v_cache": caches[1]}
    out = torch.empty(s["q"].shape, dtype=torch.float64, device=s["q"].device)
    first = list(range(case["rows"] + 1)) if op == "decode" else s["cu_host"]
    for r, length in enumerate(s["lens_host"]):
        a, b = first[r], first[r + 1]
        out[a:b] = _attend64(s["q"][a:b], _rows64(s["k_cache"], s["tables"][r], length),
                             _rows64(s["v_cache"], s["tables"][r], length), length - (b - a))
    return {"out": _quant64(out) if case["fp8"] else out}


def _exact_step(case, seed):
    step = _step(case, _Values(seed))
    ls, d = step.shape.layer, step.num_decodes
    pos = step.positions.long()
    residual = torch.zeros_like(step.residual, dtype=torch.float64)
    step.layers[0]["hidden"].copy_(step.embed_table[step.ids])
    qkvs = []
    for layer in step.layers:
        _, residual = _norm64(layer["hidden"], residual, layer["w_in"])
        q, k, val = (t.unflatten(-1, (-1, HEAD_DIM)) for t in _qkv(layer["qkv"], ls.q_heads, ls.kv_heads))
        q, k, val = _rope64(q, pos, step.table), _rope64(k, pos, step.table), val.double()
        q = q * (1 + 0.1 * torch.log1p(torch.floor(pos.double() / step.LLAMA_4_ORIGINAL_MAX)))[:, None, None]
        qkvs.append(torch.cat([t.flatten(1) for t in (q, k, val)], -1))
        post, residual = _norm64(layer["o_proj"], residual, layer["w_post"])
    # the last layer's attention, over its cache with the step's own keys and values in place
    layer, attn = step.layers[-1], torch.empty(q.shape, dtype=torch.float64, device=q.device)
    cu = [0] * (step.num_prefills + 1) if step.num_prefills == 0 else step.cu_seqlens_q.tolist()
    spans = [(r, r + 1) for r in range(d)] + [(d + a, d + b) for a, b in zip(cu, cu[1:])]
    for r, (a, b) in enumerate(spans):
        if a == b:
            continue
        length = int(step.seq_lens[r])
        kr = _rows64(layer["k_cache"], step.block_tables[r], length).double()
        vr = _rows64(layer["v_cache"], step.block_tables[r], length).double()
        kr[length - (b - a):], vr[length - (b - a):] = k[a:b], val[a:b]
        attn[a:b] = _attend64(q[a:b], kr, vr, length - (b - a))
    final, residual = _norm64(step.final_in, residual, step.final_weight)
    return {"residual": residual, "final": final, "norm": _quant64(post), "attn": _quant64(attn),
            "silu": _quant64(_silu64(layer["gate_up"])), "qkv": qkvs,
            "caches": [(None, None) for _ in step.layers]}
