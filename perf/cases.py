"""The work that serving with this framework consists of, as cases that can be timed one by one.

A case is one layer's worth of one kind of work in one engine step, taken through the entry points that the models call:
the Llama path's attention module (cache write and attention), the int4 linear layers, the routed experts, the paged
attention of the mixer models and their recurrent token mixers -- each for prompt steps and for decode steps, in the data
types and with the options that the configurations use.

``listed()`` names the standing cases, ``draw(rng)`` gives further ones of the same ranges, ``prepare(case, seed)`` makes
what a program has in hand before the call (inputs from the seed, caches, states, weights, the step's metadata),
``run(state)`` is one pass, ``work(case)`` the bytes and operations that it cannot do without, ``exact(case, seed)`` its
result in 64 bits and ``tolerance(case)`` how far another correct implementation may be from it.

Lengths of a ragged step follow from the case alone (``spread``), values from the seed alone.
"""
import math
import os
import sys
from types import SimpleNamespace

import torch

_PACKAGE_ROOT = os.path.join(os.getcwd(), "vllm-splitwise_amd")
if _PACKAGE_ROOT not in sys.path:
    sys.path.insert(0, _PACKAGE_ROOT)

from splitwise_amd import _C                                                          # noqa: E402
from splitwise_amd.model_executor.input_metadata import InputMetadata, RaggedBatch    # noqa: E402
from splitwise_amd.model_executor.layers.attention import Attention                   # noqa: E402

DEV = "cuda"
BLOCK = 16                                   # tokens per cache block, the engine's default
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
EPS = 1e-6
TAPS = 4                                     # of the short convolution in front of the delta rule
TAU = 16.0                                   # of the gated linear attention's decay


# ------------------------------------------------------------------------------------------------------ the cases
def listed():
    llama7 = dict(heads=32, kv_heads=32, dim=128, dtype="bf16", cache="auto")
    return [
        # a chat with hardly anybody on the machine: two conversations decode, every launch is mostly latency
        dict(name="decode-few", kind="decode", seqs=2, ctx=700, **llama7),
        # a full co-located machine: 256 conversations of prompt 772 + what they have generated so far, Llama-2-7B
        dict(name="decode-full", kind="decode", seqs=251, ctx=857, **llama7),
        # grouped-query attention (64 query heads on 8) over the fp8 cache, longer contexts
        dict(name="decode-gqa-fp8", kind="decode", seqs=61, ctx=2011, heads=64, kv_heads=8, dim=128, dtype="f16",
             cache="fp8_e5m2"),
        # a prompt step: three prompts of about 772 tokens, Llama-2-7B
        dict(name="prompt", kind="prompt", seqs=3, new=773, **llama7),
        # the four GPTQ int4 matrices of a Llama-2-13B layer in a decode step of 61 sequences
        dict(name="int4-decode", kind="int4", rows=61, width=5120, ff=13824),
        # routed experts of a mixer model: a prompt step and a decode step (32 experts, two per token, silu-gated)
        dict(name="experts-prompt", kind="experts", rows=3989, width=2048, ff=1024, experts=32, top=2, act="glu"),
        dict(name="experts-decode", kind="experts", rows=61, width=2048, ff=1024, experts=32, top=2, act="glu"),
        # the mixer models' attention with fp32 scores and weights: a prompt step with capped scores and an output gate,
        # a decode step with a sink
        dict(name="mixer-attention-prompt", kind="attention", seqs=2, ctx=0, new=2041, heads=16, kv_heads=4, dim=128,
             softcap=30.0, window=0, sink=False, gate=True),
        dict(name="mixer-attention-decode", kind="attention", seqs=61, ctx=2041, new=1, heads=16, kv_heads=4, dim=128,
             softcap=0.0, window=0, sink=True, gate=False),
        # the gated delta rule with its convolution in front and its norm and gate behind: a prompt and a decode step
        dict(name="delta-prompt", kind="delta", seqs=2, new=2041, heads=16, kv_heads=8, dim=128),
        dict(name="delta-decode", kind="delta", seqs=61, new=1, heads=16, kv_heads=8, dim=128),
        # gated linear attention with its norm and gate: a prompt step
        dict(name="linear-prompt", kind="linear", rule="gla", seqs=2, new=2041, heads=16, dim=128),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, even over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        rows = case.get("rows") or case["seqs"] * case.get("new", 1)
        # no larger than the listed cases: a full machine's decode step, a prompt step of about 4096 rows
        if rows <= 4200 and w["bytes"] <= 3.5e9 and w["flops"] <= 1.1e11:
            return case


def _draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "int4", "experts", "experts", "attention", "attention", "delta", "delta",
                       "linear"])
    if kind in ("decode", "prompt"):
        heads, kv_heads, dim = rng.choice([(32, 32, 128), (40, 40, 128), (64, 8, 128), (16, 2, 128), (32, 8, 128), (12, 12, 64)])
        case = dict(kind=kind, heads=heads, kv_heads=kv_heads, dim=dim, dtype=rng.choice(["bf16", "bf16", "f16"]),
                    cache=rng.choice(["auto", "auto", "fp8_e5m2"]))
        if kind == "decode":
            return dict(case, seqs=_log(rng, 1, 256), ctx=_log(rng, 64, 4096))
        return dict(case, seqs=rng.randint(1, 8), new=_log(rng, 33, 2100))
    if kind == "int4":
        width, ff = rng.choice([(4096, 11008), (5120, 13824)])
        return dict(kind=kind, rows=_log(rng, 1, 256), width=width, ff=ff)
    if kind == "experts":
        return dict(kind=kind, rows=_log(rng, 1, 4100), width=rng.choice([768, 1024, 2048]), ff=rng.choice([512, 704, 1024]),
                    experts=rng.choice([8, 16, 32, 64]), top=rng.choice([1, 2, 4]), act=rng.choice(["glu", "relu2", "gelu"]))
    if kind == "attention":
        heads, kv_heads, dim = rng.choice([(16, 4, 128), (16, 8, 128), (8, 2, 128), (12, 4, 64), (16, 16, 64), (16, 4, 96)])
        decode = rng.random() < 0.5
        return dict(kind=kind, seqs=_log(rng, 1, 64) if decode else rng.randint(1, 4),
                    ctx=_log(rng, 64, 4096) if decode else rng.choice([0, 0, _log(rng, 64, 1024)]),
                    new=1 if decode else _log(rng, 40, 2050), heads=heads, kv_heads=kv_heads, dim=dim,
                    softcap=rng.choice([0.0, 30.0]), window=rng.choice([0, 0, 1024]), sink=rng.random() < 0.5,
                    gate=rng.random() < 0.5)
    decode = rng.random() < 0.4
    steps = dict(seqs=_log(rng, 1, 64) if decode else rng.randint(1, 4), new=1 if decode else _log(rng, 40, 2050))
    if kind == "delta":
        heads, kv_heads, dim = rng.choice([(16, 8, 128), (8, 8, 128), (16, 4, 64), (12, 12, 96)])
        return dict(kind=kind, heads=heads, kv_heads=kv_heads, dim=dim, **steps)
    heads, dim = rng.choice([(16, 128), (4, 128), (8, 128), (16, 64)])
    return dict(kind=kind, rule=rng.choice(["gla", "lightning", "retention"]), heads=heads, dim=dim, **steps)


def spread(mean, count):
    """``count`` lengths around ``mean``, none of them alike for the usual counts: what requests of different ages bring."""
    return [max(1, int(mean * (0.75 + 0.5 * ((i * 0.6180339887498949 + 0.31) % 1.0)))) for i in range(count)]


def _lengths(case):
    """[(tokens already there, tokens that this step brings)] per sequence."""
    if case["kind"] == "decode":
        return [(n - 1, 1) if n > 1 else (0, 1) for n in spread(case["ctx"], case["seqs"])]
    new = spread(case["new"], case["seqs"]) if case["new"] > 1 else [1] * case["seqs"]
    ctx = spread(case["ctx"], case["seqs"]) if case.get("ctx") else [0] * case["seqs"]
    return list(zip(ctx, new))


# ---------------------------------------------------------------------------------------------------- inputs by seed
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, dtype=torch.float32, scale=1.0):
    return torch.randn(*shape, generator=g, device=DEV, dtype=dtype) * scale


def _ints(values, dtype=torch.int32):
    return torch.tensor(values, dtype=dtype, device=DEV)


def _pages(g, lengths):
    """Block tables of sequences whose blocks lie anywhere in the pool -> (table int32 [S, width], blocks of the pool)."""
    need = [-(-(c + n) // BLOCK) for c, n in lengths]
    order = torch.randperm(sum(need), generator=g, device=DEV).to(torch.int32)
    table = torch.zeros(len(need), max(need), dtype=torch.int32, device=DEV)
    lo = 0
    for i, n in enumerate(need):
        table[i, :n] = order[lo:lo + n]
        lo += n
    return table, sum(need)


def _slots(table, lengths):
    """Cache slot of every token of the step, in its order."""
    out = []
    for i, (c, n) in enumerate(lengths):
        pos = torch.arange(c, c + n, device=DEV)
        out.append(table[i, pos // BLOCK].long() * BLOCK + pos % BLOCK)
    return torch.cat(out)


def _ragged(lengths, table=None, blocks=1):
    starts, owner = [0], []
    for i, (_, n) in enumerate(lengths):
        starts.append(starts[-1] + n)
        owner += [i] * n
    count = len(lengths)
    if table is None:
        table = torch.zeros(count, 1, dtype=torch.int32, device=DEV)
    return RaggedBatch(q_start=_ints(starts), ctx_len=_ints([c for c, _ in lengths]), token_seq=_ints(owner),
                       state_slot=_ints(list(range(count))), block_tables=table, num_seqs=count,
                       max_query_len=max(n for _, n in lengths), max_pages_used=table.shape[1], max_page_id=blocks - 1,
                       max_state_slot=count - 1)


# ------------------------------------------------------- the Llama path's attention module: cache write and attention
def _cache_tensors(case):
    fp8 = case["cache"] != "auto"
    return fp8, (16 if fp8 else 8), (torch.uint8 if fp8 else DTYPES[case["dtype"]])


def _prepare_llama(case, seed):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    h, kvh, d = case["heads"], case["kv_heads"], case["dim"]
    lengths = _lengths(case)
    rows = sum(n for _, n in lengths)
    fp8, x, cdt = _cache_tensors(case)
    table, blocks = _pages(g, lengths)
    shape_k, shape_v = (blocks, kvh, d // x, BLOCK, x), (blocks, kvh, d, BLOCK)
    if case["kind"] == "decode":
        key_cache, value_cache = _randn(g, *shape_k, dtype=dt), _randn(g, *shape_v, dtype=dt)
        if fp8:
            key_cache, value_cache = (t.to(torch.float8_e5m2).view(torch.uint8) for t in (key_cache, value_cache))
    else:
        key_cache, value_cache = (torch.zeros(s, dtype=cdt, device=DEV) for s in (shape_k, shape_v))
    qkv = _randn(g, rows, (h + 2 * kvh) * d, dtype=dt)       # one projection's output: q, k and v are column ranges
    total = [c + n for c, n in lengths]
    decode = case["kind"] == "decode"
    md = InputMetadata(
        is_prompt=not decode, slot_mapping=_slots(table, lengths), prompt_lens=None if decode else _ints(total),
        max_seq_len=None if decode else max(total),
        start_loc=None if decode else _ints([sum(total[:i]) for i in range(len(total))]),
        max_context_len=max(total) if decode else None, context_lens=_ints(total) if decode else None,
        block_tables=table if decode else None, use_cuda_graph=False,
        kv_cache_dtype=case["cache"], mean_context_len=sum(total) / len(total) if decode else None)
    layer = Attention(h, d, d ** -0.5, kvh)
    return SimpleNamespace(run=_run_llama, layer=layer, q=qkv[:, :h * d], k=qkv[:, h * d:(h + kvh) * d],
                           v=qkv[:, (h + kvh) * d:], key_cache=key_cache, value_cache=value_cache, md=md, table=table)


def _run_llama(s):
    out = s.layer(s.q, s.k, s.v, s.key_cache, s.value_cache, s.md)
    return {"out": out, "key_cache": s.key_cache, "value_cache": s.value_cache}


def _exact_llama(case, seed):
    s = _prepare_llama(case, seed)
    h, kvh, d = case["heads"], case["kv_heads"], case["dim"]
    fp8 = case["cache"] != "auto"
    scale, rep = d ** -0.5, h // kvh
    q, k, v = (t.double().view(t.shape[0], -1, d) for t in (s.q, s.k, s.v))
    out, row = torch.empty_like(q), 0
    for i, (c, n) in enumerate(_lengths(case)):
        ks, vs = k[row:row + n], v[row:row + n]
        if case["kind"] == "decode":
            # what this step's token looks like in the cache, after what the cache holds
            if fp8:
                ks, vs = (t.to(DTYPES[case["dtype"]]).to(torch.float8_e5m2).double() for t in (ks, vs))
            if c > 0:
                blocks = s.table[i, :-(-c // BLOCK)].long()
                kc, vc = s.key_cache[blocks], s.value_cache[blocks]
                if fp8:
                    kc, vc = kc.view(torch.float8_e5m2), vc.view(torch.float8_e5m2)
                kc = kc.double().permute(0, 3, 1, 2, 4).reshape(-1, kvh, d)[:c]
                vc = vc.double().permute(0, 3, 1, 2).reshape(-1, kvh, d)[:c]
                ks, vs = torch.cat([kc, ks]), torch.cat([vc, vs])
        for head in range(kvh):
            qh = q[row:row + n, head * rep:(head + 1) * rep].transpose(0, 1)                 # [rep, n, d]
            score = torch.matmul(qh, ks[:, head].t()) * scale
            if n > 1:
                score.masked_fill_(torch.ones(n, n, dtype=torch.bool, device=DEV).triu(1), -math.inf)
            out[row:row + n, head * rep:(head + 1) * rep] = torch.matmul(score.softmax(-1), vs[:, head]).transpose(0, 1)
        row += n
    return {"out": out.view(row, h * d), "key_cache": None, "value_cache": None}


def _work_llama(case):
    h, kvh, d = case["heads"], case["kv_heads"], case["dim"]
    lengths = _lengths(case)
    rows, elt = sum(n for _, n in lengths), 1 if case["cache"] != "auto" else 2
    act = rows * (2 * h + 2 * kvh) * d * 2                                                   # q, k, v, out
    pairs = sum(n * c + n * (n + 1) // 2 for c, n in lengths)
    return {"bytes": act + 2 * kvh * d * elt * (rows + sum(c for c, _ in lengths)), "flops": 4 * pairs * h * d}


# --------------------------------------------------------------------------------- the int4 matrices of a Llama layer
def _int4_shapes(case):
    w, f = case["width"], case["ff"]
    return [(w, 3 * w), (w, w), (w, 2 * f), (f, w)]          # qkv, o, gate | up, down: (in, out)


def _make_int4(g, k, n):
    groups = k // 128
    q = torch.randint(0, 16, (k, n), generator=g, device=DEV, dtype=torch.int32)
    zero = torch.randint(0, 15, (groups, n), generator=g, device=DEV, dtype=torch.int32)     # stored: one less than used
    scales = ((torch.rand(groups, n, generator=g, device=DEV) * 0.5 + 0.75) * 0.25 * k ** -0.5).half()
    return q, zero, scales


def _pack8(v, dim):
    """Eight 4-bit numbers to a 32-bit word along ``dim``, the first in the lowest bits."""
    v = v.unflatten(dim, (-1, 8))
    at = dim + 1
    out = torch.zeros_like(v.select(at, 0))
    for i in range(8):
        out |= v.select(at, i) << (4 * i)
    return out


def _prepare_int4(case, seed):
    g = _gen(seed)
    layers = []
    for k, n in _int4_shapes(case):
        q, zero, scales = _make_int4(g, k, n)
        qweight = _pack8(q, 0).contiguous()
        _C.ops.gptq_shuffle(qweight, torch.empty((1, 1), device="meta"), 4)      # as a layer does when it is loaded
        layers.append((_randn(g, case["rows"], k, dtype=torch.float16), qweight, _pack8(zero, 1).contiguous(), scales))
    return SimpleNamespace(run=_run_int4, layers=layers, g_idx=torch.empty((1, 1), device="meta"))


def _run_int4(s):
    return [_C.ops.gptq_gemm(x, qweight, qzeros, scales, s.g_idx, True, 4) for x, qweight, qzeros, scales in s.layers]


def _exact_int4(case, seed):
    g, out = _gen(seed), []
    for k, n in _int4_shapes(case):
        q, zero, scales = _make_int4(g, k, n)
        x = _randn(g, case["rows"], k, dtype=torch.float16).double()
        w = (q - (zero + 1).repeat_interleave(128, 0)).double() * scales.double().repeat_interleave(128, 0)
        out.append(torch.matmul(x, w))
    return out


def _work_int4(case):
    m = case["rows"]
    nbytes = sum(k * n // 2 + (k // 128) * n * 2.5 + 2 * m * (k + n) for k, n in _int4_shapes(case))
    return {"bytes": nbytes, "flops": sum(2 * m * k * n for k, n in _int4_shapes(case))}


# ----------------------------------------------------------------------------------------------------- routed experts
def _prepare_experts(case, seed):
    g, bf = _gen(seed), torch.bfloat16
    rows, width, ff, experts, top = (case[k] for k in ("rows", "width", "ff", "experts", "top"))
    x = _randn(g, rows, width, dtype=bf)
    # some experts are asked for more often than others
    logits = _randn(g, rows, experts) + _randn(g, 1, experts, scale=0.5)
    weights, chosen = torch.topk(logits.softmax(-1), top, dim=-1)
    weights = (weights / weights.sum(-1, keepdim=True)).contiguous()
    up = _randn(g, experts, ff, width, dtype=bf, scale=width ** -0.5)
    gate = _randn(g, experts, ff, width, dtype=bf, scale=width ** -0.5) if case["act"] == "glu" else None
    down = _randn(g, experts, width, ff, dtype=bf, scale=ff ** -0.5)
    packed = up if gate is None else _C.mixer_ops.glu_rows(gate, up)
    return SimpleNamespace(run=_run_experts, x=x, chosen=chosen.to(torch.int32).contiguous(), weights=weights, packed=packed,
                           up=up, gate=gate, down=down, experts=experts, top=top, act=case["act"])


def _run_experts(s):
    out = torch.zeros(s.x.shape, dtype=torch.float32, device=s.x.device)
    order, start = _C.mixer_ops.group_pairs(s.chosen, s.experts)
    _C.mixer_ops.expert_ffn(out, s.x, s.packed, s.down, order, start, s.top, 1.0,
                            activation=_C.mixer_ops.ACT_GELU if s.act == "gelu" else _C.mixer_ops.ACT_RELU2,
                            pair_weight=s.weights, glu=(1.0, math.inf, 0.0) if s.act == "glu" else None)
    return out


def _exact_experts(case, seed):
    s = _prepare_experts(case, seed)
    x, out = s.x.double(), torch.zeros(s.x.shape, dtype=torch.float64, device=DEV)
    for e in range(s.experts):
        row, choice = (s.chosen == e).nonzero(as_tuple=True)
        if row.numel() == 0:
            continue
        z = torch.matmul(x[row], s.up[e].double().t())
        if s.act == "glu":
            z = torch.nn.functional.silu(torch.matmul(x[row], s.gate[e].double().t())) * z
        elif s.act == "relu2":
            z = z.clamp(min=0).square()
        else:
            z = torch.nn.functional.gelu(z)
        out.index_add_(0, row, torch.matmul(z, s.down[e].double().t()) * s.weights[row, choice].double()[:, None])
    return out


def _work_experts(case):
    rows, width, ff, experts, top = (case[k] for k in ("rows", "width", "ff", "experts", "top"))
    mats = 3 if case["act"] == "glu" else 2
    touched = experts * (1 - (1 - top / experts) ** rows)                       # experts that some row asks for, about
    return {"bytes": touched * mats * ff * width * 2 + rows * width * (2 + 4) + rows * top * 8,
            "flops": 2 * mats * rows * top * ff * width}


# ------------------------------------------------------------------------------------- the mixer models' paged attention
def _prepare_attention(case, seed):
    g, bf = _gen(seed), torch.bfloat16
    h, kvh, d = case["heads"], case["kv_heads"], case["dim"]
    lengths = _lengths(case)
    rows = sum(n for _, n in lengths)
    table, blocks = _pages(g, lengths)
    return SimpleNamespace(
        run=_run_attention, case=case, q=_randn(g, rows, h * d), key_cache=_randn(g, blocks, BLOCK, kvh * d, dtype=bf),
        value_cache=_randn(g, blocks, BLOCK, kvh * d, dtype=bf), gate=_randn(g, rows, h * d, dtype=bf) if case["gate"] else None,
        sink=_randn(g, h) if case["sink"] else False, batch=_ragged(lengths, table, blocks), table=table)


def _run_attention(s):
    c = s.case
    out = torch.empty(s.q.shape, dtype=s.key_cache.dtype, device=s.q.device)
    _C.mixer_ops.capped_attention(out, s.q, s.key_cache, s.value_cache, s.gate, s.batch, c["heads"], c["kv_heads"], c["dim"],
                                  c["dim"], c["dim"] ** -0.5, c["softcap"], window=c["window"], sink=s.sink)
    return out


def _exact_attention(case, seed):
    s = _prepare_attention(case, seed)
    h, kvh, d = case["heads"], case["kv_heads"], case["dim"]
    rep, q = h // kvh, s.q.double().view(-1, h, d)
    out, row = torch.empty_like(q), 0
    for i, (c, n) in enumerate(_lengths(case)):
        blocks = s.table[i, :-(-(c + n) // BLOCK)].long()
        ks = s.key_cache[blocks].double().reshape(-1, kvh, d)[:c + n]
        vs = s.value_cache[blocks].double().reshape(-1, kvh, d)[:c + n]
        at, seen = torch.arange(c, c + n, device=DEV)[:, None], torch.arange(c + n, device=DEV)[None]
        hidden = (seen > at) | ((at - seen >= case["window"]) if case["window"] else torch.zeros_like(seen > at))
        for head in range(h):
            score = torch.matmul(q[row:row + n, head], ks[:, head // rep].t()) * d ** -0.5
            if case["softcap"]:
                score = case["softcap"] * torch.tanh(score / case["softcap"])
            score.masked_fill_(hidden, -math.inf)
            if case["sink"]:
                sink = s.sink[head].double().expand(n, 1)
                weight = torch.cat([score, sink], 1).softmax(-1)[:, :-1]
            else:
                weight = score.softmax(-1)
            out[row:row + n, head] = torch.matmul(weight, vs[:, head // rep])
        row += n
    out = out.view(row, h * d)
    return out * torch.sigmoid(s.gate.double()) if case["gate"] else out


def _work_attention(case):
    h, kvh, d = case["heads"], case["kv_heads"], case["dim"]
    most = case["window"] or 1 << 30
    pairs = sum(min(c + i + 1, most) for c, n in _lengths(case) for i in range(n))
    keys = sum(min(c + n, most + n - 1) for c, n in _lengths(case))
    rows = sum(n for _, n in _lengths(case))
    return {"bytes": keys * kvh * d * 4 + rows * h * d * (4 + 2 + (2 if case["gate"] else 0)), "flops": 4 * pairs * h * d}


# ------------------------------------------------------------------------------------------- the recurrent token mixers
def _recurrent_lengths(case):
    """Prompts start from nothing; a decoded token continues a state."""
    return [(64 if case["new"] == 1 else 0, n) for _, n in _lengths(case)]


def _prepare_delta(case, seed):
    g, bf = _gen(seed), torch.bfloat16
    h, kvh, d = case["heads"], case["kv_heads"], case["dim"]
    lengths = _recurrent_lengths(case)
    rows, count, c = sum(n for _, n in lengths), len(lengths), (2 * kvh + h) * d
    return SimpleNamespace(
        run=_run_delta, case=case, channels=c, proj=_randn(g, rows, c + 2 * h + h * d, dtype=bf),
        taps=_randn(g, c, TAPS, scale=0.4), conv_state=_randn(g, count, TAPS - 1, c),
        state=_randn(g, count, h, d, d, scale=0.1), dt_bias=_randn(g, h, scale=0.5), a_log=_randn(g, h, scale=0.3),
        norm=1.0 + _randn(g, d, scale=0.1), batch=_ragged(lengths))


def _run_delta(s):
    case, c, rows, dev = s.case, s.channels, s.proj.shape[0], s.proj.device
    h, kvh, d = case["heads"], case["kv_heads"], case["dim"]
    qkv = torch.empty(rows, c, dtype=torch.float32, device=dev)
    _C.mixer_ops.causal_conv(qkv, s.proj[:, :c], s.taps, s.conv_state, s.batch, silu=True, residual=False)
    o = torch.empty(rows, h * d, dtype=torch.float32, device=dev)
    _C.mixer_ops.gated_delta(o, qkv, s.proj[:, c:c + h], s.proj[:, c + h:c + 2 * h], s.dt_bias, s.a_log, s.state, s.batch, h,
                             kvh, d, d)
    gated = torch.empty(rows, h * d, dtype=s.proj.dtype, device=dev)
    _C.mixer_ops.head_norm_gate(gated, o, s.proj[:, c + 2 * h:], s.norm, False, EPS, h, d, gate_silu=True)
    return {"gated": gated, "conv_state": s.conv_state, "state": s.state}


def _padded(t, lengths):
    """[rows, ...] -> [longest, sequences, ...], zeros behind the shorter sequences."""
    out = t.new_zeros((max(n for _, n in lengths), len(lengths)) + t.shape[1:])
    row = 0
    for i, (_, n) in enumerate(lengths):
        out[:n, i] = t[row:row + n]
        row += n
    return out


def _unpadded(t, lengths):
    return torch.cat([t[:n, i] for i, (_, n) in enumerate(lengths)])


def _head_norm(o, d):
    return o * torch.rsqrt(o.square().mean(-1, keepdim=True) + EPS)


def _exact_delta(case, seed):
    s = _prepare_delta(case, seed)
    h, kvh, d = case["heads"], case["kv_heads"], case["dim"]
    lengths, c = _recurrent_lengths(case), s.channels
    fresh = case["new"] > 1
    proj = s.proj.double()
    conv_state = torch.zeros_like(s.conv_state.double()) if fresh else s.conv_state.double()
    taps, parts, row = s.taps.double(), [], 0
    for i, (_, n) in enumerate(lengths):
        x = torch.cat([conv_state[i], proj[row:row + n, :c]])
        parts.append(sum(x[j:j + n] * taps[:, j] for j in range(TAPS)))
        conv_state[i] = x[n:]
        row += n
    qkv = torch.nn.functional.silu(torch.cat(parts))
    unit = lambda t: t / torch.sqrt(t.square().sum(-1, keepdim=True) + 1e-6)                 # noqa: E731
    q = unit(qkv[:, :kvh * d].view(-1, kvh, d)).repeat_interleave(h // kvh, 1) * d ** -0.5
    k = unit(qkv[:, kvh * d:2 * kvh * d].view(-1, kvh, d)).repeat_interleave(h // kvh, 1)
    v = qkv[:, 2 * kvh * d:].view(-1, h, d)
    beta = torch.sigmoid(proj[:, c:c + h])
    keep = torch.exp(-s.a_log.double().exp() * torch.nn.functional.softplus(proj[:, c + h:c + 2 * h] + s.dt_bias.double()))
    live = _padded(torch.ones(row, 1, 1, 1, device=DEV, dtype=torch.float64), lengths)
    q, k, v, beta, keep = (_padded(t, lengths) for t in (q, k, v, beta, keep))
    S = torch.zeros_like(s.state.double()) if fresh else s.state.double()
    o = torch.empty_like(v)
    for t in range(q.shape[0]):
        new = keep[t][..., None, None] * S
        u = beta[t][..., None] * (v[t] - torch.matmul(k[t][..., None, :], new).squeeze(-2))
        new = new + k[t][..., None] * u[..., None, :]
        S = torch.where(live[t] > 0, new, S)
        o[t] = torch.matmul(q[t][..., None, :], new).squeeze(-2)
    o = _head_norm(_unpadded(o, lengths), d) * s.norm.double()
    gated = o.reshape(row, h * d) * torch.nn.functional.silu(proj[:, c + 2 * h:])
    return {"gated": gated, "conv_state": conv_state, "state": S}


def _work_delta(case):
    h, kvh, d = case["heads"], case["kv_heads"], case["dim"]
    lengths = _recurrent_lengths(case)
    rows, count, c = sum(n for _, n in lengths), len(lengths), (2 * kvh + h) * d
    states = count * (h * d * d + (TAPS - 1) * c) * 4 * (2 if case["new"] == 1 else 1)
    return {"bytes": rows * (c + 2 * h + 2 * h * d) * 2 + states, "flops": rows * (6 * h * d * d + 2 * TAPS * c)}


def _prepare_linear(case, seed):
    g, bf = _gen(seed), torch.bfloat16
    h, d = case["heads"], case["dim"]
    lengths = _recurrent_lengths(case)
    rows, n = sum(n for _, n in lengths), h * d
    s = SimpleNamespace(run=_run_linear, case=case, proj=_randn(g, rows, 4 * n, dtype=bf),
                        state=_randn(g, len(lengths), h, d, d, scale=0.1), batch=_ragged(lengths))
    s.decay_pre, s.decay_bias = _randn(g, rows, n, dtype=bf), 2.0 + _randn(g, n)
    # one constant decay per head, from fast to slow
    s.decay = torch.exp(-torch.exp2(-8.0 * (torch.arange(h, device=DEV) + 1) / h)).float()
    s.q32, s.k32 = _randn(g, rows, n), _randn(g, rows, n, scale=d ** -0.5)
    s.norm = 1.0 + _randn(g, n if case["rule"] == "lightning" else d, scale=0.1)
    return s


def _run_linear(s):
    case, rows, dev = s.case, s.proj.shape[0], s.proj.device
    h, d = case["heads"], case["dim"]
    n = h * d
    q, k, v, gate = (s.proj[:, i * n:(i + 1) * n] for i in range(4))
    o = torch.empty(rows, n, dtype=torch.float32, device=dev)
    gated = torch.empty(rows, n, dtype=s.proj.dtype, device=dev)
    if case["rule"] == "gla":
        _C.mixer_ops.gla(o, q, k, v, s.decay_pre, s.decay_bias, TAU, d ** -0.5, s.state, s.batch, h, d, d)
        _C.mixer_ops.head_norm_gate(gated, o, gate, s.norm, False, EPS, h, d, gate_silu=True)
    elif case["rule"] == "lightning":
        _C.mixer_ops.lightning(o, q, k, v, s.decay, s.state, s.batch, h, d, d)
        _C.mixer_ops.head_norm_gate(gated, o, gate, s.norm, True, EPS, 1, n)
    else:
        _C.mixer_ops.retention(o, s.q32, s.k32, v, s.decay, s.state, s.batch, h, d, d)
        _C.mixer_ops.head_norm_gate(gated, o, gate, None, False, EPS, h, d, gate_silu=True)
    return {"gated": gated, "state": s.state}


def _exact_linear(case, seed):
    s = _prepare_linear(case, seed)
    h, d, rule = case["heads"], case["dim"], case["rule"]
    lengths, n = _recurrent_lengths(case), case["heads"] * case["dim"]
    q, k, v, gate = (s.proj[:, i * n:(i + 1) * n].double() for i in range(4))
    silu = torch.nn.functional.silu
    if rule == "gla":
        q = q * d ** -0.5
        keep = torch.exp(torch.nn.functional.logsigmoid(s.decay_pre.double() + s.decay_bias.double()) / TAU)
        keep = keep.view(-1, h, d, 1)
    else:
        keep = s.decay.double().view(1, h, 1, 1).expand(q.shape[0], h, 1, 1)
        q, k, v = (silu(q), silu(k), silu(v)) if rule == "lightning" else (s.q32.double(), s.k32.double(), v)
    live = _padded(torch.ones(q.shape[0], 1, 1, 1, device=DEV, dtype=torch.float64), lengths)
    q, k, v = (_padded(t.view(-1, h, d), lengths) for t in (q, k, v))
    keep = _padded(keep, lengths)
    S = torch.zeros_like(s.state.double()) if case["new"] > 1 else s.state.double()
    o = torch.empty_like(v)
    for t in range(q.shape[0]):
        new = keep[t] * S + k[t][..., None] * v[t][..., None, :]
        S = torch.where(live[t] > 0, new, S)
        o[t] = torch.matmul(q[t][..., None, :], new).squeeze(-2)
    o = _unpadded(o, lengths)
    if rule == "lightning":
        gated = _head_norm(o.reshape(-1, n), n) * s.norm.double() * torch.sigmoid(gate)
    else:
        o = _head_norm(o, d) * (s.norm.double() if rule == "gla" else 1.0)
        gated = o.reshape(-1, n) * silu(gate)
    return {"gated": gated, "state": S}


def _work_linear(case):
    h, d = case["heads"], case["dim"]
    lengths = _recurrent_lengths(case)
    rows, n = sum(n for _, n in lengths), h * d
    ins = {"gla": 2 * 5, "lightning": 2 * 4, "retention": 4 * 2 + 2 * 2}[case["rule"]]
    states = len(lengths) * n * d * 4 * (2 if case["new"] == 1 else 1)
    return {"bytes": rows * n * (ins + 2) + states, "flops": rows * 4 * h * d * d}


# ------------------------------------------------------------------------------------------------------ what is called
_PREPARE = {"decode": _prepare_llama, "prompt": _prepare_llama, "int4": _prepare_int4, "experts": _prepare_experts,
            "attention": _prepare_attention, "delta": _prepare_delta, "linear": _prepare_linear}
_EXACT = {"decode": _exact_llama, "prompt": _exact_llama, "int4": _exact_int4, "experts": _exact_experts,
          "attention": _exact_attention, "delta": _exact_delta, "linear": _exact_linear}
_WORK = {"decode": _work_llama, "prompt": _work_llama, "int4": _work_int4, "experts": _work_experts,
         "attention": _work_attention, "delta": _work_delta, "linear": _work_linear}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


@torch.inference_mode()
def run(state):
    return state.run(state)


@torch.inference_mode()
def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def work(case):
    return _WORK[case["kind"]](case)


def tolerance(case):
    """About four times the distance from the 64-bit result that was measured over these ranges: results in 16 bits, whose
    last place is 2^-9 (bf16) or 2^-12 (f16) of a number, and sums in fp32."""
    kind = case["kind"]
    if kind in ("decode", "prompt"):
        # softmax weights are 16-bit numbers in the second product
        return {"rel": 0.009} if case["dtype"] == "bf16" else {"rel": 0.0012}
    if kind == "int4":
        return {"rel": 0.0012}                   # weights rounded to fp16 before the product
    return {"rel": 0.007}                        # a hidden layer or the result is rounded to bf16
