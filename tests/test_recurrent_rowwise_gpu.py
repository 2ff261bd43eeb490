"""The short convolution in runs of rows, the per-head norm in 16-byte pieces and the delta rule's decode step in one launch, and
the kernels that take calls whose operands do not lie on 16 bytes: every call is made both ways, aligned and with an operand moved
by one element, and both are compared with a plain statement in 64 bits.  fp32 sums of at most 4 products, or of a head's squares
(rtol 1e-5), rounded once where the result is bf16 (2^-7)."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _tol(dtype):
    return dict(atol=1e-5, rtol=1e-5) if dtype == torch.float32 else dict(atol=1e-4, rtol=2.0 ** -7)


def _moved(t, lead, row):
    """``t`` [rows, n] as a view with row stride ``row`` that begins ``lead`` elements into its storage."""
    at = torch.empty(t.shape[0] * row + lead + 8, dtype=t.dtype, device=DEV)
    view = at[lead:lead + t.shape[0] * row].view(t.shape[0], row)[:, :t.shape[1]]
    view.copy_(t)
    return view


@pytest.mark.parametrize("lens", [[1], [1] * 5 + [2, 3, 4, 1, 7], [15, 2, 1, 16, 33, 1, 3, 17, 2, 64], [1, 1030, 2, 31, 1, 1, 3, 100]])
@pytest.mark.parametrize("channels,taps", [(8, 4), (72, 3), (4160, 4), (264, 2)])
@pytest.mark.parametrize("x_dtype,out_dtype", [(torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16),
                                               (torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32)])
def test_convolution_in_runs(lens, channels, taps, x_dtype, out_dtype):
    from splitwise_amd import _C
    starts, owner = [0], []
    for i, n in enumerate(lens):
        starts.append(starts[-1] + n)
        owner += [i] * n
    rows, count = starts[-1], len(lens)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)          # noqa: E731
    slots = [(i * 3 + 1) % (count + 2) if (count + 2) % 3 else i + 1 for i in range(count)]
    batch = SimpleNamespace(q_start=i32(starts), ctx_len=i32([(0, 9)[i % 2] for i in range(count)]), token_seq=i32(owner),
                            state_slot=i32(slots), max_state_slot=max(slots))
    g = torch.Generator(device=DEV).manual_seed(rows + channels)
    x = torch.randn(rows, channels, generator=g, device=DEV).to(x_dtype)
    w = torch.randn(channels, taps, generator=g, device=DEV)
    state = torch.randn(count + 2, taps - 1, channels, generator=g, device=DEV)
    past = torch.zeros(count, taps - 1, channels, dtype=torch.float64, device=DEV)           # a sequence's carried inputs
    past[1::2] = state[slots][1::2].double()
    seen = [torch.cat([past[i], x[starts[i]:starts[i + 1]].double()]) for i in range(count)]
    conv = torch.cat([sum(w[:, j].double() * t[j:len(t) - taps + 1 + j] for j in range(taps)) for t in seen])
    kept = state.clone()
    for i, t in enumerate(seen):
        kept[slots[i]] = t[len(t) - taps + 1:].float()
    for silu, residual in ((True, False), (False, True)):
        ref = conv + x.double() if residual else conv
        ref = torch.nn.functional.silu(ref) if silu else ref
        res = []
        for lead in (0, 1):
            s, out = state.clone(), torch.full((rows, channels), float("nan"), dtype=out_dtype, device=DEV)
            at = _moved(x, lead, channels + 8)
            assert at.data_ptr() % 16 == lead * x.element_size()
            _C.mixer_ops.causal_conv(out, at, w, s, batch, silu=silu, residual=residual)
            res.append((out, s))
            torch.testing.assert_close(out.double(), ref, **_tol(out_dtype))
            assert torch.equal(s, kept)                        # inputs are copied, nothing is rounded
        torch.testing.assert_close(res[0][0], res[1][0], **_tol(out_dtype))


@pytest.mark.parametrize("heads,vdim", [(3, 8), (5, 40), (16, 64), (1, 72), (2, 128), (7, 200), (3, 512), (1, 520), (2, 1024), (1, 2048),
                                        (1, 4096)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_head_norm_in_pieces(heads, vdim, dtype):
    from splitwise_amd import _C
    g = torch.Generator(device=DEV).manual_seed(heads * 1000 + vdim)
    for rows in (1, 37):
        o = torch.randn(rows, heads * vdim, generator=g, device=DEV)
        o[0] *= 1e-3                                           # small enough for eps to count
        gate = torch.randn(rows, heads * vdim, generator=g, device=DEV).to(dtype) * 3
        for weight, per_head, silu in ((None, False, True), (torch.randn(vdim, generator=g, device=DEV), False, False),
                                       (torch.randn(heads * vdim, generator=g, device=DEV), True, True)):
            res = []
            for lead in (0, 1):
                out = torch.full((rows, heads * vdim), float("nan"), dtype=dtype, device=DEV)
                _C.mixer_ops.head_norm_gate(out, o, _moved(gate, lead, heads * vdim + 16), weight, per_head, 1e-5, heads, vdim,
                                            gate_silu=silu)
                res.append(out)
                x64, g64 = o.double().view(rows, heads, vdim), gate.double()
                ref = (x64 * (x64.square().mean(-1, keepdim=True) + 1e-5).rsqrt()).view(rows, -1)
                if weight is not None:
                    ref = ref * (weight if per_head else weight.repeat(heads)).double()
                ref = ref * (torch.nn.functional.silu(g64) if silu else torch.sigmoid(g64))
                torch.testing.assert_close(out.double(), ref, **_tol(dtype))
            torch.testing.assert_close(res[0], res[1], **_tol(dtype))


def _delta_rule(qkv, beta, decay, dt_bias, a_log, state, batch, heads, kv_heads, dim, vdim):
    """The rule in 64 bits, token by token -> outputs and states."""
    rows, ends, out = qkv.shape[0], state.double(), []
    q, k, v = qkv.double().split([kv_heads * dim, kv_heads * dim, heads * vdim], 1)
    unit = lambda t: t * (t.square().sum(-1, keepdim=True) + 1e-6).rsqrt()  # noqa: E731
    q, k = (unit(t.view(rows, kv_heads, dim)).repeat_interleave(heads // kv_heads, 1) for t in (q, k))
    g = torch.nn.functional.softplus(decay.double() + dt_bias.double()).view(rows, heads, -1)
    g, b = torch.exp(-a_log.double().exp()[:, None] * g), torch.sigmoid(beta.double())
    owner, slots = batch.token_seq.tolist(), batch.state_slot.tolist()
    for i, (c, lo, hi) in enumerate(zip(batch.ctx_len.tolist(), batch.q_start.tolist(), batch.q_start.tolist()[1:])):
        if c == 0 and hi > lo:
            ends[slots[i]] = 0
    for t in range(rows):
        s = g[t][..., None] * ends[slots[owner[t]]]
        u = b[t][:, None] * (v[t].view(heads, vdim) - (s * k[t][..., None]).sum(-2))
        s = s + k[t][..., None] * u[:, None, :]
        ends[slots[owner[t]]] = s
        out.append((s * q[t][..., None]).sum(-2).flatten() * dim ** -0.5)
    return torch.stack(out), ends


@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(1, 1, 4, 4), (4, 2, 24, 36), (2, 2, 64, 64), (3, 1, 100, 132), (4, 4, 128, 128),
                                                     (2, 1, 256, 256), (1, 1, 256, 8), (2, 1, 6, 260)])
@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_delta_decode_step_in_one_launch(heads, kv_heads, dim, vdim, per_channel, dtype):
    """The prologue and recurrence take the output off 16 bytes.  Sums of at most 256 products of numbers around 1 in fp32."""
    from splitwise_amd import _C
    g = torch.Generator(device=DEV).manual_seed(heads * 1000 + dim + vdim)
    seqs, slots = 9, [3, 0, 11, 5, 7, 1, 8, 2, 10]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)          # noqa: E731
    lens = [1, 1, 0, 2, 1, 1, 1, 1, 1]                         # as many rows as sequences, though not one each
    starts = [sum(lens[:i]) for i in range(seqs + 1)]
    batch = SimpleNamespace(q_start=i32(starts), ctx_len=i32([5, 0, 7, 0, 3, 9, 0, 64, 1]), max_query_len=1, max_state_slot=11,
                            token_seq=i32([i for i, n in enumerate(lens) for _ in range(n)]), state_slot=i32(slots))
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)               # noqa: E731
    qkv = rnd(seqs, 2 * kv_heads * dim + heads * vdim)
    beta, dt_bias, a_log = rnd(seqs, heads + 3).to(dtype)[:, :heads], rnd(heads * (dim if per_channel else 1)), rnd(heads) * 0.3
    decay = rnd(seqs, heads * dim if per_channel else heads).to(dtype)
    state = rnd(12, heads, dim, vdim)
    ref, ends = _delta_rule(qkv, beta, decay, dt_bias, a_log, state, batch, heads, kv_heads, dim, vdim)
    res = []
    for lead in (0, 1):
        s = state.clone()
        out = torch.full((seqs * heads * vdim + 1,), float("nan"), device=DEV)[lead:lead + seqs * heads * vdim].view(seqs, -1)
        op = _C.mixer_ops.channel_delta if per_channel else _C.mixer_ops.gated_delta
        op(out, qkv, beta, decay, dt_bias, a_log, s, batch, heads, kv_heads, dim, vdim)
        res.append((out, s))
        torch.testing.assert_close(out.double(), ref, atol=3e-5, rtol=1e-4)
        torch.testing.assert_close(s.double(), ends, atol=3e-5, rtol=1e-4)
    torch.testing.assert_close(res[0][0], res[1][0], atol=3e-5, rtol=1e-4)
    torch.testing.assert_close(res[0][1], res[1][1], atol=3e-5, rtol=1e-4)
    idle = [i for i in range(12) if i not in slots] + [11]     # slots of nobody, and of the sequence without a token
    assert torch.equal(res[0][1][idle], state[idle])


@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(2, 1, 32, 16), (3, 3, 64, 17), (6, 1, 96, 40), (4, 2, 128, 128), (2, 2, 160, 33),
                                                     (1, 1, 224, 64)])
@pytest.mark.parametrize("lens", [[32, 31, 1, 33, 64, 95, 2], [1] * 9 + [40, 16, 17, 0, 1, 3, 70], [1] * 80 + [33], [1] * 13])
def test_delta_chunks_agree_with_the_tokens(heads, kv_heads, dim, vdim, lens):
    """Runs that end at, before and behind a chunk's border, from nothing and from a state, alone and beside decoding sequences
    (which go another way in the same call), against the rule token by token: fp32 sums in another order, over states whose size
    the rule keeps around that of the values."""
    from splitwise_amd import _C
    n = len(lens)
    ctx, slots = [(0, 3, 9, 0, 64, 0, 1)[i % 7] for i in range(n)], [(4, 0, 8, 2, 1, 7, 3)[i % 7] + i // 7 * 9 for i in range(n)]
    starts = [sum(lens[:i]) for i in range(len(lens) + 1)]
    g = torch.Generator(device=DEV).manual_seed(dim + vdim)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)          # noqa: E731
    batch = SimpleNamespace(q_start=i32(starts), ctx_len=i32(ctx), max_query_len=max(lens), max_state_slot=max(slots),
                            token_seq=i32([i for i, m in enumerate(lens) for _ in range(m)]), state_slot=i32(slots))
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)               # noqa: E731
    rows = starts[-1]
    qkv, both = rnd(rows, 2 * kv_heads * dim + heads * vdim), rnd(rows, 2 * heads).to(torch.bfloat16)
    dt_bias, a_log, state = rnd(heads), rnd(heads) * 0.3, rnd(max(slots) + 9, heads, dim, vdim) * 0.1
    res = []
    ref, ends = _delta_rule(qkv, both[:, :heads], both[:, heads:], dt_bias, a_log, state, batch, heads, kv_heads, dim, vdim)
    for chunked in (True, False):
        s, out = state.clone(), torch.full((rows, heads * vdim), float("nan"), device=DEV)
        _C.mixer_ops.gated_delta(out, qkv, both[:, :heads], both[:, heads:], dt_bias, a_log, s, batch, heads, kv_heads, dim, vdim,
                                 chunked=chunked)
        res.append((out, s))
        torch.testing.assert_close(out.double(), ref, atol=2e-5, rtol=1e-4)
        torch.testing.assert_close(s.double(), ends, atol=2e-5, rtol=1e-4)
    torch.testing.assert_close(res[0][0], res[1][0], atol=2e-5, rtol=1e-4)
    torch.testing.assert_close(res[0][1], res[1][1], atol=2e-5, rtol=1e-4)
    idle = [i for i in range(state.shape[0]) if i not in slots]
    assert torch.equal(res[0][1][idle], state[idle])


@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(3, 1, 32, 24), (2, 2, 64, 16), (5, 1, 96, 130), (6, 2, 128, 72), (2, 1, 224, 20)])
@pytest.mark.parametrize("lead", [0, 1])
def test_delta_chunks_through_every_turn_of_the_walk(heads, kv_heads, dim, vdim, lead):
    """Runs of 1 to 8 chunks, whole and not, which leave the walk's loop over chunks at each of its places; one of them is NaN, and
    stays with itself.  qkv on 16 bytes and off them.  End states within 4e-7 of 64 bits, as norms: sums of at most 256 fp32
    products around 1, each rounded to 2^-24, over the few dozen tokens that a state remembers."""
    from splitwise_amd import _C
    lens = [256, 225, 191, 160, 130, 96, 64, 33]
    starts, bad = [sum(lens[:i]) for i in range(len(lens) + 1)], 5
    g = torch.Generator(device=DEV).manual_seed(dim + vdim)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)          # noqa: E731
    ctx, slots = [0, 3, 9, 0, 64, 0, 1, 5], [4, 0, 8, 2, 1, 7, 3, 5]
    batch = SimpleNamespace(q_start=i32(starts), ctx_len=i32(ctx), max_query_len=max(lens), max_state_slot=8, state_slot=i32(slots),
                            token_seq=i32([i for i, m in enumerate(lens) for _ in range(m)]))
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)               # noqa: E731
    rows, width = starts[-1], 2 * kv_heads * dim + heads * vdim
    qkv = torch.empty(rows * width + 1, device=DEV)[lead:lead + rows * width].view(rows, width)
    qkv.copy_(rnd(rows, width))
    both = rnd(rows, 2 * heads).to(torch.bfloat16)
    dt_bias, a_log, state = rnd(heads), rnd(heads) * 0.3, rnd(9, heads, dim, vdim) * 0.1
    ref, ends = _delta_rule(qkv, both[:, :heads], both[:, heads:], dt_bias, a_log, state, batch, heads, kv_heads, dim, vdim)
    qkv[starts[bad]:starts[bad + 1]] = float("nan")
    out = torch.full((rows, heads * vdim), float("nan"), device=DEV)
    _C.mixer_ops.gated_delta(out, qkv, both[:, :heads], both[:, heads:], dt_bias, a_log, state, batch, heads, kv_heads, dim, vdim,
                             chunked=True)
    good = [i for i in range(len(lens)) if i != bad]
    at = torch.cat([torch.arange(starts[i], starts[i + 1], device=DEV) for i in good])
    assert bool(out[starts[bad]:starts[bad + 1]].isnan().all()) and bool(state[slots[bad]].isnan().all())
    torch.testing.assert_close(out[at].double(), ref[at], atol=2e-5, rtol=1e-4)
    for i in good:
        err = (state[slots[i]].double() - ends[slots[i]]).norm() / ends[slots[i]].norm()
        assert float(err) < 4e-7, (i, float(err))


def test_delta_chunks_of_the_widest_rows():
    """Rows of 128 MiB: a chunk of them passes 32-bit places.  Sums of 4 products in fp32."""
    from splitwise_amd import _C
    dim, vdim, lens = 4, 1 << 25, [2, 1]
    g = torch.Generator(device=DEV).manual_seed(1)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)          # noqa: E731
    batch = SimpleNamespace(q_start=i32([0, 2, 3]), ctx_len=i32([0, 5]), max_query_len=2, max_state_slot=1, state_slot=i32([1, 0]),
                            token_seq=i32([0, 0, 1]))
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)               # noqa: E731
    qkv, both, dt_bias, a_log = rnd(sum(lens), 2 * dim + vdim), rnd(sum(lens), 2).bfloat16(), rnd(1), rnd(1) * 0.3
    state, out = rnd(2, 1, dim, vdim), torch.full((sum(lens), vdim), float("nan"), device=DEV)
    ref, ends = _delta_rule(qkv, both[:, :1], both[:, 1:], dt_bias, a_log, state, batch, 1, 1, dim, vdim)
    _C.mixer_ops.gated_delta(out, qkv, both[:, :1], both[:, 1:], dt_bias, a_log, state, batch, 1, 1, dim, vdim, chunked=True)
    for a, b in ((out, ref), (state, ends)):
        assert float((a.double() - b).abs().max()) < 2e-5


@pytest.mark.parametrize("heads,kv_heads,dim,vdim", [(4, 2, 64, 24), (2, 1, 128, 40)])
def test_decays_that_overflowed(heads, kv_heads, dim, vdim):
    """A decay gate of +inf, or one large enough for a decay of 0 in fp32, makes a head forget what was in front of the token, one of
    -inf keeps it: single tokens of long runs, next to one another and at a chunk's ends, in chunks and token by token.  (Bounds as
    for the chunks above.)"""
    from splitwise_amd import _C
    lens, inf = [70, 33, 130], float("inf")
    starts, ctx, slots = [sum(lens[:i]) for i in range(4)], [3, 0, 9], [1, 2, 0]
    g = torch.Generator(device=DEV).manual_seed(dim)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)          # noqa: E731
    batch = SimpleNamespace(q_start=i32(starts), ctx_len=i32(ctx), max_query_len=max(lens), max_state_slot=2, state_slot=i32(slots),
                            token_seq=i32([i for i, m in enumerate(lens) for _ in range(m)]))
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)               # noqa: E731
    rows = starts[-1]
    qkv, both = rnd(rows, 2 * kv_heads * dim + heads * vdim), rnd(rows, 2 * heads).to(torch.bfloat16)
    for first, m in zip(starts, lens):
        for at, head, gate in ((9, 0, inf), (12, 0, inf), (13, 0, -inf), (20, 1, 1e30), (21, 1, 3e38), (0, 1, inf), (31, 0, 500.0),
                               (32, 0, 1e9), (m - 1, 1, inf)):
            both[first + at, heads + head] = gate
    dt_bias, a_log, state = rnd(heads), rnd(heads) * 0.3, rnd(3, heads, dim, vdim) * 0.1
    ref, ends = _delta_rule(qkv, both[:, :heads], both[:, heads:], dt_bias, a_log, state, batch, heads, kv_heads, dim, vdim)
    for chunked in (True, False):
        s, out = state.clone(), torch.full((rows, heads * vdim), float("nan"), device=DEV)
        _C.mixer_ops.gated_delta(out, qkv, both[:, :heads], both[:, heads:], dt_bias, a_log, s, batch, heads, kv_heads, dim, vdim,
                                 chunked=chunked)
        torch.testing.assert_close(out.double(), ref, atol=2e-5, rtol=1e-4)
        torch.testing.assert_close(s.double(), ends, atol=2e-5, rtol=1e-4)


@pytest.mark.parametrize("rule", ["gla", "gla, strong decays", "lightning", "retention"])
@pytest.mark.parametrize("heads,dim,vdim", [(2, 32, 16), (3, 64, 17), (1, 72, 130), (2, 128, 40), (1, 160, 16), (1, 256, 33)])
def test_linear_attention_walk_agrees_with_short_runs(rule, heads, dim, vdim):
    """Runs that end at, before and behind the borders of a chunk and of its halves, in one step and in portions of at most 16
    tokens, which take the kernels of decode steps.  Sums of fp32 products in another order."""
    from splitwise_amd import _C
    ops = _C.mixer_ops
    lens = [17, 32, 33, 16, 1, 64, 95]
    g = torch.Generator(device=DEV).manual_seed(dim + vdim)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)               # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)          # noqa: E731
    rows, nk, nv = sum(lens), heads * dim, heads * vdim
    dtype = torch.float32 if rule == "retention" else torch.bfloat16
    proj = rnd(rows, 2 * nk + nv + 8).to(dtype)
    strong = rule == "gla, strong decays"
    z, bias = rnd(rows, nk).to(dtype) * (6.0 if strong else 1.0), rnd(nk)
    decay, ctx, slots = torch.linspace(0.3, 0.999, heads, device=DEV), [0, 3, 9, 0, 64, 0, 1], [4, 0, 8, 2, 1, 7, 3]
    state = rnd(9, heads, dim, vdim) * 0.1

    def step(parts, out, s):
        """parts: (sequence, tokens before it, tokens)."""
        first = [sum(lens[:i]) for i in range(len(lens))]
        pick = torch.cat([torch.arange(first[i] + lo, first[i] + lo + n, device=DEV) for i, lo, n in parts])
        starts = [sum(n for _, _, n in parts[:i]) for i in range(len(parts) + 1)]
        batch = SimpleNamespace(q_start=i32(starts), ctx_len=i32([ctx[i] + lo for i, lo, _ in parts]), max_state_slot=8,
                                max_query_len=max(n for _, _, n in parts), state_slot=i32([slots[i] for i, _, _ in parts]),
                                token_seq=i32([j for j, (_, _, n) in enumerate(parts) for _ in range(n)]))
        p, o = proj[pick], torch.empty(len(pick), nv, device=DEV)
        q, k, v = p[:, :nk], p[:, nk:2 * nk], p[:, 2 * nk:2 * nk + nv]
        if rule == "lightning":
            ops.lightning(o, q, k, v, decay, s, batch, heads, dim, vdim)
        elif rule == "retention":
            ops.retention(o, q.contiguous(), k.contiguous() * dim ** -0.5, v, decay, s, batch, heads, dim, vdim)
        else:
            ops.gla(o, q, k, v, z[pick].contiguous(), bias, 0.5 if strong else 8.0, dim ** -0.5, s, batch, heads, dim, vdim)
        out[pick] = o
    a, b = state.clone(), state.clone()
    whole, pieces = (torch.full((rows, nv), float("nan"), device=DEV) for _ in range(2))
    step([(i, 0, n) for i, n in enumerate(lens)], whole, a)
    for lo in range(0, max(lens), 13):
        step([(i, lo, min(13, n - lo)) for i, n in enumerate(lens) if n > lo], pieces, b)
    size = float(pieces.abs().max())
    torch.testing.assert_close(whole, pieces, atol=1e-5 * size, rtol=1e-4)
    torch.testing.assert_close(a, b, atol=1e-5 * float(b.abs().max()), rtol=1e-4)
