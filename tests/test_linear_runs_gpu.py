"""Linear-attention steps whose runs are cut into segments, and steps whose decoding sequences go another way than the long runs
beside them, against the rule in 64 bits token by token.  States and outputs are fp32 sums of products whose decays are
exponentials of sums: a relative error of about 2e-7 of their size in the 2-norm, 5e-6 of their root mean square for the worst."""
import ctypes
import os
import subprocess
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rule(q, k, v, keep, state, starts, fresh):
    """q, k [rows, heads, dim], v [rows, heads, vdim], keep [rows, heads, dim or 1], state [sequences, heads, dim, vdim]."""
    out, ends = torch.empty_like(v), state.clone()
    longest = max(b - a for a, b in zip(starts, starts[1:]))
    first, last = torch.tensor(starts[:-1], device=DEV), torch.tensor(starts[1:], device=DEV)
    ends[fresh] = 0
    for t in range(longest):
        live = (first + t < last).nonzero().squeeze(1)         # every sequence's token t at once
        at = first[live] + t
        s = keep[at][..., None] * ends[live] + k[at][..., None] * v[at][..., None, :]
        ends[live] = s
        out[at] = (q[at][..., None] * s).sum(-2)
    return out, ends


@pytest.mark.parametrize("rule", ["gla", "lightning", "retention"])
@pytest.mark.parametrize("heads,dim,vdim,lens", [
    (2, 128, 40, [1100, 577, 1, 30, 576]), (1, 64, 16, [5000]), (1, 40, 17, [1024, 1025]), (2, 160, 33, [1500, 3]),
    (3, 256, 20, [33, 2049]),                                              # segments
    (2, 128, 128, [1] * 130 + [40] + [2] * 70 + [17, 16, 95]),              # decoding sequences beside portions
    (4, 128, 128, [1] * 61 + [600, 1100]), (16, 64, 64, [1, 5, 0, 2] * 40 + [70]),
    # workgroups that go on to further pieces: several of them, of a run's segments, a few at most, narrow ones
    (2, 128, 128, [n for i in range(60) for n in (1, 17 + i % 17)] + [200, 64] + [30] * 20), (4, 128, 128, [1] * 100 + [2100] + [40] * 3),
    (32, 256, 33, [1] * 150 + [300, 0, 21, 50]), (32, 32, 40, [1, 18] * 130 + [97])], ids=str)
def test_segments_and_mixed_steps(rule, heads, dim, vdim, lens):
    from splitwise_amd import _C
    ops = _C.mixer_ops
    rows, n = sum(lens), len(lens)
    starts = [sum(lens[:i]) for i in range(n + 1)]
    g = torch.Generator(device=DEV).manual_seed(rows + dim)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)               # noqa: E731
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)          # noqa: E731
    ctx = [0 if i % 3 == 1 else 7 for i in range(n)]
    slots = [(i * 7 + 3) % (n + 2) if (n + 2) % 7 else i + 1 for i in range(n)]
    batch = SimpleNamespace(q_start=i32(starts), ctx_len=i32(ctx), state_slot=i32(slots), max_state_slot=n + 1, max_query_len=max(lens),
                            token_seq=i32([i for i, m in enumerate(lens) for _ in range(m)]))
    nk, nv = heads * dim, heads * vdim
    proj, z, bias = rnd(rows, 2 * nk + nv + 8).bfloat16(), rnd(rows, nk).bfloat16(), 2.0 + rnd(nk)
    decay = torch.linspace(0.3, 0.999, heads, device=DEV)
    q, k, v = proj[:, :nk], proj[:, nk:2 * nk], proj[:, 2 * nk:2 * nk + nv]
    state = rnd(n + 2, heads, dim, vdim) * 0.1
    got, out = state.clone(), torch.full((rows, nv), float("nan"), device=DEV)
    q64, k64, v64 = (t.double().view(rows, heads, -1) for t in (q, k, v))
    keep = decay.double().view(1, heads, 1).expand(rows, heads, 1)
    if rule == "gla":
        ops.gla(out, q, k, v, z, bias, 16.0, dim ** -0.5, got, batch, heads, dim, vdim)
        q64 = q64 * dim ** -0.5
        keep = torch.exp(torch.nn.functional.logsigmoid(z.double() + bias.double()) / 16.0).view(rows, heads, dim)
    elif rule == "lightning":
        ops.lightning(out, q, k, v, decay, got, batch, heads, dim, vdim)
        q64, k64, v64 = (torch.nn.functional.silu(t) for t in (q64, k64, v64))
    else:
        k32 = k.float() * dim ** -0.5
        ops.retention(out, q.float(), k32, v, decay, got, batch, heads, dim, vdim)
        k64 = k32.double().view(rows, heads, dim)
    at = torch.tensor(slots, device=DEV)
    ref, ends = _rule(q64, k64, v64, keep, state[at].double(), starts, torch.tensor([c == 0 for c in ctx], device=DEV))
    some = torch.tensor([m > 0 for m in lens], device=DEV)     # a sequence without a token leaves its state alone
    for a, b in ((out.double().view_as(ref), ref), (got[at][some].double(), ends[some])):
        off = (a - b).abs()
        assert a.isfinite().all()
        assert float(off.norm() / b.norm()) < 6e-7 and float(off.max() / b.square().mean().sqrt()) < 3e-5
    idle = [i for i in range(n + 2) if i not in slots] + [slots[i] for i in range(n) if lens[i] == 0]
    assert torch.equal(got[idle], state[idle])


@pytest.mark.parametrize("rule", ["gla", "lightning", "retention"])
@pytest.mark.parametrize("heads,dim,vdim", [(16, 128, 128), (2, 256, 260), (64, 8, 4), (16, 40, 12), (2, 96, 132), (1, 200, 1024), (2, 33, 64),
                                            (2, 64, 17)])
@pytest.mark.parametrize("lens", [[1] * 7, [5, 1, 0, 3, 5], [1] * 9 + [40, 6, 16, 2]], ids=str)
def test_few_tokens(rule, heads, dim, vdim, lens):
    """Token by token with the state in whole rows, alone and in steps of few sequences of which one walks: key sizes that fill the
    threads' rows or not, value sizes of one piece of 16 bytes, of part of a workgroup's, of several workgroups (and one that has no
    such pieces and goes by chunks).  (Some hundred outputs: one of a few may be a small difference of its terms.)"""
    test_segments_and_mixed_steps(rule, heads, dim, vdim, lens)


@pytest.fixture(scope="module")
def shares(tmp_path_factory):
    """-> up to how many tokens a sequence of the step goes token by token and up to how many it does not walk, by linear_plan.h."""
    at = tmp_path_factory.mktemp("plan")
    (at / "plan.cpp").write_text(r"""
#include "linear_plan.h"
extern "C" void shares(int per_channel, long rows, int seqs, int longest, int heads, int dim, int vdim, int* out) {
  out[1] = swm::linear_at_most(per_channel, rows, seqs, longest, heads, dim, vdim);
  out[0] = swm::linear_step_tokens(out[1], rows, seqs, longest);
}
""")
    mixers = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "vllm-splitwise_amd", "csrc", "mixers")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", mixers, str(at / "plan.cpp"), "-o", str(at / "plan.so")], check=True)
    lib = ctypes.CDLL(str(at / "plan.so"))

    def ask(per_channel, lens, heads, dim, vdim):
        out = (ctypes.c_int * 2)()
        lib.shares(per_channel, ctypes.c_long(sum(lens)), len(lens), max(lens), heads, dim, vdim, out)
        return tuple(out)
    return ask


@pytest.mark.parametrize("rule", ["gla", "lightning", "retention"])
@pytest.mark.parametrize("heads,dim,vdim", [(16, 128, 128), (2, 256, 260), (64, 8, 4), (16, 40, 12), (2, 96, 132), (1, 200, 1024), (2, 33, 64),
                                            (2, 64, 17)])
def test_few_tokens_beside_runs_by_chunks_and_runs_that_walk(rule, heads, dim, vdim, shares):
    """The three ways in one step, for the same sizes."""
    lens = ([1] * 9 + [5, 0, 3, 2]) * -(-180 * 128 // (heads * dim * 13)) + [97, 16, 6, 60]
    assert shares(rule == "gla", lens, heads, dim, vdim) == (5, 16)
    test_segments_and_mixed_steps(rule, heads, dim, vdim, lens)


@pytest.mark.parametrize("rule", ["lightning", "retention"])
@pytest.mark.parametrize("portion", [1, 2, 3, 5])
def test_portions_of_few_tokens_add_up(rule, portion):
    """1600 tokens in portions of as many as go token by token, one decay per head.  A token rounds the state about once, by 2^-24 of
    an element at most and half of that typically; those of the last 1 / (1 - decay^2) tokens (500 at the slowest of the decays) are still
    in it: 22 x 3e-8, measured 7e-7.  (A chunk's power of the decay would be rounded alike in every portion: 3e-6 to 8e-6.)"""
    from splitwise_amd import _C
    heads, dim, seqs, total = 4, 64, 2, 1600
    g = torch.Generator(device=DEV).manual_seed(portion)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)          # noqa: E731
    q, k, v = (torch.randn(total, seqs, heads * dim, generator=g, device=DEV) for _ in range(3))
    decay, state = torch.linspace(0.3, 0.999, heads, device=DEV), torch.zeros(seqs, heads, dim, dim, device=DEV)
    q64, k64, v64 = (t.double().view(total, seqs, heads, dim) for t in (q, k, v))
    if rule == "lightning":
        q64, k64, v64 = (torch.nn.functional.silu(t) for t in (q64, k64, v64))
    end = state.double()
    for t in range(total):
        end = decay.double().view(1, heads, 1, 1) * end + k64[t][..., None] * v64[t][..., None, :]
    for first in range(0, total, portion):
        m = min(portion, total - first)
        batch = SimpleNamespace(q_start=i32([0, m, 2 * m]), ctx_len=i32([first] * seqs), state_slot=i32([0, 1]), max_state_slot=1,
                                max_query_len=m, token_seq=i32([0] * m + [1] * m))
        part = [t[first:first + m].transpose(0, 1).reshape(seqs * m, -1).contiguous() for t in (q, k, v)]
        out = torch.empty(seqs * m, heads * dim, device=DEV)
        getattr(_C.mixer_ops, rule)(out, *part, decay, state, batch, heads, dim, dim)
    assert float((state.double() - end).norm() / end.norm()) < 1.2e-6


@pytest.mark.parametrize("said", [0, 1, 3])
def test_a_run_longer_than_the_batch_says(said):
    """The longest run is a hint: a sequence that brings more is worked out all the same."""
    from splitwise_amd import _C
    heads, dim, lens = 2, 64, [1, 9, 40, 2]
    rows, n = sum(lens), len(lens)
    g = torch.Generator(device=DEV).manual_seed(said)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)          # noqa: E731
    batch = SimpleNamespace(q_start=i32([sum(lens[:i]) for i in range(n + 1)]), ctx_len=i32([3] * n), state_slot=i32(list(range(n))),
                            max_state_slot=n - 1, max_query_len=said, token_seq=i32([i for i, m in enumerate(lens) for _ in range(m)]))
    q, k, v = (torch.randn(rows, heads * dim, generator=g, device=DEV) for _ in range(3))
    decay, state = torch.linspace(0.3, 0.99, heads, device=DEV), torch.randn(n, heads, dim, dim, generator=g, device=DEV)
    got, out = state.clone(), torch.full_like(v, float("nan"))
    _C.mixer_ops.retention(out, q, k, v, decay, got, batch, heads, dim, dim)
    q64, k64, v64 = (t.double().view(rows, heads, dim) for t in (q, k, v))
    ref, ends = _rule(q64, k64, v64, decay.double().view(1, heads, 1).expand(rows, heads, 1), state.double(),
                      batch.q_start.tolist(), torch.zeros(n, dtype=torch.bool, device=DEV))
    for a, b in ((out.double().view_as(ref), ref), (got.double(), ends)):
        assert float((a - b).norm() / b.norm()) < 6e-7


@pytest.mark.parametrize("heads,dim,vdim", [(2, 128, 40), (1, 160, 16), (3, 64, 17)])
@pytest.mark.parametrize("lens", [[70, 33, 130], [1600]], ids=["runs", "segments"])
def test_gates_that_overflowed(heads, dim, vdim, lens):
    """A gate of +inf keeps a channel as it is, one of -inf or -3e38 forgets it: in single tokens of a long run, in both halves of a
    chunk and next to one another, against the rule in 64 bits and against the same tokens in portions of 13, which take the decode
    kernel.  A gate that is NaN makes its channel NaN, and with it the outputs from there on, and nothing else."""
    from splitwise_amd import _C
    n, inf = len(lens), float("inf")
    starts, rows = [sum(lens[:i]) for i in range(n + 1)], sum(lens)
    g = torch.Generator(device=DEV).manual_seed(rows + dim)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)               # noqa: E731
    nk, nv = heads * dim, heads * vdim
    proj, z, bias = rnd(rows, 2 * nk + nv).bfloat16(), rnd(rows, nk).bfloat16(), 2.0 + rnd(nk)
    for first, m in zip(starts, lens):
        for at, channel, gate in ((3, 0, -inf), (5, 1, inf), (17, 2, -inf), (20, 2, -inf), (6, 3, -3e38), (7, 3, inf), (22, 4, 1e38),
                                  (0, 5, -inf), (m - 1, 6, -inf), (31, 7, -1e38), (32, 7, -inf)):
            z[first + at, channel::dim] = gate
    q, k, v = proj[:, :nk], proj[:, nk:2 * nk], proj[:, 2 * nk:]
    state, slots, ctx = rnd(n, heads, dim, vdim) * 0.1, list(range(n)), [7, 0, 9][:n]

    def step(parts, out, s):
        """parts: (sequence, tokens before it, tokens)."""
        pick = torch.cat([torch.arange(starts[i] + lo, starts[i] + lo + m, device=DEV) for i, lo, m in parts])
        i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)      # noqa: E731
        batch = SimpleNamespace(q_start=i32([sum(m for _, _, m in parts[:i]) for i in range(len(parts) + 1)]),
                                ctx_len=i32([ctx[i] + lo for i, lo, _ in parts]), state_slot=i32([slots[i] for i, _, _ in parts]),
                                max_state_slot=n - 1, max_query_len=max(m for _, _, m in parts),
                                token_seq=i32([j for j, (_, _, m) in enumerate(parts) for _ in range(m)]))
        p, o = proj[pick], torch.empty(len(pick), nv, device=DEV)
        _C.mixer_ops.gla(o, p[:, :nk], p[:, nk:2 * nk], p[:, 2 * nk:], z[pick].contiguous(), bias, 16.0, dim ** -0.5, s, batch, heads,
                         dim, vdim)
        out[pick] = o

    whole = [(i, 0, m) for i, m in enumerate(lens)]
    keep = torch.exp(torch.nn.functional.logsigmoid(z.double() + bias.double()) / 16.0).view(rows, heads, dim)
    q64, k64, v64 = (t.double().view(rows, heads, -1) for t in (q, k, v))
    ref, ends = _rule(q64 * dim ** -0.5, k64, v64, keep, state.double(), starts, torch.tensor([c == 0 for c in ctx], device=DEV))
    got, out = state.clone(), torch.full((rows, nv), float("nan"), device=DEV)
    step(whole, out, got)
    short, pieces = state.clone(), torch.full((rows, nv), float("nan"), device=DEV)
    for lo in range(0, max(lens), 13):
        step([(i, lo, min(13, m - lo)) for i, m in enumerate(lens) if m > lo], pieces, short)
    for a, b in ((out.double().view_as(ref), ref), (got.double(), ends), (pieces.double().view_as(ref), ref), (short.double(), ends)):
        off = (a - b).abs()
        assert a.isfinite().all()
        assert float(off.norm() / b.norm()) < 6e-7 and float(off.max() / b.square().mean().sqrt()) < 3e-5
    z[starts[-2] + 40, 9] = float("nan")                       # the first head of the last sequence
    bad, res = state.clone(), out.clone()
    step(whole, res, bad)
    spoilt = torch.zeros_like(bad, dtype=torch.bool)
    spoilt[n - 1, 0, 9] = True
    assert torch.equal(bad.isnan(), spoilt) and torch.equal(bad[~spoilt], got[~spoilt])
    late = slice(starts[-2] + 40, None)
    assert res[late, :vdim].isnan().all() and torch.equal(res[late, vdim:], out[late, vdim:])
    before = starts[-2] + 40 // 32 * 32                        # (its chunk's outputs are sums over the whole channel)
    assert torch.equal(res[:before], out[:before])
