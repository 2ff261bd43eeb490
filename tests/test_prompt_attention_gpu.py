"""Steps of the mixers' attention on the bf16 matrix cores against the attention in 64 bits and against the general kernel.

The general kernel takes a call whose queries do not lie on 16 bytes, so the same step is made with its queries moved by one
float too.  Both keep scores, weights and sums in fp32 (an error of about 1e-5 of the largest value) and round once to bf16: two
results are at most one unit in the last place, 2^-7 of the value at most, apart.  Which kernels a call goes to is asked of
attention_plan.h, which the launch code goes by."""
import ctypes
import os
import subprocess
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


PROMPT, DECODE, GENERAL = range(3)                           # enum AttentionWay
PLAN = r"""
#include "attention_plan.h"
extern "C" int way(unsigned long at, long k_stride, long v_stride, int seqs, int mql, int heads, int kv_heads, int dim, int vdim, int page,
                   int width, int window, int chunk) {
  return swm::attention_way(swm::attention_pieces(at, dim, vdim, k_stride, v_stride), seqs, mql, heads, kv_heads, dim, vdim, page,
                            width, window, chunk);
}
extern "C" int groups(long rows, int seqs, int mql, int heads, int kv_heads, int page, int width, int window, int chunk) {
  return swm::prompt_attention_groups(rows, seqs, mql, heads, kv_heads, page, width, window, chunk);
}
"""


@pytest.fixture(scope="module")
def way(tmp_path_factory):
    """-> the kernels that a call goes to."""
    at = tmp_path_factory.mktemp("plan")
    (at / "plan.cpp").write_text(PLAN)
    mixers = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "vllm-splitwise_amd", "csrc", "mixers")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", mixers, str(at / "plan.cpp"), "-o", str(at / "plan.so")],
                   check=True)
    lib = ctypes.CDLL(str(at / "plan.so"))

    def ask(q, kc, vc, batch, H, G, d, dv, window=0, chunk=0, **_):
        vc = kc if vc is None else vc
        at = q.data_ptr() | kc.data_ptr() | vc.data_ptr()
        return lib.way(ctypes.c_ulong(at), ctypes.c_long(kc.shape[2]), ctypes.c_long(vc.shape[2]), batch.num_seqs, batch.max_query_len, H,
                       G, d, dv, kc.shape[1], batch.block_tables.shape[1], window, chunk)

    def groups(batch, H, G, page, window=0, chunk=0, **_):
        """-> how many groups of waves share a workgroup's walk in the prompt kernel."""
        return lib.groups(ctypes.c_long(batch.token_seq.numel()), batch.num_seqs, batch.max_query_len, H, G, page,
                          batch.block_tables.shape[1], window, chunk)
    ask.groups = groups
    return ask


def _step(lengths, page):
    starts, owner, tables, used = [0], [], [], 2
    width = max(-(-(c + n) // page) for c, n in lengths)
    for i, (c, n) in enumerate(lengths):
        starts.append(starts[-1] + n)
        owner += [i] * n
        need = -(-(c + n) // page)
        tables.append([used + (j * 7 + 3) % need if need % 7 else used + need - 1 - j for j in range(need)] + [0] * (width - need))
        used += need
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)          # noqa: E731
    return SimpleNamespace(q_start=i32(starts), ctx_len=i32([c for c, _ in lengths]), token_seq=i32(owner),
                           state_slot=i32(list(range(len(lengths)))), block_tables=i32(tables), num_seqs=len(lengths),
                           max_query_len=max(n for _, n in lengths), max_pages_used=width, max_page_id=used - 1,
                           max_state_slot=len(lengths) - 1), used


def _statement(lengths, batch, q, kc, vc, gate, H, G, d, dv, softcap=0.0, window=0, chunk=0, sink=False, score_bias=None):
    """The attention in 64 bits, a query at a time over the keys that it sees.  vc None: values inside the key rows."""
    page, vc, out, row = kc.shape[1], kc if vc is None else vc, [], 0
    for i, (c, n) in enumerate(lengths):
        pages = batch.block_tables[i, :-(-(c + n) // page)].long()
        ks, vs = (t[pages].reshape(-1, t.shape[-1])[:c + n].double() for t in (kc, vc))
        for t in range(n):
            pos = c + t
            lo = pos // chunk * chunk if chunk else max(0, pos - window + 1) if window else 0
            for h in range(H):
                g = h // (H // G)
                k, v = ks[lo:pos + 1, g * d:(g + 1) * d], vs[lo:pos + 1, g * dv:(g + 1) * dv]
                s = (k * (q[row + t, h * d:(h + 1) * d].double() * d ** -0.5)).sum(-1)
                s = softcap * torch.tanh(s / softcap) if softcap else s
                if score_bias is not None:
                    w = torch.sigmoid(s + score_bias[h].double())
                else:
                    extra = sink[h:h + 1].double() if isinstance(sink, torch.Tensor) else s.new_zeros(1 if sink else 0)
                    w = torch.cat([s, extra]).softmax(0)[:len(s)]
                out.append((w[:, None] * v).sum(0))
        row += n
    out = torch.stack(out).view(row, H * dv)
    return out if gate is None else out * torch.sigmoid(gate.double())


@pytest.mark.parametrize("option", ["plain", "cap", "sigmoid", "learned sink"])
@pytest.mark.parametrize("H,G,d", [(4, 2, 64), (3, 1, 128)])
@pytest.mark.parametrize("lengths", [[(70, 9), (37, 40), (64, 1), (40, 1)], [(64, 1), (40, 2), (300, 1)], [(2100, 1), (33, 1)]],
                         ids=["prompt", "decode", "decode, keys shared out"])
def test_infinities_in_the_cache(H, G, d, option, lengths):
    """A key coordinate or value that overflowed to an infinity gives what fp32 products give: a score of -inf hides its key, a
    capped score of inf is the cap, a value of inf stays inf.  Queries of few bits: all but the first part of theirs is zero."""
    from splitwise_amd import _C
    batch, pages = _step(lengths, 16)
    g = torch.Generator(device=DEV).manual_seed(H * 100 + d)
    rows, inf = sum(n for _, n in lengths), float("inf")
    kc, vc = (torch.randn(pages, 16, G * d, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    q = torch.randint(1, 16, (rows, H * d), generator=g, device=DEV).float() / 8.0
    at = lambda i, pos: (int(batch.block_tables[i, pos // 16]), pos % 16)   # noqa: E731
    for i, (c, n) in enumerate(lengths):                     # (keys that every query of the sequence sees)
        p, o = at(i, 3)
        kc[p, o, 5::d] = -inf                                # queries are positive: a score of -inf
        if option != "plain" and option != "learned sink":   # (a softmax over a score of inf is NaN, there as here)
            p, o = at(i, 9)
            kc[p, o, 7::d] = inf
        p, o = at(i, 17)
        vc[p, o, 2::d], vc[p, o, 11::d] = inf, -inf
        if n == 1:                                           # the last key of all: what lies behind it is nobody's
            p, o = at(i, c)
            vc[p, o, 4::d] = inf
    kw = {"cap": dict(softcap=4.0), "learned sink": dict(sink=torch.linspace(-3.0, 2.0, H, device=DEV)),
          "sigmoid": dict(score_bias=torch.linspace(-2.0, 1.0, H, device=DEV))}.get(option, {})
    out = torch.empty(rows, H * d, dtype=torch.bfloat16, device=DEV)
    _C.mixer_ops.capped_attention(out, q, kc, vc, None, batch, H, G, d, d, d ** -0.5, **kw)
    ref = _statement(lengths, batch, q, kc, vc, None, H, G, d, d, **kw)
    assert not ref.isnan().any() and ref.isinf().any()
    torch.testing.assert_close(out.double(), ref, atol=2e-4, rtol=2.0 ** -7)


@pytest.mark.parametrize("H,G,d", [(4, 2, 128), (3, 3, 96)])
def test_an_infinity_in_shared_keys_that_one_of_two_tokens_sees(H, G, d, way):
    """An infinite value in front of the second token's window: the channels that it spoils are worked out again, those of another
    wave are not, and both are joined with the other workgroups' parts by one maximum."""
    from splitwise_amd import _C
    lengths, window = [(2100, 2), (1800, 2)], 1500
    batch, pages = _step(lengths, 16)
    g = torch.Generator(device=DEV).manual_seed(d)
    kc, vc = (torch.randn(pages, 16, G * d, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    q = torch.randn(4, H * d, generator=g, device=DEV) * 2
    for i, (c, _) in enumerate(lengths):
        at = lambda pos: (int(batch.block_tables[i, pos // 16]), pos % 16)  # noqa: E731
        first = c - window + 1                               # the first token's first key
        assert first // 32 == (first + 1) // 32
        vc[at(first)][d - 20::d] = float("inf")
        # a score of 8 for the second token in the second tile of that tile's wave, of 4 parts of 8: its running maximum stays behind
        own = q[2 * i + 1].view(G, H // G, d)[:, 0]
        kc[at(first // 32 * 32 + 4 * 8 * 32 + 5)] = (8 * d ** 0.5 * own / own.square().sum(-1, keepdim=True)).flatten().bfloat16()
    assert way(q, kc, vc, batch, H, G, d, d, window=window) == DECODE
    out = torch.empty(4, H * d, dtype=torch.bfloat16, device=DEV)
    _C.mixer_ops.capped_attention(out, q, kc, vc, None, batch, H, G, d, d, d ** -0.5, window=window)
    ref = _statement(lengths, batch, q, kc, vc, None, H, G, d, d, window=window)
    assert ref[1::2].isfinite().all() and ref[::2].isinf().any() and not ref.isnan().any()
    torch.testing.assert_close(out.double(), ref, atol=2e-4, rtol=2.0 ** -7)


@pytest.mark.parametrize("H,G,d,page", [(4, 2, 128, 16), (3, 1, 96, 12), (8, 4, 24, 8)])
@pytest.mark.parametrize("option", ["plain", "cap", "window", "chunk", "learned sink", "sigmoid"])
@pytest.mark.parametrize("lengths", [[(0, 240), (0, 40)], [(0, 255), (0, 40)], [(0, 257), (31, 66)], [(700, 33), (256, 1), (224, 40), (607, 2)],
                                     [(700, 33), (256, 1), (224, 40), (607, 2)] + [(i * 37 % 700, 1) for i in range(256)]],
                         ids=lambda v: str(v[:4]) + " and 256 more" * (len(v) > 4))
def test_two_groups_share_a_walk(H, G, d, page, option, lengths, way):
    """On both sides of the number of keys from which two groups of waves share a workgroup's stages of 32, and of the number of
    workgroups beyond which long walks go to one group; odd and even numbers of stages, rows that see keys of one group's only.  In
    front, from the second stage on, keys that weigh next to nothing or most, and a value of inf in a channel: what one group makes of
    it has to meet the other's sums.  (Tolerances as above.)"""
    from splitwise_amd import _C
    batch, pages = _step(lengths, page)
    g = torch.Generator(device=DEV).manual_seed(d + len(lengths))
    rows, inf = sum(n for _, n in lengths), float("inf")
    kc, vc = (torch.randn(pages, page, G * d, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    q = torch.randn(rows, H * d, generator=g, device=DEV)
    at = lambda i, pos: (int(batch.block_tables[i, pos // page]), pos % page)   # noqa: E731
    for i, (c, n) in enumerate(lengths):
        kc[at(i, min(34, c + n - 1))] *= 9.0
        if c > 100:
            vc[at(i, c // 32 * 32 - 20)][3::d] = inf         # the last stage but one or two that all of the sequence's rows see
    kw = {"cap": dict(softcap=4.0), "window": dict(window=290), "chunk": dict(chunk=258), "sigmoid": dict(score_bias=torch.linspace(-2.0, 1.0, H, device=DEV)),
          "learned sink": dict(sink=torch.linspace(-3.0, 2.0, H, device=DEV))}.get(option, {})
    assert way(q, kc, vc, batch, H, G, d, d, **kw) == PROMPT
    assert way.groups(batch, H, G, page, **kw) == (1 if len(lengths) > 4 or lengths[0] == (0, 240) else 2)
    out = torch.empty(rows, H * d, dtype=torch.bfloat16, device=DEV)
    _C.mixer_ops.capped_attention(out, q, kc, vc, None, batch, H, G, d, d, d ** -0.5, **kw)
    ref = _statement(lengths, batch, q, kc, vc, None, H, G, d, d, **kw)
    assert not ref.isnan().any() and (len(lengths) < 3 or ref.isinf().any())
    torch.testing.assert_close(out.double(), ref, atol=2e-4, rtol=2.0 ** -7)


def test_a_page_of_4_gib():
    """The second page of a cache begins 2^32 bytes behind the first."""
    from splitwise_amd import _C
    H = G = 16
    d, page = 128, 1 << 20
    lengths = [(0, 40)]
    batch, _ = _step(lengths, page)
    batch.block_tables.fill_(1)
    batch.max_page_id = 1
    g = torch.Generator(device=DEV).manual_seed(3)
    kc = torch.zeros(2, page, G * d, dtype=torch.bfloat16, device=DEV)       # values are the keys
    kc[1, :40] = torch.randn(40, G * d, generator=g, device=DEV).to(torch.bfloat16)
    q = torch.randn(40, H * d, generator=g, device=DEV)
    out = torch.empty(40, H * d, dtype=torch.bfloat16, device=DEV)
    _C.mixer_ops.capped_attention(out, q, kc, None, None, batch, H, G, d, d, d ** -0.5)
    near = SimpleNamespace(block_tables=torch.zeros_like(batch.block_tables))
    ref = _statement(lengths, near, q, kc[1:, :64], None, None, H, G, d, d)
    torch.testing.assert_close(out.double(), ref, atol=2e-4, rtol=2.0 ** -7)


@pytest.mark.parametrize("H,G,d,dv,page", [(4, 4, 128, 128, 16), (8, 2, 64, 96, 16), (6, 2, 40, 24, 8), (32, 1, 16, 8, 32),
                                           (3, 1, 104, 128, 12)])
@pytest.mark.parametrize("option", ["plain", "cap", "window", "chunk", "sink", "learned sink", "sigmoid", "values in the keys"])
def test_prompt_steps_agree_with_the_general_kernel(H, G, d, dv, page, option, way):
    from splitwise_amd import _C
    per_wg = 4 * (32 // (H // G))                            # tokens of a workgroup
    lengths = [(0, per_wg), (5, per_wg + 1), (0, 1), (31, max(1, per_wg - 1)), (0, 2 * per_wg + 33), (200, 32), (64, 1)]
    batch, pages = _step(lengths, page)
    g = torch.Generator(device=DEV).manual_seed(H * 100 + d)
    rows = sum(n for _, n in lengths)
    if option == "values in the keys" and G > 1:
        dv = d
    kc = torch.randn(pages, page, G * d, generator=g, device=DEV).to(torch.bfloat16)
    vc = torch.randn(pages, page, G * dv, generator=g, device=DEV).to(torch.bfloat16)
    kc[:2], vc[:2] = float("nan"), float("nan")              # pages that no table names
    if option == "values in the keys":
        dv, vc = min(d, dv) // 8 * 8, None
    else:                                                    # slots behind a sequence's end have never been written
        for i, (c, n) in enumerate(lengths):
            if (c + n) % page:
                last = int(batch.block_tables[i, (c + n) // page])
                kc[last, (c + n) % page:], vc[last, (c + n) % page:] = float("nan"), float("nan")
    q = torch.randn(rows * H * d + 4, generator=g, device=DEV) * 2
    gate = torch.randn(rows, H * dv + 3, generator=g, device=DEV).to(torch.bfloat16)[:, 3:]
    kw = {"cap": dict(softcap=4.0), "window": dict(window=37), "chunk": dict(chunk=48), "sink": dict(sink=True),
          "learned sink": dict(sink=torch.linspace(-3.0, 9.0, H, device=DEV)),
          "sigmoid": dict(score_bias=torch.linspace(-2.0, 1.0, H, device=DEV))}.get(option, {})
    outs = []
    for lead in (0, 1):                                      # aligned queries, then the same ones a float further on
        at = torch.empty(rows * H * d + 1, device=DEV)[lead:lead + rows * H * d].view(rows, H * d)
        at.copy_(q[:rows * H * d].view(rows, H * d))
        assert at.data_ptr() % 16 == 4 * lead
        assert way(at, kc, vc, batch, H, G, d, dv, **kw) == (GENERAL if lead else PROMPT)
        out = torch.full((rows, H * dv), float("nan"), dtype=torch.bfloat16, device=DEV)
        _C.mixer_ops.capped_attention(out, at, kc, vc, gate if option != "plain" else None, batch, H, G, d, dv, d ** -0.5,
                                      **kw)
        outs.append(out.float())
    torch.testing.assert_close(outs[0], outs[1], atol=2e-4, rtol=2.0 ** -7)
    ref = _statement(lengths, batch, at, kc, vc, gate if option != "plain" else None, H, G, d, dv, **kw)
    torch.testing.assert_close(outs[0].double(), ref, atol=2e-4, rtol=2.0 ** -7)
    assert outs[0].isfinite().all() and outs[0].abs().max() > 0.1


@pytest.mark.parametrize("H,G,d,dv", [(4, 1, 32, 32), (8, 2, 64, 56), (6, 2, 96, 96), (16, 4, 128, 128), (5, 1, 128, 104)])
def test_finished_rows_go_out_alike_whatever_the_alignment(H, G, d, dv, way):
    """Gates and results on 16 bytes and off them, gates at sigmoid's ends: the same bits four times, those of the 64-bit statement
    within the bound above."""
    from splitwise_amd import _C
    lengths = [(0, 40), (5, 3), (0, 33), (17, 1)]
    batch, pages = _step(lengths, 16)
    g = torch.Generator(device=DEV).manual_seed(H * dv)
    rows = sum(n for _, n in lengths)
    kc, vc = (torch.randn(pages, 16, G * n, generator=g, device=DEV).to(torch.bfloat16) for n in (d, dv))
    q = torch.randn(rows, H * d, generator=g, device=DEV)
    gate = torch.randn(rows, H * dv, generator=g, device=DEV).to(torch.bfloat16) * 4
    gate[1, :8] = torch.tensor([float("inf"), -float("inf"), 80.0, -80.0, 88.5, -88.5, 3e38, -3e38])
    assert way(q, kc, vc, batch, H, G, d, dv) == PROMPT
    outs = []
    for gate_at, out_at in ((0, 0), (0, 3), (1, 0), (1, 3)):
        wide = torch.full((rows, H * dv + 8), 7.0, dtype=torch.bfloat16, device=DEV)
        out = wide[:, out_at:out_at + H * dv]
        at = torch.empty(rows, H * dv + 8, dtype=torch.bfloat16, device=DEV)[:, gate_at:gate_at + H * dv]
        at.copy_(gate)
        _C.mixer_ops.capped_attention(out, q, kc, vc, at, batch, H, G, d, dv, d ** -0.5)
        assert (wide[:, :out_at] == 7).all() and (wide[:, out_at + H * dv:] == 7).all()
        outs.append(out.float())
    for other in outs[1:]:
        assert torch.equal(outs[0], other)
    ref = _statement(lengths, batch, q, kc, vc, gate, H, G, d, dv)
    torch.testing.assert_close(outs[0].double(), ref, atol=2e-4, rtol=2.0 ** -7)


def test_every_gate_weighs_as_in_the_general_kernel(way):
    """A first token sees its own value alone, so that its result is value times sigmoid(gate) rounded once: the general kernel's bits
    for every bf16 gate there is, and with large values those whose sigmoid is no normal number any more (2^-126 is reached at -87.3)."""
    from splitwise_amd import _C
    H, G, d, lengths = 16, 4, 128, [(0, 33)] * 32
    batch, pages = _step(lengths, 16)
    g = torch.Generator(device=DEV).manual_seed(5)
    rows, first = 32 * 33, torch.arange(0, 32 * 33, 33, device=DEV)
    kc = torch.randn(pages, 16, G * d, generator=g, device=DEV).to(torch.bfloat16)
    vc = (torch.randn(pages, 16, G * d, generator=g, device=DEV) * 2.0 ** 40).to(torch.bfloat16)
    q = torch.randn(rows * H * d + 1, generator=g, device=DEV)
    gate = torch.zeros(rows, H * d, dtype=torch.bfloat16, device=DEV)
    gate[first] = torch.arange(-32768, 32768, device=DEV).to(torch.int16).view(torch.bfloat16).view(32, H * d)
    outs = []
    for lead in (0, 1):
        at = q[lead:lead + rows * H * d].view(rows, H * d)
        assert way(at, kc, vc, batch, H, G, d, d) == (GENERAL if lead else PROMPT)
        out = torch.empty(rows, H * d, dtype=torch.bfloat16, device=DEV)
        _C.mixer_ops.capped_attention(out, at, kc, vc, gate, batch, H, G, d, d, d ** -0.5)
        outs.append(out[first].float())
    torch.testing.assert_close(outs[0], outs[1], atol=0, rtol=0, equal_nan=True)
    value = vc[batch.block_tables[:, 0].long(), 0].double().view(32, G, 1, d).expand(32, G, H // G, d).reshape(32, H * d)
    ref = value * torch.sigmoid(gate[first].double())
    seen = (gate[first].double() > -88.5) & ref.abs().isfinite()             # (from -88.7 on e^-gate overflows in fp32)
    assert float(((outs[0].double() - ref).abs() / ref.abs())[seen].max()) < 2.0 ** -8 * 1.001


@pytest.mark.parametrize("H,G,d,dv,page", [(4, 4, 128, 128, 16), (8, 2, 64, 96, 16), (6, 2, 40, 24, 8), (8, 1, 16, 8, 32),
                                           (5, 1, 104, 128, 12)])
@pytest.mark.parametrize("option", ["plain", "cap", "window", "chunk", "sink", "learned sink", "sigmoid", "values in the keys"])
@pytest.mark.parametrize("long", [0, 1, 2])
def test_decode_steps_agree_with_the_general_kernel(H, G, d, dv, page, option, long, way):
    """Few query rows per sequence and key/value head: one or two sets of four, one or several workgroups per sequence (the
    step's longest context decides), contexts at the edges of the 32-key tiles.  Same bound as above."""
    from splitwise_amd import _C
    most = 8 // (H // G)                                     # tokens of a sequence
    lengths = [[(0, 1), (5, 1), (30, 1), (31, 1), (32, most), (200, 1), (256, most)], [(900, 1), (2300, most), (31, 1)],
               [(4001, 1)]][long]
    batch, pages = _step(lengths, page)
    g = torch.Generator(device=DEV).manual_seed(H * 100 + d + long)
    rows = sum(n for _, n in lengths)
    few = H == G and long == 2 and option in ("window", "chunk")             # one query row that sees few keys
    if option == "values in the keys" and G > 1:
        dv = d
    kc = torch.randn(pages, page, G * d, generator=g, device=DEV).to(torch.bfloat16)
    vc = torch.randn(pages, page, G * dv, generator=g, device=DEV).to(torch.bfloat16)
    kc[:2], vc[:2] = float("nan"), float("nan")              # pages that no table names
    if option == "values in the keys":
        dv, vc = min(d, dv) // 8 * 8, None
    else:                                                    # slots behind a sequence's end have never been written
        for i, (c, n) in enumerate(lengths):
            if (c + n) % page:
                last = int(batch.block_tables[i, (c + n) // page])
                kc[last, (c + n) % page:], vc[last, (c + n) % page:] = float("nan"), float("nan")
            if option == "window" and c > 3 * page + 37:     # pages behind a window may be somebody else's by now
                batch.block_tables[i, :(c - 36) // page] = 0
    q = torch.randn(rows * H * d + 4, generator=g, device=DEV) * 2
    gate = torch.randn(rows, H * dv + 3, generator=g, device=DEV).to(torch.bfloat16)[:, 3:]
    kw = {"cap": dict(softcap=4.0), "window": dict(window=37), "chunk": dict(chunk=48), "sink": dict(sink=True),
          "learned sink": dict(sink=torch.linspace(-3.0, 9.0, H, device=DEV)),
          "sigmoid": dict(score_bias=torch.linspace(-2.0, 1.0, H, device=DEV))}.get(option, {})
    outs = []
    for lead in (0, 1):                                      # aligned queries, then the same ones a float further on
        at = torch.empty(rows * H * d + 1, device=DEV)[lead:lead + rows * H * d].view(rows, H * d)
        at.copy_(q[:rows * H * d].view(rows, H * d))
        assert way(at, kc, vc, batch, H, G, d, dv, **kw) == (GENERAL if lead or few else DECODE)
        out = torch.full((rows, H * dv), float("nan"), dtype=torch.bfloat16, device=DEV)
        _C.mixer_ops.capped_attention(out, at, kc, vc, gate if option != "plain" else None, batch, H, G, d, dv, d ** -0.5,
                                      **kw)
        outs.append(out.float())
    torch.testing.assert_close(outs[0], outs[1], atol=2e-4, rtol=2.0 ** -7)
    ref = _statement(lengths, batch, at, kc, vc, gate if option != "plain" else None, H, G, d, dv, **kw)
    torch.testing.assert_close(outs[0].double(), ref, atol=2e-4, rtol=2.0 ** -7)
    # (a mean over up to 4002 keys of values of spread 1: 4002^-1/2 = 0.016 at least, the largest of them more)
    assert outs[0].isfinite().all() and outs[0].abs().max() > 0.016


@pytest.mark.parametrize("G,d,most", [(3, 128, 512), (8, 64, 256), (2, 96, 160), (3, 104, 512), (5, 40, 256), (1, 16, 160), (300, 32, 320), (150, 64, 1024)])
@pytest.mark.parametrize("option", ["plain", "cap", "learned sink", "sigmoid"])
def test_one_query_row_on_both_sides_of_the_rule(G, d, most, option, way):
    """One new token per sequence, one head per key/value head: up to `most` keys the vector kernel, the matrix cores beyond."""
    from splitwise_amd import _C
    page = 8
    kw = {"cap": dict(softcap=4.0), "learned sink": dict(sink=torch.linspace(-3.0, 9.0, G, device=DEV)),
          "sigmoid": dict(score_bias=torch.linspace(-2.0, 1.0, G, device=DEV))}.get(option, {})
    for longest, expected in ((most, GENERAL), (most + 1, DECODE)):
        lengths = [(longest - 1, 1), (0, 1), (min(31, longest - 1), 1), (most // 2, 1)]
        batch, pages = _step(lengths, page)
        g = torch.Generator(device=DEV).manual_seed(G * 100 + d)
        kc, vc = (torch.randn(pages, page, G * d, generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
        q = torch.randn(len(lengths), G * d, generator=g, device=DEV) * 2
        assert way(q, kc, vc, batch, G, G, d, d) == expected
        out = torch.full((len(lengths), G * d), float("nan"), dtype=torch.bfloat16, device=DEV)
        _C.mixer_ops.capped_attention(out, q, kc, vc, None, batch, G, G, d, d, d ** -0.5, **kw)
        ref = _statement(lengths, batch, q, kc, vc, None, G, G, d, d, **kw)
        torch.testing.assert_close(out.double(), ref, atol=2e-4, rtol=2.0 ** -7)
