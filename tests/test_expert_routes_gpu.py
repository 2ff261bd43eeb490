"""The bf16 experts' three kernels (weights streamed for few rows, tiles of 64 x 64 and of 128 x 128) at the sizes where they
can go wrong: tiles' and stages' remainders, experts without rows, one expert with nearly all, more than 64 experts.

The reference takes the products in 64 bits and rounds the hidden layer to bf16 as the kernels do.  A hidden value on the
border between two bf16 numbers may be rounded the other way, by 2^-8 of itself; that bounds every output."""
import math
import os
import re

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _routes(pairs, experts, n):
    """What the rule beside the kernels says for a product of n weight rows, by its own numbers."""
    source = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "vllm-splitwise_amd", "csrc", "mixers", "expert_ffn.hip")
    with open(source) as f:
        numbers = dict(re.findall(r"constexpr int (kFewPairs|kManyPairs|kManyTiles) = (\d+);", f.read()))
    few, many, tiles = (int(numbers[k]) for k in ("kFewPairs", "kManyPairs", "kManyTiles"))
    if pairs <= few * experts:
        return "few"
    return "128" if pairs >= many * experts and pairs // 128 * -(-n // 128) >= tiles else "64"


@pytest.mark.parametrize("rows,width,ff,experts,top,act,skew,route", [
    (1, 64, 32, 4, 2, "glu", 0, "few"), (13, 72, 40, 9, 2, "relu2", 0, "few"), (50, 296, 200, 70, 4, "glu", 0, "few"),
    (90, 136, 24, 32, 2, "gelu", 40, "few"), (190, 520, 264, 64, 2, "glu", 6, "few"), (6, 40, 8, 1, 1, "relu2", 0, "few"),
    (65, 64, 48, 2, 1, "gelu", 0, "64"), (200, 328, 136, 5, 2, "glu", 3, "64"), (333, 200, 72, 66, 4, "relu2", 40, "64"),
    (128, 1032, 520, 3, 2, "glu", 0, "64"), (1501, 2056, 2120, 4, 2, "glu", 0, "128"), (3300, 1800, 1304, 3, 2, "relu2", 5, "128"),
    (2049, 3080, 3080, 20, 1, "gelu", 1, "128")])
@pytest.mark.parametrize("weigh_input", [False, True])
def test_expert_kernels_at_their_edges(rows, width, ff, experts, top, act, skew, route, weigh_input):
    from splitwise_amd import _C
    ops = _C.mixer_ops
    up_rows = 32 * -(-ff // 16) if act == "glu" else ff
    assert _routes(rows * top, experts, up_rows) == route and _routes(rows * top, experts, width) == route
    g = torch.Generator(device=DEV).manual_seed(rows * 7 + width)
    bf, rnd = torch.bfloat16, lambda *s: torch.randn(*s, generator=g, device=DEV)            # noqa: E731
    x, up = rnd(rows, width).to(bf), (rnd(experts, ff, width) * width ** -0.5).to(bf)
    gate, down = (rnd(experts, ff, width) * width ** -0.5).to(bf), (rnd(experts, width, ff) * ff ** -0.5).to(bf)
    want = rnd(rows, experts)
    want[:, experts // 2] += skew                              # most rows ask for this one
    want[:, 0] -= 100.0 if experts > top else 0.0              # nobody asks for this one
    chosen = want.topk(top, -1).indices.to(torch.int32).contiguous()
    weights = torch.rand(rows, top, generator=g, device=DEV) + 0.1
    order, start = ops.group_pairs(chosen, experts)
    out = torch.zeros(rows, width, device=DEV)
    packed = ops.glu_rows(gate, up) if act == "glu" else up
    ops.expert_ffn(out, x, packed, down, order, start, top, 0.5, activation=ops.ACT_GELU if act == "gelu" else ops.ACT_RELU2,
                   pair_weight=weights, glu=(1.702, 2.0, 1.0) if act == "glu" else None, weigh_input=weigh_input)
    ref, bound = torch.zeros(rows, width, dtype=torch.float64, device=DEV), torch.zeros(rows, width, dtype=torch.float64, device=DEV)
    for e in range(experts):
        r, c = (chosen == e).nonzero(as_tuple=True)
        if r.numel() == 0:
            continue
        w = weights[r, c].double()[:, None]
        z = torch.matmul(x[r].double(), up[e].double().t()) * (w if weigh_input else 1.0)
        if act == "glu":
            a = torch.matmul(x[r].double(), gate[e].double().t()) * (w if weigh_input else 1.0)
            a = a.clamp(max=2.0)
            z = a * torch.sigmoid(1.702 * a) * (z.clamp(-2.0, 2.0) + 1.0)
        else:
            z = torch.nn.functional.gelu(z) if act == "gelu" else z.clamp(min=0).square()
        h, d = z.to(bf).double(), down[e].double().t()
        scale = 0.5 * (1.0 if weigh_input else w)
        ref.index_add_(0, r, torch.matmul(h, d) * scale)
        bound.index_add_(0, r, torch.matmul(h.abs(), d.abs()) * scale * 2.0 ** -8)
    off = (out.double() - ref).abs()
    assert out.isfinite().all() and (off <= bound + 1e-5).all()
    # nearly all hidden values round the same way: in the mean the results are much closer than the bound
    assert off.norm() <= 1e-3 * ref.norm() and math.isfinite(float(ref.norm())) and float(ref.norm()) > 0


@pytest.mark.parametrize("experts", [1, 7, 64, 65, 256])
@pytest.mark.parametrize("pairs", [0, 1, 63, 1024, 1025, 2048, 2049, 8191, 8192, 8193, 20000])
def test_pairs_in_groups(pairs, experts):
    """On both sides of the pairs that one turn of the workgroup's threads takes; experts that nobody asks for; all on one."""
    from splitwise_amd import _C
    ops = _C.mixer_ops
    g = torch.Generator(device=DEV).manual_seed(pairs + experts)
    for chosen in (torch.randint(0, experts, (pairs, 1), generator=g, device=DEV), torch.full((pairs, 1), experts - 1, device=DEV)):
        order, start = ops.group_pairs(chosen.to(torch.int32), experts)
        count = torch.bincount(chosen.flatten(), minlength=experts)
        assert start.tolist() == [0] + torch.cumsum(count, 0).tolist()
        assert torch.equal(order.sort().values, torch.arange(pairs, device=DEV, dtype=torch.int32))
        assert torch.equal(chosen.flatten()[order.long()], chosen.flatten().sort().values)
