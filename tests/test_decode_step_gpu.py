"""A small decode step's cache write and attention in one launch against the two calls one after the other: the same bits in the caches and
in the output, whatever kernel the sizes take and whatever blocks the sequences share; what it does not take is left to the two calls."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(heads, kv_heads, dim, ctx, dtype, cache, block, seed=0):
    """q, k, v as column ranges of one projection, filled caches, the slots of the sequences' last tokens, block tables, lengths."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    n = len(ctx)
    proj = torch.randn(n, (heads + 2 * kv_heads) * dim, generator=g, device=DEV).to(dtype)
    q, k, v = (t.view(n, -1, dim) for t in proj.split([heads * dim, kv_heads * dim, kv_heads * dim], dim=1))
    es = torch.finfo(dtype).bits // 8
    x = 16 // (1 if cache != "auto" else es)
    need = [-(-c // block) for c in ctx]
    order = torch.randperm(sum(need) + 2, generator=g, device=DEV).to(torch.int32)
    tables = torch.zeros(n, max(need), dtype=torch.int32, device=DEV)
    at = 0
    for i, m in enumerate(need):
        tables[i, :m] = order[at:at + m]
        at += m
    caches = [torch.randn(sum(need) + 2, kv_heads, *shape, generator=g, device=DEV).to(dtype)
              for shape in ((dim // x, block, x), (dim, block))]
    if cache != "auto":
        caches = [t.to(torch.float8_e5m2).view(torch.uint8) for t in caches]
    slots = torch.tensor([int(tables[i, (c - 1) // block]) * block + (c - 1) % block for i, c in enumerate(ctx)], device=DEV)
    return q, k, v, caches, slots, tables, torch.tensor(ctx, dtype=torch.int32, device=DEV)


def _temporaries(q, longest):
    parts = -(-longest // 512)
    sums = torch.empty(q.shape[0], q.shape[1], parts, device=DEV)
    return [sums, torch.empty_like(sums), torch.empty(q.shape[0], q.shape[1], parts, q.shape[2], dtype=q.dtype, device=DEV)]


def _both(case, cache, split, slopes=None):
    from splitwise_amd import _C
    q, k, v, caches, slots, tables, lens = case
    scale, longest, block, kv_heads = q.shape[2] ** -0.5, int(lens.max()), caches[1].shape[3], k.shape[1]
    ref, got = torch.zeros_like(q), torch.zeros_like(q)
    ours = [t.clone() for t in caches]
    _C.cache_ops.reshape_and_cache(k, v, *caches, slots, cache)
    if split:
        _C.ops.paged_attention_v2(ref, *_temporaries(q, longest), q, *caches, kv_heads, scale, tables, lens, block, longest, slopes, cache)
    else:
        _C.ops.paged_attention_v1(ref, q, *caches, kv_heads, scale, tables, lens, block, longest, slopes, cache)
    temporaries = _temporaries(q, longest) if split else [None] * 3
    assert _C.ops.paged_attention_and_cache(got, *temporaries, q, k, v, *ours, slots, scale, tables, lens, longest, cache, kv_heads, slopes)
    assert torch.equal(ref, got) and all(torch.equal(a, b) for a, b in zip(caches, ours))


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("cache", ["auto", "fp8_e5m2"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,kv_heads,dim,block", [(32, 32, 128, 16), (64, 8, 128, 32), (12, 12, 64, 16), (6, 3, 96, 8), (4, 4, 256, 32)])
def test_one_launch_is_the_two(heads, kv_heads, dim, block, dtype, cache, split):
    for ctx in ([1], [15, 16, 17, 1040], [513] * 3 + [100] * 5, [40 + 31 * i for i in range(25)]):
        _both(_case(heads, kv_heads, dim, ctx, dtype, cache, block), cache, split)
    slopes = torch.rand(heads, device=DEV)
    _both(_case(heads, kv_heads, dim, [70, 530], dtype, cache, block), cache, split, slopes)


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("seqs", [4, 5, 14, 17, 98])         # all tokens written by everyone; those that are looked up
@pytest.mark.parametrize("heads,kv_heads,dim", [(8, 8, 128), (16, 2, 128), (6, 3, 80)])
def test_sequences_that_read_each_others_tokens(heads, kv_heads, dim, seqs, split):
    """Every sequence's table also holds the others' newest blocks, one token has no slot, and one goes into the middle of a block that
    all of them read."""
    ctx = ([700, 650, 600, 530, 33, 48, 16, 90, 700, 700, 20, 5, 64, 129] * 7)[:seqs]
    case = _case(heads, kv_heads, dim, ctx, torch.bfloat16, "auto", 16)
    q, k, v, caches, slots, tables, lens = case
    newest = (slots // 16).to(torch.int32)
    for i, c in enumerate(ctx):
        held = min(-(-c // 16) - 1, len(ctx))
        tables[i, :held] = newest.roll(i)[:held]
    slots[3] = -1
    slots[5 % seqs] = int(newest[0]) * 16 + 2
    _both(case, "auto", split)


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("heads,kv_heads,dim", [(1, 1, 64), (4, 1, 64)])        # the vector kernel, the matrix cores
def test_blocks_that_look_alike(heads, kv_heads, dim, split):
    """Block numbers beyond the lookup's 8192 bits: sequence i reads blocks whose numbers differ by 8192 from those that the others' tokens
    go to, the one above or the one below, and two of the others' own."""
    ctx = [700 - 16 * (i % 7) for i in range(24)]
    q, k, v, _, _, tables, lens = _case(heads, kv_heads, dim, ctx, torch.bfloat16, "auto", 16)
    blocks = 3 * 8192
    g = torch.Generator(device=DEV).manual_seed(1)
    caches = [torch.randn(blocks, kv_heads, *shape, generator=g, device=DEV).to(torch.bfloat16) for shape in ((dim // 8, 16, 8), (dim, 16))]
    newest = [8192 + 100 + 5 * i if i % 2 else 2 * 8192 + 100 + 5 * i for i in range(24)]
    for i, c in enumerate(ctx):
        row = [(b + 8192) % blocks for b in newest[:i] + newest[i + 1:]] + [newest[i - 1], newest[i - 2]] + list(range(20 * i, 20 * i + 20))
        last = (c - 1) // 16
        tables[i, :last] = torch.tensor(row[:last], dtype=torch.int32)
        tables[i, last] = newest[i]
    slots = torch.tensor([newest[i] * 16 + (c - 1) % 16 for i, c in enumerate(ctx)], device=DEV)
    _both((q, k, v, caches, slots, tables, lens), "auto", split)


@torch.inference_mode()
@pytest.mark.parametrize("heads,kv_heads", [(8, 8), (8, 2)])
def test_layer_with_rotary(heads, kv_heads):
    """A layer that is handed the rotary module rotates and writes the cache in a launch of its own: the same bits as rotating first and
    then the layer without it, which writes the cache in the attention's."""
    from splitwise_amd.model_executor.input_metadata import InputMetadata
    from splitwise_amd.model_executor.layers.attention import Attention
    from splitwise_amd.model_executor.layers.basic import RotaryEmbedding
    dim, ctx = 128, [40, 700, 1100]
    q, k, v, caches, slots, tables, lens = _case(heads, kv_heads, dim, ctx, torch.bfloat16, "auto", 16)
    layer, rotary = Attention(heads, dim, dim ** -0.5, kv_heads), RotaryEmbedding(dim, dim, 2048, 10000.0, True, torch.bfloat16).to(DEV)
    md = InputMetadata(is_prompt=False, slot_mapping=slots, prompt_lens=None, max_seq_len=None, start_loc=None, max_context_len=max(ctx),
                       context_lens=lens, block_tables=tables, use_cuda_graph=False, kv_cache_dtype="auto")
    positions, results = lens.long() - 1, []
    for handed_over in (True, False):
        a, b, c, to = q.flatten(1).clone(), k.flatten(1).clone(), v.flatten(1), [t.clone() for t in caches]
        if handed_over:
            out = layer(a, b, c, *to, md, rotary=rotary, positions=positions)
        else:
            out = layer(*rotary(positions, a, b), c, *to, md)
        results.append([out, a, *to])
    assert all(torch.equal(x, y) for x, y in zip(*results)) and not torch.equal(results[0][2], caches[0])


@pytest.mark.parametrize("longest", [256, 257])
@pytest.mark.parametrize("seqs", [4, 24])                    # all tokens written by everyone; those that are looked up
def test_waves_of_short_contexts(seqs, longest):
    """On either side of the length from which a launch has 8 waves whatever it writes."""
    _both(_case(12, 12, 64, ([longest, 1, 64, 65, 200, 255] * 4)[:seqs], torch.float16, "auto", 16), "auto", False)


@pytest.mark.parametrize("split", [False, True])
def test_lds_just_under_64_kb(split):
    """Eleven query heads a kv head, eight waves: 64192 bytes of LDS, and tokens that are looked up (in some of them)."""
    _both(_case(22, 2, 128, [40 + 31 * i for i in range(25)], torch.bfloat16, "auto", 16), "auto", split)


def test_what_is_left_to_the_two_calls():
    from splitwise_amd import _C
    def call(case, cache="auto", **other):
        q, k, v, caches, slots, tables, lens = case
        a = dict(q=q, k=k, v=v, kc=caches[0], vc=caches[1], slots=slots) | other
        before = [t.clone() for t in caches]
        done = _C.ops.paged_attention_and_cache(torch.zeros_like(a["q"]), None, None, None, a["q"], a["k"], a["v"], a["kc"], a["vc"], a["slots"],
                                                0.1, tables, lens, int(lens.max()), cache, k.shape[1], None)
        assert done or all(torch.equal(x, y) for x, y in zip(before, caches))
        return done
    small = lambda: _case(4, 4, 64, [20, 40], torch.float16, "auto", 16)      # noqa: E731
    assert call(small())
    assert call(_case(4, 4, 64, [20] * 128, torch.float16, "auto", 16))
    assert not call(_case(4, 4, 64, [20] * 129, torch.float16, "auto", 16))                # tokens
    assert not call(_case(32, 32, 64, [20] * 33, torch.float16, "auto", 16))               # sequences x heads
    q, k, v, caches, slots, tables, lens = _case(4, 4, 64, [20] * 40, torch.float16, "auto", 16)
    assert not call((q[:39], k, v, caches, slots, tables[:39], lens[:39]))                 # more tokens than sequences, and too many for all
    case = small()
    assert not call(case, slots=case[4].int())
    assert not call(case, k=case[1].transpose(0, 1).contiguous().transpose(0, 1))
    assert not call(case, v=case[2][:, :, :32])
    assert not call(case, kc=torch.cat([case[3][0]] * 2, 1)[:, :4])                        # heads of a wider cache
    assert not call(_case(4, 4, 64, [20, 40], torch.float16, "auto", 4))                   # blocks that the attention refuses


@torch.inference_mode()                                      # (as the workers capture theirs)
def test_layer_in_a_graph():
    """The layer's decode step as it is called, captured and replayed on other inputs, for a split and an unsplit context."""
    from splitwise_amd.model_executor.input_metadata import InputMetadata
    from splitwise_amd.model_executor.layers.attention import Attention
    heads, kv_heads, dim = 8, 8, 128
    for ctx in ([40, 300], [1500, 90, 16]):
        q, k, v, caches, slots, tables, lens = _case(heads, kv_heads, dim, ctx, torch.bfloat16, "auto", 16)
        layer = Attention(heads, dim, dim ** -0.5, kv_heads)
        md = InputMetadata(is_prompt=False, slot_mapping=slots, prompt_lens=None, max_seq_len=None, start_loc=None, max_context_len=max(ctx),
                           context_lens=lens, block_tables=tables, use_cuda_graph=True, kv_cache_dtype="auto")
        call = lambda: layer(q.flatten(1), k.flatten(1), v.flatten(1), *caches, md)      # noqa: E731
        call()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = call()
        for seed in (1, 2, 3):
            case = _case(heads, kv_heads, dim, ctx, torch.bfloat16, "auto", 16, seed=seed)
            for to, new in zip((q, k, v, *caches), (*case[:3], *case[3])):
                to.copy_(new)
            graph.replay()
            got = [out.clone()] + [t.clone() for t in caches]
            for to, new in zip(caches, case[3]):
                to.copy_(new)
            eager = call()
            assert torch.equal(got[0], eager) and all(torch.equal(a, b) for a, b in zip(got[1:], caches))
