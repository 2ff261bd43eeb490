"""A prompt run's cache write and attention in one launch against the two calls one after the other: the same bits in the caches and in
the output, whatever form the launch has, and what it does not take is left to the two calls."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(heads, kv_heads, dim, lens, dtype, cache, block, seed=0, stray=0, shift=0):
    """Tensors of one step: q, k, v as column ranges of one projection, caches, slots (prompts behind one another, `shift` slots on, some
    tokens without a slot, one of them far from its neighbours), starts, lengths; `stray` rows that belong to no sequence."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    rows = sum(lens) + stray
    proj = torch.randn(rows, (heads + 2 * kv_heads) * dim, generator=g, device=DEV).to(dtype)
    q, k, v = (t.view(rows, -1, dim) for t in proj.split([heads * dim, kv_heads * dim, kv_heads * dim], dim=1))
    fp8 = cache != "auto"
    x, ct = (16, torch.uint8) if fp8 else (8, dtype)
    blocks = (rows + shift) // block + 3
    slots = torch.arange(rows, device=DEV) + shift
    slots[rows // 2] = -1
    slots[rows // 3] = (blocks - 1) * block + 1
    caches = [torch.zeros(blocks, kv_heads, dim // x, block, x, dtype=ct, device=DEV),
              torch.zeros(blocks, kv_heads, dim, block, dtype=ct, device=DEV)]
    starts = torch.tensor([sum(lens[:i]) for i in range(len(lens))], dtype=torch.int32, device=DEV)
    return q, k, v, caches, slots, starts, torch.tensor(lens, dtype=torch.int32, device=DEV)


def _both(case, cache, scale, slopes=None, window=None, taken=True):
    from splitwise_amd import _C
    q, k, v, caches, slots, starts, lens = case
    ref, got = torch.zeros_like(q), torch.zeros_like(q)
    ours = [t.clone() for t in caches]
    _C.cache_ops.reshape_and_cache(k, v, *caches, slots, cache)
    _C.ops.prefill_attention(ref, q, k, v, starts, lens, int(lens.max()), scale, slopes, window)
    assert _C.ops.prefill_attention_and_cache(got, q, k, v, starts, lens, int(lens.max()), scale, slopes, window, *ours, slots,
                                              cache) is taken
    if taken:
        assert torch.equal(ref, got)
    for a, b in zip(caches, ours):
        assert torch.equal(a, b) if taken else not b.any()
    assert caches[0].any() and caches[1].any()


@pytest.mark.parametrize("cache", ["auto", "fp8_e5m2"])
@pytest.mark.parametrize("heads,kv_heads,dim", [(12, 12, 64), (16, 2, 128), (6, 3, 80), (4, 4, 96), (5, 1, 112), (8, 8, 256)])
@pytest.mark.parametrize("lens", [[1], [37, 15, 16], [130, 300, 257]])
def test_one_launch_is_the_two(heads, kv_heads, dim, lens, cache):
    for dtype, shift, block in ((torch.bfloat16, 0, 16), (torch.float16, 5, 32)):
        _both(_case(heads, kv_heads, dim, lens, dtype, cache, block, stray=9, shift=shift), cache, dim ** -0.5)


@pytest.mark.parametrize("cache", ["auto", "fp8_e5m2"])
def test_wide_launches(cache):
    # 256 rows a workgroup (8 waves: two tiles of the write): 2048 tokens and more, 384 workgroups and more; an odd number of tiles
    _both(_case(48, 3, 128, [2050], torch.bfloat16, cache, 16, shift=3), cache, 128 ** -0.5)
    # 128 rows: more workgroups than the GPU has places for
    _both(_case(32, 8, 128, [773, 699, 1000], torch.bfloat16, cache, 16), cache, 128 ** -0.5)


def test_slopes_and_window():
    case = _case(8, 4, 64, [70, 200], torch.float16, "auto", 16)
    _both(case, "auto", 0.125, slopes=torch.rand(8, device=DEV), window=None)
    _both(_case(8, 4, 64, [70, 200], torch.float16, "auto", 16), "auto", 0.125, window=33)


def test_what_is_left_to_the_two_calls():
    _both(_case(4, 4, 64, [40], torch.float16, "fp8_e5m2", 8), "fp8_e5m2", 0.125, taken=False)      # blocks of 8 in an fp8 cache
    _both(_case(4, 4, 64, [40], torch.float16, "auto", 4), "auto", 0.125, taken=False)
    from splitwise_amd import _C
    q, k, v, caches, slots, starts, lens = _case(4, 4, 64, [40], torch.float16, "auto", 16)
    call = lambda q, k, v, slots: _C.ops.prefill_attention_and_cache(torch.zeros_like(q), q, k, v, starts, lens, 40, 0.125, None, None,     # noqa: E731
                                                                     *caches, slots, "auto")
    assert not call(q.float(), k.float(), v.float(), slots)
    assert not call(q, k, v, slots.int())
    assert not call(q, k.transpose(0, 1).contiguous().transpose(0, 1), v, slots)
    assert not call(q[:, :, :32], k, v, slots)
    assert not call(q, k, v[:20], slots)
    assert not caches[0].any() and not caches[1].any()


@torch.inference_mode()                                      # (as the workers capture theirs)
def test_layer_in_a_graph():
    """The layer's prompt step as it is called, captured and replayed on other inputs."""
    from splitwise_amd.model_executor.input_metadata import InputMetadata
    from splitwise_amd.model_executor.layers.attention import Attention
    heads, kv_heads, dim, lens = 8, 4, 128, [100, 61]
    q, k, v, caches, slots, starts, n = _case(heads, kv_heads, dim, lens, torch.bfloat16, "auto", 16)
    layer = Attention(heads, dim, dim ** -0.5, kv_heads)
    md = InputMetadata(is_prompt=True, slot_mapping=slots, prompt_lens=n, max_seq_len=max(lens), start_loc=starts, max_context_len=None,
                       context_lens=None, block_tables=None, use_cuda_graph=False, kv_cache_dtype="auto")
    call = lambda: layer(q.flatten(1), k.flatten(1), v.flatten(1), *caches, md)      # noqa: E731
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for seed in (1, 2, 3):
        case = _case(heads, kv_heads, dim, lens, torch.bfloat16, "auto", 16, seed=seed)
        for to, new in zip((q, k, v), case[:3]):
            to.copy_(new)
        for t in caches:
            t.zero_()
        graph.replay()
        got = [out.clone()] + [t.clone() for t in caches]
        for t in caches:
            t.zero_()
        eager = call()
        assert torch.equal(got[0], eager) and all(torch.equal(a, b) for a, b in zip(got[1:], caches))
