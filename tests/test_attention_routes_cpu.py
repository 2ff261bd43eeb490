"""Which launches a step of the Llama path's attention module asks for: the operators are stood in for by recorders."""
from types import SimpleNamespace

import pytest
import torch

from splitwise_amd import _C
from splitwise_amd.model_executor.input_metadata import InputMetadata
from splitwise_amd.model_executor.layers.attention import Attention


class _Calls(list):
    def __init__(self, monkeypatch):
        super().__init__()
        def entry(name, answer=None):
            return lambda *args: (self.append(name), answer)[1]
        ops = {n: entry(n) for n in ("paged_attention_v1", "paged_attention_v2", "prefill_attention", "rotary_embedding_and_cache")}
        ops |= {n: entry(n, True) for n in ("prefill_attention_and_cache", "paged_attention_and_cache")}
        monkeypatch.setattr(_C, "ops", SimpleNamespace(**ops))
        monkeypatch.setattr(_C, "cache_ops", SimpleNamespace(reshape_and_cache=entry("reshape_and_cache")))


def _meta(*shape, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=dtype, device="meta")


def _step(calls, heads, kv_heads, dim, rows, md, block=16, **kw):
    calls.clear()
    Attention(heads, dim, 1.0, kv_heads)(_meta(rows, heads * dim), _meta(rows, kv_heads * dim), _meta(rows, kv_heads * dim),
                                         _meta(9, kv_heads, dim // 8, block, 8), _meta(9, kv_heads, dim, block), md, **kw)
    return list(calls)


def _prompt(lens, cache):
    return InputMetadata(is_prompt=True, slot_mapping=_meta(sum(lens)), prompt_lens=_meta(len(lens)), max_seq_len=max(lens),
                         start_loc=_meta(len(lens)), max_context_len=None, context_lens=None, block_tables=None, use_cuda_graph=False,
                         kv_cache_dtype=cache)


ONE, TWO = ["prefill_attention_and_cache"], ["reshape_and_cache", "prefill_attention"]


@pytest.mark.parametrize("heads,kv_heads,dim,lens,auto,fp8", [
    (32, 32, 128, [17], ONE, ONE), (32, 32, 128, [773] * 3, ONE, TWO), (32, 32, 128, [1000], ONE, ONE), (32, 32, 128, [2000] * 2, ONE, TWO),
    (32, 32, 128, [2049] * 8, TWO, TWO), (32, 32, 128, [773] * 8, TWO, TWO), (32, 32, 128, [120] * 32, ONE, TWO), (32, 32, 128, [4100], TWO, TWO),
    (32, 32, 128, [33] * 64, TWO, TWO), (32, 32, 128, [33] * 8, ONE, TWO), (64, 8, 128, [300] * 2, ONE, ONE), (64, 8, 128, [2049] * 8, TWO, TWO),
    (16, 16, 256, [120] * 32, ONE, TWO), (12, 12, 64, [700] * 4, ONE, ONE), (16, 2, 128, [33] * 64, ONE, ONE), (16, 2, 128, [4095], ONE, ONE)])
def test_prompt_steps(heads, kv_heads, dim, lens, auto, fp8, monkeypatch):
    calls = _Calls(monkeypatch)
    assert _step(calls, heads, kv_heads, dim, sum(lens), _prompt(lens, "auto")) == auto
    assert _step(calls, heads, kv_heads, dim, sum(lens), _prompt(lens, "fp8_e5m2")) == fp8


@pytest.mark.parametrize("block,auto,fp8", [(8, ONE, TWO), (16, ONE, ONE), (32, ONE, ONE)])
def test_prompt_steps_do_not_ask_for_a_launch_that_refuses_their_blocks(block, auto, fp8, monkeypatch):
    calls = _Calls(monkeypatch)
    assert _step(calls, 12, 12, 64, 40, _prompt([40], "auto"), block) == auto
    assert _step(calls, 12, 12, 64, 40, _prompt([40], "fp8_e5m2"), block) == fp8


def _decode(seqs, ctx, cache):
    return InputMetadata(is_prompt=False, slot_mapping=_meta(seqs), prompt_lens=None, max_seq_len=None, start_loc=None, max_context_len=ctx,
                         context_lens=_meta(seqs), block_tables=_meta(seqs, 9), use_cuda_graph=False, kv_cache_dtype=cache)


BESIDE, SPLIT, UNSPLIT = ["paged_attention_and_cache"], ["reshape_and_cache", "paged_attention_v2"], ["reshape_and_cache", "paged_attention_v1"]


@pytest.mark.parametrize("heads,kv_heads,dim,seqs,ctx,auto,fp8", [
    (32, 32, 128, 2, 700, BESIDE, BESIDE), (32, 32, 128, 32, 700, BESIDE, UNSPLIT), (32, 32, 128, 16, 700, BESIDE, BESIDE),
    (32, 32, 128, 33, 700, UNSPLIT, UNSPLIT), (32, 32, 128, 2, 4096, BESIDE, BESIDE), (32, 32, 128, 3, 4096, SPLIT, SPLIT),
    (32, 32, 128, 8, 15000, SPLIT, SPLIT), (64, 8, 128, 64, 2011, BESIDE, BESIDE), (64, 8, 128, 65, 2011, BESIDE, UNSPLIT), (64, 8, 128, 65, 2049, UNSPLIT, UNSPLIT), (64, 8, 128, 128, 2048, BESIDE, UNSPLIT),
    (64, 8, 128, 12, 2875, BESIDE, BESIDE), (64, 8, 128, 12, 7000, SPLIT, SPLIT), (64, 8, 128, 2, 2875, BESIDE, BESIDE), (16, 2, 128, 24, 3000, BESIDE, BESIDE),
    (16, 2, 128, 24, 28000, SPLIT, SPLIT), (32, 32, 128, 1, 16384, BESIDE, BESIDE), (32, 32, 128, 1, 16385, SPLIT, SPLIT), (12, 12, 64, 128, 300, UNSPLIT, UNSPLIT), (4, 4, 64, 128, 300, BESIDE, BESIDE),
    (4, 4, 64, 129, 300, UNSPLIT, UNSPLIT)])
def test_decode_steps(heads, kv_heads, dim, seqs, ctx, auto, fp8, monkeypatch):
    calls = _Calls(monkeypatch)
    assert _step(calls, heads, kv_heads, dim, seqs, _decode(seqs, ctx, "auto")) == auto
    assert _step(calls, heads, kv_heads, dim, seqs, _decode(seqs, ctx, "fp8_e5m2")) == fp8


def test_decode_steps_that_rotate(monkeypatch):
    """A model that hands its rotary module over (the Llama models): rotation and cache write in one launch, the attention in the next."""
    calls = _Calls(monkeypatch)
    rotary = SimpleNamespace(fusable_with_cache_write=lambda dtype: True, cos_sin_cache=None, is_neox_style=True)
    kw = dict(rotary=rotary, positions=_meta(2))
    assert _step(calls, 32, 32, 128, 2, _decode(2, 700, "auto"), **kw) == ["rotary_embedding_and_cache", "paged_attention_v1"]
    assert _step(calls, 32, 32, 128, 3, _decode(3, 4096, "auto"), **kw) == ["rotary_embedding_and_cache", "paged_attention_v2"]


class _Held(torch.Tensor):
    """A CPU tensor that says that it is on the GPU, for the operators' checks in front of the library."""
    is_cuda = property(lambda self: True)


@pytest.mark.parametrize("dtype,taken", [(torch.float32, True), (torch.bfloat16, False), (torch.float64, False)])
def test_slopes_of_another_type_are_left_to_the_two_calls(dtype, taken, monkeypatch):
    """The kernel reads the slopes as fp32; paged attention alone refuses others, and so the one launch may not take them."""
    from contextlib import nullcontext
    calls = []
    monkeypatch.setattr(_C, "load_library", lambda: SimpleNamespace(sw_paged_attention_and_cache=lambda *args: calls.append(args) or 0))
    monkeypatch.setattr(_C, "_on_device_of", lambda t: nullcontext())
    monkeypatch.setattr(_C, "_stream", lambda t: None)
    held = lambda *shape, dtype=torch.bfloat16: torch.zeros(shape, dtype=dtype).as_subclass(_Held)      # noqa: E731
    q, k, v, slopes = held(2, 4, 64), held(2, 4, 64), held(2, 4, 64), held(4, dtype=dtype)
    kc, vc, tables, lens = held(5, 4, 8, 16, 8), held(5, 4, 64, 16), held(2, 2, dtype=torch.int32), held(2, dtype=torch.int32)
    assert _C.paged_attention_and_cache(held(2, 4, 64), None, None, None, q, k, v, kc, vc, held(2, dtype=torch.int64), 0.125, tables, lens, 20,
                                        "auto", 4, slopes) is taken
    assert len(calls) == taken
    if not taken:
        with pytest.raises(RuntimeError, match="alibi_slopes must be float32"):
            _C.paged_attention_v1(held(2, 4, 64), q, kc, vc, 4, 0.125, tables, lens, 16, 20, slopes, "auto")
