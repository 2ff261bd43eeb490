"""The native side of small steps' operators (csrc/host/step_ops.cpp) against the Python functions it stands in front of: the same
bits for every form it takes, and whatever it does not take is left to Python, refusals included."""
import ctypes
import dataclasses
import inspect

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _gen():
    return torch.Generator(device="cuda").manual_seed(3)


def _randn(*shape, dtype=torch.float32):
    return torch.randn(*shape, device="cuda", generator=_gen()).to(dtype)


def _batch(lens, ctx):
    from splitwise_amd.model_executor.input_metadata import RaggedBatch
    start = [0]
    for n in lens:
        start.append(start[-1] + n)
    i32 = dict(dtype=torch.int32, device="cuda")
    pages = max(-(-(c + n) // 16) for c, n in zip(ctx, lens))
    tables = torch.arange(len(lens) * pages, **i32).view(len(lens), pages)
    return RaggedBatch(q_start=torch.tensor(start, **i32), ctx_len=torch.tensor(ctx, **i32),
                       token_seq=torch.tensor([i for i, n in enumerate(lens) for _ in range(n)], **i32),
                       state_slot=torch.arange(len(lens), **i32), block_tables=tables, num_seqs=len(lens),
                       max_query_len=max(lens), max_pages_used=pages, max_page_id=len(lens) * pages - 1,
                       max_state_slot=len(lens) - 1)


STEPS = {"decode": ([1, 1, 1], [5, 40, 17]), "portions": ([40, 3, 33], [0, 9, 16])}
H, KVH, D = 4, 2, 64


def _call(name, step):
    """-> (module, function name, arguments by position, keywords, tensors that the call writes)"""
    from splitwise_amd import _C, _C_mixers as m
    lens, ctx = STEPS[step]
    b, rows = _batch(lens, ctx), sum(lens)
    n = H * D
    proj = _randn(rows, 4 * n + 8, dtype=BF)
    q, k, v, gate = (proj[:, i * n:(i + 1) * n] for i in range(4))
    o = torch.zeros(rows, n, device="cuda")
    state = _randn(len(lens), H, D, D)
    if name == "causal_conv":
        conv_state = _randn(len(lens), 3, n)
        out = torch.zeros(rows, n, device="cuda")
        return m, name, (out, q, _randn(n, 4), conv_state, b), dict(silu=True, residual=False), [out, conv_state]
    if name == "gated_delta":
        qkv = _randn(rows, 2 * KVH * D + n)
        return m, name, (o, qkv, proj[:, 4 * n:4 * n + H], proj[:, 4 * n + H:], _randn(H), _randn(H), state, b, H, KVH, D, D), {}, \
            [o, state]
    if name == "head_norm_gate":
        out = torch.zeros(rows, n, device="cuda", dtype=BF)
        return m, name, (out, _randn(rows, n), gate, _randn(D), False, 1e-6, H, D), dict(gate_silu=True), [out]
    if name == "gla":
        return m, name, (o, q, k, v, _randn(rows, n, dtype=BF), _randn(n), 16.0, D ** -0.5, state, b, H, D, D), {}, [o, state]
    if name == "lightning":
        return m, name, (o, q, k, v, torch.rand(H, device="cuda"), state, b, H, D, D), {}, [o, state]
    if name == "retention":
        return m, name, (o, _randn(rows, n), _randn(rows, n), v, torch.rand(H, device="cuda"), state, b, H, D, D), {}, [o, state]
    if name == "expert_ffn":
        x, up, down = _randn(rows, 64, dtype=BF), _randn(4, 96, 64, dtype=BF), _randn(4, 64, 48, dtype=BF)
        order, start = m.group_pairs((torch.arange(rows, device="cuda", dtype=torch.int32) % 4).view(rows, 1), 4)
        out = torch.zeros(rows, 64, device="cuda")
        return m, name, (out, x, up, down, order, start, 1, 1.0), dict(pair_weight=torch.rand(rows, 1, device="cuda"),
                                                                    glu=(1.0, float("inf"), 0.0)), [out]
    if name == "capped_attention":
        caches = [_randn(b.max_page_id + 1, 16, KVH * D, dtype=BF) for _ in range(2)]
        out = torch.zeros(rows, n, device="cuda", dtype=BF)
        return m, name, (out, _randn(rows, n), *caches, gate, b, H, KVH, D, D, D ** -0.5, 30.0), \
            dict(sink=_randn(H) if step == "decode" else True), [out]
    kc = _randn(8 * len(lens), KVH, D // 8, 16, 8, dtype=BF)
    vc = _randn(8 * len(lens), KVH, D, 16, dtype=BF)
    q3, k3, v3 = q.view(rows, H, D), k[:, :KVH * D].view(rows, KVH, D), v[:, :KVH * D].view(rows, KVH, D)
    if name == "reshape_and_cache":
        return _C, name, (k3, v3, kc, vc, torch.arange(rows, device="cuda"), "auto"), {}, [kc, vc]
    if name == "paged_attention_v1":
        out = torch.zeros(len(lens), H, D, device="cuda", dtype=BF)
        return _C, name, (out, q3[:len(lens)], kc, vc, KVH, D ** -0.5, b.block_tables, b.ctx_len + 1, 16, max(ctx) + 1, None,
                          "auto"), {}, [out]
    if name.startswith("paged_attention_and_cache"):
        few, longest = len(lens), max(ctx) + 1 + (600 if name.endswith("split") else 0)      # (two parts)
        out, temporaries = torch.zeros(few, H, D, device="cuda", dtype=BF), [None] * 3
        if name.endswith("split"):
            sums = torch.zeros(few, H, 2, device="cuda")
            temporaries = [sums, torch.zeros_like(sums), torch.zeros(few, H, 2, D, device="cuda", dtype=BF)]
        return _C, "paged_attention_and_cache", (out, *temporaries, q3[:few], k3[:few], v3[:few], kc, vc,
                                                 (b.ctx_len + b.block_tables[:, 0] * 16).long(), D ** -0.5, b.block_tables, b.ctx_len + 1, longest,
                                                 "auto", KVH, None), {}, [out, kc, vc]
    out = torch.zeros(rows, H, D, device="cuda", dtype=BF)
    if name == "prefill_attention_and_cache":
        return _C, name, (out, q3, k3, v3, b.q_start[:-1], torch.tensor(lens, dtype=torch.int32, device="cuda"), max(lens), D ** -0.5,
                          None, 8, kc, vc, torch.arange(rows, device="cuda"), "auto"), {}, [out, kc, vc]
    return _C, name, (out, q3, k3, v3, b.q_start[:-1], torch.tensor(lens, dtype=torch.int32, device="cuda"), max(lens), D ** -0.5,
                      None, 8), {}, [out]


class _Seen:
    """The extension, with what it answered."""
    def __init__(self, inner):
        self.inner, self.answers = inner, []

    def __getattr__(self, name):
        def run(*args):
            self.answers.append(getattr(self.inner, name)(*args))
            return self.answers[-1]
        return run


class _None:
    def __getattr__(self, name):
        return lambda *args: None


NAMES = ["causal_conv", "gated_delta", "head_norm_gate", "gla", "lightning", "retention", "expert_ffn", "capped_attention",
         "reshape_and_cache", "paged_attention_v1", "prefill_attention", "prefill_attention_and_cache", "paged_attention_and_cache",
         "paged_attention_and_cache split"]


@pytest.mark.parametrize("step", list(STEPS))
@pytest.mark.parametrize("name", NAMES)
def test_native_call_is_the_python_call(name, step, monkeypatch):
    module, name, args, kw, written = _call(name, step)
    module.load_library()
    before = [t.clone() for t in written]
    seen = _Seen(module._native)
    monkeypatch.setattr(module, "_native", seen)
    getattr(module, name)(*args, **kw)
    assert seen.answers == [0]
    native = [t.clone() for t in written]
    for t, old in zip(written, before):
        t.copy_(old)
    monkeypatch.setattr(module, "_native", _None())
    getattr(module, name)(*args, **kw)
    for a, b, old in zip(native, written, before):
        assert torch.equal(a, b) and not torch.equal(a, old)


def _spoil(t):
    """Forms of a tensor that an operator may not be given, or only in other code."""
    yield t.cpu()
    yield t.double() if t.is_floating_point() else t.long()
    if t.dim() > 1 and t.shape[0] > 1:
        yield t[:-1]
    yield torch.stack([t, t], -1)[..., 0]


class _Recorder:
    """Stands for the library in Python's part of a call: writes down what would be launched and launches nothing."""
    def __init__(self, lib, signatures):
        self.lib, self.signatures, self.calls = lib, signatures, []

    def __getattr__(self, name):
        if name not in self.signatures or name.endswith("_floats"):
            return getattr(self.lib, name)

        def entry(*args):
            self.calls.append((name,) + args)
            return 0
        return entry


@pytest.mark.parametrize("name", NAMES)
def test_nothing_is_taken_that_python_refuses(name, monkeypatch):
    """Every tensor of a call (and of the step's layout) spoilt in turn, every number changed: what the extension takes, Python
    takes, and both ask the library for the same.  Nothing is launched: the extension is bound to callbacks here."""
    module, name, args, kw, _ = _call(name, "decode")
    lib = module.load_library()
    native, recorder = module._native, _Recorder(lib, module._SIGNATURES)
    asked, real, stubs = [], {}, {}
    for entry, argtypes in module._SIGNATURES.items():
        if entry.endswith("_floats"):
            continue
        kind = ctypes.CFUNCTYPE(ctypes.c_int, *argtypes)
        stubs[entry] = kind(lambda *a, entry=entry: asked.append((entry,) + a) or 0)
        real[entry] = ctypes.cast(getattr(lib, entry), ctypes.c_void_p).value

    def plain(calls, known):
        out = []
        for entry, *a in calls:
            kinds = module._SIGNATURES[entry]
            out.append((entry,) + tuple(
                (v or 0) if k is ctypes.c_void_p and (v or 0) in known else "scratch" if k is ctypes.c_void_p
                else ctypes.c_float(v).value if k is ctypes.c_float else v for k, v in zip(kinds, a)))
        return out

    names = list(inspect.signature(getattr(module, name)).parameters)
    full = {**dict(zip(names, args)), **kw}
    forms = [full]
    for key, value in full.items():
        if isinstance(value, torch.Tensor):
            forms += [{**full, key: x} for x in _spoil(value)]
        elif dataclasses.is_dataclass(value):
            for f in ("q_start", "ctx_len", "token_seq", "state_slot", "block_tables"):
                forms += [{**full, key: dataclasses.replace(value, **{f: x})} for x in _spoil(getattr(value, f))]
            forms += [{**full, key: dataclasses.replace(value, **{f: 9999})} for f in ("max_state_slot", "max_page_id", "max_pages_used")]
            forms += [{**full, key: dataclasses.replace(value, max_query_len=0)}]
        elif isinstance(value, (int, float)) and not isinstance(value, bool):
            forms += [{**full, key: x} for x in (value + 1, -value, float(value), 1 << 40)]
    stream = torch.cuda.current_stream().cuda_stream
    taken = refused = 0
    try:
        native.bind({e: ctypes.cast(f, ctypes.c_void_p).value for e, f in stubs.items()})
        monkeypatch.setattr(module, "load_library", lambda: recorder)
        for form in forms:
            held = [t for v in form.values() for t in (vars(v).values() if dataclasses.is_dataclass(v) else (v,))
                    if isinstance(t, torch.Tensor)]
            known = {0, stream} | {t.data_ptr() for t in held}
            recorder.calls.clear()
            asked.clear()
            monkeypatch.setattr(module, "_native", _None())
            try:
                getattr(module, name)(**form)
                alone = plain(recorder.calls, known)
            except Exception:                                         # noqa: BLE001
                alone = None
            monkeypatch.setattr(module, "_native", native)
            recorder.calls.clear()
            try:
                getattr(module, name)(**form)
            except Exception:                                         # noqa: BLE001
                assert alone is None
            if asked:
                taken += 1
                assert not recorder.calls and plain(asked, known) == alone
            elif not alone:                   # (an exception, or the answer that the call is for other functions)
                refused += 1
    finally:
        native.bind(real)
    assert taken >= 2 and refused >= 2


@pytest.mark.parametrize("rows,top,experts", [(1, 1, 1), (5, 2, 4), (300, 3, 7)])
def test_group_pairs(rows, top, experts, monkeypatch):
    from splitwise_amd import _C_mixers as m
    chosen = torch.randint(0, experts, (rows, top), device="cuda", dtype=torch.int32, generator=_gen())
    m.load_library()
    seen = _Seen(m._native)
    monkeypatch.setattr(m, "_native", seen)
    native = m.group_pairs(chosen, experts)
    assert type(seen.answers[0]) is tuple
    monkeypatch.setattr(m, "_native", _None())
    alone = m.group_pairs(chosen, experts)
    assert torch.equal(native[1], alone[1]) and native[0].dtype == torch.int32
    for e in range(experts):                                          # the order inside an expert is free
        lo, hi = int(alone[1][e]), int(alone[1][e + 1])
        assert torch.equal(native[0][lo:hi].sort().values, alone[0][lo:hi].sort().values)
