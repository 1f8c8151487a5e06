"""The native call path of the factories (csrc/h3_call.cpp): what it takes and
what it leaves to the checked Python path."""
from __future__ import annotations

import contextlib
import ctypes
import importlib
import types

import pytest
import torch

BF = torch.bfloat16
EPS = 1e-6


@pytest.fixture()
def native():
    return importlib.import_module("minimaxh3_on_k100-ai_amd._h3call")


def test_plan_arguments_are_checked(native):
    for args in [(0, "", (), None), (0, "b3", (1,), None), (0, "b3", [0], None), (0, "b3", (0,), (1, 0, 5)),
                 (0, "b3", (0,), (0, 3, 5)), (0, "b3" * 17, (0,), None), (0, "t2" * 11, tuple(range(11)), None)]:
        with pytest.raises((ValueError, TypeError)):
            native.plan(*args)
    with pytest.raises(ValueError):
        native.call(object(), 1)


def test_other_than_plain_cuda_tensors_are_not_taken(native):
    """No address is called: wrong counts, types and devices return False
    before the launch."""
    plan = native.plan(0, "b3b1s0", (0, 1, 2), None)
    x, w = torch.zeros(1, 2, 8, dtype=BF), torch.zeros(8, dtype=BF)
    for args in [(x, w), (x, w, 1.0, 2), (x, w, 1.0), (x, 3, 1.0), (None, w, 1.0), (x, w, "a"),
                 (torch.nn.Buffer(x), w, 1.0)]:
        assert native.call(plan, *args) is False


@pytest.mark.parametrize("case", ["missing", "does not load", "another torch"])
def test_factories_work_without_the_native_module(pkg, monkeypatch, case):
    """With the library there and the native module not usable, factories are
    made as before it existed, with one warning, and call through ctypes."""
    name = "minimaxh3_on_k100-ai_amd._h3call"
    real = importlib.import_module

    def no_module(module, *a):
        if module != name:
            return real(module, *a)
        if case == "another torch":
            return types.SimpleNamespace(torch_version="0.0.1", plan=None, call=None)
        raise ImportError("undefined symbol" if case == "does not load" else f"No module named {name!r}")

    called = []
    monkeypatch.setattr(pkg._lib.importlib, "import_module", no_module)
    monkeypatch.setattr(pkg._lib, "_fast_calls", {})
    monkeypatch.setattr(pkg._lib, "LIBRARY_PATH", pkg._lib.Path(__file__))  # there
    monkeypatch.setattr(pkg._lib, "launch", lambda name, *a: called.append(name))
    monkeypatch.setattr(pkg._lib, "check_cuda", lambda *t: torch.device("cuda:0"))
    pkg._lib._call_module.cache_clear()
    try:
        with pytest.warns(RuntimeWarning, match="_h3call") as warned:
            swiglu, _ = pkg.make_swiglu(), pkg.make_attention()
        assert len(warned) == 1
        x = torch.zeros(1, 2, 8, dtype=BF)
        swiglu(x, x, x)
    finally:
        pkg._lib._call_module.cache_clear()
    assert called == ["launch_h3_swiglu_exact"]


# Every factory with a native call, and tensors of its arguments' ranks.
CALLS = [
    ("make_swiglu", "x3 x3 x3"), ("make_rms", "x3 x1 e x3", dict(width=None)),
    ("make_rms_modulate", "x3 x1 e x3 x3 x3"),
    ("make_gated_residual", "x3 x3 x3 x3"), ("make_gated_residual_rms_modulate", "x3 x3 x3 x1 e x3 x3 x3 x3"),
    ("make_rms_modulate_indexed", "x3 x1 e x2 x2 i x3", dict(check_indices=False)),
    ("make_gated_residual_rms_modulate_indexed", "x3 x2 x3 x1 e x2 x2 i x3 x3", dict(check_indices=False)),
    ("make_gated_residual_indexed", "x3 x2 x3 i x3", dict(check_indices=False)), ("make_rope", "x3 x2 x2 x3"),
    ("make_qk_norm_rope", "x4 x1 e x2 x2 x4"), ("make_qkv_norm_rope_pack", "x4 x4 x4 x1 x1 e c p x4 x4 x4"),
    ("make_qkv_norm_rope_pack_fp8", "x4 x4 x4 x1 x1 e c p q q x4 f f"),
    ("make_qkv_norm_rope_pack_fp8_vamax", "x4 x4 x4 x1 x1 e c p q q x4 f f a"),
    ("make_qkv_norm_rope_pack_fp8x2_vamax", "x4 x4 x4 x1 x1 e c p q q q q x4 f f a"),
    ("make_qk_norm_rope_interleaved", "x4 x1 e x2 x2 x4"),
    ("make_qk_norm_rope_interleaved_qk", "x4 x4 x1 x1 e x2 x2 x4 x4"), ("make_rope_cache", "d2 f x2 x2"),
    ("make_attention", "x4 x4 x4 e x4"), ("make_attention", "x4 x4 x4 e x4", dict(split_last_round=False)),
    ("make_attention_fp8", "q q q f f f e x4"), ("make_attention_fp8x2", "q q q q q f f f e x4"),
    ("make_attention_fp8pv", "x4 x4 q f e x4"), ("quantize_fp8_per_head", "x4 k q f a"),
]


@pytest.mark.parametrize("status", [1, 98, 700])
@pytest.mark.parametrize("factory,kinds,options", [(c + ({},))[:3] for c in CALLS])
def test_a_launch_that_returns_an_error_is_not_repeated(pkg, monkeypatch, factory, kinds, options, status):
    """A launcher's status can be an error an earlier call left, with its kernel
    queued all the same: it is raised, and the entry point is not called again."""
    shape = {"1": (128,), "2": (1, 128), "3": (1, 1, 128), "4": (1, 1, 1, 128)}
    make = {"x": lambda k: torch.zeros(shape[k[1]], dtype=BF), "e": lambda k: EPS,
            "i": lambda k: torch.zeros(1, 1).long(),
            "c": lambda k: torch.zeros(1, 96, dtype=BF), "p": lambda k: torch.zeros(1).long(),
            "q": lambda k: torch.zeros(1, 1, 1, 128, dtype=torch.float8_e4m3fn), "f": lambda k: torch.zeros(1),
            "a": lambda k: torch.zeros(1, 64), "d": lambda k: torch.zeros(1, 3).double(), "k": lambda k: False}
    args = [make[k[0]](k) for k in kinds.split()]
    native, direct = [], []
    monkeypatch.setattr(pkg._lib, "fast", lambda name, *a, **kw: lambda *args: native.append(name) or status)
    monkeypatch.setattr(pkg._lib, "call", lambda name, *a: direct.append(name) or 0)
    monkeypatch.setattr(pkg._lib, "check_cuda", lambda *t: torch.device("cuda:0"))
    monkeypatch.setattr(pkg._lib, "planned_workspace", lambda *sizes: 0)
    attention = importlib.import_module("minimaxh3_on_k100-ai_amd.h3_attention")
    pointwise = importlib.import_module("minimaxh3_on_k100-ai_amd.h3_pointwise")
    attention._slots_fast.cache_clear()
    monkeypatch.setattr(pointwise, "_positions", lambda p, device: p)
    if factory == "make_qkv_norm_rope_pack":  # compares the device of its positions itself
        monkeypatch.setattr(pkg._lib, "check_cuda", lambda *t: t[0].device)
    if factory == "make_attention":
        monkeypatch.setattr(torch, "empty", lambda *a, device=None, **kw: torch.zeros(*a, **kw))
    fn = getattr(pkg, factory) if factory.startswith("quantize") else getattr(pkg, factory)(**options)
    try:
        with pytest.raises(pkg._lib.LaunchError) as e:
            fn(*args)
    finally:
        attention._slots_fast.cache_clear()
    assert e.value.status == status and len(native) == 1 and direct == []


def test_python_path_launches_what_the_native_call_left(pkg, monkeypatch):
    called = []
    monkeypatch.setattr(pkg._lib, "call", lambda name, *a: called.append(name) or 0)
    monkeypatch.setattr(torch.cuda, "device", lambda d: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d: types.SimpleNamespace(cuda_stream=0))
    pkg._lib.launch_after(False, "launch_h3_swiglu_exact", torch.device("cuda:0"))
    assert called == ["launch_h3_swiglu_exact"]


@pytest.mark.gpu
def test_native_call_returns_the_status_of_its_one_launch(pkg, native, device):
    statuses = [0, 1, 98, 700]
    calls = []
    signature = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, *[pkg._lib.NineToothedTensor] * 3)
    launcher = signature(lambda *a: calls.append(a) or statuses[len(calls) - 1])
    plan = native.plan(ctypes.cast(launcher, ctypes.c_void_p).value, "b3b3b3", (0, 1, 2), None)
    x = torch.zeros(1, 2, 8, dtype=BF, device=device)
    assert [native.call(plan, x, x, x) for _ in statuses] == [True, 1, 98, 700]
    assert native.call(plan, x, x, x.float()) is False and len(calls) == len(statuses)


@pytest.mark.gpu
def test_an_error_left_by_another_call_is_raised_after_one_launch(pkg, device):
    """In place, so that a second launch would show: the gated residual reports
    the thread's earlier error (a device that does not exist) and ran once."""
    hip = ctypes.CDLL("libamdhip64.so")
    x = torch.ones(1, 64, 1024, dtype=BF, device=device)
    kernel = pkg.make_gated_residual()
    kernel(x.clone(), x, x, x.clone())  # bound
    torch.cuda.synchronize()
    one = torch.ones_like(x)
    torch.cuda.synchronize()
    assert hip.hipSetDevice(4096) != 0
    with pytest.raises(pkg._lib.LaunchError):
        kernel(x, one, one, x)
    torch.cuda.synchronize()
    assert torch.equal(x, one * 2)
    kernel(x, one, one, x)
    torch.cuda.synchronize()
    assert torch.equal(x, one * 3)


@pytest.mark.gpu
def test_plain_calls_skip_the_python_path(pkg, device, monkeypatch):
    """With the ctypes launch disabled: plain calls of every kind of argument
    (table, index with and without its batch dim, workspace, fixed size) still
    launch, and calls that need a conversion or a check reach it."""
    def no_launch(*args):
        raise AssertionError("python path")

    gen = torch.Generator("cpu").manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=gen).to(BF).to(device)
    x, y, w, out = r(1, 9, 520), r(1, 9, 520), r(520), torch.empty(1, 9, 520, dtype=BF, device=device)
    tab, index = r(3, 520), torch.tensor([0, 0, 1, 1, 1, 2, 2, 2, 2], device=device)
    q, k, v = (r(7, 1, 2, 128) for _ in range(3))
    outs = [torch.empty_like(q) for _ in range(3)]
    cache, w128, pos = r(7, 96), r(128), torch.arange(7, device=device)
    att = [r(1, 2, 300, 128) for _ in range(3)] + [0.1, torch.empty(1, 2, 300, 128, dtype=BF, device=device)]
    attention = pkg.make_attention()
    attention(*att)  # plans the shape
    want_att = att[4].clone()
    swiglu, rms = pkg.make_swiglu(), pkg.make_rms(width=520)
    mod, pack = pkg.make_rms_modulate_indexed(check_indices=False), pkg.make_qkv_norm_rope_pack()
    mod(x, w, EPS, tab, tab, index, out)
    want_mod = out.clone()
    pack(q, k, v, w128, w128, EPS, cache, pos.int(), *outs)  # int32 positions: converted in Python
    want_pack = [t.clone() for t in outs]
    monkeypatch.setattr(pkg._lib, "launch", no_launch)
    swiglu(x, y, out)
    rms(x, w, 0, out)
    for ix in (index, index.view(1, 9)):
        out.zero_()
        mod(x, w, EPS, tab, tab, ix, out)
        assert torch.equal(out, want_mod)
    for t in outs:
        t.zero_()
    pack(q, k, v, w128, w128, EPS, cache, pos, *outs)
    assert all(torch.equal(a, b) for a, b in zip(outs, want_pack))
    att[4].zero_()
    attention(*att)
    assert torch.equal(att[4], want_att)
    for call in [lambda: pack(q, k, v, w128, w128, EPS, cache, pos.int(), *outs),
                 lambda: rms(x, w, torch.tensor(EPS), out),
                 lambda: swiglu(torch.nn.Parameter(x).view(1, 9, 520).as_subclass(_Sub), y, out)]:
        with pytest.raises(AssertionError, match="python path"):
            call()
    for call in [lambda: rms(r(1, 9, 128), r(128), EPS, r(1, 9, 128)), lambda: swiglu(x.float(), y, out),
                 lambda: swiglu(x[0], y, out), lambda: swiglu(x.cpu(), y, out),
                 lambda: attention(att[0][..., :64], *att[1:])]:
        with pytest.raises(ValueError):
            call()


@pytest.mark.gpu
def test_lo_code_strides_are_still_compared(pkg, device):
    """The two-term pack refuses lo codes whose strides differ from the hi
    codes', also where they only differ in a dim of size 1."""
    r = lambda *s: torch.randn(*s, device=device).to(BF)
    q, k, v = (r(5, 1, 2, 128) for _ in range(3))
    codes = [torch.empty(5, 1, 2, 128, dtype=torch.float8_e4m3fn, device=device) for _ in range(4)]
    codes[1] = codes[1].as_strided((5, 1, 2, 128), (256, 512, 128, 1))
    d, amax = torch.empty(2, device=device), torch.empty(2, 64, device=device)
    with pytest.raises(ValueError, match="strides"):
        pkg.make_qkv_norm_rope_pack_fp8x2_vamax()(q, k, v, r(128), r(128), EPS, r(5, 96),
                                                  torch.arange(5, device=device), *codes, torch.empty_like(v), d,
                                                  d.clone(), amax)


class _Sub(torch.Tensor):
    pass


@pytest.mark.gpu
def test_calls_use_the_current_stream(pkg, device):
    """A call under a side stream is captured there."""
    x = torch.randn(1, 64, 1024, device=device).to(BF)
    out = torch.zeros_like(x)
    swiglu = pkg.make_swiglu()
    swiglu(x, x, out)
    torch.cuda.synchronize()
    want = out.clone()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            swiglu(x, x, out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
