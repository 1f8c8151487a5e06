"""launch_h3_attention_planned: the plan's 64- and 128-query units with the keys
split over a workgroup's waves (attention16_short_kernel), against the float64
oracle, and the entry point's argument checks."""
from __future__ import annotations

import ctypes

import pytest
import torch

from conftest import attention_error
from test_attention_gpu import MAX_ABS, REL_RMS, _bhsd, _dominant_keys, gpu_reference_fp32

BF = torch.bfloat16
_BUF = ctypes.create_string_buffer(1 << 16)


@pytest.mark.parametrize("shapes", [
    ([1, 2, 8, 64], [1, 2, 8, 64], [1, 2, 8, 64], [0]),    # head dim
    ([1, 2, 8, 72], [1, 2, 8, 128], [1, 2, 8, 72], [0]),   # k and q differ
    ([1, 2, 8, 128], [1, 2, 0, 128], [1, 2, 8, 128], [0]),  # no keys
    ([1, 2, 8, 128], [1, 2, 8, 128], [1, 2, 9, 128], [0]),  # out length
])
def test_planned_entry_rejects_bad_shapes(shapes):
    import importlib
    L = importlib.import_module("minimaxh3_on_k100-ai_amd")._lib

    def t(shape):
        strides = [1] * len(shape)
        for i in range(len(shape) - 2, -1, -1):
            strides[i] = strides[i + 1] * max(shape[i + 1], 1)
        return L.raw_tensor((ctypes.addressof(_BUF) + 255) & ~255, shape, strides)

    q, k, o, ws = (t(s) for s in shapes)
    assert L.call("launch_h3_attention_planned", 0, q, k, k, L.scalar(0.1), o, ws) == L.HIP_ERROR_INVALID_VALUE
    assert L.attention_planned_workspace_bytes(0, 1, 5, 5, 128) == 0
    assert L.attention_planned_workspace_bytes(1, 1, 5, 5, 64) == 0


def _kernels(fn):
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    return [e.name for e in prof.events() if "attention" in e.name]


@pytest.mark.gpu
@pytest.mark.parametrize("D", [128, 72])
@pytest.mark.parametrize("B,H,Sq,Sk,scale,QW", [
    (1, 3, 1, 129, 0.1, 2),        # one query; one key past a tile: waves without keys in the second
    (2, 3, 63, 255, 0.1, 2),       # the last query of a unit and the last key of a tile missing
    (1, 2, 64, 128, -0.1, 2),      # one whole tile, one whole unit, negative scale
    (1, 2, 65, 193, 0.1, 2),       # one query past a unit
    (1, 2, 130, 1000, 0.0, 2),     # zero scale; the last wave of the partial tile without keys
    (2, 7, 1200, 1100, 0.1, 4),    # 266 units of 64 queries on 256 CUs: 128-query units
    (1, 16, 1537, 257, -0.1, 4),   # 13 units a head, the last of one query
])
def test_short_units_match_fp64(pkg, oracle, device, D, B, H, Sq, Sk, scale, QW):
    """Both unit sizes at the edges of their tiles, in buffers whose
    neighbouring head is NaN: within the operator's bar of float64, two
    launches bitwise equal, doubling V doubles the output bitwise."""
    gen = torch.Generator("cpu").manual_seed(Sq * 5 + Sk + D)
    bufs = [torch.full((B, s, H + 1, D), float("nan")) for s in (Sq, Sk, Sk)]
    for b in bufs:
        b[:, :, :H] = torch.randn(b[:, :, :H].shape, generator=gen)
    q, k, v = (_bhsd(b.to(BF)[:, :, :H]) for b in bufs)
    qd, kd, vd = (_bhsd(b.to(BF).to(device)[:, :, :H]) for b in bufs)
    out = torch.full((B, Sq, H, D), float("nan"), dtype=BF, device=device)
    out1, out2 = torch.full_like(out, float("nan")), torch.full_like(out, float("nan"))
    attn = pkg.make_attention(head_dim=D)
    names = _kernels(lambda: attn(qd, kd, vd, scale, _bhsd(out)))
    if torch.cuda.get_device_properties(device).multi_processor_count == 256:
        neg = "true" if scale < 0 else "false"
        assert len(names) == 1 and f"attention16_short_kernel<{neg}, {D}, {QW}>" in names[0], names
    attn(qd, kd, vd, scale, _bhsd(out1))
    attn(qd, kd, vd * 2, scale, _bhsd(out2))
    torch.cuda.synchronize()
    mx, rel = attention_error(_bhsd(out).cpu(), oracle.attention(q, k, v, scale))
    assert mx <= MAX_ABS and rel <= REL_RMS, (mx, rel)
    assert torch.equal(out, out1) and torch.equal(out2, out * 2)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [128, 72])
@pytest.mark.parametrize("case", ["overflow", "dominated", "denominator", "huge_values"])
def test_short_units_reference_maximum(pkg, oracle, device, D, case):
    """A key far above the first tile's maxima, in a later tile and one key
    group: exact where its weight dominates, recomputed with the running
    maximum where p, a denominator or O leaves its range."""
    keys = [320, 324, 328, 332] if case == "denominator" else [333]
    q, k, v = _dominant_keys(700, keys, 127.0, 0.25 if case == "denominator" else 1.96875)
    if case == "overflow":
        k[0, 0, 333, 0] = 100.0
    elif case == "dominated":
        k[0, 0, 333, 0] = 24.0
    elif case == "huge_values":
        k[0, 0, 300:, 0] = 10.0
        v = (v.float().sign() * 1e33 + v.float() * 1e31).to(BF)
    q, k, v = (t[..., :D].contiguous() for t in (q, k, v))
    scale = 128 ** -0.5
    want = oracle.attention(q.double(), k.double(), v.double(), scale)
    out = torch.full(q.shape, float("nan"), dtype=BF, device=device)
    pkg.make_attention(head_dim=D)(q.to(device), k.to(device), v.to(device), scale, out)
    torch.cuda.synchronize()
    got = out.cpu()
    assert torch.isfinite(got.float()).all()
    if case in ("overflow", "dominated"):
        assert torch.equal(got, torch.full_like(got, 1.96875))
    rel = float((got.double() - want).norm() / want.norm())
    assert rel <= REL_RMS, rel


@pytest.mark.gpu
@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("D,B,H,Sq,Sk,planned,kernel,masked", [
    (128, 1, 1, 256, 256, True, "attention16_short_kernel", (64, 96)),   # the third of four key groups of a tile
    (128, 1, 1, 256, 256, True, "attention16_short_kernel", (0, 128)),   # every group of the first tile
    (128, 1, 16, 1537, 300, True, "attention16_short_kernel", (0, 64)),  # the first of two groups
    (72, 1, 1, 256, 256, True, "attention16_short_kernel", (64, 96)),
    (72, 1, 16, 1537, 300, True, "attention16_short_kernel", (0, 128)),
    (128, 1, 1, 256, 6400, True, "attention16_kernel", (0, 3200)),       # whole pieces and the first tile of one
    (72, 2, 3, 1000, 3001, True, "attention16_kernel", (0, 1600)),
    (128, 1, 2, 300, 150, False, "attention16_kernel", (0, 64)),         # a unit's first tile
    (128, 1, 14, 8192, 150, False, "attention16_small_kernel", (0, 64)),
    (72, 1, 2, 300, 150, False, "attention_fwd_kernel", (0, 64)),
    (72, 1, 16, 4096, 150, False, "attention_fwd_kernel", (0, 64)),
])
def test_keys_at_minus_infinity(pkg, device, sign, D, B, H, Sq, Sk, planned, kernel, masked):
    """Keys masked through a channel of K at -inf, all that a wave's key group, a
    workgroup's key piece or a unit takes its first maximum from: their weight
    is 0, and the result is that of the other keys. With every key masked it is
    NaN, as a softmax over no keys."""
    gen = torch.Generator(device).manual_seed(Sk + D)
    q, k, v = (torch.randn(B, H, s, D, generator=gen, device=device).to(BF) for s in (Sq, Sk, Sk))
    q[..., 0] = 1.0
    keep = torch.ones(Sk, dtype=torch.bool, device=device)
    keep[masked[0]:masked[1]] = False
    k[:, :, ~keep, 0] = float("-inf") * sign
    out = torch.full_like(q, 3.0)
    attn = pkg.make_attention(head_dim=D, split_last_round=planned)
    names = _kernels(lambda: attn(q, k, v, sign * D ** -0.5, out))
    if torch.cuda.get_device_properties(device).multi_processor_count == 256:
        assert kernel + "<" in names[0], names
    want = gpu_reference_fp32(q, k[:, :, keep].contiguous(), v[:, :, keep].contiguous(), sign * D ** -0.5)
    assert torch.isfinite(out.float()).all()
    mx, rel = attention_error(out, want)
    assert mx <= MAX_ABS and rel <= REL_RMS, (mx, rel)
    k[..., 0] = float("-inf") * sign
    attn(q, k, v, sign * D ** -0.5, out)
    assert torch.isnan(out.float()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("D", [128, 72])
@pytest.mark.parametrize("H,Sq,Sk,low", [
    (1, 256, 700, 333),    # four key groups to a tile: keys 5 and 333 in different ones
    (16, 1537, 700, 333),  # two
    (1, 256, 6400, 3400),  # the pieces of a key split
])
def test_merge_keeps_keys_far_above_their_own_reference(pkg, oracle, device, D, H, Sq, Sk, low):
    """Key 5 sits 126.5 log2 units above the zeros and sets its part's reference
    maximum; key `low`, two units below it, is in a part whose first tile has
    zeros only. Its weight there (2^124.5) needs no recompute, and the merge has
    to bring it back by 2^-126.5, below the smallest normal number."""
    gen = torch.Generator("cpu").manual_seed(Sk)
    q, k = torch.zeros(1, H, Sq, D), torch.zeros(1, H, Sk, D)
    v = (torch.rand(1, H, Sk, D, generator=gen) * 2 - 1).to(BF)  # |p v| < 2^125: no recompute for O either
    q[..., 0] = 16.0
    k[:, :, 5, 0], k[:, :, low, 0] = 62.0, 61.0  # 126.50 and 124.46 log2 units
    q, k = q.to(BF), k.to(BF)
    scale = 128 ** -0.5
    out = torch.full(q.shape, float("nan"), dtype=BF, device=device)
    attn = pkg.make_attention(head_dim=D)
    names = _kernels(lambda: attn(q.to(device), k.to(device), v.to(device), scale, out))
    if torch.cuda.get_device_properties(device).multi_processor_count == 256:
        assert ("short" in names[0]) == (Sk == 700) and len(names) == (1 if Sk == 700 else 2), names
    want = oracle.attention(q[:, :, :1].double(), k.double(), v.double(), scale).expand(q.shape)
    mx, rel = attention_error(out.cpu(), want)
    assert mx <= MAX_ABS and rel <= REL_RMS, (mx, rel)


@pytest.mark.gpu
@pytest.mark.parametrize("H,Sq,Sk,kernel", [
    (1, 256, 704, "attention16_short_kernel<false, 72, 2>"), (16, 1537, 715, "attention16_short_kernel<false, 72, 4>"),
    (1, 256, 6410, "attention16_kernel<false, true, 72>"), (16, 4096, 705, "attention_fwd_kernel<false, true, 72"),
])
def test_vision_denominator_sums_the_unrounded_weights(pkg, device, H, Sq, Sk, kernel):
    """Head dim 72: the reference's order on every path, bf16 weights on V over
    the fp32 sum of the weights before that rounding. One key of 16 weighs 1 and
    the others 0.5019, which rounds to 0.5: V = 1 comes out as (1 + 15 / 2) /
    (1 + 15 * 0.5019) = 0.9967, not as 1."""
    q, k = torch.zeros(1, H, Sq, 72), torch.zeros(1, H, Sk, 72)
    q[..., 0] = 1.0
    k[:, :, 5::16, 0] = 1.0
    q, k, v = (t.to(BF).to(device) for t in (q, k, torch.ones(1, H, Sk, 72)))
    out = torch.full_like(q, float("nan"))
    attn = pkg.make_attention(head_dim=72)
    scale = 0.99453 * 0.6931471805599453
    names = _kernels(lambda: attn(q, k, v, scale, out))
    if torch.cuda.get_device_properties(device).multi_processor_count == 256:
        assert kernel in names[0], names
    weight = 2.0 ** -0.99453
    high = len(range(5, Sk, 16))
    want = torch.tensor((high + (Sk - high) * 0.5) / (high + (Sk - high) * weight)).to(BF).item()
    assert want == 0.99609375 and bool((out == want).all()), out.float().aminmax()
