"""Head dim 72 on the buffer path: the padding of the 72-dim rows and the
running maximum on each of its kernels -- unsplit launches (attention_fwd_kernel),
the key split of a partly filled last round (attention16_kernel) and the short
launches (attention16_short_kernel) -- against the fp32 / fp64 references of the
operator."""
from __future__ import annotations

import pytest
import torch

from conftest import attention_error
from test_attention_gpu import MAX_ABS, REL_RMS, _bhsd, gpu_reference_fp32
from test_attention_planned import _kernels

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
D = 72


FWD, SPLIT = "attention_fwd_kernel<{}, true, 72, false>", "attention16_kernel<{}, true, 72>"


def _assert_kernel(device, names, kernel, negative):
    """The launch ran `kernel` (the plans are those of 256 CUs)."""
    if torch.cuda.get_device_properties(device).multi_processor_count == 256:
        assert kernel.format("true" if negative else "false") in names[0], names
        assert len(names) == (2 if kernel == SPLIT else 1), names  # the split's merge


@pytest.mark.parametrize("B,H,Sq,Sk,sign,split", [
    (1, 16, 4097, 4097, 1.0, True),    # 272 units on 256 CUs: the last 16 split along the keys
    (2, 3, 1000, 3001, -1.0, True),    # one partial round, ragged keys, negative scale
    (1, 2, 255, 64, 1.0, False),       # one whole key tile
    (1, 2, 257, 65, -1.0, False),      # one key past it
    (1, 1, 16, 63, 1.0, False),        # a partial tile only
    (1, 16, 3501, 3501, -1.0, False),  # 224 units: ragged queries and keys, negative scale
    (1, 16, 4000, 63, 1.0, False),     # a nearly full chip with a partial tile only
    (3, 16, 1280, 1024, 1.0, False),   # whole tiles, several batch entries
])
def test_vision_attention_plans(pkg, device, B, H, Sq, Sk, sign, split):
    """Every plan at its edges, in a fused projection whose neighbours are NaN
    (no value outside a head's 72 dims may reach the result): within the
    operator's bar, and doubling V doubles the output bitwise."""
    nbytes = pkg._lib.attention_planned_workspace_bytes(B, H, Sq, Sk, D)
    if torch.cuda.get_device_properties(device).multi_processor_count == 256:
        assert (nbytes > 0) == split, nbytes
    gen = torch.Generator("cpu").manual_seed(Sq + 3 * Sk)
    # Rows of H heads in an H + 1 head buffer of NaN; 144-byte head rows.
    bufs = [torch.full((B, s, H + 1, D), float("nan")) for s in (Sq, Sk, Sk)]
    for b in bufs:
        b[:, :, :H] = torch.randn(b[:, :, :H].shape, generator=gen)
    q, k, v = (_bhsd(b.to(BF).to(device)[:, :, :H]) for b in bufs)
    out = torch.full((B, Sq, H, D), float("nan"), dtype=BF, device=device)
    out2 = torch.full_like(out, float("nan"))
    attn = pkg.make_attention(head_dim=D)
    names = _kernels(lambda: attn(q, k, v, sign * D ** -0.5, _bhsd(out)))
    _assert_kernel(device, names, SPLIT if split else FWD, sign < 0)
    attn(q, k, v * 2, sign * D ** -0.5, _bhsd(out2))
    torch.cuda.synchronize()
    mx, rel = attention_error(_bhsd(out), gpu_reference_fp32(q, k, v, sign * D ** -0.5))
    assert mx <= MAX_ABS and rel <= REL_RMS, (mx, rel)
    assert torch.equal(out2, out * 2)


@pytest.mark.parametrize("Sk,planned,kernel", [
    (700, True, "attention16_short_kernel<{}, 72, 2>"), (6400, True, SPLIT), (700, False, FWD)])
@pytest.mark.parametrize("case", ["dominated", "late_logit", "denominator", "huge_values"])
def test_vision_attention_running_maximum(pkg, oracle, device, case, Sk, planned, kernel):
    """A later key far above the first tile's maximum raises the running one: its
    V row comes out exactly where it dominates, and nothing overflows where
    weights against the first tile's maximum, their sum or O would."""
    gen = torch.Generator("cpu").manual_seed(9)
    q = torch.zeros(1, 1, 300, D)
    k = torch.zeros(1, 1, Sk, D)
    v = torch.randn(1, 1, Sk, D, generator=gen)
    q[..., 0] = 16.0
    scale = 0.1803369  # times log2 e: 0.2601710
    if case == "dominated":
        k[0, 0, 333, 0] = 10.0
        v[0, 0, 333] = 1.96875
    elif case == "late_logit":
        k[0, 0, 500, 0] = 50.0
    elif case == "denominator":
        k[0, 0, [320, 324, 328, 332], 0] = 30.5  # 127.0 log2 units each
        v[0, 0, [320, 324, 328, 332]] = 0.25
    else:
        k[0, 0, 300:, 0] = 5.0
        v = v.sign() * 1e33 + v * 1e31
    q, k, v = (t.to(BF) for t in (q, k, v))
    want = oracle.attention(q.double(), k.double(), v.double(), scale)
    out = torch.full(q.shape, float("nan"), dtype=BF, device=device)
    attn = pkg.make_attention(head_dim=D, split_last_round=planned)
    names = _kernels(lambda: attn(q.to(device), k.to(device), v.to(device), scale, out))
    _assert_kernel(device, names, kernel, False)
    got = out.cpu()
    assert torch.isfinite(got.float()).all()
    if case == "dominated":
        assert torch.equal(got, torch.full_like(got, 1.96875))
    rel = float((got.double() - want).norm() / want.norm())
    assert rel <= REL_RMS, rel
