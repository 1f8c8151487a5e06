"""Head dim 72 on the buffer path (attention16_kernel): the padding of the
72-dim rows, the denominator taken from V's padding dim, the key split of a
partly filled last round and the overflow fallback, against the fp32 / fp64
references of the operator."""
from __future__ import annotations

import pytest
import torch

from conftest import attention_error
from test_attention_gpu import MAX_ABS, REL_RMS, _bhsd, gpu_reference_fp32

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
D = 72


@pytest.mark.parametrize("B,H,Sq,Sk,sign,split", [
    (1, 16, 4097, 4097, 1.0, True),    # 272 units on 256 CUs: the last 16 split along the keys
    (2, 3, 1000, 3001, -1.0, True),    # one partial round, ragged keys, negative scale
    (1, 2, 255, 64, 1.0, False),       # one whole key tile
    (1, 2, 257, 65, -1.0, False),      # one key past it
    (1, 1, 16, 63, 1.0, False),        # a partial tile only
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
    attn(q, k, v, sign * D ** -0.5, _bhsd(out))
    attn(q, k, v * 2, sign * D ** -0.5, _bhsd(out2))
    torch.cuda.synchronize()
    mx, rel = attention_error(_bhsd(out), gpu_reference_fp32(q, k, v, sign * D ** -0.5))
    assert mx <= MAX_ABS and rel <= REL_RMS, (mx, rel)
    assert torch.equal(out2, out * 2)


@pytest.mark.parametrize("case", ["dominated", "late_logit", "denominator", "huge_values"])
def test_vision_attention_reference_maximum(pkg, oracle, device, case):
    """A later key far above the first tile's maximum: its V row comes out
    exactly where it dominates; where p, the denominator (finite weights that
    sum past FLT_MAX) or O overflows, the unit is recomputed with the running
    maximum."""
    gen = torch.Generator("cpu").manual_seed(9)
    q = torch.zeros(1, 1, 300, D)
    k = torch.zeros(1, 1, 700, D)
    v = torch.randn(1, 1, 700, D, generator=gen)
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
    pkg.make_attention(head_dim=D)(q.to(device), k.to(device), v.to(device), scale, out)
    torch.cuda.synchronize()
    got = out.cpu()
    assert torch.isfinite(got.float()).all()
    if case == "dominated":
        assert torch.equal(got, torch.full_like(got, 1.96875))
    rel = float((got.double() - want).norm() / want.norm())
    assert rel <= REL_RMS, rel
