"""The RMS family's 16-byte launch shapes at the sizes where the rule that picks
them changes (rows_by_block) and at the edges of their groups: bitwise against
the oracle's fixed order, on rows taken from every part of the launch."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
EPS = 1e-6


def _randn(gen, *shape, scale=1.0, mean=0.0):
    return (torch.randn(*shape, generator=gen) * scale + mean).to(BF)


# One launch per side of every bound: 1536 rows, 2048 / 3072 rows of W8 > 512,
# 8192 gated rows; W8 = 65 (one group past a wave), 512 / 513, 672 (a half last
# wave group), 768 and 1024 (exact), 1023.
SIZES = [(1535, 520), (1536, 520), (1536, 4096), (1537, 4104), (2048, 5376), (2049, 5376), (3072, 8184), (3073, 8192),
         (1600, 6144), (8191, 5376), (8192, 5376)]


# Per-row views take one launch shape whatever the size.
@pytest.mark.parametrize("rows,W,mods", [(*s, m) for s in SIZES for m in ("broadcast", "per_token")] +
                         [(1537, 4104, "per_row"), (2049, 5376, "per_row")])
def test_rms_family_launch_shapes_bitwise(pkg, oracle, device, rows, W, mods):
    gen = torch.Generator("cpu").manual_seed(rows + W)
    R = 3
    B, S = (3, rows // 3) if rows % 3 == 0 else (1, rows)
    x, y = _randn(gen, B, S, W), _randn(gen, B, S, W)
    w = _randn(gen, W, scale=0.1, mean=1.0)
    tables = [_randn(gen, R, W, scale=0.1) for _ in range(3)]
    # Runs of rows, one boundary inside a block of eight rows.
    index = (torch.arange(B * S) * R // (B * S)).view(B, S)
    if mods == "broadcast":
        index = torch.zeros(B, S, dtype=torch.int64)
    gate, scale, shift = (t[index] for t in tables)  # [B, S, W]
    d = lambda t: t.to(device)
    xd, yd, wd = d(x), d(y), d(w)
    outs = [torch.full((B, S, W), float("nan"), dtype=BF, device=device) for _ in range(4)]
    mod, res, norm, plain = outs
    if mods == "per_token":
        gt, sc, sh = (d(t) for t in tables)
        pkg.make_rms_modulate_indexed()(xd, wd, EPS, sc, sh, d(index), mod)
        pkg.make_gated_residual_rms_modulate_indexed()(xd, gt, yd, wd, EPS, sc, sh, d(index), res, norm)
    else:
        views = [d(t) for t in (gate, scale, shift)]
        if mods == "broadcast":
            views = [d(t)[:1].unsqueeze(0).expand(B, S, W) for t in tables]
        gt, sc, sh = views
        pkg.make_rms_modulate()(xd, wd, EPS, sc, sh, mod)
        pkg.make_gated_residual_rms_modulate()(xd, gt, yd, wd, EPS, sc, sh, res, norm)
    pkg.make_rms(width=None)(xd, wd, EPS, plain)
    torch.cuda.synchronize()
    for t in outs:
        assert not torch.isnan(t).any()
    rows_at = torch.unique(torch.cat([torch.arange(9), torch.arange(S - 9, S), S // R + torch.arange(-9, 9),
                                      torch.randint(0, S, (32,), generator=gen)]).clamp(0, S - 1))
    pick = lambda t: t[:, rows_at].contiguous()
    want_res, want_norm = oracle.gated_residual_rms_modulate(pick(x), pick(gate), pick(y), w, EPS, pick(scale),
                                                             pick(shift))
    want = {"mod": oracle.rms_modulate(pick(x), w, EPS, pick(scale), pick(shift)), "res": want_res,
            "norm": want_norm, "plain": oracle.rms_norm(pick(x), w, EPS)}
    for name, got in zip(("mod", "res", "norm", "plain"), outs):
        assert torch.equal(pick(got.cpu()), want[name]), name


def test_rms_row_kernel_past_the_x_extent_of_a_grid(pkg, device):
    """2^24 rows and more, one block of 256 threads each, are more than the
    2^32 - 1 threads a launch holds along x. The batch is broadcast (stride 0),
    so that only the outputs take memory: every batch entry is the first one's
    bits, which a small launch gives as well."""
    B, S, W, R = 4097, 4099, 520, 5
    assert B * S > 1 << 24
    if torch.cuda.mem_get_info(device)[0] < 48 << 30:
        pytest.skip("48 GiB of device memory needed")
    gen = torch.Generator("cpu").manual_seed(11)
    x, y, scale, shift = (_randn(gen, 1, S, W).to(device) for _ in range(4))
    w, tables = _randn(gen, W).to(device), [_randn(gen, R, W).to(device) for _ in range(3)]
    index = torch.randint(0, R, (1, S), generator=gen).to(device)
    big = lambda t: t.expand(B, *t.shape[1:])

    def check(got, want):
        for b in range(0, B, 256):
            part = got[b:b + 256]
            assert bool((part == want).all()), b

    out, small = torch.zeros(B, S, W, dtype=BF, device=device), torch.zeros(1, S, W, dtype=BF, device=device)
    rms = pkg.make_rms_modulate()
    rms(x, w, EPS, scale, shift, small)
    rms(big(x), w, EPS, big(scale), big(shift), out)  # per-row modulation views
    check(out, small)
    gated = pkg.make_gated_residual_rms_modulate_indexed(check_indices=False)
    res, small_res = torch.zeros_like(out), torch.zeros_like(small)
    gated(x, tables[0], y, w, EPS, tables[1], tables[2], index, small_res, small)
    out.zero_()
    gated(big(x), tables[0], big(y), w, EPS, tables[1], tables[2], big(index), res, out)
    check(res, small_res)
    check(out, small)


@pytest.mark.parametrize("rows,W", [(64, 5376), (2000, 5376), (5726, 5376), (9000, 3072)])
def test_outputs_in_place_of_inputs(pkg, device, rows, W):
    """Outputs over the inputs they replace (RMSNorm into x, the residual into x
    and the norm into y, RoPE and the SwiGLU product into their inputs): the bits
    of separate outputs, on the one-row-per-block and the persistent launches."""
    gen = torch.Generator("cpu").manual_seed(rows)
    x, y = (_randn(gen, 1, rows, W).to(device) for _ in range(2))
    w = _randn(gen, W, scale=0.1, mean=1.0).to(device)
    table = [_randn(gen, 3, W, scale=0.1).to(device) for _ in range(3)]
    index = (torch.arange(rows, device=device) * 3 // rows).view(1, rows)
    gate, scale, shift = (t[:1].unsqueeze(0).expand(1, rows, W) for t in table)
    new = lambda: torch.zeros_like(x)
    rms, mod, gated = pkg.make_rms(width=None), pkg.make_rms_modulate(), pkg.make_gated_residual_rms_modulate()
    imod, igated = pkg.make_rms_modulate_indexed(False), pkg.make_gated_residual_rms_modulate_indexed(False)
    ops = [(lambda x, y, r, o: rms(x, w, EPS, o), "x"), (lambda x, y, r, o: mod(x, w, EPS, scale, shift, o), "x"),
           (lambda x, y, r, o: imod(x, w, EPS, table[1], table[2], index, o), "x"),
           (lambda x, y, r, o: gated(x, gate, y, w, EPS, scale, shift, r, o), "xy"),
           (lambda x, y, r, o: igated(x, table[0], y, w, EPS, table[1], table[2], index, r, o), "xy"),
           (lambda x, y, r, o: pkg.make_swiglu()(x, y, o), "x")]
    for op, over in ops:
        r, o, xi, yi = new(), new(), x.clone(), y.clone()
        op(x, y, r, o)
        op(xi, yi, xi, yi if over == "xy" else xi)
        if over == "xy":
            assert torch.equal(xi, r) and torch.equal(yi, o)
        else:
            assert torch.equal(xi, o)
    heads = x.view(rows, W // 128, 128)
    cos, sin = (_randn(gen, rows, 48).to(device) for _ in range(2))
    o, xi = torch.zeros_like(heads), heads.clone()
    pkg.make_rope()(heads, cos, sin, o)
    pkg.make_rope()(xi, cos, sin, xi)
    assert torch.equal(xi, o)
