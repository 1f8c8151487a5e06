"""H3 pointwise ops with the reference's per-step bf16 rounding, on gfx950.

Drop-in for tools/h3_pointwise.py: the same `make_*` factories, keyword
arguments and returned-callable argument orders. Outputs are preallocated by the
caller; each call enqueues one kernel of libh3mi355x.so on the current torch
stream and returns None. Tile keywords of the reference (rows, cols, block,
num_warps, block_tokens, ranks) are accepted for signature compatibility; the
gfx950 kernels choose their own launch shapes, and the results do not depend
on them.
"""
from __future__ import annotations

import torch

from . import _lib

__all__ = [
    "make_swiglu", "make_rms", "make_rms_modulate", "make_gated_residual",
    "make_gated_residual_rms_modulate", "make_rope", "make_qk_norm_rope",
    "make_qk_norm_rope_interleaved", "make_qk_norm_rope_interleaved_qk", "make_rope_cache", "modulation_columns", "make_rms_modulate_indexed",
    "make_gated_residual_rms_modulate_indexed", "make_gated_residual_indexed", "qkv_by_rank",
    "make_qkv_norm_rope_pack", "make_qkv_norm_rope_pack_fp8", "make_qkv_norm_rope_pack_fp8_vamax",
    "make_qkv_norm_rope_pack_fp8_noalloc", "make_qkv_norm_rope_pack_fp8x2_vamax",
]


def _bf16_only(dtype) -> None:
    """The reference's `dtype` keyword (ninetoothed.bfloat16 by default): the
    gfx950 kernels are bf16 kernels."""
    if dtype is None:
        return
    name = str(getattr(dtype, "name", dtype)).lower()
    if name not in ("bfloat16", "torch.bfloat16", "bf16"):
        raise ValueError(f"only bfloat16 kernels are built for gfx950, got dtype={dtype!r}")


def _bf16(*tensors: torch.Tensor) -> torch.device:
    device = _lib.check_cuda(*tensors)
    _lib.check_dtype(torch.bfloat16, *tensors)
    return device


def _ndim(n: int, **tensors: torch.Tensor) -> None:
    for name, t in tensors.items():
        if t.dim() != n:
            raise ValueError(f"{name} must be {n}-D, got shape {tuple(t.shape)}")


def make_swiglu(caller="torch", output_dir=None, archs=None, rows=1, cols=1024, num_warps=4, dtype=None):
    """out = bf16(up * bf16(g / (1 + exp(-g)))) on [B, S, F] (tools/h3_pointwise.py:18-34)."""
    _bf16_only(dtype)
    fast = _lib.fast("launch_h3_swiglu_exact", "b3b3b3")

    def kernel(up, gate, out):
        status = fast(up, gate, out)
        if status is True:
            return
        _ndim(3, up=up, gate=gate, out=out)
        device = _bf16(up, gate, out)
        _lib.launch_after(status, "launch_h3_swiglu_exact", device, _lib.tensor(up), _lib.tensor(gate),
                          _lib.tensor(out))

    return kernel


def make_rms(caller="torch", output_dir=None, archs=None, width=5376, dtype=None):
    """RMSNorm with bf16 rounding per step on [B, S, width] (tools/h3_pointwise.py:46-70)."""
    _bf16_only(dtype)
    if width is not None and width <= 0:
        raise ValueError("width must be positive")
    name = {128: "launch_h3_rms_exact_128", 5376: "launch_h3_rms_exact_5376"}.get(width, "launch_h3_rms_exact")
    fast = _lib.fast(name, "b3b1s0b3", fix=None if width is None else (0, 2, width))

    def kernel(x, weight, eps, out):
        status = fast(x, weight, eps, out)
        if status is True:
            return
        _ndim(3, x=x, out=out)
        _ndim(1, weight=weight)
        if width is not None and x.shape[-1] != width:
            raise ValueError(f"this kernel was made for width {width}, got {x.shape[-1]}")
        device = _bf16(x, weight, out)
        _lib.launch_after(status, name, device, _lib.tensor(x), _lib.tensor(weight), _lib.scalar(eps),
                          _lib.tensor(out))

    return kernel


def make_rms_modulate(caller="torch", output_dir=None, archs=None, dtype=None):
    """RMSNorm + AdaLN: bf16(bf16(bf16(rms(x) w) bf16(1 + scale)) + shift)
    (tools/h3_pointwise.py:83-108), any width."""
    _bf16_only(dtype)
    fast = _lib.fast("launch_h3_rms_modulate_exact", "b3b1s0b3b3b3")

    def kernel(x, weight, eps, scale, shift, out):
        status = fast(x, weight, eps, scale, shift, out)
        if status is True:
            return
        _ndim(3, x=x, scale=scale, shift=shift, out=out)
        _ndim(1, weight=weight)
        device = _bf16(x, weight, scale, shift, out)
        _lib.launch_after(status, "launch_h3_rms_modulate_exact", device, _lib.tensor(x), _lib.tensor(weight),
                          _lib.scalar(eps), _lib.tensor(scale), _lib.tensor(shift), _lib.tensor(out))

    return kernel


def make_gated_residual(caller="torch", output_dir=None, archs=None, block=(4, 512), num_warps=8, dtype=None):
    """out = bf16(x + bf16(gate * y)) (tools/h3_pointwise.py:121-136)."""
    _bf16_only(dtype)
    fast = _lib.fast("launch_h3_gated_residual_exact", "b3b3b3b3")

    def kernel(x, gate, y, out):
        status = fast(x, gate, y, out)
        if status is True:
            return
        _ndim(3, x=x, gate=gate, y=y, out=out)
        device = _bf16(x, gate, y, out)
        _lib.launch_after(status, "launch_h3_gated_residual_exact", device, _lib.tensor(x), _lib.tensor(gate),
                          _lib.tensor(y), _lib.tensor(out))

    return kernel


def make_gated_residual_rms_modulate(caller="torch", output_dir=None, archs=None, num_warps=4, dtype=None):
    """residual = bf16(x + bf16(gate * y)); out = rms_modulate(residual)
    (tools/h3_pointwise.py:150-182)."""
    _bf16_only(dtype)
    fast = _lib.fast("launch_h3_gated_residual_rms_modulate_exact", "b3b3b3b1s0b3b3b3b3")

    def kernel(x, gate, y, weight, eps, scale, shift, residual, out):
        status = fast(x, gate, y, weight, eps, scale, shift, residual, out)
        if status is True:
            return
        _ndim(3, x=x, gate=gate, y=y, scale=scale, shift=shift, residual=residual, out=out)
        _ndim(1, weight=weight)
        device = _bf16(x, gate, y, weight, scale, shift, residual, out)
        _lib.launch_after(status, "launch_h3_gated_residual_rms_modulate_exact", device, _lib.tensor(x),
                          _lib.tensor(gate), _lib.tensor(y), _lib.tensor(weight), _lib.scalar(eps), _lib.tensor(scale),
                          _lib.tensor(shift), _lib.tensor(residual), _lib.tensor(out))

    return kernel


# ------------------------------------------------- per-token AdaLN rows (indexed)
#
# A DiT block's AdaLN sites over all tokens in one launch each, token (b, s)
# taking row index[b, s] of the modulation tables. The reference launches each
# op once per run-length segment of the indices, on broadcast views of the
# segment's row (patches/InfiniLM.patch:1353-1397, segments built on the host
# at :1765-1793); the results are the same bits.

MODULATION_COLUMNS = ("shift_msa", "scale_msa", "gate_msa", "shift_mlp", "scale_mlp", "gate_mlp")


def modulation_columns(modulation: torch.Tensor, hidden: int) -> dict:
    """The six [R, hidden] column blocks of the AdaLN modulation matrix
    [R, 6 * hidden], by name, in the reference's column order
    (patches/InfiniLM.patch:1359-1364,1375): views, no copies."""
    if modulation.dim() != 2 or modulation.shape[1] != 6 * hidden:
        raise ValueError(f"modulation must be [R, 6 * {hidden}], got {tuple(modulation.shape)}")
    return {name: modulation[:, i * hidden:(i + 1) * hidden] for i, name in enumerate(MODULATION_COLUMNS)}


def _token_index(index: torch.Tensor, x: torch.Tensor, table_rows: int, check: bool) -> torch.Tensor:
    """The per-token row index as the kernels take it: int64 [B, S]. Accepts
    [S] (B == 1) or [B, S], int32 or int64 (the dtypes the reference accepts,
    patches/InfiniLM.patch:1772-1775). With `check`, an index outside
    [0, table_rows) raises (one device-to-host read of its min and max), as the
    reference's narrow of the modulation row would."""
    if index.device != x.device:
        raise ValueError(f"index must be on {x.device}, got {index.device}")
    if index.dtype not in (torch.int32, torch.int64):
        raise ValueError(f"AdaLN indices must be int32 or int64, got {index.dtype}")
    if index.dim() == 1 and x.shape[0] == 1:
        index = index.unsqueeze(0)
    if tuple(index.shape) != tuple(x.shape[:2]):
        raise ValueError(f"index must be [B, S] = {tuple(x.shape[:2])} (or [S] for B == 1), got "
                         f"{tuple(index.shape)}")
    if index.dtype != torch.int64:
        index = index.to(torch.int64)
    if check and index.numel() > 0:
        lo, hi = (int(v) for v in torch.aminmax(index))
        if lo < 0 or hi >= table_rows:
            raise ValueError(f"AdaLN index out of range: [{lo}, {hi}] not within [0, {table_rows})")
    return index


def make_rms_modulate_indexed(check_indices: bool = True):
    """RMSNorm + AdaLN over [B, S, W] with scale/shift rows index[b, s] of [R, W]
    tables: one launch for every segment of the indices. Returns
    kernel(x, weight, eps, scale, shift, index, out). check_indices=False skips
    the range check (no host synchronisation; out-of-range indices are clamped
    by the kernel)."""
    fast = _lib.fast("launch_h3_rms_modulate_indexed", "b3b1s0b2b2i2b3")

    def kernel(x, weight, eps, scale, shift, index, out):
        status = False if check_indices else fast(x, weight, eps, scale, shift, index, out)
        if status is True:
            return
        _ndim(3, x=x, out=out)
        _ndim(2, scale=scale, shift=shift)
        _ndim(1, weight=weight)
        device = _bf16(x, weight, scale, shift, out)
        index = _token_index(index, x, scale.shape[0], check_indices)
        _lib.launch_after(status, "launch_h3_rms_modulate_indexed", device, _lib.tensor(x), _lib.tensor(weight),
                          _lib.scalar(eps), _lib.tensor(scale), _lib.tensor(shift), _lib.tensor(index),
                          _lib.tensor(out))

    return kernel


def make_gated_residual_rms_modulate_indexed(check_indices: bool = True):
    """residual = bf16(x + bf16(gate * y)); out = rms_modulate(residual), with
    gate/scale/shift rows index[b, s] of [R, W] tables. Returns
    kernel(x, gate, y, weight, eps, scale, shift, index, residual, out)."""
    fast = _lib.fast("launch_h3_gated_residual_rms_modulate_indexed", "b3b2b3b1s0b2b2i2b3b3")

    def kernel(x, gate, y, weight, eps, scale, shift, index, residual, out):
        status = False if check_indices else fast(x, gate, y, weight, eps, scale, shift, index, residual, out)
        if status is True:
            return
        _ndim(3, x=x, y=y, residual=residual, out=out)
        _ndim(2, gate=gate, scale=scale, shift=shift)
        _ndim(1, weight=weight)
        device = _bf16(x, gate, y, weight, scale, shift, residual, out)
        index = _token_index(index, x, scale.shape[0], check_indices)
        _lib.launch_after(status, "launch_h3_gated_residual_rms_modulate_indexed", device, _lib.tensor(x),
                          _lib.tensor(gate), _lib.tensor(y), _lib.tensor(weight), _lib.scalar(eps), _lib.tensor(scale),
                          _lib.tensor(shift), _lib.tensor(index), _lib.tensor(residual), _lib.tensor(out))

    return kernel


def make_gated_residual_indexed(check_indices: bool = True):
    """out = bf16(x + bf16(gate * y)) with the gate row index[b, s] of a [R, W]
    table. Returns kernel(x, gate, y, index, out)."""
    fast = _lib.fast("launch_h3_gated_residual_indexed", "b3b2b3i2b3")

    def kernel(x, gate, y, index, out):
        status = False if check_indices else fast(x, gate, y, index, out)
        if status is True:
            return
        _ndim(3, x=x, y=y, out=out)
        _ndim(2, gate=gate)
        device = _bf16(x, gate, y, out)
        index = _token_index(index, x, gate.shape[0], check_indices)
        _lib.launch_after(status, "launch_h3_gated_residual_indexed", device, _lib.tensor(x), _lib.tensor(gate),
                          _lib.tensor(y), _lib.tensor(index), _lib.tensor(out))

    return kernel


def make_rope(caller="torch", output_dir=None, archs=None, dtype=None):
    """Rotate-half RoPE on channels 0..95 of [S, H, 128], cos/sin [S, 48]
    (tools/h3_pointwise.py:199-231). Returns launch(x, cos, sin, out)."""
    _bf16_only(dtype)
    fast = _lib.fast("launch_h3_rope_exact", "b3b2b2b3", (0, 0, 0, 1, 2, 3, 3, 3))

    def launch(x, cos, sin, out):
        status = fast(x, cos, sin, out)
        if status is True:
            return
        _ndim(3, x=x, out=out)
        _ndim(2, cos=cos, sin=sin)
        device = _bf16(x, cos, sin, out)
        xa, oa = _lib.tensor(x), _lib.tensor(out)
        _lib.launch_after(status, "launch_h3_rope_exact", device, xa, xa, xa, _lib.tensor(cos), _lib.tensor(sin), oa,
                          oa, oa)

    return launch


def _qk_launch(x0, x1, xp, w0, w1, wp, eps, cos, sin, y0, y1, yp, status=False):
    _ndim(4, x0=x0, x1=x1, xp=xp, y0=y0, y1=y1, yp=yp)
    _ndim(1, w0=w0, w1=w1, wp=wp)
    _ndim(2, cos=cos, sin=sin)
    device = _bf16(x0, x1, xp, w0, w1, wp, cos, sin, y0, y1, yp)
    _lib.launch_after(status, "launch_h3_qk_norm_rope", device, _lib.tensor(x0), _lib.tensor(x1), _lib.tensor(xp),
                      _lib.tensor(w0), _lib.tensor(w1), _lib.tensor(wp), _lib.scalar(eps), _lib.tensor(cos),
                      _lib.tensor(sin), _lib.tensor(y0), _lib.tensor(y1), _lib.tensor(yp))


def _qk_raw(x0, x1, xp, w0, w1, wp, eps, cos, sin, y0, y1, yp):
    _qk_launch(x0, x1, xp, w0, w1, wp, eps, cos, sin, y0, y1, yp)


def make_qk_norm_rope(caller="torch", output_dir=None, archs=None, rows=8, num_warps=1, block_tokens=1, ranks=1,
                      dtype=None):
    """Per-head RMSNorm (weight [128]) + rotate-half RoPE on x [T, P, Hs, 128]
    (any strides) into out [T, P, Hs, 128] (any strides), cos/sin [T, 48]
    (tools/h3_pointwise.py:262-294,370-402). caller="torch" returns
    launch(x, weight, eps, cos, sin, out); any other caller returns the raw
    12-argument kernel (x, x, x, w, w, w, eps, cos, sin, out, out, out)."""
    _bf16_only(dtype)
    if block_tokens != 1 and ranks != 1:
        raise ValueError("qk_norm_rope: block_tokens > 1 needs ranks == 1")
    if caller != "torch":
        return _qk_raw
    fast = _lib.fast("launch_h3_qk_norm_rope", "b4b1s0b2b2b4", (0, 0, 0, 1, 1, 1, 2, 3, 4, 5, 5, 5))

    def launch(x, weight, eps, cos, sin, out):
        status = fast(x, weight, eps, cos, sin, out)
        if status is True:
            return
        _qk_launch(x, x, x, weight, weight, weight, eps, cos, sin, out, out, out, status)

    return launch


def qkv_by_rank(projected: torch.Tensor, ranks: int):
    """The q, k and v parts of the fused projection [T, 3, P * Hs, 128] as
    [T, P, Hs, 128] views by destination rank, as InfiniLM builds them
    (patches/InfiniLM.patch:1089-1097). Views, no copies."""
    if projected.dim() != 4 or projected.shape[1] != 3 or projected.shape[2] % ranks != 0:
        raise ValueError(f"projected must be [T, 3, P * Hs, D] with P = {ranks}, got {tuple(projected.shape)}")
    T, _, width, D = projected.shape
    hs = width // ranks
    parts = []
    for i in range(3):
        part = projected[:, i]
        s0, s1, s2 = part.stride()
        parts.append(part.as_strided((T, ranks, hs, D), (s0, hs * s1, s1, s2)))
    return tuple(parts)


def make_qkv_norm_rope_pack(dtype=None):
    """q/k per-head RMSNorm + rotate-half RoPE and the v copy of one head group
    in one launch, cos/sin rows gathered from the [N, 96] RoPE cache through the
    token positions (patches/InfiniLM.patch:1071-1110). Returns
    kernel(q, k, v, q_weight, k_weight, eps, cache, positions, q_out, k_out, v_out):
    q, k, v and the outputs [T, P, Hs, 128] with any strides (see qkv_by_rank;
    the outputs are typically send buffers [P, T, Hs, 128] permuted to
    [T, P, Hs, 128]); positions int64 [T] (int32 is widened)."""
    _bf16_only(dtype)
    fast = _lib.fast("launch_h3_qkv_norm_rope_pack", "b4b4b4b1b1s0t2l1b4b4b4")

    def kernel(q, k, v, q_weight, k_weight, eps, cache, positions, q_out, k_out, v_out):
        status = fast(q, k, v, q_weight, k_weight, eps, cache, positions, q_out, k_out, v_out)
        if status is True:
            return
        _ndim(4, q=q, k=k, v=v, q_out=q_out, k_out=k_out, v_out=v_out)
        _ndim(1, q_weight=q_weight, k_weight=k_weight, positions=positions)
        _ndim(2, cache=cache)
        if cache.shape[1] != 96:
            raise ValueError(f"the RoPE cache must be [N, 96], got {tuple(cache.shape)}")
        device = _bf16(q, k, v, q_weight, k_weight, cache, q_out, k_out, v_out)
        if positions.device != device or positions.dtype not in (torch.int32, torch.int64):
            raise ValueError("positions must be an int32 or int64 tensor on the device of q")
        if positions.dtype != torch.int64:
            positions = positions.to(torch.int64)
        _lib.launch_after(status, "launch_h3_qkv_norm_rope_pack", device, _lib.tensor(q), _lib.tensor(k),
                          _lib.tensor(v), _lib.tensor(q_weight), _lib.tensor(k_weight), _lib.scalar(eps),
                          _lib.tensor(cache[:, :48]), _lib.tensor(cache[:, 48:]), _lib.tensor(positions),
                          _lib.tensor(q_out), _lib.tensor(k_out), _lib.tensor(v_out))

    return kernel


def _positions(positions: torch.Tensor, device) -> torch.Tensor:
    if positions.device != device or positions.dtype not in (torch.int32, torch.int64):
        raise ValueError("positions must be an int32 or int64 tensor on the device of q")
    return positions if positions.dtype == torch.int64 else positions.to(torch.int64)


def make_qkv_norm_rope_pack_fp8(dtype=None):
    """make_qkv_norm_rope_pack with q and k written as e4m3fn codes for the fp8
    attention: codes = e4m3fn(sat(bf16(y) * 448 / bound)), bound =
    fp32(sqrt(128) * 1.03125) * max|weight| (an upper bound of |y| for any
    input, so no absmax pass). Returns kernel(q, k, v, q_weight, k_weight, eps,
    cache, positions, q8, k8, v_out, q_descale, k_descale): q8, k8
    torch.float8_e4m3fn (or uint8) [T, P, Hs, 128]; q_descale, k_descale fp32
    [P * Hs] receive bound / 448; v_out bf16 (quantise it with
    quantize_fp8_per_head). No counterpart in the reference."""
    _bf16_only(dtype)
    fast = _lib.fast("launch_h3_qkv_norm_rope_pack_fp8", "b4b4b4b1b1s0t2l1u4u4b4f1f1")

    def kernel(q, k, v, q_weight, k_weight, eps, cache, positions, q8, k8, v_out, q_descale, k_descale,
               _entry="launch_h3_qkv_norm_rope_pack_fp8", _extra=(), _status=False):
        if not _extra:
            _status = fast(q, k, v, q_weight, k_weight, eps, cache, positions, q8, k8, v_out, q_descale, k_descale)
            if _status is True:
                return
        _ndim(4, q=q, k=k, v=v, q8=q8, k8=k8, v_out=v_out)
        _ndim(1, q_weight=q_weight, k_weight=k_weight, positions=positions, q_descale=q_descale,
              k_descale=k_descale)
        _ndim(2, cache=cache)
        if cache.shape[1] != 96:
            raise ValueError(f"the RoPE cache must be [N, 96], got {tuple(cache.shape)}")
        device = _bf16(q, k, v, q_weight, k_weight, cache, v_out)
        _lib.check_cuda(q, q8, k8, q_descale, k_descale)
        for name, t in (("q8", q8), ("k8", k8)):
            if t.dtype not in (torch.float8_e4m3fn, torch.uint8):
                raise ValueError(f"{name} must be float8_e4m3fn or uint8, got {t.dtype}")
        _lib.check_dtype(torch.float32, q_descale, k_descale)
        positions = _positions(positions, device)
        _lib.launch_after(_status, _entry, device, _lib.tensor(q), _lib.tensor(k), _lib.tensor(v),
                          _lib.tensor(q_weight), _lib.tensor(k_weight), _lib.scalar(eps), _lib.tensor(cache[:, :48]),
                          _lib.tensor(cache[:, 48:]), _lib.tensor(positions), _lib.tensor(q8), _lib.tensor(k8),
                          _lib.tensor(v_out), _lib.tensor(q_descale), _lib.tensor(k_descale), *_extra)

    return kernel


def make_qkv_norm_rope_pack_fp8_vamax(dtype=None):
    """make_qkv_norm_rope_pack_fp8 that also folds V's per-head amax while it
    copies v: kernel(q, k, v, q_weight, k_weight, eps, cache, positions, q8,
    k8, v_out, q_descale, k_descale, v_amax) with v_amax fp32 [P * Hs, 64]
    (contiguous), cleared and then filled by the launch: the maximum over a
    head's 64 slots is the amax of |v| over that head's rows (head p * Hs + h).
    Pass it to quantize_fp8_per_head(v, amax_slots=...) so that V's
    quantisation reads v once. No counterpart in the reference; the v copy it
    extends is patches/InfiniLM.patch:1063-1069,1104."""
    _bf16_only(dtype)
    base = make_qkv_norm_rope_pack_fp8()
    fast = _lib.fast("launch_h3_qkv_norm_rope_pack_fp8_vamax", "b4b4b4b1b1s0t2l1u4u4b4f1f1c2")

    def kernel(q, k, v, q_weight, k_weight, eps, cache, positions, q8, k8, v_out, q_descale, k_descale, v_amax):
        status = fast(q, k, v, q_weight, k_weight, eps, cache, positions, q8, k8, v_out, q_descale, k_descale, v_amax)
        if status is True:
            return
        _ndim(2, v_amax=v_amax)
        _lib.check_cuda(q, v_amax)
        _lib.check_dtype(torch.float32, v_amax)
        heads = q.shape[1] * q.shape[2]
        if v_amax.shape != (heads, _lib.AMAX_SLOTS) or not v_amax.is_contiguous():
            raise ValueError(f"v_amax must be a contiguous fp32 [{heads}, {_lib.AMAX_SLOTS}] tensor")
        base(q, k, v, q_weight, k_weight, eps, cache, positions, q8, k8, v_out, q_descale, k_descale,
             _entry="launch_h3_qkv_norm_rope_pack_fp8_vamax", _extra=(_lib.tensor(v_amax),),
             _status=status)

    return kernel


def make_qkv_norm_rope_pack_fp8x2_vamax(dtype=None):
    """make_qkv_norm_rope_pack_fp8_vamax with q and k also as the lo codes of
    the two-term split, for make_attention_fp8x2: kernel(q, k, v, q_weight,
    k_weight, eps, cache, positions, q8, q8_lo, k8, k8_lo, v_out, q_descale,
    k_descale, v_amax); q8, k8 as in make_qkv_norm_rope_pack_fp8; q8_lo, k8_lo
    e4m3fn (or uint8) with the shapes and strides of q8, k8. No counterpart in
    the reference."""
    _bf16_only(dtype)
    fast = _lib.fast("launch_h3_qkv_norm_rope_pack_fp8x2_vamax", "b4b4b4b1b1s0t2l1u4u4u4u4b4f1f1c2")

    def kernel(q, k, v, q_weight, k_weight, eps, cache, positions, q8, q8_lo, k8, k8_lo, v_out, q_descale,
               k_descale, v_amax):
        status = False
        if q8_lo.stride() == q8.stride() and k8_lo.stride() == k8.stride():
            status = fast(q, k, v, q_weight, k_weight, eps, cache, positions, q8, q8_lo, k8, k8_lo, v_out, q_descale,
                          k_descale, v_amax)
            if status is True:
                return
        _ndim(4, q8_lo=q8_lo, k8_lo=k8_lo)
        _ndim(2, v_amax=v_amax)
        _lib.check_cuda(q, q8_lo, k8_lo, v_amax)
        for name, lo, hi in (("q8_lo", q8_lo, q8), ("k8_lo", k8_lo, k8)):
            if lo.dtype not in (torch.float8_e4m3fn, torch.uint8):
                raise ValueError(f"{name} must be float8_e4m3fn or uint8, got {lo.dtype}")
            if lo.shape != hi.shape or lo.stride() != hi.stride():
                raise ValueError(f"{name} must have the shape and strides of its hi codes")
        _lib.check_dtype(torch.float32, v_amax)
        heads = q.shape[1] * q.shape[2]
        if v_amax.shape != (heads, _lib.AMAX_SLOTS) or not v_amax.is_contiguous():
            raise ValueError(f"v_amax must be a contiguous fp32 [{heads}, {_lib.AMAX_SLOTS}] tensor")
        _ndim(4, q=q, k=k, v=v, q8=q8, k8=k8, v_out=v_out)
        _ndim(1, q_weight=q_weight, k_weight=k_weight, positions=positions, q_descale=q_descale,
              k_descale=k_descale)
        _ndim(2, cache=cache)
        if cache.shape[1] != 96:
            raise ValueError(f"the RoPE cache must be [N, 96], got {tuple(cache.shape)}")
        device = _bf16(q, k, v, q_weight, k_weight, cache, v_out)
        _lib.check_cuda(q, q8, k8, q_descale, k_descale)
        for name, t in (("q8", q8), ("k8", k8)):
            if t.dtype not in (torch.float8_e4m3fn, torch.uint8):
                raise ValueError(f"{name} must be float8_e4m3fn or uint8, got {t.dtype}")
        _lib.check_dtype(torch.float32, q_descale, k_descale)
        positions = _positions(positions, device)
        _lib.launch_after(status, "launch_h3_qkv_norm_rope_pack_fp8x2_vamax", device, _lib.tensor(q), _lib.tensor(k),
                          _lib.tensor(v), _lib.tensor(q_weight), _lib.tensor(k_weight), _lib.scalar(eps),
                          _lib.tensor(cache[:, :48]), _lib.tensor(cache[:, 48:]), _lib.tensor(positions),
                          _lib.tensor(q8), _lib.tensor(q8_lo), _lib.tensor(k8), _lib.tensor(k8_lo), _lib.tensor(v_out),
                          _lib.tensor(q_descale), _lib.tensor(k_descale), _lib.tensor(v_amax))

    return kernel


def make_qkv_norm_rope_pack_fp8_noalloc(dtype=None):
    """make_qkv_norm_rope_pack_fp8_vamax and quantize_fp8_per_head(v_out,
    amax_slots=...) in one call that allocates nothing: V's amax slots live in
    a static array of the library. kernel(q, k, v, q_weight, k_weight, eps,
    cache, positions, q8, k8, v_out, q_descale, k_descale, v8, v_descale) for
    one rank (q/k/v [T, 1, Hs, 128], Hs <= NOALLOC_MAX_HEADS, int64 positions
    on the device: nothing is converted); v8 float8_e4m3fn (or uint8)
    [1, Hs, T, 128], e.g. the S-contiguous view quantize_fp8_per_head(...,
    transposed=True) makes; v_descale fp32 [Hs]. Results bitwise those of the
    two calls. Calls that overlap on one device race on the shared slots.
    No counterpart in the reference: it serves callers that cannot allocate
    (graph capture, fixed serving loops)."""
    _bf16_only(dtype)
    base = make_qkv_norm_rope_pack_fp8()

    def kernel(q, k, v, q_weight, k_weight, eps, cache, positions, q8, k8, v_out, q_descale, k_descale, v8,
               v_descale):
        _ndim(4, q=q, v8=v8)
        _ndim(1, v_descale=v_descale)
        T, P, Hs, D = q.shape
        if P != 1:
            raise ValueError(f"the allocation-free pack takes one rank's heads ([T, 1, Hs, 128]), got P = {P}")
        if Hs > _lib.NOALLOC_MAX_HEADS:
            raise ValueError(f"the allocation-free pack's static slot array holds {_lib.NOALLOC_MAX_HEADS} heads, "
                             f"got {Hs}")
        if positions.dtype != torch.int64:
            raise ValueError("the allocation-free pack takes int64 positions (a conversion would allocate)")
        _lib.check_cuda(q, v8, v_descale)
        if v8.dtype not in (torch.float8_e4m3fn, torch.uint8):
            raise ValueError(f"v8 must be float8_e4m3fn or uint8, got {v8.dtype}")
        _lib.check_dtype(torch.float32, v_descale)
        if tuple(v8.shape) != (1, Hs, T, D) or tuple(v_descale.shape) != (Hs,) or not v_descale.is_contiguous():
            raise ValueError(f"v8 must be [1, {Hs}, {T}, {D}] and v_descale a contiguous fp32 [{Hs}] tensor")
        base(q, k, v, q_weight, k_weight, eps, cache, positions, q8, k8, v_out, q_descale, k_descale,
             _entry="launch_h3_qkv_norm_rope_pack_fp8_noalloc",
             _extra=(_lib.tensor(v8.view(torch.uint8)), _lib.tensor(v_descale)))

    return kernel


def make_qk_norm_rope_interleaved(dtype=None):
    """Per-head RMSNorm then interleaved-pair RoPE over all 128 channels (pair i =
    channels 2i, 2i+1; cos/sin [T, 64]); the rounding steps of make_qk_norm_rope.
    Returns launch(x, weight, eps, cos, sin, out). No counterpart in the
    reference; it serves the 32/48/48 interleaved RoPE layout."""
    _bf16_only(dtype)
    fast = _lib.fast("launch_h3_qk_norm_rope_interleaved", "b4b1s0b2b2b4")

    def launch(x, weight, eps, cos, sin, out):
        status = fast(x, weight, eps, cos, sin, out)
        if status is True:
            return
        _ndim(4, x=x, out=out)
        _ndim(1, weight=weight)
        _ndim(2, cos=cos, sin=sin)
        device = _bf16(x, weight, cos, sin, out)
        _lib.launch_after(status, "launch_h3_qk_norm_rope_interleaved", device, _lib.tensor(x), _lib.tensor(weight),
                          _lib.scalar(eps), _lib.tensor(cos), _lib.tensor(sin), _lib.tensor(out))

    return launch


def make_qk_norm_rope_interleaved_qk(dtype=None):
    """make_qk_norm_rope_interleaved for q and k in one launch (one pass over
    both; the table rows are read once for the two). Returns
    launch(q, k, q_weight, k_weight, eps, cos, sin, q_out, k_out), bitwise equal
    to the two single-tensor launches. No counterpart in the reference."""
    _bf16_only(dtype)
    fast = _lib.fast("launch_h3_qk_norm_rope_interleaved_qk", "b4b4b1b1s0b2b2b4b4")

    def launch(q, k, q_weight, k_weight, eps, cos, sin, q_out, k_out):
        status = fast(q, k, q_weight, k_weight, eps, cos, sin, q_out, k_out)
        if status is True:
            return
        _ndim(4, q=q, k=k, q_out=q_out, k_out=k_out)
        _ndim(1, q_weight=q_weight, k_weight=k_weight)
        _ndim(2, cos=cos, sin=sin)
        device = _bf16(q, k, q_weight, k_weight, cos, sin, q_out, k_out)
        _lib.launch_after(status, "launch_h3_qk_norm_rope_interleaved_qk", device, _lib.tensor(q), _lib.tensor(k),
                          _lib.tensor(q_weight), _lib.tensor(k_weight), _lib.scalar(eps), _lib.tensor(cos),
                          _lib.tensor(sin), _lib.tensor(q_out), _lib.tensor(k_out))

    return launch


def make_rope_cache(caller="torch", output_dir=None, archs=None, block_tokens=64, num_warps=4, dtype=None):
    """H3's RoPE table: position [T, 3] fp64 and power [16] fp32 to cos/sin
    [T, 48] bf16 views (tools/h3_pointwise.py:405-442).
    Returns kernel(position, power, cos, sin)."""
    _bf16_only(dtype)
    fast = _lib.fast("launch_h3_rope_cache", "d2f1b2b2")

    def kernel(position, power, cos, sin):
        status = fast(position, power, cos, sin)
        if status is True:
            return
        _ndim(2, position=position, cos=cos, sin=sin)
        _ndim(1, power=power)
        device = _lib.check_cuda(position, power, cos, sin)
        _lib.check_dtype(torch.float64, position)
        _lib.check_dtype(torch.float32, power)
        _lib.check_dtype(torch.bfloat16, cos, sin)
        _lib.launch_after(status, "launch_h3_rope_cache", device, _lib.tensor(position), _lib.tensor(power),
                          _lib.tensor(cos), _lib.tensor(sin))

    return kernel
