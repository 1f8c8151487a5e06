"""ctypes binding to libh3mi355x.so (the C ABI declared in include/h3mi355x.h).

Tensors cross the boundary as NineToothedTensor {data, shape, strides} with
element strides, scalars as {&double, NULL, NULL}, and every launch goes to the
current torch stream of the tensors' device, mirroring how the reference's
InfiniCore launchers fill the struct (patches/InfiniCore.patch:1062-1089).
There is no fallback: a missing library or a non-zero status raises.

`fast` binds an entry point through the native module _h3call (csrc/h3_call.cpp)
for the plain case of a call; the factories try it first and take the checked
ctypes path below for everything else.
"""
from __future__ import annotations

import ctypes
import functools
import importlib
import warnings
from pathlib import Path
from typing import Sequence

import torch

LIBRARY_PATH = Path(__file__).resolve().parent / "libh3mi355x.so"

# Entry points and their NineToothedTensor argument counts (stream excluded).
ENTRY_POINTS = {
    "launch_h3_full_attention": 5,
    "launch_h3_full_attention_ws": 6,
    "launch_h3_vision_attention_72": 5,
    "launch_h3_attention_planned": 6,
    "launch_h3_full_attention_bf16_prescale": 5,
    "launch_h3_full_attention_fp8": 8,
    "launch_h3_full_attention_fp8pv": 6,
    "launch_h3_quantize_fp8_per_head": 3,
    "launch_h3_quantize_fp8_per_head_slots": 4,
    "launch_h3_quantize_fp8_two_term": 4,
    "launch_h3_full_attention_fp8x2": 10,
    "launch_h3_swiglu_exact": 3,
    "launch_h3_rms_exact": 4,
    "launch_h3_rms_exact_128": 4,
    "launch_h3_rms_exact_5376": 4,
    "launch_h3_rms_modulate_exact": 6,
    "launch_h3_rope_exact": 8,
    "launch_h3_gated_residual_exact": 4,
    "launch_h3_gated_residual_rms_modulate_exact": 9,
    "launch_h3_rms_modulate_indexed": 7,
    "launch_h3_gated_residual_rms_modulate_indexed": 10,
    "launch_h3_gated_residual_indexed": 5,
    "launch_h3_qk_norm_rope": 12,
    "launch_h3_qk_norm_rope_interleaved": 6,
    "launch_h3_qk_norm_rope_interleaved_qk": 9,
    "launch_h3_qkv_norm_rope_pack": 12,
    "launch_h3_qkv_norm_rope_pack_fp8": 14,
    "launch_h3_qkv_norm_rope_pack_fp8_vamax": 15,
    "launch_h3_qkv_norm_rope_pack_fp8x2_vamax": 17,
    "launch_h3_qkv_norm_rope_pack_fp8_noalloc": 16,
    "launch_h3_rope_cache": 4,
    "launch_h3_calibration_stream": 4,
    "launch_h3_calibration_row_copy": 4,
    "launch_h3_calibration_mfma": 3,
    "launch_h3_calibration_mfma_16x16x32": 3,
    "launch_h3_calibration_mfma_fp8": 3,
}

HIP_ERROR_INVALID_VALUE = 1

# Slots per head of a producer-folded amax (H3_AMAX_SLOTS in include/h3mi355x.h).
AMAX_SLOTS = 64
# Heads of the allocation-free pack's static slot array (H3_NOALLOC_MAX_HEADS).
NOALLOC_MAX_HEADS = 1024


class NineToothedTensor(ctypes.Structure):
    _fields_ = [("data", ctypes.c_void_p),
                ("shape", ctypes.POINTER(ctypes.c_uint64)),
                ("strides", ctypes.POINTER(ctypes.c_int64))]


class LaunchError(RuntimeError):
    """A launcher returned a non-zero hipError_t."""

    def __init__(self, name: str, status: int):
        self.status = status
        super().__init__(f"{name} failed with hipError {status} ({_error_string(status)})")


_lib = None
_hip = None


def library() -> ctypes.CDLL:
    """The loaded libh3mi355x.so; raises if it was not built."""
    global _lib
    if _lib is None:
        if not LIBRARY_PATH.exists():
            raise ImportError(f"{LIBRARY_PATH} is missing: build it with __graft_entry__.build() "
                              "(hipcc --offload-arch=gfx950); there is no non-HIP fallback")
        _lib = ctypes.CDLL(str(LIBRARY_PATH))
    return _lib


_bound: dict = {}


def entry(name: str):
    """The typed ctypes function for an entry point (AttributeError if the
    library does not export it)."""
    fn = _bound.get(name)
    if fn is None:
        fn = getattr(library(), name)
        fn.restype = ctypes.c_int
        fn.argtypes = [ctypes.c_void_p] + [NineToothedTensor] * ENTRY_POINTS[name]
        _bound[name] = fn
    return fn


_fast_calls: dict = {}  # the bound calls, one per distinct argument list of `fast`


def _not_taken(*args) -> bool:
    return False


@functools.lru_cache(maxsize=None)
def _call_module():
    """The native module, or None where it is missing, does not load or was built
    against another torch (it reads tensors through that torch's headers): every
    call then goes through ctypes, with the same kernels and about 10 to 30 us
    more host time."""
    try:
        native = importlib.import_module(__package__ + "._h3call")
    except ImportError as e:
        reason = str(e)
    else:
        if native.torch_version == torch.__version__:
            return native
        reason = f"built against torch {native.torch_version}, running {torch.__version__}"
    warnings.warn(f"_h3call.so is not used ({reason}): calls go through ctypes. __graft_entry__.build() builds it.",
                  RuntimeWarning, stacklevel=3)
    return None


def fast(name: str, kinds: str, order: tuple | None = None, fix: tuple | None = None):
    """A callable that calls entry point `name` once when every argument is as
    `kinds` says (csrc/h3_call.cpp: a kind and a rank per argument) and returns
    True, or its status where that is not 0; False if it did not call it. Unless
    True, the ctypes path runs the checks and hands the result on to
    `launch_after`, which raises a status and launches after False. order: the launcher's
    arguments by index of the call's; fix: (argument, dim, size) that must hold.
    Without the library it takes no call, and the ctypes path raises at first
    use; without the native module it takes none, and the ctypes path launches."""
    key = (name, kinds, order, fix)
    bound = _fast_calls.get(key)
    if bound is None:
        if not LIBRARY_PATH.exists():
            return _not_taken
        native = _call_module()
        if native is None:
            return _not_taken
        address = ctypes.cast(getattr(library(), name), ctypes.c_void_p).value
        order = tuple(range(len(kinds) // 2)) if order is None else order
        bound = _fast_calls[key] = functools.partial(native.call, native.plan(address, kinds, order, fix))
    return bound


def _workspace_query(name: str, *sizes: int) -> int:
    fn = _bound.get(name)
    if fn is None:
        fn = getattr(library(), name)
        fn.restype = ctypes.c_int64
        fn.argtypes = [ctypes.c_int64] * len(sizes)
        _bound[name] = fn
    n = int(fn(*sizes))
    if n < 0:
        raise LaunchError(name, 100)
    return n


def attention_workspace_bytes(B: int, H: int, Sq: int, Sk: int) -> int:
    """h3_full_attention_workspace_bytes on the current device (0: no split)."""
    return _workspace_query("h3_full_attention_workspace_bytes", B, H, Sq, Sk)


@functools.lru_cache(maxsize=4096)
def planned_workspace(device_index: int, B: int, H: int, Sq: int, Sk: int, head_dim: int) -> int:
    """attention_planned_workspace_bytes on a device, kept by its sizes."""
    with torch.cuda.device(device_index):
        return attention_planned_workspace_bytes(B, H, Sq, Sk, head_dim)


def attention_planned_workspace_bytes(B: int, H: int, Sq: int, Sk: int, head_dim: int) -> int:
    """h3_attention_planned_workspace_bytes on the current device (0: none used)."""
    return _workspace_query("h3_attention_planned_workspace_bytes", B, H, Sq, Sk, head_dim)


def _error_string(status: int) -> str:
    global _hip
    try:
        if _hip is None:
            _hip = ctypes.CDLL("libamdhip64.so")
            _hip.hipGetErrorString.restype = ctypes.c_char_p
            _hip.hipGetErrorString.argtypes = [ctypes.c_int]
        return _hip.hipGetErrorString(status).decode()
    except OSError:
        return "unknown"


class _Arg:
    """Owns the shape/stride arrays behind one NineToothedTensor."""

    __slots__ = ("struct", "_keep")

    def __init__(self, data: int, shape: Sequence[int], strides: Sequence[int] | None, keep=None):
        if strides is None:
            self._keep = (ctypes.c_double(0.0), keep)
            self.struct = NineToothedTensor(data, None, None)
            return
        n = len(shape)
        shape_arr = (ctypes.c_uint64 * max(n, 1))(*shape)
        stride_arr = (ctypes.c_int64 * max(n, 1))(*strides)
        self._keep = (shape_arr, stride_arr, keep)
        self.struct = NineToothedTensor(data, shape_arr, stride_arr)


def tensor(t: torch.Tensor) -> _Arg:
    return _Arg(t.data_ptr(), tuple(t.shape), tuple(t.stride()), keep=t)


def scalar(value: float) -> _Arg:
    box = ctypes.c_double(float(value))
    arg = _Arg(ctypes.addressof(box), (), None, keep=box)
    return arg


def raw_tensor(data: int, shape: Sequence[int], strides: Sequence[int]) -> _Arg:
    """A NineToothedTensor over raw memory (host-side validation tests)."""
    return _Arg(data, shape, strides)


def call(name: str, stream: int, *args: _Arg) -> int:
    """Calls an entry point and returns its status (no exception)."""
    return entry(name)(ctypes.c_void_p(stream), *(a.struct for a in args))


def launch(name: str, device: torch.device, *args: _Arg) -> None:
    """Calls an entry point on the current stream of `device`; raises on error."""
    with torch.cuda.device(device):
        stream = torch.cuda.current_stream(device).cuda_stream
        status = call(name, stream, *args)
    if status != 0:
        raise LaunchError(name, status)


def launch_after(status: bool | int, name: str, device: torch.device, *args: _Arg) -> None:
    """`launch` of what `fast` did not call (status False); raises the status of
    what it did, without launching again."""
    if status is not False:
        raise LaunchError(name, status)
    launch(name, device, *args)


def check_cuda(*tensors: torch.Tensor) -> torch.device:
    """All tensors on one GPU; returns that device."""
    device = tensors[0].device
    if device.type != "cuda":
        raise ValueError("H3 kernels run on the GPU: tensors must be on a cuda device")
    for t in tensors[1:]:
        if t.device != device:
            raise ValueError(f"all tensors must be on {device}, got {t.device}")
    return device


def check_dtype(dtype: torch.dtype, *tensors: torch.Tensor) -> None:
    for t in tensors:
        if t.dtype != dtype:
            raise ValueError(f"expected {dtype}, got {t.dtype}")
