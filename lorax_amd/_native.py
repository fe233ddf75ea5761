"""ctypes binding of liblorax_hip.so with the call signatures of the reference's pybind
module ``punica_kernels`` (server/punica_kernels/punica_kernels/punica_ops.cc:446-459):
``dispatch_bgmv``, ``sgmv_cutlass``, ``sgmv_shrink`` and ``sgmv_cutlass_tmp_size``.

The functions take torch tensors, perform the checks the reference performs with
TORCH_CHECK (punica_ops.cc:36-43, 291-411) and raise ``RuntimeError`` on any failure.
There is no other implementation behind them: if the shared library is missing every
call raises.
"""

import contextlib
import ctypes
import os
import struct
from pathlib import Path
from typing import Optional

import torch  # noqa: F401  (must be imported first so that its HIP runtime is the one in the process)

LIB_PATH = Path(__file__).resolve().parent / "liblorax_hip.so"

F16, BF16 = 0, 1
ESPACE = 5
EROUTE = 6
A_RH, A_HR = 0, 1
B_RH, B_HR = 0, 1
SHRINK_TMP_BYTES = 8 * 1024 * 1024

_c = ctypes


class BgmvProblem(ctypes.Structure):
    """lorax_bgmv_problem_t of include/lorax_hip.h."""

    _fields_ = [
        ("y", _c.c_void_p),
        ("x", _c.c_void_p),
        ("w_ptrs", _c.c_void_p),
        ("indices", _c.c_void_p),
        ("y_offset", _c.c_int64),
        ("y_stride", _c.c_int64),
        ("h_out", _c.c_int32),
        ("plan", _c.c_void_p),
        ("num_groups", _c.c_int32),
        ("h_in", _c.c_int32),
        ("a_stack", _c.c_void_p),
        ("b_stack", _c.c_void_p),
    ]


class SgmvShrinkProblem(ctypes.Structure):
    """lorax_sgmv_shrink_problem_t of include/lorax_hip.h."""

    _fields_ = [("v", _c.c_void_p), ("w_ptrs", _c.c_void_p)]


class SgmvShrinkGroup(ctypes.Structure):
    """lorax_sgmv_shrink_group_t of include/lorax_hip.h."""

    _fields_ = [("problems", _c.POINTER(SgmvShrinkProblem)), ("num_problems", _c.c_int32), ("r", _c.c_int32),
                ("s_start", _c.c_void_p), ("s_end", _c.c_void_p), ("num_segments", _c.c_int32), ("tiles", _c.c_void_p)]


class SgmvLoraProblem(ctypes.Structure):
    """lorax_sgmv_lora_problem_t of include/lorax_hip.h."""

    _fields_ = [("y", _c.c_void_p), ("a_ptrs", _c.c_void_p), ("b_ptrs", _c.c_void_p), ("y_offset", _c.c_int64),
                ("y_stride", _c.c_int64), ("h_out", _c.c_int32)]


class AdapterEntry(ctypes.Structure):
    """lorax_adapter_entry_t of include/lorax_hip.h."""

    _fields_ = [("adapter", _c.c_int64), ("a_addr", _c.c_int64), ("b_addr", _c.c_int64), ("rank", _c.c_int32),
                ("reserved", _c.c_int32)]


class TableGroup(ctypes.Structure):
    """lorax_table_group_t of include/lorax_hip.h."""

    _fields_ = [("layer_type", _c.c_int32), ("rank", _c.c_int32), ("use_sgmv", _c.c_int32),
                ("num_segments", _c.c_int32), ("num_chunks", _c.c_int32), ("num_long_segments", _c.c_int32),
                ("a_ptr_off", _c.c_int64), ("b_ptr_off", _c.c_int64), ("starts_off", _c.c_int64),
                ("ends_off", _c.c_int64), ("indices_off", _c.c_int64), ("plan_off", _c.c_int64),
                ("shrink_tiles_off", _c.c_int64), ("expand_tiles_off", _c.c_int64),
                ("num_shrink_tiles", _c.c_int32), ("shrink_tile_rows", _c.c_int32),
                ("num_expand_tiles", _c.c_int32), ("expand_tile_rows", _c.c_int32),
                ("segments_id", _c.c_int32), ("num_tokens", _c.c_int32)]


class LayerSlice(ctypes.Structure):
    """lorax_layer_slice_t of include/lorax_hip.h."""

    _fields_ = [("layer_type", _c.c_int32), ("width", _c.c_int32), ("y_offset", _c.c_int64)]


class SgmvTiles(ctypes.Structure):
    """lorax_sgmv_tiles_t of include/lorax_hip.h."""

    _fields_ = [("tiles", _c.c_void_p), ("num_tiles", _c.c_int32), ("tile_rows", _c.c_int32)]


class SgmvExpandProblem(ctypes.Structure):
    """lorax_sgmv_expand_problem_t of include/lorax_hip.h."""

    _fields_ = [("y", _c.c_void_p), ("v", _c.c_void_p), ("w_ptrs", _c.c_void_p), ("s_start", _c.c_void_p),
                ("s_end", _c.c_void_p), ("num_segments", _c.c_int32), ("r", _c.c_int32), ("h_out", _c.c_int32),
                ("y_offset", _c.c_int64), ("y_stride", _c.c_int64), ("tiles", _c.POINTER(SgmvTiles))]


TILES_SHRINK, TILES_EXPAND, TILES_EXPAND_BATCH = 0, 1, 2


class TilePlan:
    """A row-tile plan of an SGMV launch: `records` is an int32 [num_tiles, 4] tensor on the launch's device
    (seg, row0, row_end, index per tile), `tile_rows` the bound of the tiles' heights."""

    __slots__ = ("records", "num_tiles", "tile_rows")

    def __init__(self, records: torch.Tensor, tile_rows: int):
        if records.dtype != torch.int32 or records.dim() != 2 or records.size(1) != 4 or not records.is_contiguous():
            raise RuntimeError("tile records must be a contiguous int32 [num_tiles, 4] tensor")
        self.records = records
        self.num_tiles = records.size(0)
        self.tile_rows = int(tile_rows)

    def c_struct(self, device) -> "SgmvTiles":
        if self.records.device != device:
            raise RuntimeError(f"tile plan on {self.records.device}, launch on {device}")
        # (a plan without tiles has no storage; any non-null address marks it as a plan)
        addr = self.records.data_ptr() if self.num_tiles > 0 else 16
        return SgmvTiles(addr, self.num_tiles, self.tile_rows)


MAX_BGMV_PROBLEMS = 16
MAX_BGMV_TOKENS = 65535  # rows of a BGMV launch and records of one routing plan (capi.hip: bgmv_batch)
MAX_FUSED_BGMV_PROBLEMS = 4

_SIGNATURES = {
    "lorax_bgmv": (
        _c.c_int,
        [_c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_int64, _c.c_int32, _c.c_int32,
         _c.c_int64, _c.c_int64, _c.c_int64, _c.c_float, _c.c_int32, _c.c_void_p],
    ),
    "lorax_bgmv_multi": (
        _c.c_int,
        [_c.c_void_p, _c.c_int32, _c.c_int64, _c.c_int32, _c.c_int64, _c.c_float, _c.c_int32,
         _c.c_int32, _c.c_void_p],
    ),
    "lorax_bgmv_lora_multi": (
        _c.c_int,
        [_c.POINTER(BgmvProblem), _c.c_int32, _c.c_int64, _c.c_int32, _c.c_int32, _c.c_int64, _c.c_float,
         _c.c_int32, _c.c_void_p],
    ),
    "lorax_sgmv_shrink": (
        _c.c_int,
        [_c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_int64,
         _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int64, _c.c_float, _c.c_void_p, _c.c_int64, _c.c_int32,
         _c.c_void_p],
    ),
    "lorax_sgmv_shrink_static": (
        _c.c_int,
        [_c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_int64,
         _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int64, _c.c_float, _c.c_int32, _c.c_void_p],
    ),
    "lorax_sgmv_shrink_multi": (
        _c.c_int,
        [_c.POINTER(SgmvShrinkProblem), _c.c_int32, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_int64,
         _c.c_int32, _c.c_int32, _c.c_int64, _c.c_float, _c.c_int32, _c.c_void_p, _c.c_int64, _c.POINTER(SgmvTiles),
         _c.c_int32, _c.c_void_p],
    ),
    "lorax_sgmv_shrink_groups": (
        _c.c_int,
        [_c.POINTER(SgmvShrinkGroup), _c.c_int32, _c.c_void_p, _c.c_int64, _c.c_int32, _c.c_int64, _c.c_float, _c.c_int32,
         _c.c_void_p, _c.c_int64, _c.c_int32, _c.c_void_p],
    ),
    "lorax_sgmv_shrink_groups_parts": (
        _c.c_int,
        [_c.POINTER(SgmvShrinkGroup), _c.c_int32, _c.c_void_p, _c.c_int64, _c.c_int32, _c.c_int64, _c.c_int32, _c.c_void_p,
         _c.c_int64, _c.c_int32],
    ),
    "lorax_sgmv_shrink_groups_parts_of": (
        _c.c_int,
        [_c.POINTER(SgmvShrinkGroup), _c.c_int32, _c.c_void_p, _c.c_int64, _c.c_int32, _c.c_int64, _c.c_int32, _c.c_void_p,
         _c.c_int64, _c.c_int32, _c.c_void_p],
    ),
    "lorax_sgmv_expand_planned": (
        _c.c_int,
        [_c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_int64, _c.c_int32,
         _c.c_int32, _c.c_int64, _c.c_int64, _c.c_int64, _c.c_int32, _c.POINTER(SgmvTiles), _c.c_int32, _c.c_void_p],
    ),
    "lorax_sgmv_expand_multi": (
        _c.c_int,
        [_c.POINTER(SgmvExpandProblem), _c.c_int32, _c.c_int64, _c.c_int64, _c.c_int32, _c.c_int32, _c.c_void_p],
    ),
    "lorax_sgmv_plan_tiles": (
        _c.c_int,
        [_c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_int64, _c.c_int32, _c.c_int32, _c.c_void_p, _c.c_int32,
         _c.POINTER(_c.c_int32), _c.POINTER(_c.c_int32)],
    ),
    "lorax_set_fixed_order_shrink": (_c.c_int, [_c.c_int32]),
    "lorax_sgmv_lora_multi": (
        _c.c_int,
        [_c.POINTER(SgmvLoraProblem), _c.c_int32, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_int64,
         _c.c_int32, _c.c_int32, _c.c_int64, _c.c_float, _c.c_int32, _c.c_void_p],
    ),
    "lorax_sgmv_expand": (
        _c.c_int,
        [_c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_int64,
         _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int64, _c.c_int64, _c.c_int64, _c.c_int32, _c.c_void_p,
         _c.c_int64, _c.c_int32, _c.c_void_p],
    ),
    "lorax_sgmv_tmp_size": (_c.c_size_t, [_c.c_int32]),
    "lorax_build_batch_tables": (
        _c.c_int,
        [_c.c_void_p, _c.c_int64, _c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_int32, _c.c_void_p, _c.c_void_p,
         _c.POINTER(_c.c_int32), _c.c_void_p, _c.c_int64, _c.POINTER(_c.c_int64), _c.POINTER(TableGroup), _c.c_int32,
         _c.POINTER(_c.c_int32)],
    ),
    "lorax_decode_in_one_launch": (_c.c_int, [_c.c_void_p, _c.c_int32, _c.c_int64, _c.c_int32]),
    "lorax_shrink_summed_rank": (_c.c_int, [_c.c_void_p, _c.c_int32, _c.c_int64, _c.c_int32]),
    "lorax_prefill_in_one_launch": (_c.c_int, [_c.c_int32, _c.c_int32, _c.c_int64, _c.c_int32]),
    "lorax_layer_update": (
        _c.c_int,
        [_c.c_void_p, _c.c_int32, _c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_void_p, _c.c_int64, _c.c_void_p, _c.c_int64,
         _c.c_int32, _c.c_int64, _c.c_void_p, _c.c_int64, _c.c_void_p, _c.c_int64, _c.c_int32, _c.c_int32, _c.c_void_p],
    ),
    "lorax_stacked_update": (
        _c.c_int,
        [_c.c_void_p, _c.c_int32, _c.c_void_p, _c.c_int32, _c.c_void_p, _c.c_int64, _c.c_void_p, _c.c_int64, _c.c_int32,
         _c.c_void_p, _c.c_int64, _c.c_int32, _c.c_int32, _c.c_void_p],
    ),
    "lorax_init": (_c.c_int, [_c.c_int32]),
    "lorax_workspace_bytes": (_c.c_size_t, []),
    "lorax_last_error": (_c.c_char_p, []),
    "lorax_version": (_c.c_char_p, []),
}

EXPORTED_SYMBOLS = tuple(_SIGNATURES)

_lib: Optional[ctypes.CDLL] = None
_load_error: Optional[str] = None
_initialised_devices = set()


def _load() -> Optional[ctypes.CDLL]:
    global _lib, _load_error
    if _lib is not None or _load_error is not None:
        return _lib
    path = os.environ.get("LORAX_HIP_LIBRARY", str(LIB_PATH))
    try:
        lib = ctypes.CDLL(path)
        for name, (restype, argtypes) in _SIGNATURES.items():
            fn = getattr(lib, name)
            fn.restype = restype
            fn.argtypes = argtypes
        _lib = lib
    except (OSError, AttributeError) as exc:
        _load_error = f"{path}: {exc}"
    return _lib


def available() -> bool:
    """True iff liblorax_hip.so is loaded with every expected symbol."""
    return _load() is not None


def load_error() -> Optional[str]:
    _load()
    return _load_error


def lib() -> ctypes.CDLL:
    handle = _load()
    if handle is None:
        raise RuntimeError(
            f"liblorax_hip.so is not available ({_load_error}); build it with `python -m lorax_amd.build`. "
            "There is no non-HIP implementation of the LoRA kernels in this package."
        )
    return handle


def version() -> str:
    return lib().lorax_version().decode()


def _raise_last(rc: int):
    msg = lib().lorax_last_error().decode() or f"error code {rc}"
    raise RuntimeError(msg)


def init(device) -> None:
    """lorax_init: per-device set-up of the library (idempotent; call it outside graph capture)."""
    index = torch.device(device).index
    if index is None:
        index = torch.cuda.current_device()
    if index in _initialised_devices:
        return
    rc = lib().lorax_init(index)
    if rc != 0:
        _raise_last(rc)
    _initialised_devices.add(index)


def _ready(t: torch.Tensor) -> None:
    """init() for t's device unless it has been done or the stream is capturing (the launches then do what is missing)."""
    if t.get_device() not in _initialised_devices and not torch.cuda.is_current_stream_capturing():
        init(t.device)


_DTYPE_CODES = {torch.float16: F16, torch.bfloat16: BF16}


def _dtype_code(t: torch.Tensor) -> int:
    return _DTYPE_CODES.get(t.dtype, -1)


def _check_input(t: torch.Tensor, name: str, dim: int) -> None:
    if not isinstance(t, torch.Tensor):
        raise RuntimeError(f"{name} must be a torch.Tensor")
    if not t.is_cuda:
        raise RuntimeError(f"{name} must be a CUDA tensor")
    if not t.is_contiguous():
        raise RuntimeError(f"{name} must be contiguous")
    if t.dim() != dim:
        raise RuntimeError(f"{name} must be a {dim}D tensor")


# torch's own accessors build a Stream object and a guard object per call, 2 to 3 us each; these are the calls beneath.
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_current_device = getattr(torch._C, "_cuda_getDevice", None)
_unguarded = contextlib.nullcontext()


def _stream(t: torch.Tensor) -> int:
    if _raw_stream is not None:
        return _raw_stream(t.get_device())
    return torch.cuda.current_stream(t.device).cuda_stream


def _on_device(t: torch.Tensor):
    """Context in which t's device is the current one."""
    if _current_device is not None and _current_device() == t.get_device():
        return _unguarded
    return torch.cuda.device(t.device)


def _check_same(y: torch.Tensor, x: torch.Tensor, *rest: torch.Tensor) -> None:
    if y.dtype != x.dtype:
        raise RuntimeError(f"y and x must share one dtype, got {y.dtype} and {x.dtype}")
    for t in rest:
        if t.device != x.device:
            raise RuntimeError(f"all tensors must be on one device, got {t.device} and {x.device}")
    if y.device != x.device:
        raise RuntimeError(f"all tensors must be on one device, got {y.device} and {x.device}")


def sgmv_cutlass_tmp_size(num_problems: int) -> int:
    """sgmv_tmp_size, sgmv/sgmv_cutlass.cuh:54-58."""
    return int(lib().lorax_sgmv_tmp_size(int(num_problems)))


def bgmv(y, x, w_ptr, indicies, layer_idx, scale, y_offset=0, y_slice_size=None) -> None:
    """lorax_bgmv with an optional column window [y_offset, y_offset + y_slice_size) of y."""
    _check_input(y, "y", 2)
    _check_input(x, "x", 2)
    _check_input(w_ptr, "w_ptr", 1)
    _check_input(indicies, "indicies", 1)
    _check_same(y, x, w_ptr, indicies)
    if w_ptr.dtype != torch.int64 or indicies.dtype != torch.int64:
        raise RuntimeError("w_ptr and indicies must be int64 tensors")
    if indicies.size(0) != x.size(0):
        raise RuntimeError(f"CHECK_EQ(indicies.size(0), x.size(0)) failed. {indicies.size(0)} vs {x.size(0)}")
    if y.size(0) != x.size(0):
        raise RuntimeError(f"CHECK_EQ(y.size(0), x.size(0)) failed. {y.size(0)} vs {x.size(0)}")
    h_out = y.size(1) if y_slice_size is None else int(y_slice_size)
    with _on_device(x):
        rc = lib().lorax_bgmv(
            y.data_ptr(), x.data_ptr(), w_ptr.data_ptr(), indicies.data_ptr(), x.size(0), x.size(1), h_out,
            int(y_offset), y.size(1), int(layer_idx), float(scale), _dtype_code(x), _stream(x),
        )
    if rc != 0:
        _raise_last(rc)


PLAN_RECORD_WORDS = 8


def bgmv_multi(problems, layer_idx, scale=1.0, accumulate=True, plans=None) -> None:
    """lorax_bgmv_multi: `problems` is a list of up to 16 tuples (y, x, w_ptr, indicies, y_offset, y_slice_size)
    that share the token count and the direction; shrink problems share x.shape and may differ in rank
    (y's width), expand problems may differ in rank (x's width) and output width.  y_slice_size None means
    the whole width of y.
    `plans`, if given, holds one routing plan per problem: an int64 device tensor [num_groups, 8]; w_ptr and
    indicies of a planned problem may then be None (the kernels read the plan only).  Plans over stacked weights:
    bgmv_stacked."""
    if not 1 <= len(problems) <= MAX_BGMV_PROBLEMS:
        raise RuntimeError(f"between 1 and {MAX_BGMV_PROBLEMS} problems per launch, got {len(problems)}")
    arr = (BgmvProblem * len(problems))()
    x0 = problems[0][1]
    for i, (y, x, w_ptr, indicies, y_offset, y_slice_size) in enumerate(problems):
        _check_input(y, "y", 2)
        _check_input(x, "x", 2)
        planned_only = plans is not None and w_ptr is None and indicies is None  # the plan holds the routing
        if planned_only:
            _check_same(y, x)
        else:
            _check_input(w_ptr, "w_ptr", 1)
            _check_input(indicies, "indicies", 1)
            _check_same(y, x, w_ptr, indicies)
            if w_ptr.dtype != torch.int64 or indicies.dtype != torch.int64:
                raise RuntimeError("w_ptr and indicies must be int64 tensors")
        if x.size(0) != x0.size(0) or x.dtype != x0.dtype or x.device != x0.device:
            raise RuntimeError("all problems of one launch must have inputs of one row count, dtype and device")
        if (not planned_only and indicies.size(0) != x.size(0)) or y.size(0) != x.size(0):
            raise RuntimeError(
                f"CHECK_EQ(indicies.size(0), x.size(0)) / CHECK_EQ(y.size(0), x.size(0)) failed. "
                f"{'-' if planned_only else indicies.size(0)}, {y.size(0)} vs {x.size(0)}"
            )
        h_out = y.size(1) if y_slice_size is None else int(y_slice_size)
        plan_ptr, num_groups = None, 0
        if plans is not None:
            plan = plans[i]
            _check_input(plan, "plan", 2)
            if plan.dtype != torch.int64 or plan.size(1) != PLAN_RECORD_WORDS or plan.device != x.device:
                raise RuntimeError(f"plan must be an int64 [num_groups, {PLAN_RECORD_WORDS}] tensor on the device of x")
            plan_ptr, num_groups = plan.data_ptr(), plan.size(0)
            if num_groups == 0:
                plan_ptr = x.data_ptr()  # an empty plan has no storage; any non-null address will do
        arr[i] = BgmvProblem(y.data_ptr(), x.data_ptr(), None if planned_only else w_ptr.data_ptr(),
                             None if planned_only else indicies.data_ptr(), int(y_offset),
                             y.size(1), h_out, plan_ptr, num_groups, x.size(1), None, None)
    with _on_device(x0):
        rc = lib().lorax_bgmv_multi(arr, len(problems), x0.size(0), x0.size(1), int(layer_idx), float(scale),
                                    1 if accumulate else 0, _dtype_code(x0), _stream(x0))
    if rc != 0:
        _raise_last(rc)


# BgmvProblem for struct.pack: ctypes takes 1.5 us to fill one
_BGMV_PROBLEM = "4Q2qi4xQ2i2Q"
assert struct.calcsize(_BGMV_PROBLEM) == ctypes.sizeof(BgmvProblem)


def bgmv_stacked(y, x, jobs, plan, scale=1.0) -> None:
    """The planned shrink launch and the planned expand launch (lorax_bgmv_multi) of up to 16 projections over stacked
    weights: `jobs` holds (lora_a [n, r, h_in], lora_b [n, width, r], r, y_offset, width) per projection, `plan` is the
    batch's routing plan over stack entries.  The operands are checked once for both launches."""
    if not 1 <= len(jobs) <= MAX_BGMV_PROBLEMS:
        raise RuntimeError(f"between 1 and {MAX_BGMV_PROBLEMS} problems per launch, got {len(jobs)}")
    _check_input(y, "y", 2)
    _check_input(x, "x", 2)
    _check_input(plan, "plan", 2)
    _check_same(y, x, plan)
    if plan.dtype != torch.int64 or plan.size(1) != PLAN_RECORD_WORDS:
        raise RuntimeError(f"plan must be an int64 [num_groups, {PLAN_RECORD_WORDS}] tensor on the device of x")
    rows, h_in = x.shape
    y_rows, y_stride = y.shape
    if y_rows != rows:
        raise RuntimeError(f"CHECK_EQ(y.size(0), x.size(0)) failed. {y_rows} vs {rows}")
    groups = plan.size(0)
    x_ptr, y_ptr = x.data_ptr(), y.data_ptr()
    plan_ptr = plan.data_ptr() if groups > 0 else x_ptr  # an empty plan has no storage; any non-null address will do
    v = torch.empty((rows * sum(r for _, _, r, _, _ in jobs),), dtype=x.dtype, device=x.device)
    v_ptr = v.data_ptr()
    shrink, expand = [], []
    for a, b, r, y_offset, width in jobs:
        _check_stack(a, x)
        _check_stack(b, x)
        shrink += (v_ptr, x_ptr, 0, 0, 0, r, r, plan_ptr, groups, h_in, a.data_ptr(), 0)
        expand += (y_ptr, v_ptr, 0, 0, y_offset, y_stride, width, plan_ptr, groups, r, 0, b.data_ptr())
        v_ptr += rows * r * 2
    layout = struct.Struct(_BGMV_PROBLEM * len(jobs))
    shrink, expand = layout.pack(*shrink), layout.pack(*expand)
    code, stream = _dtype_code(x), _stream(x)
    with _on_device(x):
        launch = lib().lorax_bgmv_multi
        rc = launch(shrink, len(jobs), rows, h_in, 0, scale, 0, code, stream)
        if rc == 0:
            rc = launch(expand, len(jobs), rows, jobs[0][2], 0, 1.0, 1, code, stream)
    if rc != 0:
        _raise_last(rc)


_DECODE_JOB = struct.Struct("3i")  # lorax_decode_job_t


def decode_in_one_launch(jobs, num_tokens: int, h_in: int) -> bool:
    """lorax_decode_in_one_launch: whether a decode batch's projections go out as single-launch updates (bgmv_lora_multi, one
    per rank) rather than as a shrink and an expand launch.  `jobs`: (rank, columns, routing records) per projection."""
    packed = b"".join([_DECODE_JOB.pack(*job) for job in jobs])
    return lib().lorax_decode_in_one_launch(packed, len(jobs), num_tokens, h_in) != 0


_SHRINK_PLAN = struct.Struct("4i")  # lorax_shrink_plan_t


def shrink_summed_rank(groups, num_tokens: int, h_in: int) -> int:
    """lorax_shrink_summed_rank: the summed rank up to which projections go to sgmv_shrink_groups as one group.  `groups`:
    (rank, projections, TilePlan or None) per rank group of the call that has rows for the segment kernels."""
    packed = b"".join([_SHRINK_PLAN.pack(r, n, tiles.num_tiles if tiles is not None else 0, tiles.tile_rows if tiles is not None else 0)
                       for r, n, tiles in groups])
    return lib().lorax_shrink_summed_rank(packed, len(groups), num_tokens, h_in)


def bgmv_lora_fits(rank: int, h_in: int, h_out: int) -> bool:
    """True where the single-launch shrink+expand (lorax_bgmv_lora_multi) is the better choice whatever the batch: the
    adapter's A slab is small and one workgroup covers all output columns of the projection."""
    return decode_in_one_launch([(rank, h_out, MAX_BGMV_TOKENS)], MAX_BGMV_TOKENS, h_in)


def _check_stack(stack, x) -> None:
    if not isinstance(stack, torch.Tensor) or stack.dim() != 3 or not stack.is_contiguous() or stack.dtype != x.dtype \
            or stack.device != x.device:
        raise RuntimeError("stacked weights must be a contiguous [num_adapters, rows, cols] tensor of the input's "
                           "dtype on its device")


def bgmv_lora_multi(problems, rank, layer_idx, scale=1.0, stacks=None) -> None:
    """lorax_bgmv_lora_multi: `problems` is a list of up to 4 tuples (y, x, plan, y_offset, y_slice_size) that
    share x.shape; y[:, window] += (x @ A^T) @ B^T per planned token chunk, rank 8 or 16.
    `stacks`: per problem a pair (lora_a [num_adapters, r, h_in], lora_b [num_adapters, h_out, r]) of stacked weight
    tensors; the plan's address words then hold entry numbers and layer_idx must be 0."""
    if not 1 <= len(problems) <= MAX_FUSED_BGMV_PROBLEMS:
        raise RuntimeError(f"between 1 and {MAX_FUSED_BGMV_PROBLEMS} problems per launch, got {len(problems)}")
    arr = (BgmvProblem * len(problems))()
    x0 = problems[0][1]
    for i, (y, x, plan, y_offset, y_slice_size) in enumerate(problems):
        _check_input(y, "y", 2)
        _check_input(x, "x", 2)
        _check_input(plan, "plan", 2)
        _check_same(y, x, plan)
        if x.shape != x0.shape or x.dtype != x0.dtype or x.device != x0.device:
            raise RuntimeError("all problems of one launch must have inputs of one shape, dtype and device")
        if y.size(0) != x.size(0):
            raise RuntimeError(f"CHECK_EQ(y.size(0), x.size(0)) failed. {y.size(0)} vs {x.size(0)}")
        if plan.dtype != torch.int64 or plan.size(1) != PLAN_RECORD_WORDS:
            raise RuntimeError(f"plan must be an int64 [num_groups, {PLAN_RECORD_WORDS}] tensor on the device of x")
        h_out = y.size(1) if y_slice_size is None else int(y_slice_size)
        plan_ptr = plan.data_ptr() if plan.size(0) > 0 else x.data_ptr()
        a_stack = b_stack = None
        if stacks is not None:
            if int(layer_idx) != 0:
                raise RuntimeError("stacked weights hold one layer: layer_idx must be 0")
            _check_stack(stacks[i][0], x)
            _check_stack(stacks[i][1], x)
            if stacks[i][0].shape[1:] != (rank, x.size(1)) or stacks[i][1].shape[1:] != (h_out, rank):
                raise RuntimeError(f"stacked weights of problem {i} do not have the shapes [n, {rank}, {x.size(1)}] "
                                   f"and [n, {h_out}, {rank}]")
            a_stack, b_stack = stacks[i][0].data_ptr(), stacks[i][1].data_ptr()
        arr[i] = BgmvProblem(y.data_ptr(), x.data_ptr(), None, None, int(y_offset), y.size(1), h_out, plan_ptr,
                             plan.size(0), 0, a_stack, b_stack)
    with _on_device(x0):
        rc = lib().lorax_bgmv_lora_multi(arr, len(problems), x0.size(0), x0.size(1), int(rank), int(layer_idx),
                                         float(scale), _dtype_code(x0), _stream(x0))
    if rc != 0:
        _raise_last(rc)


def dispatch_bgmv(y, x, w_ptr, indicies, layer_idx, scale) -> None:
    """dispatch_bgmv, punica_ops.cc:291-334."""
    bgmv(y, x, w_ptr, indicies, layer_idx, scale)


def _check_sgmv(y, x, w_ptr, s_start, s_end, tmp) -> None:
    _check_input(y, "y", 2)
    _check_input(x, "x", 2)
    _check_input(w_ptr, "w_ptr", 1)
    _check_input(s_start, "s_start", 1)
    _check_input(s_end, "s_end", 1)
    _check_input(tmp, "tmp", 1)
    _check_same(y, x, w_ptr, s_start, s_end, tmp)
    if w_ptr.dtype != torch.int64:
        raise RuntimeError("w_ptr must be an int64 tensor")
    if s_start.dtype != torch.int32 or s_end.dtype != torch.int32:
        raise RuntimeError("s_start and s_end must be int32 tensors")
    if not (w_ptr.size(0) == s_start.size(0) == s_end.size(0)):
        raise RuntimeError(
            f"w_ptr, s_start and s_end must have one entry per segment, got {w_ptr.size(0)}, "
            f"{s_start.size(0)}, {s_end.size(0)}"
        )
    if y.size(0) != x.size(0):
        raise RuntimeError(f"CHECK_EQ(y.size(0), x.size(0)) failed. {y.size(0)} vs {x.size(0)}")


def sgmv_expand(y, x, w_ptr, s_start, s_end, tmp, layer_idx, y_offset=0, y_slice_size=None,
                transposed: bool = False, accumulate: bool = True, tiles: Optional[TilePlan] = None) -> None:
    """lorax_sgmv_expand with an optional column window of y.  `transposed`: w_ptr addresses [L, h_out, r]
    stacks (B^T) instead of the reference's [L, r, h_out].  accumulate=False overwrites the segments' rows.
    `tiles`: a row-tile plan of the segment tables (transposed stacks only: lorax_sgmv_expand_planned)."""
    _check_sgmv(y, x, w_ptr, s_start, s_end, tmp)
    h_out = y.size(1) if y_slice_size is None else int(y_slice_size)
    if tiles is not None and transposed:
        plan = tiles.c_struct(x.device)
        with _on_device(x):
            rc = lib().lorax_sgmv_expand_planned(
                y.data_ptr(), x.data_ptr(), w_ptr.data_ptr(), s_start.data_ptr(), s_end.data_ptr(), s_start.size(0),
                x.size(0), x.size(1), h_out, int(y_offset), y.size(1), int(layer_idx), 1 if accumulate else 0,
                ctypes.byref(plan), _dtype_code(x), _stream(x),
            )
        if rc != 0:
            _raise_last(rc)
        return
    with _on_device(x):
        rc = lib().lorax_sgmv_expand(
            y.data_ptr(), x.data_ptr(), w_ptr.data_ptr(), s_start.data_ptr(), s_end.data_ptr(), s_start.size(0),
            x.size(0), x.size(1), h_out, B_HR if transposed else B_RH, int(y_offset), y.size(1), int(layer_idx),
            1 if accumulate else 0, tmp.data_ptr(),
            tmp.numel() * tmp.element_size(), _dtype_code(x), _stream(x),
        )
    if rc != 0:
        _raise_last(rc)


MAX_SGMV_EXPAND_PROBLEMS = 16


def sgmv_expand_multi(problems, layer_idx, accumulate: bool = True) -> None:
    """lorax_sgmv_expand_multi: up to 16 expands over transposed stacks in one launch.  `problems` is a list of tuples
    (y, v, w_ptr, s_start, s_end, y_offset, y_slice_size, tiles) of one row count, dtype and device whose elements of y
    are disjoint; ranks (v's width) may differ, tiles is a row-tile plan or None."""
    if not 1 <= len(problems) <= MAX_SGMV_EXPAND_PROBLEMS:
        raise RuntimeError(f"between 1 and {MAX_SGMV_EXPAND_PROBLEMS} problems per launch, got {len(problems)}")
    arr = (SgmvExpandProblem * len(problems))()
    v0 = problems[0][1]
    plans = []  # keeps the host structs alive until the call has read them
    for i, (y, v, w_ptr, s_start, s_end, y_offset, y_slice_size, tiles) in enumerate(problems):
        _check_sgmv(y, v, w_ptr, s_start, s_end, s_start)
        if v.size(0) != v0.size(0) or v.dtype != v0.dtype or v.device != v0.device:
            raise RuntimeError("all problems of one launch must have inputs of one row count, dtype and device")
        plan = None
        if tiles is not None:
            plans.append(tiles.c_struct(v.device))
            plan = ctypes.pointer(plans[-1])
        h_out = y.size(1) if y_slice_size is None else int(y_slice_size)
        arr[i] = SgmvExpandProblem(y.data_ptr(), v.data_ptr(), w_ptr.data_ptr(), s_start.data_ptr(), s_end.data_ptr(),
                                   s_start.size(0), v.size(1), h_out, int(y_offset), y.size(1), plan)
    with _on_device(v0):
        rc = lib().lorax_sgmv_expand_multi(arr, len(problems), v0.size(0), int(layer_idx), 1 if accumulate else 0,
                                           _dtype_code(v0), _stream(v0))
    if rc != 0:
        _raise_last(rc)


def _sgmv_shrink(y, x, w_ptr, s_start, s_end, tmp, layer_idx, a_layout, scale: float = 1.0) -> None:
    _check_sgmv(y, x, w_ptr, s_start, s_end, tmp)
    _ready(x)
    with _on_device(x):
        rc = lib().lorax_sgmv_shrink(
            y.data_ptr(), x.data_ptr(), w_ptr.data_ptr(), s_start.data_ptr(), s_end.data_ptr(), s_start.size(0),
            x.size(0), x.size(1), y.size(1), a_layout, int(layer_idx), float(scale), tmp.data_ptr(),
            tmp.numel() * tmp.element_size(), _dtype_code(x), _stream(x),
        )
    if rc != 0:
        _raise_last(rc)


def sgmv_cutlass(y, x, w_ptr, s_start, s_end, tmp, layer_idx) -> None:
    """dispatch_sgmv_cutlass, punica_ops.cc:338-367: weights are [L, d_in, d_out]; d_in < d_out is the
    expand configuration, anything else the shrink one (sgmv_cutlass.cuh:86,132)."""
    if isinstance(x, torch.Tensor) and isinstance(y, torch.Tensor) and x.dim() == 2 and y.dim() == 2:
        if x.size(1) < y.size(1):
            return sgmv_expand(y, x, w_ptr, s_start, s_end, tmp, layer_idx)
    return _sgmv_shrink(y, x, w_ptr, s_start, s_end, tmp, layer_idx, A_HR)


def sgmv_shrink(y, x, w_ptr, s_start, s_end, tmp, layer_idx, scale: float = 1.0) -> None:
    """dispatch_sgmv_shrink, punica_ops.cc:369-411: weights are [L, d_out, d_in], tmp is 8 MiB of uint8.
    `scale` (not in the reference's binding) multiplies the sums before they are rounded."""
    if isinstance(tmp, torch.Tensor) and tmp.dtype != torch.uint8:
        raise RuntimeError(f"CHECK_EQ(tmp.scalar_type(), at::ScalarType::Byte) failed. {tmp.dtype}")
    return _sgmv_shrink(y, x, w_ptr, s_start, s_end, tmp, layer_idx, A_RH, scale)


def sgmv_shrink_static(y, x, w_ptr, s_start, s_end, layer_idx, a_layout=A_RH, scale: float = 1.0) -> None:
    """lorax_sgmv_shrink_static: sgmv_shrink / the shrink direction of sgmv_cutlass without a tmp tensor; the
    library's own static device array serves as split-K scratch, so the call allocates nothing."""
    _check_sgmv(y, x, w_ptr, s_start, s_end, s_start)
    with _on_device(x):
        rc = lib().lorax_sgmv_shrink_static(
            y.data_ptr(), x.data_ptr(), w_ptr.data_ptr(), s_start.data_ptr(), s_end.data_ptr(), s_start.size(0),
            x.size(0), x.size(1), y.size(1), a_layout, int(layer_idx), float(scale), _dtype_code(x), _stream(x),
        )
    if rc != 0:
        _raise_last(rc)


MAX_SGMV_SHRINK_PROBLEMS = 4


def sgmv_shrink_multi(ys, x, w_ptrs, s_start, s_end, tmp, layer_idx, scale: float = 1.0,
                      accumulate: bool = True, tiles: Optional[TilePlan] = None) -> None:
    """lorax_sgmv_shrink_multi: sgmv_shrink for up to 4 projections (outputs `ys`, pointer tables `w_ptrs`) that
    share x, the segment tables and the rank; one launch that reads x once where the kernels allow it.
    accumulate=False overwrites the rows of the segments (no zero-fill of the outputs needed).
    `tiles`: a row-tile plan of the segment tables (plan_tiles, or the batch tables' own)."""
    if not 1 <= len(ys) <= MAX_SGMV_SHRINK_PROBLEMS or len(ys) != len(w_ptrs):
        raise RuntimeError(f"between 1 and {MAX_SGMV_SHRINK_PROBLEMS} outputs with one pointer table each")
    if isinstance(tmp, torch.Tensor) and tmp.dtype != torch.uint8:
        raise RuntimeError(f"CHECK_EQ(tmp.scalar_type(), at::ScalarType::Byte) failed. {tmp.dtype}")
    arr = (SgmvShrinkProblem * len(ys))()
    for i, (y, w_ptr) in enumerate(zip(ys, w_ptrs)):
        _check_sgmv(y, x, w_ptr, s_start, s_end, tmp)
        if y.size(1) != ys[0].size(1):
            raise RuntimeError("the projections of one call share the rank")
        arr[i] = SgmvShrinkProblem(y.data_ptr(), w_ptr.data_ptr())
    _ready(x)
    plan = tiles.c_struct(x.device) if tiles is not None else None
    with _on_device(x):
        rc = lib().lorax_sgmv_shrink_multi(
            arr, len(ys), x.data_ptr(), s_start.data_ptr(), s_end.data_ptr(), s_start.size(0), x.size(0), x.size(1),
            ys[0].size(1), int(layer_idx), float(scale), 1 if accumulate else 0, tmp.data_ptr(),
            tmp.numel() * tmp.element_size(), ctypes.byref(plan) if plan is not None else None, _dtype_code(x),
            _stream(x),
        )
    if rc != 0:
        _raise_last(rc)


MAX_SGMV_SHRINK_GROUPS = 16


def _shrink_groups(groups, x, tmp):
    """The C descriptors of `groups`, checked, and what they point to."""
    if not 1 <= len(groups) <= MAX_SGMV_SHRINK_GROUPS:
        raise RuntimeError(f"between 1 and {MAX_SGMV_SHRINK_GROUPS} groups per call, got {len(groups)}")
    if isinstance(tmp, torch.Tensor) and tmp.dtype != torch.uint8:
        raise RuntimeError(f"CHECK_EQ(tmp.scalar_type(), at::ScalarType::Byte) failed. {tmp.dtype}")
    arr, keep = (SgmvShrinkGroup * len(groups))(), []
    for i, (ys, w_ptrs, s_start, s_end, tiles) in enumerate(groups):
        if not 1 <= len(ys) <= MAX_SGMV_SHRINK_PROBLEMS or len(ys) != len(w_ptrs):
            raise RuntimeError(f"between 1 and {MAX_SGMV_SHRINK_PROBLEMS} outputs with one pointer table each")
        problems = (SgmvShrinkProblem * len(ys))()
        for k, (y, w_ptr) in enumerate(zip(ys, w_ptrs)):
            _check_sgmv(y, x, w_ptr, s_start, s_end, tmp)
            if y.size(1) != ys[0].size(1):
                raise RuntimeError("the projections of one group share the rank")
            problems[k] = SgmvShrinkProblem(y.data_ptr(), w_ptr.data_ptr())
        plan = tiles.c_struct(x.device) if tiles is not None else None
        keep.append((problems, plan))
        arr[i] = SgmvShrinkGroup(problems, len(ys), ys[0].size(1), s_start.data_ptr(), s_end.data_ptr(), s_start.size(0),
                                 ctypes.addressof(plan) if plan is not None else None)
    return arr, keep


def sgmv_shrink_groups(groups, x, tmp, layer_idx, scale: float = 1.0, accumulate: bool = True) -> None:
    """lorax_sgmv_shrink_groups: sgmv_shrink_multi for up to 16 groups over the same x, in one launch where they qualify.
    `groups` is a list of tuples (ys, w_ptrs, s_start, s_end, tiles) as sgmv_shrink_multi takes them."""
    arr, _keep = _shrink_groups(groups, x, tmp)
    _ready(x)
    with _on_device(x):
        rc = lib().lorax_sgmv_shrink_groups(arr, len(groups), x.data_ptr(), x.size(0), x.size(1), int(layer_idx), float(scale),
                                            1 if accumulate else 0, tmp.data_ptr(), tmp.numel() * tmp.element_size(),
                                            _dtype_code(x), _stream(x))
    if rc != 0:
        _raise_last(rc)


def sgmv_shrink_groups_parts(groups, x, tmp, layer_idx, accumulate: bool = True) -> int:
    """lorax_sgmv_shrink_groups_parts: the parts of the hidden dimension that sgmv_shrink_groups cuts for these arguments, 0
    where it issues one call per group."""
    arr, _keep = _shrink_groups(groups, x, tmp)
    return lib().lorax_sgmv_shrink_groups_parts(arr, len(groups), x.data_ptr(), x.size(0), x.size(1), int(layer_idx),
                                                1 if accumulate else 0, tmp.data_ptr(), tmp.numel() * tmp.element_size(),
                                                _dtype_code(x))


def sgmv_shrink_groups_parts_of(groups, x, tmp, layer_idx, accumulate: bool = True) -> list:
    """lorax_sgmv_shrink_groups_parts_of: those parts of every group, 0 = it has no tiles; empty where the call goes out group by
    group."""
    arr, _keep = _shrink_groups(groups, x, tmp)
    parts = (_c.c_int32 * len(groups))()
    together = lib().lorax_sgmv_shrink_groups_parts_of(arr, len(groups), x.data_ptr(), x.size(0), x.size(1), int(layer_idx),
                                                       1 if accumulate else 0, tmp.data_ptr(), tmp.numel() * tmp.element_size(),
                                                       _dtype_code(x), parts)
    return list(parts) if together > 0 else []


def plan_tiles(s_start, s_end, num_tokens: int, kind: int, rank: int = 0):
    """lorax_sgmv_plan_tiles on host copies of the segment tables (sequences of int): returns (records as a numpy
    int32 [num_tiles, 4] array, tile_rows).  `rank`: the LoRA rank of the launch, 0 = unknown."""
    import numpy as np

    starts = np.ascontiguousarray(s_start, dtype=np.int32)
    ends = np.ascontiguousarray(s_end, dtype=np.int32)
    if starts.shape != ends.shape or starts.ndim != 1:
        raise RuntimeError("s_start and s_end must be one-dimensional and of one length")
    n, rows = _c.c_int32(0), _c.c_int32(0)
    capacity = max(16, int(num_tokens) // 16 + 2 * starts.shape[0])
    while True:
        records = np.empty((capacity, 4), dtype=np.int32)
        rc = lib().lorax_sgmv_plan_tiles(starts.ctypes.data, ends.ctypes.data, starts.shape[0], int(num_tokens),
                                         int(kind), int(rank), records.ctypes.data, capacity, ctypes.byref(n),
                                         ctypes.byref(rows))
        if rc == ESPACE:
            capacity = int(n.value)
            continue
        if rc != 0:
            raise RuntimeError(f"lorax_sgmv_plan_tiles failed with code {rc}")
        return records[: n.value], int(rows.value)


def set_fixed_order_shrink(on: bool) -> bool:
    """lorax_set_fixed_order_shrink: the SGMV shrinks add their sums over the hidden dimension in one fixed order
    whatever the batch (slower on some shapes).  Returns the previous setting."""
    return bool(lib().lorax_set_fixed_order_shrink(1 if on else 0))


SGMV_LORA_MAX_TOKENS = 512


def sgmv_lora_fits(rank: int, h_in: int, num_tokens: int, h_out: int = 0) -> bool:
    """lorax_prefill_in_one_launch: True where the single-launch prefill update (lorax_sgmv_lora_multi) applies and pays -
    rank 8 or 16 with a small A slab, a batch short enough to be bound by launches, and an output that is not so wide (an
    LM head) that recomputing the shrink in every column slice would dominate."""
    return lib().lorax_prefill_in_one_launch(rank, h_in, num_tokens, h_out) != 0


def sgmv_lora_multi(problems, x, s_start, s_end, rank, layer_idx, scale: float = 1.0) -> None:
    """lorax_sgmv_lora_multi: `problems` is a list of up to 4 tuples (y, a_t_ptr, b_t_ptr, y_offset, y_slice_size)
    whose projections share x and the segment tables; y[s:e, window] += (x[s:e] @ A_i^T) @ B_i^T per segment,
    rank 8 or 16, at most 512 rows, in one launch."""
    if not 1 <= len(problems) <= MAX_FUSED_BGMV_PROBLEMS:
        raise RuntimeError(f"between 1 and {MAX_FUSED_BGMV_PROBLEMS} problems per launch, got {len(problems)}")
    _check_input(x, "x", 2)
    _check_input(s_start, "s_start", 1)
    _check_input(s_end, "s_end", 1)
    if s_start.dtype != torch.int32 or s_end.dtype != torch.int32 or s_start.size(0) != s_end.size(0):
        raise RuntimeError("s_start and s_end must be int32 tensors of one length")
    arr = (SgmvLoraProblem * len(problems))()
    for i, (y, a_ptr, b_ptr, y_offset, y_slice_size) in enumerate(problems):
        _check_input(y, "y", 2)
        _check_input(a_ptr, "a_ptr", 1)
        _check_input(b_ptr, "b_ptr", 1)
        _check_same(y, x, a_ptr, b_ptr, s_start, s_end)
        if a_ptr.dtype != torch.int64 or b_ptr.dtype != torch.int64:
            raise RuntimeError("a_ptr and b_ptr must be int64 tensors")
        if a_ptr.size(0) != s_start.size(0) or b_ptr.size(0) != s_start.size(0):
            raise RuntimeError("a_ptr and b_ptr must have one entry per segment")
        if y.size(0) != x.size(0):
            raise RuntimeError(f"CHECK_EQ(y.size(0), x.size(0)) failed. {y.size(0)} vs {x.size(0)}")
        h_out = y.size(1) if y_slice_size is None else int(y_slice_size)
        arr[i] = SgmvLoraProblem(y.data_ptr(), a_ptr.data_ptr(), b_ptr.data_ptr(), int(y_offset), y.size(1), h_out)
    with _on_device(x):
        rc = lib().lorax_sgmv_lora_multi(arr, len(problems), x.data_ptr(), s_start.data_ptr(), s_end.data_ptr(),
                                         s_start.size(0), x.size(0), x.size(1), int(rank), int(layer_idx),
                                         float(scale), _dtype_code(x), _stream(x))
    if rc != 0:
        _raise_last(rc)


class BatchTables:
    """What lorax_layer_update needs of one batch: the builder's group records (host), the packed tables (device) and the
    number of rows they were built for.  Owned by the batch data made from them."""

    __slots__ = ("groups", "num_groups", "packed", "rows", "prefill", "device_index", "rank_sum", "_calls")

    def __init__(self, groups, num_groups: int, packed: torch.Tensor, rows: int, prefill: bool):
        self.groups = groups
        self.num_groups = num_groups
        self.packed = packed
        self.rows = rows
        self.prefill = prefill
        self.device_index = packed.get_device()
        self.rank_sum = None  # layer type -> sum of the ranks of its groups, from the first call on
        self._calls = {}  # slices of a call -> (LayerSlice array, columns of v)

    def call(self, slices):
        """(LayerSlice array, sum of ranks) of `slices`, a tuple of (layer type, first column, end column)."""
        made = self._calls.get(slices)
        if made is None:
            if self.rank_sum is None:
                sums = {}
                for g in self.groups[: self.num_groups]:
                    sums[g.layer_type] = sums.get(g.layer_type, 0) + g.rank
                self.rank_sum = sums
            arr = (LayerSlice * len(slices))(*[LayerSlice(t, end - start, start) for t, start, end in slices])
            made = self._calls[slices] = (arr, sum(self.rank_sum[t] for t, _, _ in slices))
        return made


def layer_update(y, x, tables: BatchTables, slices, layer_idx: int) -> bool:
    """lorax_layer_update: y[:, start:end] += the LoRA update of x for every slice, all launches from one call.
    False, with nothing launched, where the single entry points have to be used: operands they would refuse or that
    need another path."""
    code = _DTYPE_CODES.get(x.dtype)
    if (code is None or y.dtype != x.dtype or x.dim() != 2 or y.dim() != 2 or not x.is_cuda or not y.is_cuda
            or not x.is_contiguous() or not y.is_contiguous()):
        return False
    rows, h_in = x.shape
    y_rows, width = y.shape
    index = tables.device_index
    if (x.get_device() != index or y.get_device() != index or y_rows != rows or rows == 0
            or not (tables.prefill or rows == tables.rows)):
        return False
    arr, columns = tables.call(slices)
    # the call's own workspace, on its stream: [shrink scratch | v] in prefill, v alone in decode
    tmp_bytes, v_bytes = 0, rows * columns * 2
    if tables.prefill:
        _ready(x)
        tmp_bytes = SHRINK_TMP_BYTES
    work = torch.empty((tmp_bytes + v_bytes,), dtype=torch.uint8, device=x.device)
    tmp = work.data_ptr()
    rc = lib().lorax_layer_update(
        tables.groups, tables.num_groups, tables.packed.data_ptr(), arr, len(arr), y.data_ptr(), width, x.data_ptr(), rows,
        h_in, layer_idx, tmp + tmp_bytes, v_bytes, tmp if tmp_bytes else None, tmp_bytes, code, index, _stream(x),
    )
    if rc == EROUTE:
        return False
    if rc != 0:
        _raise_last(rc)
    return True


_STACKED_SLICE = "2Qq2i"  # lorax_stacked_slice_t
_STACKED_SLICES = [struct.Struct(_STACKED_SLICE * n) for n in range(MAX_BGMV_PROBLEMS + 1)]


def stacked_update(y, x, slices, plan: torch.Tensor, records: int) -> bool:
    """lorax_stacked_update: y[:, first:first + width] += the update of x over stacked weights for every slice (lora_a
    [n, r, h_in], lora_b [n, width, r], first, width), all launches from one call; `plan` holds `records` routing records over
    stack entries.  False, with nothing launched, where the single operators have to be used: operands they would refuse
    or that need another path."""
    dtype = x.dtype
    code = _DTYPE_CODES.get(dtype)
    if (code is None or y.dtype != dtype or x.dim() != 2 or y.dim() != 2 or not x.is_cuda or not y.is_cuda
            or not x.is_contiguous() or not y.is_contiguous() or len(slices) > MAX_BGMV_PROBLEMS):
        return False
    rows, h_in = x.shape
    y_rows, y_stride = y.shape
    index = x.get_device()
    if (y.get_device() != index or plan.get_device() != index or y_rows != rows or rows == 0 or plan.dtype != torch.int64
            or not plan.is_contiguous()):
        return False
    fields, columns = [], 0
    for a, b, first, width in slices:
        if a.dim() != 3 or b.dim() != 3:
            return False
        r = a.size(1)
        if (a.size(2) != h_in or b.size(2) != r or b.size(1) != width or a.dtype != dtype or b.dtype != dtype
                or a.get_device() != index or b.get_device() != index or not a.is_contiguous() or not b.is_contiguous()):
            return False
        fields += (a.data_ptr(), b.data_ptr(), first, r, width)
        columns += r
    v_bytes = rows * columns * 2
    v = torch.empty((v_bytes,), dtype=torch.uint8, device=x.device)  # the call's own, on its stream
    rc = lib().lorax_stacked_update(_STACKED_SLICES[len(slices)].pack(*fields), len(slices), plan.data_ptr(), records,
                                    y.data_ptr(), y_stride, x.data_ptr(), rows, h_in, v.data_ptr(), v_bytes, code, index,
                                    _stream(x))
    if rc == EROUTE:
        return False
    if rc != 0:
        _raise_last(rc)
    return True


ENTRY_DTYPE = [("adapter", "<i8"), ("a_addr", "<i8"), ("b_addr", "<i8"), ("rank", "<i4"), ("reserved", "<i4")]


_entry_dtype = None
_table_capacity = [64 * 1024, 64]  # bytes of packed tables, number of group records


def build_batch_tables(adapter_indices, entries, entry_counts, prefill: bool):
    """lorax_build_batch_tables on numpy arrays: adapter_indices int64 [T]; entries a structured array of
    ENTRY_DTYPE, the layer types' adapters one after the other, each type sorted by adapter; entry_counts int32
    per type.  Returns (segment bounds int32 [S+1], segment owners int64 [S], packed uint8 buffer, groups)."""
    bounds, owners, packed, groups, n = batch_tables(adapter_indices, entries, entry_counts, prefill)
    return bounds, owners, packed, list(groups[:n])


def batch_tables(adapter_indices, entries, entry_counts, prefill: bool):
    """build_batch_tables with the group records as the ctypes array the builder filled and their number."""
    import numpy as np

    global _entry_dtype
    if _entry_dtype is None:
        _entry_dtype = np.dtype(ENTRY_DTYPE)  # made once: numpy takes longer to make it than the builder takes for a few rows
    adapter_indices = np.ascontiguousarray(adapter_indices, dtype=np.int64)
    entries = np.ascontiguousarray(entries, dtype=_entry_dtype)
    entry_counts = np.ascontiguousarray(entry_counts, dtype=np.int32)
    T = adapter_indices.shape[0]
    bounds = np.zeros(T + 1, dtype=np.int32)
    owners = np.zeros(max(T, 1), dtype=np.int64)
    nseg, ngroups, nbytes = _c.c_int32(0), _c.c_int32(0), _c.c_int64(0)
    capacity, group_capacity = _table_capacity
    while True:
        packed = np.empty(capacity, dtype=np.uint8)  # the builder writes every byte it reports as used
        groups = (TableGroup * group_capacity)()
        rc = lib().lorax_build_batch_tables(
            adapter_indices.ctypes.data, T, entries.ctypes.data, entry_counts.ctypes.data, entry_counts.shape[0],
            1 if prefill else 0, bounds.ctypes.data, owners.ctypes.data, ctypes.byref(nseg), packed.ctypes.data,
            capacity, ctypes.byref(nbytes), groups, group_capacity, ctypes.byref(ngroups),
        )
        if rc == ESPACE:  # remembered: the next batch of this size takes one call
            capacity = max(capacity, int(nbytes.value) * 5 // 4)
            group_capacity = max(group_capacity, int(ngroups.value) * 2)
            _table_capacity[:] = [capacity, group_capacity]
            continue
        if rc != 0:
            _raise_last(rc)
        return bounds[: nseg.value + 1], owners[: nseg.value], packed[: nbytes.value], groups, ngroups.value
