"""ctypes binding of ``libloraforge_amd.so`` (the C ABI in ``include/loraforge_amd.h``).

The library is loaded after ``torch`` so that it binds to the HIP runtime
PyTorch already loaded (both carry the soname ``libamdhip64.so.7``); pointers
and streams handed over here are therefore valid in both. There is no CPU or
PyTorch fallback: a missing library raises ``RuntimeError`` naming the build
step.
"""

from __future__ import annotations

import ctypes
import threading
from pathlib import Path

LIBRARY = Path(__file__).resolve().parent / "_lib" / "libloraforge_amd.so"
BINDING = LIBRARY.with_name("_binding.so")

LF_OK = 0
LF_EINVAL = 1
LF_EHIP = 2
LF_EXACT_WEIGHTS = 1
LF_SWIGLU_OUTPUT = 2
LF_PLAN_DECODE_CHUNKS = 4
LF_PLAN_PREFILL = 8
LF_TEST_WITHHOLD_PARTIALS = 0x100
LF_KERNEL_DECODE, LF_KERNEL_DECODE_WIDE, LF_KERNEL_DECODE_CHUNKS, LF_KERNEL_PREFILL = range(4)
NOALLOC_SCRATCH_BYTES = 8 * 1024 * 1024
ABI_VERSION = 4

# Per device index, filled by the operators' Python paths: fit for the kernels
# (gfx950), and compute units.
ARCH_OK: dict = {}
COMPUTE_UNITS: dict = {}
# Cached workspaces: (device index, stream) for the fused calls, ("rows",
# device index, stream) for the row shrink (ops/fused.py::_workspace).
WORKSPACES: dict = {}

_lock = threading.Lock()
_handle: ctypes.CDLL | None = None

c_void_p = ctypes.c_void_p
c_int64 = ctypes.c_int64
c_int32 = ctypes.c_int32
c_float_p = ctypes.c_void_p


class NF4Weight(ctypes.Structure):
    _fields_ = [
        ("qweight", c_void_p),
        ("scales", c_void_p),
        ("absmax_q", c_void_p),
        ("absmax2", c_void_p),
        ("code2", c_void_p),
        ("offset", c_void_p),
        ("dq_block", c_int64),
        ("code", c_void_p),
        ("n", c_int64),
        ("k", c_int64),
    ]


class Lora(ctypes.Structure):
    _fields_ = [
        ("a_store", c_void_p),
        ("a_offsets", c_void_p),
        ("b_store", c_void_p),
        ("b_offsets", c_void_p),
        ("b_strides", c_void_p),
        ("ranks", c_void_p),
        ("scales", c_void_p),
        ("token_slots", c_void_p),
        ("slice_offsets", c_void_p),
        ("num_slices", c_int32),
        ("max_rank", c_int32),
        ("num_slots", c_int32),
    ]


class Plan(ctypes.Structure):
    _fields_ = [("kernel", c_int32), ("tile_rows", c_int32), ("z_parts", c_int32), ("z_launch", c_int32)]


_PROTOTYPES = {
    "lf_last_error": (ctypes.c_char_p, []),
    "lf_abi_version": (ctypes.c_int, []),
    "lf_device_arch": (ctypes.c_int, [ctypes.c_int, ctypes.c_char_p, ctypes.c_int]),
    "lf_nf4_dequant": (ctypes.c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p]),
    "lf_nf4_dequant_dq": (
        ctypes.c_int,
        [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p, c_void_p, c_int64, c_void_p],
    ),
    "lf_nf4_dequant_dq_checked": (
        ctypes.c_int,
        [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p, c_void_p, c_int64, ctypes.POINTER(c_int32), c_void_p],
    ),
    "lf_nf4_prepare_scales_dq": (
        ctypes.c_int,
        [c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p, c_int64, c_void_p],
    ),
    "lf_row_shrink": (
        ctypes.c_int,
        [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_int64, c_int64, c_int32, c_int64, c_int32]
        + [c_void_p, c_int64, c_int32, c_void_p],
    ),
    "lf_row_shrink_workspace_size": (
        c_int64,
        [c_int64, c_int64, c_int64, c_int32, c_int32],
    ),
    "lf_row_expand": (
        ctypes.c_int,
        [c_void_p] * 12 + [c_int64, c_int64, c_int64, c_int64, c_int32, c_int64, c_int32, c_int32, c_void_p],
    ),
    "lf_row_expand_tiled": (
        ctypes.c_int,
        [c_void_p] * 12 + [c_int64, c_int64, c_int64, c_int64, c_int32, c_int64, c_int32, c_int32, c_int32, c_void_p],
    ),
    "lf_nf4_lora_workspace_size": (c_int64, [c_int64, c_int64, c_int64, c_int32, c_int32]),
    "lf_nf4_lora_linear": (
        ctypes.c_int,
        [
            c_void_p,
            c_int64,
            c_int64,
            ctypes.POINTER(NF4Weight),
            c_void_p,
            ctypes.POINTER(Lora),
            c_void_p,
            c_int64,
            c_void_p,
            c_int64,
            c_int32,
            c_void_p,
        ],
    ),
    "lf_nf4_lora_linear_noalloc": (
        ctypes.c_int,
        [
            c_void_p,
            c_int64,
            c_int64,
            ctypes.POINTER(NF4Weight),
            c_void_p,
            ctypes.POINTER(Lora),
            c_void_p,
            c_int64,
            c_int32,
            c_void_p,
        ],
    ),
    "lf_lora_apply": (
        ctypes.c_int,
        [c_void_p, c_int64, c_int64, c_int64, c_int64, ctypes.POINTER(Lora), c_void_p, c_int64, c_void_p, c_int64,
         c_int32, c_void_p],
    ),
    "lf_nf4_lora_plan": (
        ctypes.c_int,
        [c_int64, c_int64, c_int64, c_int32, c_int32, c_int32, c_int32, ctypes.POINTER(Plan)],
    ),
    "lf_lora_apply_plan": (
        ctypes.c_int,
        [c_int64, c_int64, c_int64, c_int32, c_int32, c_int32, ctypes.POINTER(c_int32)],
    ),
    "lf_nf4_lora_status": (ctypes.c_int, [c_void_p, c_void_p, ctypes.POINTER(c_int32)]),
    "lf_swiglu": (ctypes.c_int, [c_void_p, c_int64, c_int64, c_int64, c_void_p, c_int64, c_void_p]),
}

EXPORTS = tuple(_PROTOTYPES)


def library() -> ctypes.CDLL:
    """Load (once) and return the native library; raise if it was not built."""
    global _handle
    if _handle is not None:
        return _handle
    with _lock:
        if _handle is None:
            import torch  # noqa: F401  (binds the HIP runtime torch ships)

            if not LIBRARY.exists():
                raise RuntimeError(
                    f"loraforge_amd native library missing at {LIBRARY}; "
                    "build it with `python -c 'import __graft_entry__ as g; g.build()'` "
                    "or `python -m loraforge_amd._build`"
                )
            lib = ctypes.CDLL(str(LIBRARY))
            for name, (restype, argtypes) in _PROTOTYPES.items():
                fn = getattr(lib, name)
                fn.restype = restype
                fn.argtypes = argtypes
            if lib.lf_abi_version() != ABI_VERSION:
                raise RuntimeError("loraforge_amd native library ABI mismatch; rebuild it")
            _handle = lib
    return _handle


_binding_module = None
# The library's entry points that the native call path calls, in its order.
_BOUND = (
    "lf_nf4_lora_linear",
    "lf_nf4_lora_workspace_size",
    "lf_lora_apply",
    "lf_row_shrink",
    "lf_row_shrink_workspace_size",
    "lf_row_expand",
    "lf_nf4_dequant",
    "lf_nf4_dequant_dq_checked",
    "lf_last_error",
)


def bind(module, **replaced) -> None:
    """Hand the native call path its entry points (``replaced``: addresses that stand in for some)."""
    import torch

    from .ops.fused import LoraBatch

    stream = getattr(torch._C, "_cuda_getCurrentRawStream", None) or (lambda index: torch.cuda.current_stream(index).cuda_stream)
    device = getattr(torch._C, "_cuda_getDevice", None) or torch.cuda.current_device
    lib = library()
    addresses = tuple(replaced.get(name) or ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in _BOUND)
    module.init(addresses, stream, device, ARCH_OK, WORKSPACES, COMPUTE_UNITS, LoraBatch)


def binding():
    """The operators' native call path (``csrc/host/binding.cpp``), bound to the loaded library.

    Its functions return None for any call they do not take; the operator's
    Python code then serves or refuses it. ``ARCH_OK`` and ``COMPUTE_UNITS``
    tell it which devices were found fit, ``WORKSPACES`` is the cache that it
    finds the current stream's workspace in.
    """
    global _binding_module
    if _binding_module is not None:
        return _binding_module
    import importlib.machinery
    import importlib.util

    import torch  # noqa: F401  (the module links to torch's libraries)

    library()
    with _lock:
        if _binding_module is None:
            if not BINDING.exists():
                raise RuntimeError(f"loraforge_amd native binding missing at {BINDING}; build it with `python -m loraforge_amd._build`")
            loader = importlib.machinery.ExtensionFileLoader("_binding", str(BINDING))
            module = importlib.util.module_from_spec(importlib.util.spec_from_file_location("_binding", str(BINDING), loader=loader))
            loader.exec_module(module)
            bind(module)
            _binding_module = module
    return _binding_module


def check(status: int) -> None:
    """Map a C status to the reference's exception types."""
    if status == LF_OK:
        return
    message = (library().lf_last_error() or b"").decode(errors="replace")
    if status == LF_EINVAL:
        raise ValueError(message)
    raise RuntimeError(message)


def ptr(tensor) -> int | None:
    """Device address of a tensor's first element (None for None)."""
    return None if tensor is None else tensor.data_ptr()


def stream_of(device) -> int:
    import torch

    return torch.cuda.current_stream(device).cuda_stream
