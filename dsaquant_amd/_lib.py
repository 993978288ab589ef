"""ctypes binding of libvdmq.so (the C ABI in include/vdmq.h)."""
from __future__ import annotations

import ctypes
import importlib
import os
import subprocess
import sys
import warnings
from pathlib import Path
from typing import Optional

_PKG = Path(__file__).resolve().parent
LIB_PATH = _PKG / "libvdmq.so"
CSRC = _PKG / "csrc"

_LIB: Optional[ctypes.CDLL] = None
host = None  # the extension module _vdmq_host, once load() has run; None where it cannot be used: the general code serves every call

VDMQ_VERSION = 2  # include/vdmq.h; also the version of the bf6 block format
VDMQ_OUT_F16 = 0
VDMQ_OUT_BF16 = 1
VDMQ_ACT_NONE = 0
VDMQ_ACT_GELU_TANH = 1
VDMQ_LN_MODULATE = 1
VDMQ_LN_AFFINE = 2
VDMQ_LINEAR_BF6_MIN_K = 640
HOST_INTERFACE = 2  # the arguments of _vdmq_host's functions (kInterface in vdmq_host.cpp)


class GemmLaunchInfo(ctypes.Structure):
    """vdmq_gemm_launch_info of include/vdmq.h."""
    _fields_ = [("kernel", ctypes.c_int), ("tile_m", ctypes.c_int), ("tile_n", ctypes.c_int), ("group_m", ctypes.c_int),
                ("group_n", ctypes.c_int), ("contiguous_runs", ctypes.c_int), ("workgroups", ctypes.c_int64)]


KERNEL_GEMM_W4A4, KERNEL_GEMM_BF6, KERNEL_GEMM_BF6_PERSISTENT, KERNEL_LINEAR_RESIDENT, KERNEL_GEMM_BF6_KSPLIT, KERNEL_GEMM_BF6_PAIR = 1, 2, 3, 4, 5, 6

# name -> (restype, argtypes); every symbol include/vdmq.h declares
_i64, _p, _f32, _int = ctypes.c_int64, ctypes.c_void_p, ctypes.c_float, ctypes.c_int
SIGNATURES = {
    "vdmq_version": (_int, []),
    "vdmq_arch": (ctypes.c_char_p, []),
    "vdmq_last_error": (ctypes.c_char_p, []),
    "vdmq_k_padded": (_i64, [_i64]),
    "vdmq_quantize_act": (_int, [_p, _i64, _i64, _i64, _f32, _p, _p, _p]),
    "vdmq_quantize_act_ex": (_int, [_p, _i64, _i64, _i64, _f32, _int, _p, _p, _p]),
    "vdmq_quantize_act_ln": (_int, [_p, _i64, _i64, _i64, _f32, _int, _p, _p, _i64, _i64, _f32, _p, _p, _p]),
    "vdmq_ln_f16": (_int, [_p, _i64, _i64, _i64, _f32, _int, _p, _p, _i64, _i64, _p, _i64, _p]),
    "vdmq_linear_ln_w4a4": (_int, [_p, _i64, _i64, _i64, _f32, _int, _p, _p, _i64, _i64, _f32, _p, _p, _p, _p, _int, _i64, _i64, _p, _i64, _p]),
    "vdmq_gelu_tanh_f16": (_int, [_p, _p, _i64, _p]),
    "vdmq_gemm_w4a4": (_int, [_p, _p, _p, _p, _p, _p, _int, _i64, _i64, _i64, _i64, _p]),
    "vdmq_gemm_w4a4_ex": (_int, [_p, _p, _p, _p, _p, _p, _i64, _i64, _p, _i64, _p, _int, _i64, _i64, _i64, _i64, _p]),
    "vdmq_gemm_w4a4_acc": (_int, [_p, _p, _p, _i64, _i64, _i64, _p]),
    "vdmq_gemm_w4a4_split": (_int, [_p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _i64, _p]),
    "vdmq_gemm_w4a4_bf6_split": (_int, [_p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _i64, _p]),
    "vdmq_last_gemm_launch": (_int, [ctypes.POINTER(GemmLaunchInfo)]),
    "vdmq_workspace_bytes": (_i64, [_i64, _i64]),
    "vdmq_linear_w4a4": (_int, [_p, _i64, _i64, _i64, _f32, _p, _p, _p, _p, _int, _i64, _i64, _p, _i64, _p]),
    "vdmq_linear_w4a4_ex": (_int, [_p, _i64, _i64, _i64, _f32, _int, _p, _p, _p, _p, _int, _i64, _i64, _p, _i64, _p]),
    "vdmq_linear_w4a4_noalloc": (_int, [_p, _i64, _i64, _i64, _f32, _p, _p, _p, _p, _int, _i64, _i64, _p]),
    "vdmq_weight_v1_to_native": (_int, [_p, _p, _i64, _i64, _p]),
    "vdmq_weight_native_to_v1": (_int, [_p, _p, _i64, _i64, _p]),
    "vdmq_wscale_v1_to_plain": (_int, [_p, _p, _i64, _i64, _p]),
    "vdmq_wscale_plain_to_v1": (_int, [_p, _p, _i64, _i64, _p]),
    "vdmq_act_native_to_v1": (_int, [_p, _p, _i64, _i64, _p, _p, _p]),
    "vdmq_act_v1_to_native": (_int, [_p, _p, _i64, _i64, _p, _p, _p]),
    "vdmq_row_scale": (_int, [_p, _i64, _i64, _f32, _p, _p]),
    "vdmq_quantize_weight_native": (_int, [_p, _p, _p, _i64, _i64, _p]),
    "vdmq_pack_weight": (_int, [_p, _p, _p, _p, _p, _p, _i64, _i64, _p]),
    "vdmq_bf6_bytes": (_i64, [_i64, _i64]),
    "vdmq_quantize_act_bf6": (_int, [_p, _i64, _i64, _i64, _f32, _int, _p, _p, _p]),
    "vdmq_quantize_act_ln_bf6": (_int, [_p, _i64, _i64, _i64, _f32, _int, _p, _p, _i64, _i64, _f32, _p, _p, _p]),
    "vdmq_workspace_bytes_bf6": (_i64, [_i64, _i64]),
    "vdmq_bf6_pays": (_int, [_i64, _i64, _i64]),
    "vdmq_linear_w4a4_bf6": (_int, [_p, _i64, _i64, _i64, _f32, _int, _p, _p, _p, _p, _int, _i64, _i64, _p, _i64, _p]),
    "vdmq_linear_bf6_workspace": (_i64, [_i64, _i64, _i64, _int, _int, _i64, _i64, _int]),
    "vdmq_linear_bf6": (_int, [_p, _i64, _i64, _i64, _f32, _int, _p, _p, _p, _p, _int, _i64, _i64, _p, _i64, _p]),
    "vdmq_linear_bf6_ex": (_int, [_p, _i64, _i64, _i64, _f32, _int, _int, _f32, _p, _p, _i64, _i64, _p, _p, _p, _p, _i64, _i64, _p, _i64, _i64, _i64,
                                  _p, _int, _i64, _i64, _p, _i64, _p]),
    "vdmq_native_to_bf6": (_int, [_p, _i64, _i64, _p, _p]),
    "vdmq_weight_v1_to_bf6": (_int, [_p, _p, _i64, _i64, _p]),
    "vdmq_bf6_to_weight_v1": (_int, [_p, _p, _i64, _i64, _p]),
    "vdmq_gemm_w4a4_bf6": (_int, [_p, _p, _p, _p, _p, _p, _int, _i64, _i64, _i64, _i64, _p]),
    "vdmq_gemm_w4a4_bf6_ex": (_int, [_p, _p, _p, _p, _p, _p, _i64, _i64, _p, _i64, _p, _int, _i64, _i64, _i64, _i64, _p]),
    "vdmq_gemm_w4a4_bf6_acc": (_int, [_p, _p, _p, _i64, _i64, _i64, _p]),
    "vdmq_attention_f16": (_int, [_p, _p, _p, _p, _p, _p, _p, _p, _i64, _i64, _i64, _i64, _i64, _f32, _p]),
    "vdmq_rms_norm_rope_f16": (_int, [_p, _i64, _p, _p, _p, _i64, _p, _p, _i64, _i64, _f32, _p, _i64, _i64, _p]),
    "vdmq_row_squares_f32": (_int, [_p, _i64, _p, _p, _i64, _p, _i64, _i64, _p]),
    "vdmq_scale_rows": (_int, [_p, _i64, _p, _p, _p, _p, _i64, _p, _p, _p, _int, _i64, _i64, _p]),
    "vdmq_modulate_rows_f16": (_int, [_p, _p, _p, _p, _i64, _i64, _p]),
    "vdmq_rope_table": (_int, [_p, _i64, _i64, _i64, _i64, _p]),
    "vdmq_timestep_embedding_f16": (_int, [_p, _p, _i64, _i64, _p]),
    "vdmq_copy_u128": (_int, [_p, _p, _i64, _p]),
    "vdmq_stream_probe": (_int, [_p, _p, _i64, _int, _int, _p]),
    "vdmq_mfma_probe_operand_bytes": (_i64, []),
    "vdmq_mfma_probe": (_int, [_int, _p, _i64, _i64, _p, ctypes.POINTER(ctypes.c_double), _p]),
}


class VdmqError(RuntimeError):
    """A native precondition failed (the reference raises RuntimeError from TORCH_CHECK)."""


def build(verbose: bool = False) -> Path:
    """Compile libvdmq.so for gfx950 with hipcc, and the extension module for this interpreter (``make -C dsaquant_amd/csrc``)."""
    cmd = ["make", "-C", str(CSRC), "-j", str(min(8, os.cpu_count() or 1)), "-B", f"PYTHON={sys.executable}"]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if verbose or res.returncode != 0:
        print(res.stdout)
    if res.returncode != 0:
        raise RuntimeError("building libvdmq.so failed")
    return LIB_PATH


def load() -> ctypes.CDLL:
    """Load the built library; raises if it is missing (no fallback exists)."""
    global _LIB, host
    if _LIB is not None:
        return _LIB
    if not LIB_PATH.exists():
        raise FileNotFoundError(
            f"{LIB_PATH} is missing: build it with `python -c 'import __graft_entry__ as g; g.build()'` "
            f"or `make -C {CSRC}`")
    import torch  # noqa: F401  (the extension module below needs its libraries, and the HIP runtime that serves both is the one loaded first)

    lib = ctypes.CDLL(str(LIB_PATH))
    for name, (restype, argtypes) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = restype
        fn.argtypes = argtypes
    if lib.vdmq_version() != VDMQ_VERSION:
        raise RuntimeError(f"{LIB_PATH} has interface version {lib.vdmq_version()}, this package expects {VDMQ_VERSION}: rebuild it (make -C {CSRC})")
    host = _load_host(lib, torch.__version__)
    _LIB = lib
    return lib


def _load_host(lib: ctypes.CDLL, torch_version: str):
    """The host side of the package's own calls (vdmq_host.cpp, built with the library); None, with a warning, where there is none
    for this interpreter, torch and package: its calls then run through ctypes, with the same results and 4 ... 12 us more each."""
    try:
        module = importlib.import_module("._vdmq_host", __package__)
        built = getattr(module, "interface", None), getattr(module, "torch_version", None)
        reason = None if built == (HOST_INTERFACE, torch_version.split("+")[0]) else f"it is of interface {built[0]} and torch {built[1]}"
    except ImportError as exc:
        reason = str(exc)
    if reason is not None:
        warnings.warn(f"the extension module _vdmq_host cannot be used ({reason}): build it with `make -C {CSRC} PYTHON={sys.executable}`", RuntimeWarning, 3)
        return None
    module.init(*(ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in ("vdmq_linear_bf6_ex", "vdmq_linear_bf6_workspace", "vdmq_pack_weight")))
    return module


def last_gemm_launch() -> GemmLaunchInfo:
    """What the library chose for the last GEMM launched on this thread."""
    info = GemmLaunchInfo()
    check(load().vdmq_last_gemm_launch(ctypes.byref(info)))
    return info


def check(rc: int) -> None:
    if rc != 0:
        msg = load().vdmq_last_error()
        raise VdmqError(f"vdmq error {rc}: {msg.decode() if msg else ''}")
