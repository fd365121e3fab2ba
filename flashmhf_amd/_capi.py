"""Bindings of libmhffn_hip.so (declared in include/mhffn.h): ``lib()`` is the C ABI through ctypes, for benchmarks and
tests that hand over raw pointers; ``native()`` is the extension module the torch operators call.

torch only supplies device memory and the current stream -- the same launch discipline as the reference's
launcher (kernels/thunderkittens/flash_ffn_moe.cu:991).  There is no CPU fallback: if the library has not
been built, loading raises and every operator that needs it fails loudly.
"""
import ctypes
import importlib.util
import os

import torch
from torch.autograd import forward_ad

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "_lib", "libmhffn_hip.so")
NATIVE_PATH = os.path.join(_HERE, "_lib", "_native.so")

DTYPE_BF16, DTYPE_F32 = 0, 1
OK = 0
(ERR_NULL_POINTER, ERR_DTYPE, ERR_HEAD_DIM, ERR_EXPERT_DIM, ERR_SHAPE, ERR_WORKSPACE, ERR_LAUNCH, ERR_ALIGNMENT,
 ERR_STATIC_SCRATCH) = range(-1, -10, -1)
STATIC_SCRATCH_BYTES = 96 << 20

EXPORTS = (
    "mhffn_strerror", "mhffn_is_supported", "mhffn_check_dims", "mhffn_launch_plan", "mhffn_launch_forms", "mhffn_fwd_workspace_bytes",
    "mhffn_bwd_workspace_bytes", "mhffn_bwd_workspace_min_bytes", "mhffn_fwd", "mhffn_bwd", "mhffn_fwd_phases", "mhffn_bwd_phases",
    "mhffn_fwd_layout", "mhffn_bwd_layout", "mhffn_bwd_static", "mhffn_gate_fwd", "mhffn_gate_bwd",
    "mhffn_gate_fwd_typed", "mhffn_gate_bwd_workspace_bytes", "mhffn_gate_bwd_into", "mhffn_rope_fwd", "mhffn_rope_bwd",
    "mhffn_product_preferred", "mhffn_product_faster", "mhffn_product_tile", "mhffn_product",
    "mhffn_product_pair_faster", "mhffn_product_pair",
)
PRODUCT_NT, PRODUCT_NN, PRODUCT_TN = 0, 1, 2
TOKENS_BHSD, TOKENS_BSHD = 0, 1     # layout of Q, O, dO, dQ
FWD_MAIN, FWD_ALL = 1, 1
BWD_DQDR, BWD_DKDUDV, BWD_REDUCE, BWD_ALL = 1, 2, 4, 7
ONE_PART = 256
FORM_WEIGHTS_PAST_CACHES, FORM_TOKEN_HALVES, FORM_GATE_FWD_WHOLE_ROWS, FORM_GATE_BWD_WHOLE_ROWS, FORM_FWD_PADDED, FORM_DQDR_PADDED = 1, 2, 4, 8, 16, 32


class Dims(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in ("B", "H", "Hkuv", "S", "d_h", "E", "d_e")]


class Plan(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int) for n in ("fwd_tile_rows", "fwd_parts", "dqdr_tile_rows", "dqdr_parts", "dkdudv_slices")]


_lib = None


def lib():
    """Loads the library once.  Raises ImportError (never falls back) when it is missing."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise ImportError(
                f"{LIB_PATH} not found: build it with `python -m flashmhf_amd.build` (hipcc, gfx950). "
                "flashmhf_amd has no CPU or eager fallback.")
        L = ctypes.CDLL(LIB_PATH)
        vp, dp = ctypes.c_void_p, ctypes.POINTER(Dims)
        L.mhffn_strerror.restype = ctypes.c_char_p
        L.mhffn_strerror.argtypes = [ctypes.c_int]
        L.mhffn_is_supported.argtypes = [ctypes.c_int] * 3
        L.mhffn_check_dims.argtypes = [dp, ctypes.c_int]
        for f in (L.mhffn_fwd_workspace_bytes, L.mhffn_bwd_workspace_bytes, L.mhffn_bwd_workspace_min_bytes):
            f.restype = ctypes.c_size_t
            f.argtypes = [dp, ctypes.c_int]
        L.mhffn_launch_plan.argtypes = [dp, ctypes.c_int, ctypes.c_size_t, ctypes.c_size_t, ctypes.c_int, ctypes.POINTER(Plan)]
        L.mhffn_launch_forms.argtypes = [dp, ctypes.c_int, ctypes.c_size_t, ctypes.c_size_t, ctypes.c_int]
        L.mhffn_fwd.argtypes = [vp] * 6 + [vp, ctypes.c_size_t, dp, ctypes.c_int, vp]
        L.mhffn_bwd.argtypes = [vp] * 6 + [vp] * 5 + [ctypes.c_int, vp, ctypes.c_size_t, dp, ctypes.c_int, vp]
        L.mhffn_fwd_phases.argtypes = L.mhffn_fwd.argtypes + [ctypes.c_int]
        L.mhffn_bwd_phases.argtypes = L.mhffn_bwd.argtypes + [ctypes.c_int]
        L.mhffn_fwd_layout.argtypes = [vp] * 6 + [vp, ctypes.c_size_t, dp, ctypes.c_int, ctypes.c_int, vp, ctypes.c_int]
        L.mhffn_bwd_layout.argtypes = ([vp] * 6 + [vp] * 5 + [ctypes.c_int, vp, ctypes.c_size_t, dp, ctypes.c_int,
                                                              ctypes.c_int, vp, ctypes.c_int])
        L.mhffn_bwd_static.argtypes = [vp] * 6 + [vp] * 5 + [ctypes.c_int, dp, ctypes.c_int, ctypes.c_int, vp]
        L.mhffn_gate_fwd.argtypes = [vp, vp, ctypes.c_float, vp, vp, vp, dp, vp]
        L.mhffn_gate_bwd.argtypes = [vp, vp, ctypes.c_float, vp, vp, ctypes.c_int, vp, vp, vp, vp, dp, vp]
        L.mhffn_gate_fwd_typed.argtypes = [vp, vp, ctypes.c_int, ctypes.c_float, vp, ctypes.c_int, vp, vp, dp, vp]
        L.mhffn_gate_bwd_workspace_bytes.restype = ctypes.c_size_t
        L.mhffn_gate_bwd_workspace_bytes.argtypes = [dp]
        L.mhffn_gate_bwd_into.argtypes = [vp, vp, ctypes.c_int, ctypes.c_float, vp, ctypes.c_int, vp, ctypes.c_int, vp, vp, vp, vp,
                                          vp, ctypes.c_size_t, dp, vp]
        L.mhffn_rope_fwd.argtypes = [vp] * 5 + [ctypes.c_int] * 4 + [vp]
        L.mhffn_rope_bwd.argtypes = [vp] * 3 + [ctypes.POINTER(ctypes.c_long)] + [vp] * 3 + [ctypes.c_int] * 4 + [vp]
        L.mhffn_product_preferred.argtypes = [ctypes.c_int] * 2
        L.mhffn_product_faster.argtypes = [ctypes.c_int] * 5
        L.mhffn_product_tile.argtypes = [ctypes.c_int] * 5
        L.mhffn_product.argtypes = [ctypes.c_int] * 2 + [vp] * 3 + [ctypes.c_int] * 3 + [vp]
        L.mhffn_product_pair_faster.argtypes = [ctypes.c_int] * 4
        L.mhffn_product_pair.argtypes = [vp] * 5 + [ctypes.c_int] * 3 + [vp]
        _lib = L
    return _lib


_native = None


def native():
    """The torch side of the operators (csrc/mhffn_torch.cpp), loaded once.  Raises ImportError when it is missing."""
    global _native
    if _native is None:
        if not os.path.exists(NATIVE_PATH):
            raise ImportError(f"{NATIVE_PATH} not found: build it with `python -m flashmhf_amd.build`. "
                              "flashmhf_amd has no CPU or eager fallback.")
        spec = importlib.util.spec_from_file_location("flashmhf_amd._lib._native", NATIVE_PATH)
        _native = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(_native)
    return _native


def native_nodes():
    """Whether the operators may record the native autograd nodes.  A trace keeps only calls that it knows (the native ones
    would become constants), and functorch transforms and forward mode have to meet a torch.autograd.Function, which runs
    or refuses them: under these the operators go through their Python Functions."""
    return not (torch._C._is_tracing() or torch._C._are_functorch_transforms_active() or forward_ad._current_level >= 0)


def traced(t):
    """`t`, an output of a native call inside a Function's forward, as a tensor that a running trace knows."""
    return t.clone() if torch._C._is_tracing() else t


def launch_plan(dims, dtype, one_part=False):
    """What the operators run for these extents (they hand over the workspaces that are asked for)."""
    p = Plan()
    raise_for_code(lib().mhffn_launch_plan(dims, dtype, lib().mhffn_fwd_workspace_bytes(dims, dtype),
                                           lib().mhffn_bwd_workspace_bytes(dims, dtype), ONE_PART if one_part else 0, p),
                   "mhffn_launch_plan")
    return p


def launch_forms(dims, dtype, one_part=False):
    """... and the FORM_* bits of its kernels."""
    L = lib()
    forms = L.mhffn_launch_forms(dims, dtype, L.mhffn_fwd_workspace_bytes(dims, dtype), L.mhffn_bwd_workspace_bytes(dims, dtype),
                                 ONE_PART if one_part else 0)
    raise_for_code(min(forms, OK), "mhffn_launch_forms")
    return forms


def strerror(code):
    return lib().mhffn_strerror(code).decode()


def raise_for_code(code, what):
    """Maps return codes to the exception types the reference raises for the same condition:
    TypeError for dtypes (kernels/triton/flash_mlp_moe.py:761-766), ValueError for the expert dim (:758-759),
    RuntimeError for everything a TORCH_CHECK would catch (kernels/thunderkittens/flash_ffn_moe.cu:943-958)."""
    if code == OK:
        return
    msg = f"{what}: {strerror(code)} (code {code})"
    if code == ERR_DTYPE:
        raise TypeError(msg)
    if code in (ERR_EXPERT_DIM, ERR_HEAD_DIM):
        raise ValueError(msg)
    raise RuntimeError(msg)


def torch_dtype_code(dt):
    if dt == torch.bfloat16:
        return DTYPE_BF16
    if dt == torch.float32:
        return DTYPE_F32
    return -1
