"""ctypes binding of libmoe_hip.so (C ABI declared in include/moe_hip.h), and the torch extension module over the same
library (csrc/torch_layer.cpp: the autograd functions).  No compute happens here."""
from __future__ import annotations

import ctypes
import os

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libmoe_hip.so")

ABI_VERSION = 2   # MOE_HIP_ABI_VERSION of include/moe_hip.h this binding was written against
MOE_BF16, MOE_F16, MOE_F32 = 0, 1, 2
_DTYPES = {torch.bfloat16: MOE_BF16, torch.float16: MOE_F16, torch.float32: MOE_F32}

_P, _L, _I, _F, _Z = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int, ctypes.c_float, ctypes.c_size_t
_CODES = {"p": _P, "l": _L, "i": _I, "f": _F, "z": _Z}

# name -> (restype code, argument codes); one letter per argument in declaration order
_SIGNATURES = {
    "moe_hip_abi_version": ("i", ""),
    "moe_hip_strerror": ("s", "i"),
    "moe_profile_enable": ("i", "i"),
    "moe_profile_select": ("i", "p"),
    "moe_profile_count": ("i", ""),
    "moe_profile_get": ("i", "ipip"),
    "moe_router_logits": ("i", "plplipllip"),
    "moe_router_topk": ("i", "ppppliiip"),
    "moe_router_forward": ("i", "plpli" + "pppp" + "lliiip"),
    "moe_router_forward_sorted": ("i", "plpli" + "pppp" + "lliii" + "pppp" + "pzp"),
    "moe_router_topk_bwd": ("i", "ppppp" + "liiip"),
    "moe_gates_bwd": ("i", "plpli" + "ppppppp" + "ll" + "iii" + "p"),
    "moe_router_weight_grad_workspace_bytes": ("z", "lli"),
    "moe_router_weight_grad": ("i", "plppllliipzp"),
    "moe_gemm_debug_tile": ("i", "lillii"),
    "moe_gemm_debug_tile_plan_blocks": ("l", "ilili"),
    "moe_gemm_debug_tile_plan": ("i", "ipiilllii" + "pp"),
    "moe_gemm_debug_plan_blocks": ("l", "lili"),
    "moe_gemm_debug_launch_count": ("l", ""),
    "moe_gemm_debug_plan": ("i", "piilllii" + "pp"),
    "moe_sort_workspace_bytes": ("z", "li"),
    "moe_sort_by_expert": ("i", "piliippippplpppzp"),
    "moe_sort_static_max_bytes": ("z", ""),
    "moe_sort_by_expert_static": ("i", "piliippippplppp"),
    "moe_expert_offsets": ("i", "pilipip"),
    "moe_padded_block_indices": ("i", "piiipilpp"),
    "moe_scatter2scatter_workspace_bytes": ("z", "lilli"),
    "moe_scatter2scatter": ("i", "pll" + "plll" + "plll" + "plll" + "if" + "pll" + "pi" + "pi" + "i" + "lll" + "iiii" + "pzp"),
    "moe_linear_lora_bwd_workspace_bytes": ("z", "lilli"),
    "moe_linear_lora_bwd": ("i", "pli" + "pi" + "pli" + "plll" + "plll" + "plll" + "if" + "plll" + "plll" + "pl" + "pi" + "pi" + "i" + "lll" + "i" + "pzp"),
    "moe_group_bwd_ab_workspace_bytes": ("z", "lillii"),
    "moe_group_bwd_ab": ("i", "pll" + "pll" + "plll" + "plll" + "if" + "plll" + "plll" + "pi" + "i" + "lll" + "i" + "pzp"),
    "moe_group_bwd_w": ("i", "pll" + "pll" + "plll" + "pi" + "i" + "lll" + "i" + "p"),
    "moe_group_rows": ("i", "pl" + "pl" + "pi" + "i" + "pi" + "ll" + "i" + "p"),
    "moe_combine": ("i", "pl" + "pl" + "pi" + "p" + "i" + "ll" + "i" + "p" + "pl" + "i" + "p"),
    "moe_combine_dgates": ("i", "pl" + "pl" + "pi" + "p" + "i" + "ll" + "i" + "p"),
    "moe_swiglu_pair": ("i", "pllpplllplpipiilllii" + "p"),
    "moe_swiglu": ("i", "ppplip"),
    "moe_swiglu_bwd": ("i", "ppppplip"),
    "moe_mlp_workspace_bytes": ("z", "lilli"),
    "moe_mlp_saved_bytes": ("z", "li"),
    "moe_mlp_fwd": ("i", "pl" + "ppp" + "pp" + "if" + "pppp" + "l" + "pi" + "pi" + "i" + "lll" + "iii" + "p" + "pzp"),
    "moe_mlp_bwd": ("i", "plii" + "p" + "pl" + "ppp" + "pp" + "pp" + "if" + "ppp" + "pp" + "pli" + "pi" + "pi" + "i" + "lll" + "ii" + "p" + "pzp"),
}

EXPORTED_SYMBOLS = tuple(_SIGNATURES)


def _load() -> ctypes.CDLL:
    if not os.path.exists(LIB_PATH):
        raise ImportError(
            f"{LIB_PATH} not found: the HIP extension must be built first "
            f"(python -c 'import __graft_entry__ as g; g.build()' or make -C {os.path.join(_HERE, 'csrc')})")
    lib = ctypes.CDLL(LIB_PATH)
    lib.moe_hip_abi_version.restype = ctypes.c_int
    if lib.moe_hip_abi_version() != ABI_VERSION:   # before the symbol table: an older library lacks entry points
        raise ImportError(f"{LIB_PATH} has ABI version {lib.moe_hip_abi_version()}, this binding needs {ABI_VERSION}: rebuild the library")
    for name, (res, args) in _SIGNATURES.items():
        fn = getattr(lib, name)  # AttributeError if the library does not export a declared symbol
        fn.restype = ctypes.c_char_p if res == "s" else _CODES[res]
        fn.argtypes = [_CODES[c] for c in args]
    return lib


lib = _load()
try:
    from . import _native as native   # noqa: E402  (resolves libmoe_hip.so to the library loaded above)
except ImportError as e:
    raise ImportError(f"{os.path.join(_HERE, '_native.so')} is missing or does not fit: build it with "
                      f"python -c 'import __graft_entry__ as g; g.build()' ({e})") from e


def entry(name: str):
    """The native function, or inside torch.jit.trace the same function as an operator, which a trace can record."""
    return getattr(torch.ops.moe_hip if torch.jit.is_tracing() else native, name)


def check(status: int, what: str) -> None:
    if status != 0:
        raise RuntimeError(f"{what} failed: {lib.moe_hip_strerror(status).decode()} (status {status})")


def dtype_code(t: torch.Tensor) -> int:
    try:
        return _DTYPES[t.dtype]
    except KeyError:
        raise TypeError(f"unsupported dtype {t.dtype}: the HIP kernels take bfloat16, float16 or float32") from None


def require_gpu(*tensors: torch.Tensor) -> torch.device:
    dev = None
    for t in tensors:
        if t is None:
            continue
        if not t.is_cuda:
            raise RuntimeError("moe_distributed_training_amd runs on the GPU only (got a CPU tensor); there is no host fallback")
        if dev is None:
            dev = t.device
        elif t.device != dev:
            raise RuntimeError("all tensors must live on the same device")
    return dev


def stream_ptr(dev: torch.device) -> int:
    return torch.cuda.current_stream(dev).cuda_stream


def ptr(t):
    return 0 if t is None else t.data_ptr()


def is64(t: torch.Tensor) -> int:
    if t.dtype == torch.int64:
        return 1
    if t.dtype == torch.int32:
        return 0
    raise TypeError(f"index tensors must be int32 or int64, got {t.dtype}")


def workspace(nbytes: int, dev: torch.device) -> torch.Tensor:
    return torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=dev)
