"""The expert-MLP caller of the MoE layer: w1 / w3 grouped GEMMs, SiLU * mul, w2 grouped GEMM, weighted combine.

Follows ``scattermoe_permute_and_compute`` of the reference (megablocks_utils/config_utils.py:99-185) and the weight
views it builds (``get_mlp_weights`` :28-35, ``get_mlp_weights_lora`` :37-61).  For bf16 tensors of Mixtral-like
shape the three projections run as two fused launches (dual-weight GEMM with SwiGLU epilogue, then w2) through
``moe_mlp_fwd`` / ``moe_mlp_bwd`` of libmoe_hip.so; everything else goes through the same three
``parallel_linear(_lora)`` calls the reference makes, which use the generic HIP kernels.  The sequences of library calls
and their autograd nodes are in csrc/torch_layer.cpp.
"""
from __future__ import annotations

from typing import NamedTuple, Optional, Tuple

import torch
import torch.nn as nn

from .._lib import entry, native, require_gpu
from ..scattermoe_utils.kernels import ops
from ..scattermoe_utils.parallel_experts import parallel_linear
from ..scattermoe_utils.parallel_linear_lora import parallel_linear_lora


# ---------------------------------------------------------------------------------------------------------------
# weight views (reference config_utils.py:28-61)
# ---------------------------------------------------------------------------------------------------------------
def resolve_dtensor(t):
    """The local shard of a DTensor parameter, anything else unchanged (config_utils.py:32,58-59 strip the DTensor
    wrapper the same way before the kernels see the weights)."""
    return t.to_local() if hasattr(t, "to_local") else t


def get_mlp_weights(w: torch.Tensor, ffn_hidden_size: int, hidden_size: int, name: str = "w1") -> torch.Tensor:
    """Storage (E*ffn, hidden) -> the (E, K, N) view the kernels take: w1/w3 (E, hidden, ffn) K-contiguous,
    w2 (E, ffn, hidden) N-contiguous."""
    w = resolve_dtensor(w).view(-1, ffn_hidden_size, hidden_size)
    return w.permute(0, 2, 1) if name in ("w1", "w3") else w


def get_mlp_weights_lora(w: torch.Tensor, lora_A: torch.Tensor, lora_B: torch.Tensor, r: int,
                         ffn_hidden_size: int, hidden_size: int, name: str = "w1"):
    """Adapter storage of the reference (lora_A.weight kept transposed as (E*hidden, r), lora_B.weight (E*ffn, r),
    megablocks_utils/peft_utils.py:37-38,68-70) -> (W, A (E,K,r), B (E,r,N)) views, swapped for w2 (:51-56)."""
    W = get_mlp_weights(w, ffn_hidden_size, hidden_size, name)
    A = resolve_dtensor(lora_A).view(-1, hidden_size, r)
    B = resolve_dtensor(lora_B).view(-1, ffn_hidden_size, r).permute(0, 2, 1)
    if name == "w2":
        A, B = B.permute(0, 2, 1), A.permute(0, 2, 1)
    return W, A, B


class LoraViews(NamedTuple):
    a1: torch.Tensor
    b1: torch.Tensor
    a3: torch.Tensor
    b3: torch.Tensor
    a2: torch.Tensor
    b2: torch.Tensor


def fused_expert_mlp(x, w1, w2, w3, k, sorted_scattered_idxs, expert_offsets, lora: Optional[LoraViews] = None,
                     lora_alpha: float = 1.0, gates: Optional[torch.Tensor] = None, grouped_out: bool = False):
    """Expert MLP on expert-grouped assignments.  x (rows, d); w1, w2, w3 (E, f, d) in the reference's storage
    layout; ``k`` = fan-out of x rows (top_k, or 1 for pre-dispatched rows).  With ``gates`` (T, k) the k expert
    rows of each token are combined and (T, d) is returned; otherwise one row per assignment, in grouped order
    when ``grouped_out`` else at its flat position."""
    return entry("expert_mlp")(x, w1, w2, w3, k, sorted_scattered_idxs, expert_offsets, [] if lora is None else list(lora),
                               lora_alpha, gates, grouped_out)


def scattermoe_permute_and_compute(x, w1, w2, w3, ffn_hidden_size, hidden_size, top_k, bin_ids, indices, num_experts,
                                   lora_pointers=None, moe_expert_model_parallelism=True, expert_offsets=None,
                                   lora_views: Optional[LoraViews] = None, lora_alpha: float = 1.0):
    """Functional form of the reference caller (config_utils.py:99-185).

    x (rows, hidden); w1, w2, w3 storage (E*ffn, hidden); ``bin_ids`` / ``indices`` = sorted expert ids and sorted
    flat positions; ``lora_pointers[name] = (A.weight, B.weight, r, alpha, hidden, ffn)`` as peft_utils.py:127-132
    (or ``lora_views`` / ``lora_alpha``: the six factor views already in (E, K, r) / (E, r, N) form).
    Expert-parallel mode treats x as pre-dispatched rows (fan-out 1) and scatters the output back to ``indices``;
    otherwise the fan-out is top_k and the output stays in grouped order (the caller's ops.scatter combines it)."""
    with torch.no_grad():
        if expert_offsets is None:
            expert_offsets = ops.expert_offsets_from_sorted(bin_ids, num_experts)
    fan = 1 if moe_expert_model_parallelism else top_k
    grouped_out = not moe_expert_model_parallelism
    W = {n: w.view(-1, ffn_hidden_size, hidden_size) for n, w in (("w1", w1), ("w2", w2), ("w3", w3))}
    lora = None
    alpha = 1.0
    if lora_pointers is not None:
        v = {}
        for n in ("w1", "w2", "w3"):
            A, B, r, alpha, hs, fs = lora_pointers[n]
            _, v["a" + n[1]], v["b" + n[1]] = get_mlp_weights_lora(W[n], A, B, r, fs, hs, n)
        lora = LoraViews(v["a1"], v["b1"], v["a3"], v["b3"], v["a2"], v["b2"])
    elif lora_views is not None:
        lora, alpha = lora_views, lora_alpha
    if native.mlp_fast_path(x, W["w1"], W["w2"], W["w3"], [] if lora is None else list(lora)):
        return fused_expert_mlp(x, W["w1"], W["w2"], W["w3"], fan, indices, expert_offsets, lora, alpha, None, grouped_out)
    # generic route: the reference's three calls (:127-166)
    def proj(inp, name, kk, gin, gout):
        Wv = get_mlp_weights(W[name], ffn_hidden_size, hidden_size, name)
        if lora is None:
            return parallel_linear(inp, Wv, kk, bin_ids, indices, None, expert_offsets, None, gin, gout)
        a, b = getattr(lora, "a" + name[1]), getattr(lora, "b" + name[1])
        return parallel_linear_lora(inp, Wv, a, b, a.size(2), alpha, kk, bin_ids, indices, None, expert_offsets, None,
                                    gin, gout)
    h1 = proj(x, "w1", fan, False, True)
    h3 = proj(x, "w3", fan, False, True)
    h = entry("swiglu")(h1, h3)
    return proj(h, "w2", 1, True, grouped_out)


# ---------------------------------------------------------------------------------------------------------------
# whole layer: router -> sort -> expert MLP -> weighted combine, one autograd node
# ---------------------------------------------------------------------------------------------------------------
def moe_layer_forward(x, wg, w1, w2, w3, top_k=2, lora: Optional[LoraViews] = None, lora_alpha: float = 1.0,
                      normalize: bool = True):
    """x (T, d) bf16 -> (out (T, d), expert_weights (T, k) fp32, expert_indices (T, k) int32).
    wg (E, d) router weight; w1, w2, w3 (E, f, d) expert weights in the reference's storage layout."""
    return _layer(x, wg, w1, w2, w3, w1.size(0), w1.size(1), top_k, [] if lora is None else list(lora), lora_alpha, normalize, False)


def _layer(x, wg, w1, w2, w3, E, f, top_k, lora, lora_alpha, normalize, storage):
    if x.size(0) == 0:   # an empty batch routes nothing: empty outputs, and backward leaves every parameter's grad unset
        require_gpu(x, wg, w1, w2, w3)
        return (x.clone(), torch.zeros((0, top_k), dtype=torch.float32, device=x.device),
                torch.zeros((0, top_k), dtype=torch.int32, device=x.device))
    return entry("layer")(x, wg, w1, w2, w3, E, f, top_k, lora, lora_alpha, bool(normalize), storage)


class ScatterMoEBlock(nn.Module):
    """Drop-in for a Mixtral sparse-MoE block built the way the reference builds it: router weight (E, d), expert
    weights w1, w2, w3 stored (E*f, d) (megablocks_utils/sparse_mlp2.py:22-36, HF w2 transposed on load,
    shard_moe_utils.py:153-157), optional LoRA factors stored as peft_utils.py:37-38,68-70 does.  Returns
    ``(hidden, None)`` like the patched ParallelMLP.forward (config_utils.py:75-92); with ``bias=True`` the block owns an
    output bias (megablocks' ``ParallelMLP.bias``) and follows that method's bias branch (config_utils.py:80-84):
    ``(hidden, bias)`` when ``return_bias`` is set, otherwise the single tensor ``hidden + bias``."""

    def __init__(self, hidden_size, ffn_hidden_size, num_experts, top_k=2, lora_r=0, lora_alpha=16.0,
                 dtype=torch.bfloat16, device=None, bias=False, return_bias=False):
        super().__init__()
        self.return_bias = return_bias
        self.bias = nn.Parameter(torch.zeros(hidden_size, dtype=dtype, device=device)) if bias else None
        self.hidden_size, self.ffn_hidden_size = hidden_size, ffn_hidden_size
        self.num_experts, self.top_k, self.lora_r, self.lora_alpha = num_experts, top_k, lora_r, lora_alpha
        kw = dict(dtype=dtype, device=device)
        self.router = nn.Parameter(torch.empty(num_experts, hidden_size, **kw))
        self.w1 = nn.Parameter(torch.empty(num_experts * ffn_hidden_size, hidden_size, **kw))
        self.w2 = nn.Parameter(torch.empty(num_experts * ffn_hidden_size, hidden_size, **kw))
        self.w3 = nn.Parameter(torch.empty(num_experts * ffn_hidden_size, hidden_size, **kw))
        for p in (self.router, self.w1, self.w2, self.w3):
            nn.init.normal_(p, std=0.02)
        if lora_r > 0:
            for n in ("w1", "w2", "w3"):
                a = nn.Parameter(torch.empty(num_experts * hidden_size, lora_r, **kw))
                b = nn.Parameter(torch.zeros(num_experts * ffn_hidden_size, lora_r, **kw))
                nn.init.normal_(a, std=0.02)
                self.register_parameter(f"lora_A_{n}", a)
                self.register_parameter(f"lora_B_{n}", b)
            for p in (self.router, self.w1, self.w2, self.w3) + (() if self.bias is None else (self.bias,)):
                p.requires_grad_(False)

    def lora_views(self) -> Optional[LoraViews]:
        if self.lora_r == 0:
            return None
        v = {}
        for n in ("w1", "w2", "w3"):
            _, a, b = get_mlp_weights_lora(getattr(self, n), getattr(self, f"lora_A_{n}"), getattr(self, f"lora_B_{n}"),
                                           self.lora_r, self.ffn_hidden_size, self.hidden_size, n)
            v["a" + n[1]], v["b" + n[1]] = a, b
        return LoraViews(v["a1"], v["b1"], v["a3"], v["b3"], v["a2"], v["b2"])

    def forward(self, hidden_states: torch.Tensor):
        shape = hidden_states.shape
        x = hidden_states.reshape(-1, shape[-1])
        E, f = self.num_experts, self.ffn_hidden_size
        lora = []
        if self.lora_r > 0:   # the factors in their storage, in the order a1, b1, a3, b3, a2, b2 (w2's are swapped, see lora_views)
            lora = [resolve_dtensor(t) for t in (self.lora_A_w1, self.lora_B_w1, self.lora_A_w3, self.lora_B_w3, self.lora_B_w2, self.lora_A_w2)]
        out = _layer(x, resolve_dtensor(self.router), resolve_dtensor(self.w1), resolve_dtensor(self.w2), resolve_dtensor(self.w3), E, f,
                     self.top_k, lora, self.lora_alpha, True, True)[0]
        out = out.view(shape)
        if self.bias is not None:
            if self.return_bias:
                return out, self.bias
            return out + self.bias
        return out, None
