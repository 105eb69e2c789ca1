"""Adapter-free siblings the reference imports from scattermoe (megablocks_utils/config_utils.py:19-23,124-125):
``ParallelLinear`` / ``parallel_linear`` / ``ParallelExperts``.  Same kernels as the LoRA path with A = B = None;
the backward additionally produces the expert weight gradient dW[e] = X_e^T dY_e."""
from __future__ import annotations

import torch
import torch.nn as nn

from .._lib import entry


class ParallelLinear:
    """One autograd node (C++); its backward returns the gradients of ``x``, ``expert_weights`` and ``gates``."""

    @staticmethod
    def apply(x, expert_weights, k, sorted_expert_idxs, sorted_scattered_idxs, padded_block_idxs, expert_offsets,
              gates=None, grouped_in=False, grouped_out=False):
        return entry("linear")(x, expert_weights, None, None, 1, 0, k, sorted_expert_idxs, sorted_scattered_idxs,
                               expert_offsets, gates, grouped_in, grouped_out)


def parallel_linear(inputs, expert_weights, k, sorted_expert_idxs, sorted_scattered_idxs, padded_block_idxs,
                    expert_offsets, gates=None, grouped_in=False, grouped_out=False):
    return ParallelLinear.apply(inputs, expert_weights, k, sorted_expert_idxs, sorted_scattered_idxs,
                                padded_block_idxs, expert_offsets, gates, grouped_in, grouped_out)


class ParallelExperts(nn.Module):
    """``weight`` (num_experts, output_size, input_size), N(0, 0.02) init; forward multiplies by weight^T."""

    def __init__(self, num_experts, input_size, output_size, device=None, dtype=None) -> None:
        super().__init__()
        self.weight = nn.Parameter(torch.empty(num_experts, output_size, input_size, device=device, dtype=dtype))
        self.num_experts, self.input_size, self.output_size = num_experts, input_size, output_size
        self.reset_parameters()

    def extra_repr(self):
        return f"num_experts={self.num_experts}, input_size={self.input_size}, output_size={self.output_size}"

    def reset_parameters(self) -> None:
        nn.init.normal_(self.weight, std=0.02)

    def forward(self, inputs, k, sorted_expert_idxs, sorted_scattered_idxs, padded_block_idxs, expert_offsets,
                gates=None, grouped_in=False, grouped_out=False):
        return parallel_linear(inputs, self.weight.permute(0, 2, 1), k, sorted_expert_idxs, sorted_scattered_idxs,
                               padded_block_idxs, expert_offsets, gates=gates, grouped_in=grouped_in,
                               grouped_out=grouped_out)
