"""LoRA-enabled grouped linear over ragged expert groups as an autograd Function.

Mirrors scattermoe_utils/parallel_linear_lora.py of the reference: ``ParallelLinearLora`` (:11-149) and the entry
point ``parallel_linear_lora`` (:151-187), same positional arguments.  Differences, on purpose:
  * backward returns one gradient per forward input (14), with ``d_gates`` in the ``gates`` slot -- the reference
    returns 15 values (:136-149), which only works while ``gates`` is None;
  * adapter gradients are the full reductions of the definition (reference ops.py:284-289);
  * ``use_khd`` is accepted and ignored: there is one native implementation.
"""
from __future__ import annotations

from .._lib import entry


class ParallelLinearLora:
    """``apply`` with the reference's 14 positional inputs; one autograd node (C++) whose backward returns the gradients of
    ``x``, both adapter factors and ``gates``."""

    @staticmethod
    def apply(x, expert_weights, expert_lora_A, expert_lora_B, lora_r, lora_alp, k, sorted_expert_idxs,
              sorted_scattered_idxs, padded_block_idxs, expert_offsets, gates=None, grouped_in=False, grouped_out=False):
        return entry("linear")(x, expert_weights, expert_lora_A, expert_lora_B, lora_r, lora_alp, k, sorted_expert_idxs,
                               sorted_scattered_idxs, expert_offsets, gates, grouped_in, grouped_out)


def parallel_linear_lora(inputs, expert_weights, expert_lora_A, expert_lora_B, lora_r, lora_alp, k,
                         sorted_expert_idxs, sorted_scattered_idxs, padded_block_idxs, expert_offsets,
                         gates=None, grouped_in=False, grouped_out=False, use_khd=True):
    """Drop-in for the reference entry point (:151-187); ``use_khd`` has no effect."""
    return ParallelLinearLora.apply(inputs, expert_weights, expert_lora_A, expert_lora_B, lora_r, lora_alp, k,
                                    sorted_expert_idxs, sorted_scattered_idxs, padded_block_idxs, expert_offsets,
                                    gates, grouped_in, grouped_out)
