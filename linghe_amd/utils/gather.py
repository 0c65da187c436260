"""Gather + pad + blockwise-FP8 quant entry point (reference:
linghe/utils/gather.py:960-1113).  Name, argument order, defaults, output
tensors and layouts are the reference's; ``fp8_dtype`` is a keyword-only
extension (the reference always emits e4m3fn).
"""
from __future__ import annotations

import ctypes

import torch

from .. import _lib


def triton_batch_block_pad_permute_with_indices(
    xs, token_count_per_expert, indices, splits, probs=None, round_scale=False, *,
    fp8_dtype=torch.float8_e4m3fn, plan=None
):
    """
    select and quant, used in megatron 0.12 flex moe
    Args:
        xs: [bs, dim] bf16
        token_count_per_expert: device int tensor [n_experts]
        indices: int32 [sum of the counts each rounded up to 16]: expert e's region holds
            the source rows of its tokens followed by padding entries (ignored)
        splits: python int list of token_count_per_expert
        probs: route weights, [bs, n_experts]
        round_scale: whether round scale to power of 2
        plan: optional linghe_amd.utils.silu.ExpertPlan of the same counts built with pad=16

    Returns:
        x_q [M, dim], x_scale [M, dim/128] (per expert [dim/128, padded count]),
        xt_q [M, dim] (per expert [dim, padded count]), xt_scale [blocks, dim],
        prob_output [M] or None
    """
    assert xs.is_contiguous()
    m, N = xs.shape
    assert N % 128 == 0
    _lib.require_device_bf16(xs, "xs")
    n_experts = token_count_per_expert.size(0)
    M = indices.shape[0]
    device = xs.device
    blocks, padded = _lib.native.expert_blocks(splits)
    counts = token_count_per_expert
    if m == 0 or M == 0:
        return _lib.native.batched_pad_permute_quant(xs, counts, 0, None, 0, blocks, indices, probs, 0, 0, 0,
                                                     fp8_dtype, 0, _lib.stream_of(xs))
    assert M == padded, f"indices holds {M} entries, the counts rounded up to 16 add up to {padded}"
    if indices.dtype != torch.int32:
        raise TypeError(f"indices must be int32, got {indices.dtype}")
    assert indices.is_contiguous() and token_count_per_expert.is_contiguous()
    if counts.dtype == torch.int64:
        is64 = 1
    elif counts.dtype == torch.int32:
        is64 = 0
    else:
        raise TypeError(f"token_count_per_expert must be int32 or int64, got {counts.dtype}")
    pbf16 = 0
    if probs is not None:
        assert probs.is_contiguous() and probs.shape == (m, n_experts)
        if probs.dtype == torch.bfloat16:
            pbf16 = 1
        elif probs.dtype != torch.float32:
            raise TypeError(f"probs must be float32 or bfloat16, got {probs.dtype}")
    table, shape = None, 0
    if plan is not None:
        if plan.blocks != blocks or plan.pad != 16 or plan.table.device != device:
            raise ValueError("plan does not belong to these splits / this layout (pad=16) / this device")
        table, shape = plan.table, ctypes.addressof(plan.shape)
    return _lib.native.batched_pad_permute_quant(xs, counts, is64, table, shape, blocks, indices, probs, pbf16, 1,
                                                 int(bool(round_scale)), fp8_dtype, _lib.fp8_kind(fp8_dtype),
                                                 _lib.stream_of(xs))
