"""SwiGLU + blockwise-FP8 quant entry points (reference: linghe/utils/silu.py
:279-335, :424-464, :797-950, :1293-1393).  Names, argument order, defaults,
output tensors and scale layouts are the reference's; ``fp8_dtype`` is a
keyword-only extension (the reference always emits e4m3fn).
"""
from __future__ import annotations

import ctypes

import torch

from .. import _lib


_PlanShape = ctypes.c_int64 * 5


class ExpertPlan:
    """Device-side table of the 128-row blocks of one set of per-expert counts.

    The per-expert entry points find each workgroup's tile by a prefix scan over
    ``counts``; handing them a plan (keyword ``plan``) replaces that scan by one
    16-byte read and sizes the launch for exactly the workgroups that have a tile.
    Build it once per set of counts (``build_expert_plan``) and reuse it for every
    per-expert call of the layer: forward, backward, quantiser.  No counterpart in
    the reference, whose kernels are launched on a grid derived from the host-side
    ``splits`` instead.
    """

    __slots__ = ("table", "shape", "blocks", "pad")

    def __init__(self, table: torch.Tensor, shape):
        self.table = table
        self.shape = shape            # ctypes int64[5]: row blocks, whole / halved / quartered ones, pad
        self.blocks = int(shape[0])
        self.pad = int(shape[4])


def build_expert_plan(counts: torch.Tensor, splits, pad: int = 1) -> ExpertPlan:
    """counts: device int32/int64 [n_experts]; splits: the same numbers as a python list;
    pad: 1 for the layouts with the experts back to back (SwiGLU, blockwise quantiser), 16 for
    gather + pad + quant (every expert's region of the outputs rounded up to 16 rows)."""
    shape = _PlanShape()
    flag = 1 if counts.dtype == torch.int64 else 0 if counts.dtype == torch.int32 else -1
    table = _lib.native.expert_plan(counts, flag, splits, pad, ctypes.addressof(shape),
                                     _lib.stream_of(counts) if counts.is_cuda else 0)
    if table is None:
        _counts_flag(counts)  # raises
    return ExpertPlan(table, shape)


def _check_plan(plan: ExpertPlan, blocks: int, device) -> None:
    if plan.blocks != blocks:
        raise ValueError(f"plan was built for {plan.blocks} row blocks, splits give {blocks}")
    if plan.pad != 1:
        raise ValueError("plan was built for the padded layout of gather + pad + quant")
    if plan.table.device != device:
        raise ValueError("plan lives on another device")


def _counts_flag(counts: torch.Tensor) -> int:
    if counts.dtype == torch.int64:
        return 1
    if counts.dtype == torch.int32:
        return 0
    raise TypeError(f"counts must be int32 or int64, got {counts.dtype}")


def _tiles_of(plan, blocks: int, counts: torch.Tensor, device):
    """Where the native call finds its tiles: counts and their flag, or a plan's table and the address of its shape."""
    if plan is None:
        return counts, _counts_flag(counts), None, 0
    _check_plan(plan, blocks, device)
    return None, 0, plan.table, ctypes.addressof(plan.shape)


def _weight_flag(weight: torch.Tensor) -> int:
    if weight.dtype == torch.float32:
        return 0
    if weight.dtype == torch.bfloat16:
        return 1
    raise TypeError(f"weight must be float32 or bfloat16, got {weight.dtype}")


def triton_weighted_silu_forward(x, weight=None, out=None, asm=False):
    """
    compute silu(x)*weight, used in bf16/fp16 training with MoE
    Args:
        x: input tensor, bf16 [M, 2n] (gate | up)
        weight: tokenwise weight [M, 1] or [M], fp32 or bf16
        asm: accepted for compatibility (the reference's alternative exp2 path); ignored
    Returns:
        out: output tensor, bf16 [M, n]
    """
    assert x.is_contiguous()
    _lib.require_device_bf16(x, "x")
    M, N = x.shape
    assert N % 256 == 0
    wflag = 0
    if weight is not None:
        assert weight.is_contiguous() and weight.numel() == M
        wflag = _weight_flag(weight)
    new = _lib.native.swiglu(x, weight, wflag, out, _lib.stream_of(x))
    return new if out is None else out


def triton_weighted_silu_backward(g, x, weight=None):
    """
    backward of triton_weighted_silu_forward
    Args:
        g: gradient tensor, bf16 [M, n]
        x: input tensor, bf16 [M, 2n]
        weight: weight tensor [M, 1] or [M]

    Returns:
        - dx: gradient of x, bf16 [M, 2n]
        - dw: gradient of weight (weight's shape and dtype), None without weight
    """
    assert g.is_contiguous() and x.is_contiguous()
    _lib.require_device_bf16(x, "x")
    _lib.require_device_bf16(g, "g")
    M, N = x.shape
    assert N % 256 == 0
    assert g.shape == (M, N // 2)
    wflag = 0
    if weight is not None:
        assert weight.is_contiguous() and weight.numel() == M
        wflag = _weight_flag(weight)
    return _lib.native.swiglu_bwd(g, x, weight, wflag, _lib.stream_of(x))


def triton_silu_and_block_quant_forward(
    x, out=None, scale=None, round_scale=False, output_mode=2, *, fp8_dtype=torch.float8_e4m3fn
):
    """
    fused silu and blockwise quantization, used in shared expert
    Args:
        x: input tensor, bf16 [M, 2n] (gate | up)
        round_scale: whether round scale to power of 2
        output_mode: one of {0, 1, 2}
            0: only output non-transposed quantized tensor
            1: only output transposed quantized tensor
            2: output both

    Returns:
        - out: quantized tensor [M, n]
        - scale: quantization scale [n/128, M]
        - transpose_output: quantized tensor of transposed output [n, M]
        - transpose_scale: quantization scale of transposed output [ceil(M/128), n]
    """
    assert x.is_contiguous()
    _lib.require_device_bf16(x, "x")
    M, N = x.shape
    n = N // 2
    assert output_mode in (0, 1, 2)
    assert n % 128 == 0 and N == 2 * n
    return _lib.native.swiglu_quant(x, out, scale, int(bool(round_scale)), output_mode, fp8_dtype,
                                    _lib.fp8_kind(fp8_dtype) if M else 0, _lib.stream_of(x))


def triton_silu_and_block_quant_backward(g, x, round_scale=False, *, fp8_dtype=torch.float8_e4m3fn):
    """
    backward of triton_silu_and_block_quant_forward
    Args:
        g: gradient, bf16 [M, n]
        x: input tensor, bf16 [M, 2n]
        round_scale: whether round to power of 2

    Returns:
        - dx: quantized non-transposed gradient [M, 2n]
        - dx_scale: scales of quantization non-transposed gradient [2n/128, M]
        - transpose_dx: quantized transposed gradient [2n, M]
        - transpose_dx_scale: scales of quantization transposed gradient [M/128, 2n]
    """
    assert g.is_contiguous()
    assert x.is_contiguous()
    M, N = x.shape
    n = N // 2
    assert M % 128 == 0 and N % 256 == 0
    assert g.shape == (M, n)
    _lib.require_device_bf16(x, "x")
    _lib.require_device_bf16(g, "g")
    return _lib.native.swiglu_quant_bwd(g, x, int(bool(round_scale)), fp8_dtype,
                                        _lib.fp8_kind(fp8_dtype) if M else 0, _lib.stream_of(x))


def triton_batch_weighted_silu_and_block_quant_forward(
    x,
    weight,
    counts,
    splits=None,
    out=None,
    scale=None,
    round_scale=False,
    output_mode=2,
    *,
    fp8_dtype=torch.float8_e4m3fn,
    plan=None,
):
    """
    silu and blockwise quantize activation in routed experts
    Args:
        x: activation tensor in routed experts, bf16 [M, 2n]
        weight: router prob tensor [M, 1]
        counts: device tensor of token count per expert
        splits: python int list of token count per expert
        round_scale: whether round scale to power of 2
        output_mode: one of {0, 1, 2}
        plan: optional ExpertPlan built from the same counts (same results, no scan of the counts)

    Returns (per-expert packed layouts):
        - out: quantized tensor [M, n]
        - scale: per expert [n/128, count_e] blocks, allocated [M, n/128]
        - transpose_output: per expert [n, count_e] blocks, allocated [M, n]
        - transpose_scale: [sum ceil(count_e/128), n]
    """
    assert splits is not None, "batch mode need splits to launch kernels"
    assert x.is_contiguous() and weight.is_contiguous()
    _lib.require_device_bf16(x, "x")
    M, N = x.shape
    n = N // 2
    assert N <= 8192
    assert n % 128 == 0 and N == 2 * n
    assert output_mode in (0, 1, 2)
    assert weight.numel() == M
    device = x.device
    blocks, _ = _lib.native.expert_blocks(splits)
    tiles, wflag, kind = (None, 0, None, 0), 0, 0
    if M > 0:
        tiles = _tiles_of(plan, blocks, counts, device)
        wflag, kind = _weight_flag(weight), _lib.fp8_kind(fp8_dtype)
    new = _lib.native.batched_swiglu_quant(x, weight, wflag, *tiles, blocks, out, scale, int(bool(round_scale)),
                                           output_mode, fp8_dtype, kind, _lib.stream_of(x))
    return new[0] if out is None else out, new[1] if scale is None else scale, new[2], new[3]


def triton_batch_weighted_silu_and_block_quant_backward(
    g, x, weight, counts, splits=None, round_scale=False, *, fp8_dtype=torch.float8_e4m3fn, plan=None
):
    """
    backward of triton_batch_weighted_silu_and_block_quant_forward
    (plan: optional ExpertPlan built from the same counts)
    Returns:
        - dx: quantized non-transposed gradient [M, 2n]
        - dx_scale: per-expert packed scales, allocated [M, 2n/128]
        - dw: gradient of weight, shape and dtype of weight
        - transpose_dx: per-expert packed transposed gradient, allocated [M, 2n]
        - transpose_dx_scale: [sum ceil(count_e/128), 2n]
    """
    M, N = x.shape
    n = N // 2
    assert n % 128 == 0
    assert g.is_contiguous()
    assert x.is_contiguous() and weight.is_contiguous()
    assert splits is not None, "batch mode need splits to launch kernels"
    _lib.require_device_bf16(x, "x")
    _lib.require_device_bf16(g, "g")
    device = x.device
    blocks, _ = _lib.native.expert_blocks(splits)
    dw = None if type(weight) is torch.Tensor else torch.empty_like(weight)  # (a subclass may have its own)
    tiles, wflag, kind = (None, 0, None, 0), 0, 0
    if blocks != 0:
        tiles = _tiles_of(plan, blocks, counts, device)
        wflag, kind = _weight_flag(weight), _lib.fp8_kind(fp8_dtype)
    new = _lib.native.batched_swiglu_quant_bwd(g, x, weight, wflag, dw, *tiles, blocks, int(bool(round_scale)),
                                               fp8_dtype, kind, _lib.stream_of(x))
    return new if dw is None else (new[0], new[1], dw, new[3], new[4])
