"""Float SpMM on VOID tiles (void/ops.py:148-213): C = A @ B on the MFMA
kernels of libvoid_amd.so: void_spmm_bf16 / void_spmm_f16 when the tiles and
B share a 16-bit dtype, void_spmm_f32 (fp32 tiles and B) otherwise."""

from __future__ import annotations

import ctypes
from typing import Optional

import torch

from . import _lib, _runtime

# Longest work item of the float kernel: it holds an item's block columns in
# one register per lane.
F32_CHUNK = 64


_K16 = {torch.bfloat16: "void_spmm_bf16", torch.float16: "void_spmm_f16"}


def _rings_reach(a, c: torch.Tensor, tile_bytes: int) -> bool:
    """Whether the rings' 31-bit offsets reach A's tiles and all of C."""
    return (a.n_blocks * tile_bytes < _runtime.RING_LIMIT
            and a.shape[0] * c.stride(0) * c.element_size() < _runtime.RING_LIMIT)


def float_spmm(a, b: torch.Tensor, *, out: Optional[torch.Tensor] = None, bias: Optional[torch.Tensor] = None,
               activation: int = _lib.ACT_NONE, bias_per_row: bool = False, round_before_bias: bool = False,
               plan: Optional["_runtime.DevicePlan"] = None) -> torch.Tensor:
    """activation(A @ B + bias) for a float VOIDTensor A; the output has B's
    dtype (f32, bf16 or f16), as the reference's kernels write.  bias is [N]
    (per column), or [M] with bias_per_row (fusion.py:202-304);
    round_before_bias gives the bits of a bias added to the stored product.  ``plan``
    (work items of at most 64 tiles) replaces the default partition."""
    if b.dim() != 2:
        raise ValueError("B must be 2-D")
    M, K = a.shape
    if K != b.shape[0]:
        raise ValueError(f"A is {M}x{K} but B has {b.shape[0]} rows")
    _runtime.require_gpu(b, "B")
    N = b.shape[1]
    out_dtype = b.dtype if b.dtype in (torch.float32, torch.bfloat16, torch.float16) else torch.float32
    if out is None:
        out = torch.empty(M, N, dtype=out_dtype, device=b.device)
    elif out.shape != (M, N):
        raise ValueError(f"out must be [{M}, {N}]")
    if a.n_blocks == 0:
        out.zero_()
        if bias is not None:
            out[:] = (bias[:, None] if bias_per_row else bias[None, :]).to(out.dtype)
        return out
    _runtime.require_gpu(a.values, "A")
    if a.values.device != b.device:
        raise ValueError(f"A on {a.values.device}, B on {b.device}")
    if bias is not None:
        if bias.shape != ((M,) if bias_per_row else (N,)):
            raise ValueError(f"bias must be [{M if bias_per_row else N}]")
        bias = _runtime.vector_f32(bias, b.device)
    lib = _lib.lib()
    target = out if (out.stride(1) == 1 and out.stride(0) >= N) else torch.empty_like(out)
    # 16-bit tiles times a B of the same dtype run on the 16-bit MFMA (the
    # reference's tl.dot takes them as they are); everything else on the fp32
    # kernel, whose products of widened 16-bit values are the same numbers.
    entry = "void_spmm_f32"
    bk = None
    if a.values.dtype == b.dtype and b.dtype in _K16 and _rings_reach(a, target, 2048):
        bk = _runtime.ring_rows(b, a.n_blocks, a)
    if bk is not None:
        entry = _K16[b.dtype]
        dbsr = a.device_bsr(b.dtype)
    else:
        # A 16-bit column-major B is transposed before it is widened (half the bytes).
        wide = b
        if b.dtype is not torch.float32:
            wide = (b if b.stride(1) == 1 else _runtime.contiguous_2d(b)).to(torch.float32)
        bk = _runtime.ring_rows(wide, a.n_blocks, a) if _rings_reach(a, target, 4096) else None
        if bk is None:
            bk = _runtime.contiguous_2d(wide)
        dbsr = a.device_bsr()
    flags = _lib.DENSE_PADDED_B if _runtime.aligned_rows(bk) else 0
    if round_before_bias:
        flags |= _lib.DENSE_ROUND_BEFORE_BIAS
    if plan is None:
        plan = dbsr.plan(F32_CHUNK)
    elif plan.chunk > F32_CHUNK:
        raise ValueError(f"the float kernel takes work items of at most {F32_CHUNK} tiles, got {plan.chunk}")
    stream = _runtime.raw_stream(out.device)
    ws, ws_bytes = plan.workspace(N, out.device, stream)
    # Fields in the struct's order.
    dense = _lib.DenseArgs(bk.data_ptr(), bk.stride(0), 0, N, 1.0, None, bias.data_ptr() if bias is not None else None,
                           target.data_ptr(), target.stride(0), _runtime.out_code(target.dtype), activation,
                           bias_per_row, flags)
    st = getattr(lib, entry)(dbsr.desc_ref(), ctypes.byref(dense), plan.cplan_ref(),
                             ws.data_ptr() if ws is not None else None, ws_bytes, stream)
    _lib.check(st, entry)
    if target is not out:
        out.copy_(target)
    return out


def void_spmm(a, b: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """C = A @ B for a float VOIDTensor (ops.py:148-213); C has B's dtype."""
    from .int_quant import Int8VOIDTensor
    from .fp8 import FP8VOIDTensor
    if isinstance(a, (Int8VOIDTensor, FP8VOIDTensor)):
        raise TypeError("void_spmm takes a float VOIDTensor; use void_spmm_int8 / void_spmm_fp8 for quantised tiles")
    return float_spmm(a, b, out=out)


# The reference's tensor-core threshold on K (ops.py:28); on gfx950 every
# 32-wide tile feeds the MFMA.
MIN_TENSOR_CORE_K = 16


def compute_optimal_tile_n(N: int) -> int:
    """The reference's TILE_N rule (ops.py:31-42), kept for its callers; the
    gfx950 kernels compute 128-column panels whatever N."""
    if N >= 128:
        return 128
    if N >= 64:
        return 64
    if N >= 32:
        return 32
    if N >= 16:
        return 16
    return 1 << max(0, (int(N) - 1).bit_length())


__all__ = ["void_spmm", "float_spmm", "compute_optimal_tile_n", "MIN_TENSOR_CORE_K"]
