"""Differentiable float SpMM on VOID tiles (void/autograd.py:99-352).

Forward: C = A @ B on the fp32 kernel (void_spmm_f32).  Backward:
  dL/dB        = A^T @ dL/dC, the same kernel on the transposed tiles with
                 block rows and columns swapped (autograd.py:175-189);
  dL/dA_values = dL/dC @ B^T on the nonzero tiles only, the SDDMM kernel
                 void_sddmm_f32 (autograd.py:191-215).
The block structure's device ordering is computed once per structure and
kept with the module, together with its Stream-K plans; only the tile values
are regathered, since an optimiser updates them in place.  A step of modules
neither plans nor waits for the device, however many there are (4096 x 4096,
3277 tiles, fp32, 1024 tokens: 545 us a step when each built its plans anew, 335
us with the plans kept).
"""

from __future__ import annotations

import threading
import weakref
from collections import OrderedDict
from typing import Any, Optional, Tuple

import torch
from torch.autograd import Function, forward_ad

from . import _runtime
from .format import VOIDTensor, build_bsr_layout
from .ops import float_spmm


class _Structure:
    """The block-row order of a tile set (forward, SDDMM) and of its transpose
    (gradient of B), with the plans that live in them."""

    def __init__(self, key: tuple, block_rows: torch.Tensor, block_cols: torch.Tensor, shape: Tuple[int, int]):
        self.key, self.rows, self.cols, self.shape = key, block_rows, block_cols, tuple(shape)
        self.layout = self._build(block_rows, block_cols, *self.shape)
        self._transposed = None

    @staticmethod
    def _build(rows, cols, M, K):
        return build_bsr_layout(rows, cols, (M + 31) // 32, (K + 31) // 32, rows.device)

    @property
    def transposed(self):
        if self._transposed is None:
            with _LOCK:
                if self._transposed is None:
                    self._transposed = self._build(self.cols, self.rows, *self.shape[::-1])
        return self._transposed


# A structure lives as long as the module that used it last (_OWNED), a forward
# whose backward is still to come (ctx), or among the last MAX_RECENT used
# (VOIDSpMMFunction called on bare tensors); _ALIVE finds it.  Its key is the
# structure tensors' identity and in-place version; it holds the tensors
# themselves, so their memory cannot be handed to other structure tensors
# (same address, version 0) while it lives.  Its device arrays go back to the
# allocator, which waits for the streams they were recorded on
# (BsrLayout.on_stream).
MAX_RECENT = 64
_ALIVE: "weakref.WeakValueDictionary[tuple, _Structure]" = weakref.WeakValueDictionary()
_OWNED: "weakref.WeakKeyDictionary[torch.nn.Module, _Structure]" = weakref.WeakKeyDictionary()
_RECENT: "OrderedDict[tuple, _Structure]" = OrderedDict()
_LOCK = threading.RLock()


def _structure(block_rows: torch.Tensor, block_cols: torch.Tensor, shape: Tuple[int, int],
               owner: Optional[torch.nn.Module] = None) -> _Structure:
    key = (_runtime.source_key(block_rows, block_cols), block_rows.numel(), block_rows.stride(), block_cols.stride(),
           block_rows.dtype, block_cols.dtype, tuple(shape), block_rows.device)
    if owner is not None:
        s = _OWNED.get(owner)
        if s is not None and s.key == key:
            return s
    with _LOCK:
        s = _ALIVE.get(key)
        if s is None:
            s = _ALIVE[key] = _Structure(key, block_rows, block_cols, shape)
        if owner is not None:
            _OWNED[owner] = s
        else:
            _RECENT[key] = s
            _RECENT.move_to_end(key)
            while len(_RECENT) > MAX_RECENT:
                _RECENT.popitem(last=False)
    return s


def _layout(block_rows: torch.Tensor, block_cols: torch.Tensor, shape: Tuple[int, int]):
    """The block-row order of a tile set, with its plans."""
    return _structure(block_rows, block_cols, shape).layout


def _vt(values, block_rows, block_cols, shape, tile_size, n_blocks, layout=None, cls=VOIDTensor) -> VOIDTensor:
    """The tiles as a VOIDTensor whose device copy (fp32 or 16-bit, as the SpMM
    needs) is built on first use in a layout's order."""
    if layout is not None and torch.cuda.is_current_stream_capturing():
        # The layout and its plans may be dropped while the graph lives.
        raise RuntimeError("the differentiable SpMM cannot be captured in a HIP graph; capture void_spmm instead")
    return cls(values=values, block_rows=block_rows, block_cols=block_cols,
               morton_codes=torch.empty(0, dtype=torch.int64, device=values.device), shape=tuple(shape),
               tile_size=tuple(tile_size), nnz_original=0, n_blocks=n_blocks, density=0.0, dtype=values.dtype,
               _bsr_layout=layout)


class _TransposedTiles(VOIDTensor):
    """A^T over A's own tiles: the device copy gathers them transposed."""

    def device_bsr(self, dtype: torch.dtype = torch.float32):
        values = self.values.detach().to(dtype)
        none = torch.empty(0, dtype=torch.float32, device=values.device)
        return _runtime.make_device_bsr(values, none, self.block_rows, self.block_cols, self.shape, self.tile_size,
                                        values.device, True, layout=self._bsr_layout, transpose=True)


def _row_major_grad(grad: torch.Tensor) -> torch.Tensor:
    """grad row-major; itself where it has no storage to copy from (a batched
    gradient: is_grads_batched) or has to stay differentiable (create_graph)."""
    if torch.is_grad_enabled() or not torch._C._has_storage(grad):
        return grad
    return _runtime.contiguous_2d(grad)


class VOIDSpMMFunction(Function):
    """C = A @ B with gradients for the tile values and for B (autograd.py:99-216)."""

    @staticmethod
    def forward(ctx: Any, a_values, a_block_rows, a_block_cols, a_shape, a_tile_size, a_n_blocks, b, row_bias=None,
                owner=None):
        # row_bias [M]: added to C's rows as a constant (SparseLinear gives it
        # its gradient with _RowBias); owner: the module that keeps the structure.
        ctx.structure = None
        if a_n_blocks and a_values.is_cuda:
            ctx.structure = _structure(a_block_rows, a_block_cols, a_shape, owner)
        vt = _vt(a_values.detach(), a_block_rows, a_block_cols, a_shape, a_tile_size, a_n_blocks,
                 ctx.structure and ctx.structure.layout)
        c = float_spmm(vt, b, bias=row_bias, bias_per_row=row_bias is not None, round_before_bias=row_bias is not None)
        ctx.save_for_backward(a_values, a_block_rows, a_block_cols, b)
        ctx.a_shape, ctx.a_tile_size, ctx.a_n_blocks = tuple(a_shape), tuple(a_tile_size), a_n_blocks
        return c

    @staticmethod
    def backward(ctx: Any, grad_output: torch.Tensor):
        a_values, rows, cols, b = ctx.saved_tensors
        M, K = ctx.a_shape
        grad_a = grad_b = None
        # One row-major copy of a token-major gradient serves both products
        # (rows of whole 16-byte chunks where the SpMM would copy it to such).
        grad, padded, at = grad_output, False, None
        if ctx.needs_input_grad[6]:
            at = _vt(a_values.detach(), cols, rows, (K, M), ctx.a_tile_size[::-1], ctx.a_n_blocks,
                     ctx.structure and ctx.structure.transposed, cls=_TransposedTiles)
            if grad_output.shape[1] * grad_output.element_size() % 16 and ctx.a_n_blocks:
                grad = _runtime.ring_rows(grad_output, ctx.a_n_blocks, at, zero_tail=True)
                padded = grad is not None
        if not padded:
            grad = _runtime.contiguous_2d(grad_output)
        if at is not None:
            grad_b = float_spmm(at, grad).to(b.dtype)
            if b.stride(0) == 1 and b.stride(1) >= K > 1:
                # A column-major B (X.t() of token-major activations) gets a
                # gradient of its own layout, which autograd then takes as it is.
                grad_b = _runtime.contiguous_2d(grad_b.t()).t()
        if ctx.needs_input_grad[0]:
            grad_a = _runtime.sddmm_tiles(grad, b, rows, cols, (M, K), a_values.dtype,
                                          layout=ctx.structure and ctx.structure.layout, grad_padded=padded)
        return grad_a, None, None, None, None, None, grad_b, None, None


class _RowBias(Function):
    """The graph's edge to a bias [M] that C already holds: C = (A @ B) + bias[:, None]
    with the addition done in the SpMM's epilogue.  A node of its own, so that
    the bias's gradient alone runs no SpMM and takes batched and differentiable
    gradients, as a separate addition's does; the row-major copy that its sum
    reads (13 us on 2048 x 14336 bf16, 127 us down the columns of the
    token-major one) goes on to the SpMM's backward."""

    @staticmethod
    def forward(ctx: Any, c: torch.Tensor, bias: torch.Tensor):
        ctx.mark_dirty(c)
        return c

    @staticmethod
    def backward(ctx: Any, grad_output: torch.Tensor):
        grad = _row_major_grad(grad_output)
        return grad, grad.sum(1) if ctx.needs_input_grad[1] else None


class VOIDSpMM(torch.nn.Module):
    """A VOID matrix as a module with trainable tile values (autograd.py:219-285)."""

    def __init__(self, void_tensor: VOIDTensor, requires_grad: bool = True):
        super().__init__()
        if requires_grad:
            self.values = torch.nn.Parameter(void_tensor.values.clone())
        else:
            self.register_buffer("values", void_tensor.values.clone())
        self.register_buffer("block_rows", void_tensor.block_rows)
        self.register_buffer("block_cols", void_tensor.block_cols)
        self.shape = void_tensor.shape
        self.tile_size = void_tensor.tile_size
        self.n_blocks = void_tensor.n_blocks

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        squeeze = x.dim() == 1
        if squeeze:
            x = x.unsqueeze(1)
        y = VOIDSpMMFunction.apply(self.values, self.block_rows, self.block_cols, self.shape, self.tile_size,
                                   self.n_blocks, x, None, self)
        return y.squeeze(1) if squeeze else y

    def get_void_tensor(self) -> VOIDTensor:
        return VOIDTensor(values=self.values.data, block_rows=self.block_rows, block_cols=self.block_cols,
                          morton_codes=torch.empty(0, device=self.values.device), shape=self.shape,
                          tile_size=self.tile_size, nnz_original=0, n_blocks=self.n_blocks, density=0.0)


def _observed(m: torch.nn.Module) -> bool:
    """Whether calling m runs more than its class's forward (hooks, a replaced forward)."""
    return bool(m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks
                or "forward" in m.__dict__ or torch.nn.modules.module._has_any_global_hook())


# C of this many bytes (by element size) takes the bias in the SpMM's epilogue.
# Below, an addition of its own, whose autograd nodes cost the host less (a
# 16-bit bias is also widened for the epilogue).  Steps with the epilogue and
# with the addition, us: fp32 4096 x 1024 236 and 276 (307 and 303 where the
# host, in its slower mode, bounds both), 2048 x 2048 206 and 220; bf16
# 4096 x 2048 199 and 189, 8192 x 2048 246 and 260, 14336 x 2048 466 and 603.
BIAS_EPILOGUE_BYTES = {4: 1 << 24, 2: 1 << 25}


class SparseLinear(torch.nn.Module):
    """nn.Linear with a VOID weight: y = x W^T + b (autograd.py:288-352)."""

    def __init__(self, in_features: int, out_features: int, void_tensor: VOIDTensor, bias: bool = True,
                 dtype: Optional[torch.dtype] = None):
        super().__init__()
        if tuple(void_tensor.shape) != (out_features, in_features):
            raise ValueError(f"weight is {tuple(void_tensor.shape)}, expected ({out_features}, {in_features})")
        self.in_features = in_features
        self.out_features = out_features
        self.sparse_weight = VOIDSpMM(void_tensor, requires_grad=True)
        dtype = dtype or void_tensor.dtype
        if bias:
            self.bias = torch.nn.Parameter(torch.zeros(out_features, dtype=dtype))
        else:
            self.register_parameter("bias", None)

    def _bias_in_epilogue(self, x: torch.Tensor) -> bool:
        """Whether w(x) + bias may be one SpMM with the same bits (the product
        rounded before the bias).  Everything else, forward-mode tangents of the
        bias among it, takes the addition of its own."""
        w, bias = self.sparse_weight, self.bias
        esz = x.element_size()
        return (x.dtype in (torch.float32, torch.bfloat16, torch.float16)
                and x.numel() // self.in_features * self.out_features * esz >= BIAS_EPILOGUE_BYTES[esz]
                and type(bias) in (torch.Tensor, torch.nn.Parameter) and x.is_cuda
                and bias.dtype == x.dtype and bias.device == x.device and bias.shape == (self.out_features,)
                and type(w) is VOIDSpMM and w.n_blocks > 0 and not _observed(w)
                and forward_ad.unpack_dual(bias).tangent is None)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        x_flat = x.reshape(-1, self.in_features)
        w, bias = self.sparse_weight, self.bias
        if bias is not None and self._bias_in_epilogue(x):
            y = VOIDSpMMFunction.apply(w.values, w.block_rows, w.block_cols, w.shape, w.tile_size, w.n_blocks,
                                       x_flat.T, bias.detach(), w)
            if bias.requires_grad and torch.is_grad_enabled():
                y = _RowBias.apply(y, bias)
            y = y.T
        else:
            y = w(x_flat.T).T
            if bias is not None:
                y = y + bias
        return y.reshape(x.shape[:-1] + (self.out_features,))

    def extra_repr(self) -> str:
        return f"in_features={self.in_features}, out_features={self.out_features}, bias={self.bias is not None}"


__all__ = ["VOIDSpMMFunction", "VOIDSpMM", "SparseLinear"]
