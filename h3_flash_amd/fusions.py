"""Row-wise fusions of the MiniMax H3 DiT block on MI355X (HIP, gfx950).

Same function names, arguments and return values as the reference's Triton
wrappers (src/h3_flash/runtime/kernels/fusions.py):

* :func:`fused_rmsnorm_modulate` (fusions.py:194-215)
* :func:`fused_residual_gate_rmsnorm_modulate` (fusions.py:218-248)
* :func:`fused_swiglu` (fusions.py:251-265)
* :func:`fused_qknorm_rope` (fusions.py:268-293), from :mod:`h3_flash_amd.prologue`

Activations are bf16 (the dtype the H3 block runs in); weights and
modulation tables may be bf16 or fp32, table indices int32 or int64. Table
indices outside the table are clamped to it (the reference reads out of
bounds there). Every call is one HIP launch on the current stream.
"""

from __future__ import annotations

import torch

from . import _ext
from .prologue import fused_qknorm_rope

__all__ = [
    "fused_qknorm_rope",
    "fused_residual_gate_rmsnorm_modulate",
    "fused_rmsnorm_modulate",
    "fused_swiglu",
]


def _rows(x: torch.Tensor, name: str, columns: int) -> torch.Tensor:
    """(N, columns) bf16 device view with a contiguous last dimension."""

    if x.dtype != torch.bfloat16:
        raise TypeError(f"{name} must be bfloat16, got {x.dtype}")
    if not x.is_cuda:
        raise RuntimeError(f"{name} must be on a ROCm device, got {x.device}")
    flat = x.reshape(-1, columns)
    return flat if flat.stride(-1) == 1 else flat.contiguous()


def _vector(t: torch.Tensor, columns: int, device: torch.device, name: str) -> torch.Tensor:
    if t.shape[-1] != columns or t.numel() != columns:
        raise ValueError(f"{name} must have {columns} elements, got shape {tuple(t.shape)}")
    t = t.reshape(columns)
    if t.device != device:
        t = t.to(device)
    if t.dtype not in (torch.bfloat16, torch.float32):
        t = t.float()
    return t if t.is_contiguous() else t.contiguous()


def _tables(tables: list[torch.Tensor], columns: int, device: torch.device) -> list[torch.Tensor]:
    out = []
    for t in tables:
        if t.dim() != 2 or t.shape[1] != columns:
            raise ValueError(f"modulation tables must be (rows, {columns}), got {tuple(t.shape)}")
        out.append(t if t.device == device else t.to(device))
    dtype = torch.bfloat16 if all(t.dtype == torch.bfloat16 for t in out) else torch.float32
    out = [t if t.dtype == dtype else t.to(dtype) for t in out]
    # _row_addressable (fusions.py:190-191): the last dimension must be
    # contiguous; broadcast rows (a row stride under the row, e.g. expand())
    # are written out, since the launch takes one row stride per table
    return [t if t.stride(-1) == 1 and t.stride(0) >= columns else t.contiguous() for t in out]


def _index(index: torch.Tensor, device: torch.device) -> torch.Tensor:
    index = index.reshape(-1)
    if index.device != device:
        index = index.to(device)
    if index.numel() == 0:
        raise ValueError("index must not be empty")
    if index.dtype not in (torch.int32, torch.int64):
        index = index.long()
    return index if index.is_contiguous() else index.contiguous()


def _dtype(t: torch.Tensor) -> int:
    return _ext.H3A_DTYPE_F32 if t.dtype == torch.float32 else _ext.H3A_DTYPE_BF16


def _index_args(index: torch.Tensor) -> tuple[int, int, int]:
    return index.data_ptr(), _ext.H3A_DTYPE_I64 if index.dtype == torch.int64 else _ext.H3A_DTYPE_I32, index.numel()


def fused_rmsnorm_modulate(x, weight, scale, shift, index, eps):
    """RMSNorm over the last dimension, times ``weight``, then
    ``* (1 + scale[t]) + shift[t]`` with ``t = index[row % len(index)]``."""

    columns = x.shape[-1]
    flat = _rows(x, "x", columns)
    weight = _vector(weight, columns, x.device, "weight")
    scale, shift = _tables([scale, shift], columns, x.device)
    index = _index(index, x.device)
    output = flat.new_empty((flat.shape[0], columns))
    _ext.rmsnorm_modulate.run(
        x.device, _ext.ABI_VERSION, flat.data_ptr(), output.data_ptr(), weight.data_ptr(), _dtype(weight),
        scale.data_ptr(), shift.data_ptr(), _dtype(scale), scale.stride(0), shift.stride(0),
        min(scale.shape[0], shift.shape[0]), *_index_args(index), flat.shape[0], columns,
        flat.stride(0), output.stride(0), float(eps),
    )
    return output.view(x.shape)


def fused_residual_gate_rmsnorm_modulate(residual, branch, gate, weight, scale, shift, index, eps):
    """``hidden = residual + gate[t] * branch``, then RMSNorm(hidden) * weight
    * (1 + scale[t]) + shift[t]; returns ``(hidden, normed)``."""

    columns = residual.shape[-1]
    if branch.shape != residual.shape:
        raise ValueError(f"residual {tuple(residual.shape)} and branch {tuple(branch.shape)} differ")
    residual_flat = _rows(residual, "residual", columns)
    branch_flat = _rows(branch, "branch", columns)
    if branch.device != residual.device:
        raise ValueError(f"residual and branch must be on one device, got {residual.device} and {branch.device}")
    weight = _vector(weight, columns, residual.device, "weight")
    gate, scale, shift = _tables([gate, scale, shift], columns, residual.device)
    index = _index(index, residual.device)
    rows = residual_flat.shape[0]
    hidden, normed = residual_flat.new_empty((rows, columns)), residual_flat.new_empty((rows, columns))
    _ext.residual_gate_rmsnorm_modulate.run(
        residual.device, _ext.ABI_VERSION, residual_flat.data_ptr(), branch_flat.data_ptr(), hidden.data_ptr(),
        normed.data_ptr(), weight.data_ptr(), _dtype(weight), gate.data_ptr(), scale.data_ptr(), shift.data_ptr(),
        _dtype(gate), gate.stride(0), scale.stride(0), shift.stride(0),
        min(gate.shape[0], scale.shape[0], shift.shape[0]), *_index_args(index), residual_flat.shape[0], columns,
        residual_flat.stride(0), branch_flat.stride(0), hidden.stride(0), normed.stride(0), float(eps),
    )
    return hidden.view(residual.shape), normed.view(residual.shape)


def fused_swiglu(x):
    """``value * silu(gate)`` with ``value, gate = x.chunk(2, -1)``."""

    if x.shape[-1] % 2:
        raise ValueError(f"swiglu needs an even last dimension, got {x.shape[-1]}")
    columns = x.shape[-1] // 2
    flat = _rows(x, "x", x.shape[-1])
    output = flat.new_empty((flat.shape[0], columns))
    _ext.swiglu.run(
        x.device, _ext.ABI_VERSION, flat.data_ptr(), output.data_ptr(), flat.shape[0], columns,
        flat.stride(0), output.stride(0),
    )
    return output.view(*x.shape[:-1], columns)
