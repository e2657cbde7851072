"""Linear layers of a decode step on the HIP path (``aspire_linear``, ``aspire_linear_partials``).

The projections the reference's mixed forward runs through ``nn.Linear``
(aspire/models/sparse_draft_transformer.py:149-177,276; transformer.py:490-502) for the few
token rows of a decode step: weights ``[N, K]`` read once, fp32 accumulation, one rounding to
bf16. ``linear_partials`` leaves the sum over a split of K to its consumer
(``decode_step.add_rms_norm_partials``, ``rope.qk_norm_rope_update_kv_partials``).
``supported`` says which shapes the kernels take; larger batches are library GEMM work.
"""

from __future__ import annotations

import torch

from aspire_amd import _lib

MAX_ROWS = 224


def _rows(t: torch.Tensor) -> bool:
    return (t.dtype == torch.bfloat16 and t.dim() == 2 and t.stride(1) == 1 and t.stride(0) % 8 == 0
            and t.stride(0) < 1 << 22 and t.data_ptr() % 16 == 0)


def supported(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether the kernels take ``x [rows, K]`` against ``w [N, K]``."""
    return (_rows(x) and _rows(w) and 0 < x.shape[0] <= MAX_ROWS and x.shape[1] == w.shape[1]
            and x.shape[1] % 128 == 0 and w.shape[0] % 32 == 0)


def swiglu_pays(rows: int, n: int) -> bool:
    """Whether ``linear(..., swiglu=True)`` is the shorter way to ``n`` columns, against the library's product and
    ``silu_mul``. Past 128 rows a workgroup holds 48 columns and a CU one workgroup, so more than 256 x 48
    take a second round. Own over library time at 136 to 224 rows, weights cold: 12,288 columns 0.82 to 0.93
    (K 2,048 to 5,120), 12,416 1.16 to 1.34, 14,336 1.14 to 1.32, 17,408 1.00 to 1.16, 25,600 1.24 to 1.55; up to 128
    rows 0.4 to 1.0, but 1.1 for 25,600 x 5,120."""
    return rows <= 128 or n <= 256 * 48


def _check(x, w, what):
    _lib.require_cuda(x, w, what=what)
    if not supported(x, w):
        raise ValueError(f"{what}: x [rows <= {MAX_ROWS}, K] and w [N, K] must be bf16 with 16-byte aligned rows, "
                         "K a multiple of 128 and N of 32")


def linear(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor, *, swiglu: bool = False) -> torch.Tensor:
    """``out = x @ w.T`` (bf16 ``[rows, N]``), or with ``swiglu`` ``silu(x @ w[:N/2].T) * (x @ w[N/2:].T)``
    (``[rows, N/2]``) with the reference's bf16 roundings."""
    _check(x, w, "linear")
    _lib.require_cuda(out, what="linear")
    n = w.shape[0] // 2 if swiglu else w.shape[0]
    if out.dtype != torch.bfloat16 or out.shape != (x.shape[0], n) or out.stride(1) != 1:
        raise ValueError("linear: out must be bf16 [rows, N] (N / 2 with swiglu) with contiguous rows")
    rc = _lib.lib().aspire_linear(_lib.ptr(x), x.stride(0), _lib.ptr(w), w.stride(0), _lib.ptr(out), out.stride(0),
                                  x.shape[0], n, x.shape[1], 1 if swiglu else 0, _lib.stream_of(x))
    _lib.check(rc, "linear")
    return out


def linear_splits(rows: int, n: int, k: int) -> int:
    """Slabs ``linear_partials`` writes for these sizes (0: not supported)."""
    return int(_lib.lib().aspire_linear_splits(rows, n, k))


def linear_partials(x: torch.Tensor, w: torch.Tensor, workspace: torch.Tensor) -> torch.Tensor:
    """``[S, rows, N]`` fp32 in ``workspace`` (a flat fp32 buffer): ``x @ w.T`` is their sum over S."""
    _check(x, w, "linear_partials")
    _lib.require_cuda(workspace, what="linear_partials")
    rows, n, k = x.shape[0], w.shape[0], x.shape[1]
    s = linear_splits(rows, n, k)
    if workspace.dtype != torch.float32 or not workspace.is_contiguous() or workspace.numel() < s * rows * n:
        raise ValueError(f"linear_partials: workspace must hold {s * rows * n} contiguous floats")
    rc = _lib.lib().aspire_linear_partials(_lib.ptr(x), x.stride(0), _lib.ptr(w), w.stride(0), _lib.ptr(workspace),
                                           workspace.numel(), rows, n, k, _lib.stream_of(x))
    _lib.check(rc, "linear_partials")
    return workspace.view(-1)[: s * rows * n].view(s, rows, n)


__all__ = ["MAX_ROWS", "supported", "swiglu_pays", "linear", "linear_splits", "linear_partials"]
