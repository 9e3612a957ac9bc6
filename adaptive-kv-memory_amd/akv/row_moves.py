"""Token-row moves over several tensors in one launch (``akv_rows_move``).

The tiers of a cache layer are many small tensors -- keys, values, codes, scales, zeros,
outlier values, positions, importance -- whose token rows are joined, kept, gathered,
appended and scattered together at every update.  A ``RowMoves`` collects such jobs on
tensors laid out (B, H, T, C), or (T,), and runs them as one launch on the current stream."""
from __future__ import annotations

import ctypes
from typing import Optional

import torch
from torch.autograd import forward_ad

from . import _native as nat

SAME, KEEP, GATHER, SCATTER = range(4)
_COPY, _WIDEN, _FILL, _COUNT = range(4)
_FLOATS = (torch.float16, torch.bfloat16, torch.float32)


def movable(out_dtype: torch.dtype, *tensors: torch.Tensor) -> bool:
    """Whether ``RowMoves`` can stand in for torch's own cat / indexing of these tensors into
    ``out_dtype``: same dtype, or a 16-bit float to float32, and nothing that has to see the
    operation (autograd in either direction, functorch levels, tensor subclasses)."""
    for t in tensors:
        if type(t) is not torch.Tensor or t.dtype not in _FLOATS or (t.dtype != out_dtype and out_dtype != torch.float32):
            return False
        if (t.requires_grad and torch.is_grad_enabled()) or torch._C._functorch.is_functorch_wrapped_tensor(t):
            return False
    return out_dtype in _FLOATS and forward_ad._current_level < 0


class RowMoves:
    def __init__(self):
        self._jobs = []
        self._hold = []

    @staticmethod
    def _layout(t: torch.Tensor):
        e = t.element_size()
        if t.dim() == 1:
            return 1, 1, 1, 0, 0, t.stride(0) * e
        if t.shape[3] > 1 and t.stride(3) != 1:
            raise ValueError("row moves take rows of consecutive elements")
        return t.shape[0], t.shape[1], t.shape[3], t.stride(0) * e, t.stride(1) * e, t.stride(2) * e

    def copy(self, dst: torch.Tensor, src: torch.Tensor, n: int, rows: int = SAME, at: int = 0, value: float = 1.0):
        """``n`` rows of ``src`` to the rows of ``dst`` from ``at`` on (SCATTER: to the listed
        rows); float32 destinations take 16-bit floats widened, and float32 times ``value``."""
        if n == 0:
            return
        B, H, C, sb, sh, st = self._layout(src)
        b, h, c, db, dh, dt = self._layout(dst)
        if (b, h, c) != (B, H, C):
            raise ValueError(f"row moves between {tuple(src.shape)} and {tuple(dst.shape)}")
        token = 0 if src.dim() == 1 else 2
        rows_in, rows_out = src.shape[token], dst.shape[token]
        if n > (rows_in if rows != SCATTER else rows_out) or at + (n if rows != SCATTER else 0) > rows_out:
            raise ValueError("row moves past a tensor's rows")
        widen = src.dtype != dst.dtype or value != 1.0
        if widen and (dst.dtype != torch.float32 or src.dtype not in _FLOATS):
            raise TypeError(f"row moves do not convert {src.dtype} to {dst.dtype}")
        self._hold.append((src, dst))
        self._jobs.append(nat.RowsJob(
            src.data_ptr(), dst.data_ptr() + at * dt, sb, sh, st, db, dh, dt, n,
            rows_out if rows == SCATTER else rows_in, 0, 0, B, H, C, src.element_size(),
            _WIDEN if widen else _COPY, rows, nat.dtype_code(src.dtype) if widen else 0, value))

    def fill(self, dst: torch.Tensor, n: int, value: float, at: int = 0):
        """``value`` into ``n`` entries of a float32 vector."""
        self._vector(dst, n, at, torch.float32, _FILL, 0, 0, value)

    def count(self, dst: torch.Tensor, n: int, start: int, step: int = 1, at: int = 0):
        """start, start + step, ... into ``n`` entries of an int64 or int32 vector."""
        self._vector(dst, n, at, dst.dtype, _COUNT, start, step, 0.0)

    def _vector(self, dst, n, at, dtype, kind, start, step, value):
        if n == 0:
            return
        if dst.dim() != 1 or dst.dtype != dtype or at + n > dst.shape[0]:
            raise ValueError("fill and count take vectors that hold the entries")
        e = dst.element_size()
        self._hold.append(dst)
        self._jobs.append(nat.RowsJob(None, dst.data_ptr() + at * e * dst.stride(0), 0, 0, 0, 0, 0, e * dst.stride(0),
                                      n, n, start, step, 1, 1, 1, e, kind, SAME, 0, value))

    def run(self, idx: Optional[torch.Tensor] = None, n_idx: int = 0):
        """Launch the collected jobs; ``idx``: the first ``n_idx`` entries of an int64 list."""
        if not self._jobs:
            return
        if idx is not None and (idx.dtype != torch.int64 or (n_idx > 1 and idx.stride(-1) != 1) or n_idx > idx.numel()):
            raise ValueError("row moves take an int64 list of consecutive entries")
        jobs = (nat.RowsJob * len(self._jobs))(*self._jobs)
        hold = self._hold[0]
        like = hold if isinstance(hold, torch.Tensor) else hold[1]
        nat.check(nat.load().akv_rows_move(jobs, len(self._jobs), idx.data_ptr() if n_idx else None, n_idx,
                                           nat.stream_of(like)), "row moves")
        self._jobs, self._hold = [], []
