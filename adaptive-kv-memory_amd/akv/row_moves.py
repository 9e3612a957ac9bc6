"""Token-row moves over several tensors in one launch (``akv_rows_move``).

The tiers of a cache layer are many small tensors -- keys, values, codes, scales, zeros,
outlier values, positions, importance -- whose token rows are joined, kept, gathered,
appended and scattered together at every update.  A ``RowMoves`` collects such jobs on
tensors laid out (B, H, T, C), or (T,), and runs them as one launch on the current stream."""
from __future__ import annotations

import ctypes
import struct
from typing import Optional

import torch
from torch.autograd import forward_ad
from torch.utils._device import DeviceContext

from . import _native as nat

SAME, KEEP, GATHER, SCATTER = range(4)
_COPY, _WIDEN, _FILL, _COUNT = range(4)
_FLOATS = (torch.float16, torch.bfloat16, torch.float32)


_dispatch_modes, _function_modes = torch._C._len_torch_dispatch_stack, torch._C._len_torch_function_stack
_jit_tracing, _function_mode, _compiling = torch._C._is_tracing, torch._C._get_function_stack_at, torch.compiler.is_compiling


def observed() -> bool:
    """Whether something has to see the operations themselves: a dispatch or function mode (a
    trace, fake tensors, a logger; torch's default-device context is none of these), torch.jit
    tracing or compilation."""
    if _compiling() or _dispatch_modes() or _jit_tracing():
        return True
    n = _function_modes()
    return n != 0 and any(type(_function_mode(i)) is not DeviceContext for i in range(n))


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


# the fields of an akv_rows_job, packed in one call (a ctypes structure costs three times that)
_JOB = struct.Struct("@12q7if")
assert _JOB.size == ctypes.sizeof(nat.RowsJob)


class RowMoves:
    takes = staticmethod(movable)

    def __init__(self):
        self._jobs = []
        self._hold = []

    def copy(self, dst: torch.Tensor, src: torch.Tensor, n: int, rows: int = SAME, at: int = 0, value: float = 1.0):
        """``n`` rows of ``src`` to the rows of ``dst`` from ``at`` on (SCATTER: to the listed
        rows); float32 destinations take 16-bit floats widened, and float32 times ``value``."""
        if n == 0:
            return
        if not (src.is_cuda and dst.is_cuda):
            nat.require_device(src, dst)
        ss, ds, st, dt = src.shape, dst.shape, src.stride(), dst.stride()
        se, de = src.element_size(), dst.element_size()
        if len(ss) == 1:
            B = H = C = 1
            rows_in, rows_out = ss[0], ds[0]
            sb = sh = db = dh = 0
            s_row, d_row = st[0] * se, dt[0] * de
            fits = len(ds) == 1
        else:
            B, H, rows_in, C = ss
            rows_out = ds[2]
            sb, sh, s_row = st[0] * se, st[1] * se, st[2] * se
            db, dh, d_row = dt[0] * de, dt[1] * de, dt[2] * de
            fits = (B, H, C) == (ds[0], ds[1], ds[3]) and (C == 1 or (st[3] == 1 and dt[3] == 1))
        if not fits:
            raise ValueError(f"row moves between {tuple(ss)} {st} and {tuple(ds)} {dt}")
        if rows == SCATTER:
            past = n > rows_out or n > rows_in
        else:
            past = n > rows_in or at + n > rows_out
        if past:
            raise ValueError("row moves past a tensor's rows")
        widen = src.dtype != dst.dtype or value != 1.0
        if widen and (dst.dtype != torch.float32 or src.dtype not in _FLOATS):
            raise TypeError(f"row moves do not convert {src.dtype} to {dst.dtype}")
        self._hold.append((src, dst))
        self._jobs.append(_JOB.pack(
            src.data_ptr(), dst.data_ptr() + at * d_row, sb, sh, s_row, db, dh, d_row, n,
            rows_out if rows == SCATTER else rows_in, 0, 0, B, H, C, se,
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
        row = e * dst.stride(0)
        self._hold.append((dst, dst))
        self._jobs.append(_JOB.pack(0, dst.data_ptr() + at * row, 0, 0, 0, 0, 0, row, n, n, start, step, 1, 1, 1, e,
                                    kind, SAME, 0, value))

    def run(self, idx: Optional[torch.Tensor] = None, n_idx: int = 0):
        """Launch the collected jobs; ``idx``: the first ``n_idx`` entries of an int64 list."""
        if not self._jobs:
            return
        if idx is not None and (not idx.is_cuda or idx.dtype != torch.int64 or (n_idx > 1 and idx.stride(-1) != 1) or n_idx > idx.numel()):
            raise ValueError("row moves take an int64 list of consecutive entries on the device")
        jobs = (nat.RowsJob * len(self._jobs)).from_buffer_copy(b"".join(self._jobs))
        nat.check(nat.load().akv_rows_move(jobs, len(self._jobs), idx.data_ptr() if n_idx else None, n_idx,
                                           nat.stream_of(self._hold[0][1])), "row moves")
        self._jobs, self._hold = [], []


class _TorchMoves:
    """The same jobs as torch's own operations, one after another."""

    def __init__(self):
        self._jobs = []

    def takes(self, out_dtype: torch.dtype, *tensors: torch.Tensor) -> bool:
        return False

    def copy(self, dst, src, n, rows=SAME, at=0, value=1.0):
        self._jobs.append((self._copy, dst, src, n, rows, at, value))

    def fill(self, dst, n, value, at=0):
        self._jobs.append((lambda idx, part: part.fill_(value), dst.narrow(0, at, n)))

    def count(self, dst, n, start, step=1, at=0):
        self._jobs.append((lambda idx, part: part.copy_(
            torch.arange(n, dtype=part.dtype, device=part.device) * step + start), dst.narrow(0, at, n)))

    def run(self, idx=None, n_idx=0):
        for job, *args in self._jobs:
            job(None if idx is None else idx[:n_idx], *args)
        self._jobs = []

    @staticmethod
    def _copy(idx, dst, src, n, rows, at, value):
        ax = 0 if src.dim() == 1 else 2
        if rows == KEEP:
            mask = torch.ones(src.shape[ax], dtype=torch.bool, device=src.device)
            if idx is not None:
                mask[idx] = False
            src = src.index_select(ax, mask.nonzero().flatten()[:n])
        elif rows == GATHER:
            src = src.index_select(ax, idx[:n])
        else:
            src = src.narrow(ax, 0, n)
        if value != 1.0:
            src = src.float() * value
        if rows == SCATTER:
            dst.index_copy_(ax, idx[:n], src.to(dst.dtype))
        else:
            dst.narrow(ax, at, n).copy_(src)


def row_moves():
    """A collector of row moves, by torch's own operations where somebody looks on."""
    return _TorchMoves() if observed() else RowMoves()
