"""Opt-in ROCTX ranges (``ONDEVICEINFER_NVTX=1``), mirroring ``ondeviceinfer/profiling.py:17-49``.

On PyTorch-ROCm ``torch.cuda.nvtx`` emits ROCTX markers that rocprofv3's
marker trace records.
"""
from __future__ import annotations

import contextlib
import os

import torch

_ENABLED = os.environ.get('ONDEVICEINFER_NVTX', '0') == '1'


class _Off(contextlib.ContextDecorator):
    """Does nothing; re-entrant, and a decorator like the range it stands for."""

    def __enter__(self):
        return None

    def __exit__(self, *exc):
        return None


_OFF = _Off()


@contextlib.contextmanager
def _range(name: str):
    if not torch.cuda.is_available():
        yield
        return
    torch.cuda.nvtx.range_push(name)
    try:
        yield
    finally:
        torch.cuda.nvtx.range_pop()


def nvtx_range(name: str):
    # Off (the default): one shared no-op context, since a linear enters it on every call.
    return _range(name) if _ENABLED else _OFF
