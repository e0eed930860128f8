"""Shapes just past a line of a dispatch against their neighbours on its other
side that move as much or more: the same work may not take several times as
long because a size is a little smaller.  Each pair is timed in turn and the
best of its rounds compared, with a margin well over what rounds differ by and
well under what the line cost where it lay wrong (both stated)."""

import ctypes
import time

import numpy as np
import pytest

from tensorcrate_amd import lib

pytestmark = pytest.mark.gpu


def ratio(first, second, calls):
    """Best time of `first` over that of `second`, `calls` calls a round."""
    best = [float("inf")] * 2
    for call in (first, second):
        call()
    lib.sync()
    for _ in range(15):
        for i, call in enumerate((first, second)):
            start = time.perf_counter()
            for _ in range(calls):
                call()
            lib.sync()
            best[i] = min(best[i], time.perf_counter() - start)
    return best[0] / best[1]


def broadcast_add(kind, rows, run):
    size = lib.DTYPE_SIZE[kind]
    x, y, out = lib.Buffer(rows * run * size), lib.Buffer(run * size), lib.Buffer(rows * run * size)
    for b, n in ((x, rows * run), (y, run)):
        zero = np.zeros(1, lib.NUMPY_TYPE[kind])
        lib.call("tc_fill", b.ptr, n, size, zero.ctypes.data)
    at_x, at_y = lib.strided(0, [run, 1]), lib.strided(0, [0, 1])
    return lambda: lib.call("tc_strided_binary", kind, lib.ARITHMETIC, lib.ADD, 2, lib.dims([rows, run]), x.ptr,
                            rows * run, ctypes.byref(at_x), y.ptr, run, ctypes.byref(at_y), out.ptr)


@pytest.mark.parametrize("kind,run", [(lib.F32, 4), (lib.BF16, 8), (lib.F16, 8)])
def test_broadcasts_over_runs_of_one_word(kind, run):
    # An element a thread where the run was one word: 2.0 (f32), 3.3 (16-bit).
    rows = 10_000_000
    assert ratio(broadcast_add(kind, rows, run), broadcast_add(kind, rows // 2, run * 2), 4) < 1.5
