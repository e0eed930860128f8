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


def reduction(kind, op, shape, axis):
    """The maximum or its index along `axis`, into the leading part of `out`."""
    n, size = int(np.prod(shape)), lib.DTYPE_SIZE[kind]
    source, out = lib.Buffer(n * size), lib.Buffer(n // shape[axis] * 4)
    zero = np.zeros(1, lib.NUMPY_TYPE[kind])
    lib.call("tc_fill", source.ptr, n, size, zero.ctypes.data)
    steps = [int(np.prod(shape[k + 1:])) for k in range(len(shape))]
    kept = [k for k in range(len(shape)) if k != axis]
    split = lib.split(0, [shape[k] for k in kept], [steps[k] for k in kept], [shape[axis]], [steps[axis]])
    if op == "argmax":
        return lambda: lib.call("tc_arg_reduce", kind, source.ptr, n, ctypes.byref(split), lib.RMAX, out.ptr)
    return lambda: lib.call("tc_reduce_axes", kind, source.ptr, n, ctypes.byref(split), lib.FOLD, lib.SUM, 0, out.ptr)


@pytest.mark.parametrize("op", ["sum", "argmax"])
@pytest.mark.parametrize("columns,outers", [(2, 500_000), (8, 100_000), (15, 50_000)])
def test_narrow_columns_under_many_outer_indexes(op, columns, outers):
    # Half the elements in eight times the outer indexes, against a depth of
    # 64: a block an outer index took 4.7 to 5 times as long (2 columns), 3.1 to 3.7.
    first, second = (outers, 4, columns), (outers // 8, 64, columns)
    assert ratio(reduction(lib.F32, op, first, 1), reduction(lib.F32, op, second, 1), 20) < 1.5


@pytest.mark.parametrize("rows", [300, 3000])
def test_arg_reductions_of_a_part_round_of_words(rows):
    # 125 words a row against 128: 1.6 and 1.8 times as long where a row took
    # few lanes and they left its last whole round at different words.
    assert ratio(reduction(lib.BF16, "argmax", (rows, 1000), 1), reduction(lib.BF16, "argmax", (rows, 1024), 1), 100) < 1.3


def product(kind, m, k, n):
    size = lib.DTYPE_SIZE[kind]
    a, b, c = lib.Buffer(m * k * size), lib.Buffer(k * n * size), lib.Buffer(m * n * size)
    for x, count in ((a, m * k), (b, k * n)):
        zero = np.zeros(1, lib.NUMPY_TYPE[kind])
        lib.call("tc_fill", x.ptr, count, size, zero.ctypes.data)
    return lambda: lib.call("tc_matmul", kind, kind, lib.PLAIN, 0, m, k, n, a.ptr, b.ptr, c.ptr)


@pytest.mark.parametrize("kind,k,n", [(lib.F32, 8, 16), (lib.F32, 32, 16), (lib.BF16, 16, 10)])
def test_products_of_few_columns_over_a_short_k(kind, k, n):
    # 16 x 16 tiles of eight waves, most of them with no K to read, took 1.7, 1.4
    # and 1.3 times as long as 64 columns, which write four times as much.
    assert ratio(product(kind, 1_000_000, k, n), product(kind, 1_000_000, k, 64), 3) < 1.0
