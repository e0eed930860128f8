"""Reductions, copies and broadcasting arithmetic over more than the 256 MiB
Infinity Cache, whose loads (and the arithmetic's stores) are non-temporal, at
sizes and starts that 16 bytes do not divide: part words, last words of columns
that start earlier, several outer indexes a block.  Small whole numbers, so
every result is exact."""

import numpy as np
import pytest

from tensorcrate_amd import lib
from tensorcrate_amd.tensor import Storage, TensorView, contiguous_strides
from tests.common import KIND_NAMES, bits_equal, to_kind

pytestmark = pytest.mark.gpu

KINDS = [lib.F32, lib.BF16]
IDS = [KIND_NAMES[k] for k in KINDS]


def streamed(kind, shape, skew):
    """Whole numbers from -3 to 3, and a view of them `skew` elements into a
    storage of the type (the storage as 8-bit numbers first)."""
    n = int(np.prod(shape))
    base = np.random.default_rng(n).integers(-3, 4, 1_000_003).astype(np.int8)
    values = np.resize(base, n)
    held = np.resize(to_kind(base.astype(np.float32), kind), n)
    storage = Storage.store(kind, np.concatenate([held[:skew], held]))
    return values.reshape(shape), TensorView(storage, tuple(shape), contiguous_strides(shape), skew)


# Columns that words of four and of eight do not divide: in tiles of 64 lanes and
# of fewer, narrow, and under outer indexes of which a block takes several.
@pytest.mark.parametrize("kind", KINDS, ids=IDS)
@pytest.mark.parametrize("shape,axis", [((35001, 2045), 0), ((6_400_001, 11), 0), ((20001, 30, 119), 1),
                                        ((1_600_001, 5, 9), 1), ((35001, 2045), 1), ((250_001, 301), 1), ((3, 25_000_001), 1)])
def test_folds(kind, shape, axis):
    if kind == lib.BF16:
        shape = (shape[0] * 2, *shape[1:])
    x, view = streamed(kind, shape, 1)
    assert x.size * lib.DTYPE_SIZE[kind] > 256 << 20
    assert bits_equal(view.max_axes([axis]).to_numpy().reshape(-1), to_kind(x.max(axis).reshape(-1), kind))
    assert np.array_equal(view.argmin(axis).to_numpy(), x.argmin(axis))
    total = x.sum(axis, dtype=np.int64).reshape(-1)  # below 2^24, so exact in f32
    assert np.abs(total).max() < 1 << 24
    assert bits_equal(view.sum_axes([axis]).to_numpy().reshape(-1), to_kind(total.astype(np.float32), kind))


@pytest.mark.parametrize("kind", KINDS, ids=IDS)
def test_slices_and_joins(kind):
    x, view = streamed(kind, (40001, 2005 * 4 // lib.DTYPE_SIZE[kind]), 1)
    cols = view.shape[1]
    first, second = view.narrow(1, 3, cols // 2 - 1), view.narrow(1, cols // 2 + 2, cols // 2 - 3)
    assert bits_equal(first.contiguous().to_numpy().reshape(-1),
                      to_kind(x[:, 3:cols // 2 + 2].reshape(-1).astype(np.float32), kind))
    width = first.shape[1] + second.shape[1]
    out = Storage(kind, x.shape[0] * width)
    regions = (lib.Region * 2)(*[
        lib.region(v.storage.buffer, v.storage.len, v.shape, v.offset, v.strides, start, [width, 1])
        for v, start in ((second, 0), (first, second.shape[1]))])
    lib.call("tc_assemble", out.width, out.ptr, out.len, regions, 2)
    want = np.concatenate([x[:, cols // 2 + 2:cols // 2 * 2 - 1], x[:, 3:cols // 2 + 2]], 1)
    assert bits_equal(out.as_slice(), to_kind(want.reshape(-1).astype(np.float32), kind))


@pytest.mark.parametrize("kind", KINDS, ids=IDS)
@pytest.mark.parametrize("run", [2045, 4])
def test_broadcasts(kind, run):
    run *= 4 // lib.DTYPE_SIZE[kind] if run == 4 else 1
    rows = (270 << 20) // (run * lib.DTYPE_SIZE[kind])
    x, view = streamed(kind, (rows, run), 1)
    y, other = streamed(kind, (1, run), 3)
    got = view.elementwise(other.broadcast_to((rows, run)), lib.ADD).to_numpy()
    assert bits_equal(np.asarray(got).reshape(-1), to_kind((x + y).reshape(-1).astype(np.float32), kind))
