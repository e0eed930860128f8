"""Copies and broadcasting arithmetic over runs that start and end off 16
bytes, bit for bit against the oracle: every length around a word, part words,
slices at odd places, and assembles whose pieces go in one launch or must not."""

import numpy as np
import pytest

from oracle import binding as oracle
from tensorcrate_amd import lib
from tensorcrate_amd.tensor import Tensor
from tests.common import KINDS, KIND_NAMES, bits_equal, same_bits, to_kind

pytestmark = pytest.mark.gpu

WIDTHS = [np.uint8, np.uint16, np.float32, np.uint64]


@pytest.mark.parametrize("dtype", WIDTHS, ids=lambda d: np.dtype(d).name)
def test_slices_of_every_length_and_place(dtype):
    x = (np.arange(5 * 6 * 83) % 251).astype(dtype).reshape(5, 6, 83)
    buffer = lib.Buffer.of(x)
    for first, length in [(0, 83), (1, 82), (3, 1), (2, 2), (5, 15), (7, 16), (1, 17), (4, 31), (9, 33), (0, 64), (11, 65)]:
        out = lib.Buffer(5 * 6 * length * x.itemsize + 16)
        guard = np.full(5 * 6 * length + 16 // x.itemsize, 77, dtype)
        lib.call("tc_upload", out.ptr, guard.ctypes.data, guard.nbytes)
        lib.call("tc_strided_copy", x.itemsize, buffer.ptr, x.size, 3, lib.dims([5, 6, length]),
                 lib.ctypes.byref(lib.strided(first, [6 * 83, 83, 1])), out.ptr + x.itemsize * (length % 2))
        got = out.download(dtype, guard.size)
        body = got[length % 2:][:5 * 6 * length].reshape(5, 6, length)
        assert bits_equal(body, x[:, :, first:first + length]), (first, length)
        assert np.all(got[:length % 2] == 77) and np.all(got[length % 2 + 5 * 6 * length:] == 77)


@pytest.mark.parametrize("dtype", WIDTHS, ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("pieces", [2, 3, 8, 9, 20])
def test_concats_of_odd_pieces(dtype, pieces):
    # More pieces than a launch takes, some of them shorter than a word, with
    # the target one element off.
    rng = np.random.default_rng(pieces)
    parts = [rng.integers(0, 200, (3, int(rng.integers(1, 40)), 7)).astype(dtype) for _ in range(pieces)]
    for axis in (1, 2):
        arrays = parts if axis == 1 else [np.ascontiguousarray(p.transpose(0, 2, 1)) for p in parts]
        want = np.concatenate(arrays, axis)
        sources, regions, start = [], [], 0
        steps = [want.shape[1] * want.shape[2], want.shape[2], 1]
        for p in arrays:
            sources.append(lib.Buffer.of(p))
            regions.append(lib.region(sources[-1], p.size, p.shape, 0, [p.shape[1] * p.shape[2], p.shape[2], 1],
                                      start * steps[axis], steps))
            start += p.shape[axis]
        out = lib.Buffer((want.size + 1) * want.itemsize)
        lib.call("tc_assemble", want.itemsize, out.ptr + want.itemsize, want.size,
                 (lib.Region * pieces)(*regions), pieces)
        assert bits_equal(out.download(dtype, want.size + 1)[1:].reshape(want.shape), want), axis


def test_pieces_that_overlap_are_copied_in_order():
    # Each region writes over part of the one before, and the last reads the
    # target itself: the result is the sequential one.
    x = np.arange(400, dtype=np.float32)
    src, dst = lib.Buffer.of(x), lib.Buffer.of(np.zeros(400, np.float32))
    want = np.zeros(400, np.float32)
    regions = []
    for k, (to, length) in enumerate([(0, 200), (100, 150), (90, 33), (249, 60), (300, 100)]):
        regions.append(lib.region(src, 400, [length], 3 * k, [1], to, [1]))
        want[to:to + length] = x[3 * k:3 * k + length]
    regions.append(lib.region(dst, 400, [50], 100, [1], 5, [1]))
    want[5:55] = want[100:150].copy()
    lib.call("tc_assemble", 4, dst.ptr, 400, (lib.Region * len(regions))(*regions), len(regions))
    assert np.array_equal(dst.download(np.float32), want)
    # Rows woven through each other: boxes of two different grids.
    dst = lib.Buffer.of(np.zeros(400, np.float32))
    want = np.zeros((20, 20), np.float32)
    a = lib.region(src, 400, [10, 20], 0, [20, 1], 0, [40, 1])
    b = lib.region(src, 400, [20, 5], 7, [5, 1], 3, [20, 1])
    want[::2] = x[:200].reshape(10, 20)
    want[:, 3:8] = x[7:107].reshape(20, 5)
    lib.call("tc_assemble", 4, dst.ptr, 400, (lib.Region * 2)(a, b), 2)
    assert np.array_equal(dst.download(np.float32).reshape(20, 20), want)


@pytest.mark.parametrize("dtype,run", [(np.uint8, 2 ** 32 - 1), (np.uint8, 2 ** 32 - 15), (np.uint16, 2 ** 32 - 3)])
def test_the_last_word_of_a_run_near_2_to_32(dtype, run):
    # Its first element's index plus a word's elements is past 32 bits.
    size = np.dtype(dtype).itemsize
    source, target = lib.Buffer(run * size), lib.Buffer((run + 40) * size)
    five, nine = np.array([5], dtype), np.array([9], dtype)
    lib.call("tc_fill", source.ptr, run, size, five.ctypes.data)
    lib.call("tc_fill", target.ptr, run + 40, size, nine.ctypes.data)
    end = np.arange(20, 60, dtype=dtype)
    lib.call("tc_upload", source.ptr + (run - 40) * size, end.ctypes.data, end.nbytes)
    region = lib.region(source, run, [run], 0, [1], 3, [1])
    lib.call("tc_strided_write", size, target.ptr, run + 40, lib.ctypes.byref(region))
    got = np.empty(120, dtype)
    lib.call("tc_download", got.ctypes.data, target.ptr + (run + 40 - 120) * size, got.nbytes)
    assert got.tolist() == [5] * 43 + end.tolist() + [9] * 37
    source.free()
    target.free()
    lib.call("tc_empty_cache")


@pytest.mark.parametrize("kind", KINDS, ids=[KIND_NAMES[k] for k in KINDS])
@pytest.mark.parametrize("shape", [(3, 5, 1), (4, 3, 7), (3, 5, 8), (2, 7, 9), (3, 4, 15), (2, 3, 17), (3, 9, 64), (5, 4, 131)])
def test_broadcasts_over_odd_runs(kind, shape):
    a, b, c = shape
    rng = np.random.default_rng(a * b * c)
    x = to_kind(rng.standard_normal((a, b, c + 1)).astype(np.float32), kind)
    others = [(1, b, 1), (a, 1, c), (1, 1, c), (a, b, 1)]
    t = Tensor.from_numpy(x, kind).narrow(2, 1, c)  # every run starts one element on
    for other in others:
        y = to_kind(rng.standard_normal(other).astype(np.float32), kind)
        u = Tensor.from_numpy(y, kind).broadcast_to(shape)
        for op, left, right in ((lib.MUL, t, u), (lib.SUB, u, t)):
            got = left.elementwise(right, op).to_numpy()
            want = oracle.binary(kind, lib.ARITHMETIC, op, list(shape), left.storage.as_slice(), left.offset,
                                 list(left.strides), right.storage.as_slice(), right.offset, list(right.strides))
            assert same_bits(got, np.asarray(want), kind), (other, op)
    # Both operands apart along the runs: permuted views.
    p, q = t.permute([2, 0, 1]), t.permute([2, 0, 1])
    got = p.elementwise(q, lib.ADD).to_numpy()
    want = oracle.binary(kind, lib.ARITHMETIC, lib.ADD, list(p.shape), p.storage.as_slice(), p.offset, list(p.strides),
                         q.storage.as_slice(), q.offset, list(q.strides))
    assert same_bits(got, np.asarray(want), kind)
