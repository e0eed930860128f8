"""The general products (csrc/gemm.hip: gemm16_kernel, gemm32_kernel, and the
transposed copies before them), which take the operands the other kernels
cannot address: 2^31 bytes and more, and more tiles than one dispatch of the
register-fed kernel holds.  Rows from both ends, from the middle and from either
side of byte 2^31 are checked.

The large operand repeats a block of random values; its period divides no row.
Tolerance: relative to sum_k |a_ik b_kj|, a sum of K products in any order is
within K u = K 2^-24 of exact, and a 16-bit result within its rounding's 2^-11
(f16) or 2^-8 (bf16) of that."""

import numpy as np
import pytest

from tensorcrate_amd import lib
from tests.common import to_kind, widen

pytestmark = pytest.mark.gpu

HOST = {lib.F32: np.float32, lib.F16: np.float16, lib.BF16: np.uint16}
UNIT = {lib.F32: 2.0 ** -24, lib.F16: 2.0 ** -11, lib.BF16: 2.0 ** -8}
PERIOD = (1 << 22) - 3


class Repeated:
    """Device storage of `count` elements, element f holding block[f % PERIOD]."""

    def __init__(self, kind, count):
        self.kind, size = kind, HOST[kind](0).itemsize
        self.block = to_kind(np.random.default_rng(kind).uniform(-1, 1, PERIOD), kind)
        self.buffer = lib.Buffer(count * size)
        lib.call("tc_upload", self.buffer.ptr, self.block.ctypes.data, min(count, PERIOD) * size)
        held = min(count, PERIOD)
        while held < count:
            step = min(held // PERIOD * PERIOD, count - held)
            lib.call("tc_copy", self.buffer.ptr + held * size, self.buffer.ptr, step * size)
            held += step

    def at(self, index):
        return widen(self.kind, self.block[index % PERIOD]).astype(np.float64)


def check(kind, out_kind, form, m, k, n, large_a):
    """The product with A (or B) the large operand, at some rows (columns) of it."""
    rng = np.random.default_rng(m + n)
    many = m if large_a else n
    big = Repeated(kind, many * k)
    along_k = form != lib.LEFT if large_a else form == lib.RIGHT
    few = n if large_a else m
    small_along_k = form == lib.RIGHT if large_a else form != lib.LEFT
    small = to_kind(rng.uniform(-1, 1, (few, k) if small_along_k else (k, few)), kind)
    held = lib.Buffer.of(small)
    a, b = (big.buffer, held) if large_a else (held, big.buffer)
    out = lib.Buffer(m * n * HOST[out_kind](0).itemsize)
    nothing = np.array([np.nan if out_kind != lib.BF16 else 0x7FC0], HOST[out_kind])
    lib.call("tc_fill", out.ptr, m * n, nothing.itemsize, nothing.ctypes.data)
    lib.call("tc_matmul", kind, out_kind, form, 0, m, k, n, a.ptr, b.ptr, out.ptr)
    split = (1 << 31) // (k * HOST[kind](0).itemsize)
    picks = np.concatenate([np.arange(70), np.arange(max(split - 40, 0), split + 40), np.arange(many - 300, many),
                            rng.integers(0, many, 100)])
    picks = np.unique(picks[(picks >= 0) & (picks < many)])
    walk = np.arange(k)
    index = picks[:, None] * k + walk if along_k else walk * many + picks[:, None]
    left = big.at(index)
    right = widen(kind, small).astype(np.float64)
    right = right.T if small_along_k else right
    exact, scale = left @ right, np.abs(left) @ np.abs(right)
    if large_a:
        got = np.empty((len(picks), n), HOST[out_kind])
        for i, row in enumerate(picks):
            lib.call("tc_download", got[i].ctypes.data, out.ptr + int(row) * n * got.itemsize, n * got.itemsize)
    else:
        got = np.ascontiguousarray(out.download(HOST[out_kind], m * n).reshape(m, n)[:, picks].T)
    got = widen(out_kind, got).astype(np.float64)
    bound = (k + 2) * 2.0 ** -24 * scale + UNIT[out_kind] * np.abs(exact) + 2.0 ** -25
    assert np.all(np.abs(got - exact) <= bound), (m, k, n, large_a)
    for buffer in (big.buffer, held, out):
        buffer.free()
    lib.call("tc_empty_cache")


@pytest.mark.parametrize("form", [lib.PLAIN, lib.LEFT, lib.RIGHT], ids=["plain", "left", "right"])
@pytest.mark.parametrize("kind,out_kind", [(lib.F32, lib.F32), (lib.BF16, lib.BF16), (lib.BF16, lib.F32),
                                           (lib.F16, lib.F16), (lib.F16, lib.F32)],
                         ids=["f32", "bf16", "bf16-f32", "f16", "f16-f32"])
@pytest.mark.parametrize("large_a", [True, False], ids=["a", "b"])
@pytest.mark.parametrize("k", [1032, 1029], ids=["words", "odd"])
def test_operands_past_2_to_31_bytes(kind, out_kind, form, large_a, k):
    many = (1 << 31) // (k * HOST[kind](0).itemsize) + 301
    check(kind, out_kind, form, many if large_a else 21, k, 21 if large_a else many, large_a)


@pytest.mark.parametrize("form", [lib.PLAIN, lib.LEFT], ids=["plain", "left"])
@pytest.mark.parametrize("kind", [lib.BF16, lib.F16], ids=["bf16", "f16"])
def test_more_small_tiles_than_a_dispatch_holds(kind, form):
    check(kind, kind, form, (1 << 27) - 1, 8, 3, True)
