"""Products of operands whose rows are not whole 16-byte words (or that start
inside one): the copies of csrc/gemm_padded.hip, one operand's or both, and each
kernel over them, on both sides of the lines between them.

Tolerance: relative to sum_k |a_ik b_kj|, a sum of K products in any order is
within K u = K 2^-24 of exact, and a 16-bit result within its rounding's 2^-11
(f16) or 2^-8 (bf16) of that; an addend adds its own magnitude to the scale."""

import numpy as np
import pytest

from tensorcrate_amd import lib
from tests.common import to_kind, widen

pytestmark = pytest.mark.gpu

HOST = {lib.F32: np.float32, lib.F16: np.float16, lib.BF16: np.uint16}
UNIT = {lib.F32: 2.0 ** -24, lib.F16: 2.0 ** -11, lib.BF16: 2.0 ** -8}

# m, k, n and the elements past a word's start that A and B begin: K odd, M or N
# odd, all of them, one operand's rows aligned and the other's not (either way
# round), aligned rows at odd starts.  The first five are too few multiplications
# for copies; the next have more than a 64 x 64 tile a compute unit (256 of them)
# and less than a 256 x 256 tile; then more, K a pair of steps short of one
# element, past one, and under two steps; then at most a 64 x 64 tile a compute
# unit, in each of the register-fed kernel's tiles.
SHAPES = [(1153, 8, 1157, 0, 0), (1153, 65, 1152, 0, 0), (1152, 64, 1155, 0, 0), (1152, 72, 1152, 1, 0),
          (2047, 33, 2049, 0, 0),
          (1299, 1001, 1031, 1, 1), (1152, 1024, 1152, 1, 0), (1160, 1016, 1096, 0, 3), (1154, 1023, 1160, 0, 0),
          (4097, 127, 4098, 0, 0), (4104, 129, 4096, 0, 0), (4099, 65, 4101, 2, 1), (4096, 256, 4097, 0, 0),
          (1023, 1025, 1021, 0, 0), (513, 4097, 515, 1, 0), (200, 8191, 200, 0, 0), (64, 4097, 1030, 0, 5)]


@pytest.mark.parametrize("form", [lib.PLAIN, lib.LEFT, lib.RIGHT], ids=["plain", "left", "right"])
@pytest.mark.parametrize("kind,out_kind", [(lib.F32, lib.F32), (lib.BF16, lib.BF16), (lib.BF16, lib.F32),
                                           (lib.F16, lib.F16), (lib.F16, lib.F32)],
                         ids=["f32", "bf16", "bf16-f32", "f16", "f16-f32"])
def test_copied_operands_give_the_product(kind, out_kind, form):
    nothing = np.nan if kind != lib.BF16 else 0x7FC0
    for m, k, n, start_a, start_b in SHAPES:
        rng = np.random.default_rng(m + k + n)
        a = to_kind(rng.uniform(-1, 1, (k, m) if form == lib.LEFT else (m, k)), kind)
        b = to_kind(rng.uniform(-1, 1, (n, k) if form == lib.RIGHT else (k, n)), kind)
        wa, wb = widen(kind, a).astype(np.float64), widen(kind, b).astype(np.float64)
        wa, wb = wa.T if form == lib.LEFT else wa, wb.T if form == lib.RIGHT else wb
        exact, scale = wa @ wb, np.abs(wa) @ np.abs(wb)
        # What surrounds an operand, and what the copies' memory held, is NaN.
        da = lib.Buffer.of(np.concatenate([np.full(start_a, nothing, HOST[kind]), a.ravel(),
                                           np.full(64, nothing, HOST[kind])]))
        db = lib.Buffer.of(np.concatenate([np.full(start_b, nothing, HOST[kind]), b.ravel(),
                                           np.full(64, nothing, HOST[kind])]))
        addend = to_kind(rng.uniform(-1, 1, (m, n)), out_kind)
        for c in (None, addend):
            dc = lib.Buffer.of(c if c is not None else np.full((m, n), np.nan if out_kind != lib.BF16 else 0x7FC0,
                                                               HOST[out_kind]))
            lib.call("tc_matmul", kind, out_kind, form, int(c is not None), m, k, n,
                     da.ptr + start_a * a.itemsize, db.ptr + start_b * b.itemsize, dc.ptr)
            got = widen(out_kind, dc.download(HOST[out_kind], m * n)).reshape(m, n).astype(np.float64)
            wide = widen(out_kind, c).astype(np.float64) if c is not None else 0.0
            bound = (k + 2) * 2.0 ** -24 * (scale + np.abs(wide)) + UNIT[out_kind] * np.abs(exact + wide) + 1e-30
            if out_kind == lib.F16:
                bound = bound + 2.0 ** -25  # f16's subnormals
            assert np.all(np.abs(got - (exact + wide)) <= bound), (m, k, n, start_a, start_b, c is not None)
