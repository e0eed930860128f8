"""The 16-bit tiled kernel for products of fewer 256 x 256 tiles than compute
units (csrc/gemm_rules.hpp, launch_direct16): each tile width and number of
stages, at the edges of the tiles and at step counts below, at and past the
stages.

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

# At 256 compute units: at most 256 tiles of 128 x 64 (four stages: 1 to 9 steps
# of 64, whole and not), at most 256 of 128 x 128 (three: 1 to 7), and more (two).
SHAPES = [(1152, k, 1088) for k in (8, 64, 72, 192, 256, 264, 320, 520)] + [
    (1160, 136, 1096), (136, 640, 8008), (2048, 576, 1024),
    (2048, 40, 2048), (1928, 128, 1992), (2048, 192, 1928), (1160, 256, 2040), (1288, 392, 1304), (1992, 448, 2048),
    (2056, 8, 2048), (2184, 136, 2056), (4096, 72, 2040)]


@pytest.mark.parametrize("form", [lib.PLAIN, lib.LEFT, lib.RIGHT], ids=["plain", "left", "right"])
@pytest.mark.parametrize("kind,out_kind", [(lib.BF16, lib.BF16), (lib.BF16, lib.F32), (lib.F16, lib.F16),
                                           (lib.F16, lib.F32)], ids=["bf16", "bf16-f32", "f16", "f16-f32"])
def test_every_shape_and_step_count(kind, out_kind, form):
    for m, k, n in SHAPES:
        rng = np.random.default_rng(m + k + n)
        a = to_kind(rng.uniform(-1, 1, (k, m) if form == lib.LEFT else (m, k)), kind)
        b = to_kind(rng.uniform(-1, 1, (n, k) if form == lib.RIGHT else (k, n)), kind)
        wa, wb = widen(kind, a).astype(np.float64), widen(kind, b).astype(np.float64)
        wa, wb = wa.T if form == lib.LEFT else wa, wb.T if form == lib.RIGHT else wb
        exact, scale = wa @ wb, np.abs(wa) @ np.abs(wb)
        da, db = lib.Buffer.of(a), lib.Buffer.of(b)
        addend = to_kind(rng.uniform(-1, 1, (m, n)), out_kind)
        for c in (None, addend):
            dc = lib.Buffer.of(c if c is not None else np.full((m, n), np.nan if out_kind != lib.BF16 else 0x7FC0,
                                                               HOST[out_kind]))
            lib.call("tc_matmul", kind, out_kind, form, int(c is not None), m, k, n, da.ptr, db.ptr, dc.ptr)
            got = widen(out_kind, dc.download(HOST[out_kind], m * n)).reshape(m, n).astype(np.float64)
            wide = widen(out_kind, c).astype(np.float64) if c is not None else 0.0
            bound = (k + 2) * 2.0 ** -24 * (scale + np.abs(wide)) + UNIT[out_kind] * np.abs(exact + wide) + 1e-30
            if out_kind == lib.F16:
                bound = bound + 2.0 ** -25  # f16's subnormals
            assert np.all(np.abs(got - (exact + wide)) <= bound), (m, k, n, c is not None)
