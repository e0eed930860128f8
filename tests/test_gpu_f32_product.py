"""The in-place f32 product kernel (csrc/gemm_kernels.hpp) at the edges of its
tiles and its K steps, in both tile widths and every form.

Tolerance: relative to sum_k |a_ik b_kj|, a sum of K products in any order is
within K u = K 2^-24 of exact; an addend adds its own magnitude and rounding."""

import numpy as np
import pytest

from tensorcrate_amd import lib

pytestmark = pytest.mark.gpu

# Operands of whole 16-byte rows, more than a 64 x 64 tile a compute unit (256):
# one K step with most of it missing (K below 8 goes to another kernel), then one,
# two, three and many, whole and ragged; 128 x 64 tiles (the first seven) and 128 x
# 128, with a last tile of one row or of four columns, and whole.
SHAPES = [(1152, 8, 1152), (1156, 12, 1028), (1152, 32, 1152), (1028, 36, 1156), (1284, 64, 1028), (1156, 68, 1152), (1028, 1000, 1092),
          (2048, 32, 2048), (2048, 64, 2048), (1924, 96, 2048), (2048, 132, 1924), (1924, 260, 1988), (4100, 60, 964)]


@pytest.mark.parametrize("form", [lib.PLAIN, lib.LEFT, lib.RIGHT], ids=["plain", "left", "right"])
def test_every_tile_edge_and_step_count(form):
    rng = np.random.default_rng(form)
    for m, k, n in SHAPES:
        if form == lib.LEFT:
            k += 1 if k < 32 else -1  # neither operand's rows run along K
        a = rng.uniform(-1, 1, (k, m) if form == lib.LEFT else (m, k)).astype(np.float32)
        b = rng.uniform(-1, 1, (n, k) if form == lib.RIGHT else (k, n)).astype(np.float32)
        wa = (a.T if form == lib.LEFT else a).astype(np.float64)
        wb = (b.T if form == lib.RIGHT else b).astype(np.float64)
        exact, scale = wa @ wb, np.abs(wa) @ np.abs(wb)
        da, db = lib.Buffer.of(a), lib.Buffer.of(b)
        addend = rng.uniform(-1, 1, (m, n)).astype(np.float32)
        for c in (None, addend):
            dc = lib.Buffer.of(c if c is not None else np.full((m, n), np.nan, np.float32))
            lib.call("tc_matmul", lib.F32, lib.F32, form, int(c is not None), m, k, n, da.ptr, db.ptr, dc.ptr)
            got = dc.download(np.float32, m * n).reshape(m, n).astype(np.float64)
            wide = c.astype(np.float64) if c is not None else 0.0
            bound = (k + 2) * 2.0 ** -24 * (scale + np.abs(wide)) + 1e-30
            assert np.all(np.abs(got - (exact + wide)) <= bound), (m, k, n, c is not None)
