"""The register-fed product kernel (csrc/gemm_sliced.hpp) at the edges of its
tiles, its turns along K and its rules, in every form and type.

Tolerance: relative to sum_k |a_ik b_kj|, which cancellation cannot shrink, a
sum of K products in any order is within K u = K 2^-24 of exact, and a 16-bit
result within its rounding's 2^-11 (f16) or 2^-8 (bf16) of that; an addend
adds its own magnitude to the scale."""

import numpy as np
import pytest

from tensorcrate_amd import lib
from tests.common import Code, column_broadcast, identity_place, row_broadcast, to_kind, widen

pytestmark = pytest.mark.gpu

HOST = {lib.F32: np.float32, lib.F16: np.float16, lib.BF16: np.uint16}
UNIT = {lib.F32: 2.0 ** -24, lib.F16: 2.0 ** -11, lib.BF16: 2.0 ** -8}
IDS = {lib.F32: "f32", lib.F16: "f16", lib.BF16: "bf16"}

# 16 x 16 tiles (few of them: every K from one lane's 8 up, through a wave's
# chunks and the eight waves' turns), 32 x 32 tiles (128 of them and more,
# sides above 16) and 64 x 64 (sides above 32), whole and ragged, aligned and
# not, and long thin ones.
SHAPES = [(2, 8, 2), (16, 8, 16), (17, 31, 15), (15, 32, 33), (40, 33, 24), (33, 127, 65), (16, 1024, 48),
          (31, 1057, 16), (64, 2085, 50), (512, 96, 256), (500, 70, 301), (33, 64, 4000), (511, 4097, 263),
          (1024, 64, 512), (1000, 130, 601), (35, 77, 8200), (2048, 40, 2047), (9000, 24, 3), (2, 17, 5000)]
# Over 1024 tiles of 16 x 16, which two waves share up to K of 64 in 32 bits and of
# 128 in 16: less than a chunk, whole chunks, the last such K and the next.
SHAPES += [(17000, 8, 3), (16500, 64, 16), (16500, 65, 11), (10, 31, 17000), (16600, 128, 9), (16600, 129, 16)]


def operands(kind, form, m, k, n, seed):
    rng = np.random.default_rng(seed)
    a = to_kind(rng.uniform(-1, 1, (k, m) if form == lib.LEFT else (m, k)), kind)
    b = to_kind(rng.uniform(-1, 1, (n, k) if form == lib.RIGHT else (k, n)), kind)
    wa, wb = widen(kind, a).astype(np.float64), widen(kind, b).astype(np.float64)
    wa, wb = wa.T if form == lib.LEFT else wa, wb.T if form == lib.RIGHT else wb
    return a, b, wa @ wb, np.abs(wa) @ np.abs(wb)


@pytest.mark.parametrize("form", [lib.PLAIN, lib.LEFT, lib.RIGHT], ids=["plain", "left", "right"])
@pytest.mark.parametrize("kind,out_kind", [(lib.F32, lib.F32), (lib.BF16, lib.BF16), (lib.BF16, lib.F32),
                                           (lib.F16, lib.F16), (lib.F16, lib.F32)],
                         ids=["f32", "bf16", "bf16-f32", "f16", "f16-f32"])
def test_every_tile_edge_and_form(kind, out_kind, form):
    for m, k, n in SHAPES:
        a, b, exact, scale = operands(kind, form, m, k, n, m * 7 + k * 3 + n)
        da, db = lib.Buffer.of(a), lib.Buffer.of(b)
        addend = to_kind(np.random.default_rng(k).uniform(-1, 1, (m, n)), out_kind)
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


@pytest.mark.parametrize("kind", [lib.F32, lib.BF16, lib.F16], ids=IDS.get)
@pytest.mark.parametrize("form", [lib.PLAIN, lib.LEFT, lib.RIGHT], ids=["plain", "left", "right"])
def test_operands_at_any_address_and_values_past_the_edges(kind, form):
    # Operands one element off their allocation's alignment, between NaNs: a
    # read past a row's end, or past K, into a result would show.
    for m, k, n in ((50, 45, 39), (130, 131, 129), (600, 37, 700)):
        a, b, exact, scale = operands(kind, form, m, k, n, 5)
        held = []
        for x in (a, b):
            framed = np.full(x.size + 64, np.nan if kind != lib.BF16 else 0x7FC0, HOST[kind])
            framed[1:1 + x.size] = x.reshape(-1)
            held.append(lib.Buffer.of(framed))
        size = HOST[kind](0).itemsize
        framed = np.full(m * n + 2, 3, HOST[kind])
        dc = lib.Buffer.of(framed)
        lib.call("tc_matmul", kind, kind, form, 0, m, k, n, held[0].ptr + size, held[1].ptr + size, dc.ptr + size)
        out = dc.download(HOST[kind], m * n + 2)
        assert out[0] == 3 and out[-1] == 3
        got = widen(kind, out[1:-1]).reshape(m, n).astype(np.float64)
        bound = (k + 2) * 2.0 ** -24 * scale + UNIT[kind] * np.abs(exact) + 2.0 ** -25
        assert np.all(np.abs(got - exact) <= bound), (m, k, n)


@pytest.mark.parametrize("kind", [lib.F32, lib.BF16, lib.F16], ids=IDS.get)
@pytest.mark.parametrize("m,k,n", [(24, 40, 40), (264, 200, 512), (1000, 64, 520), (17000, 56, 16)],
                         ids=["16", "32", "64", "16 of two waves"])
def test_a_program_in_the_epilogue_gives_the_unfused_bits(kind, m, k, n):
    # Every tile's epilogue, interpreted on the first call and compiled from
    # the second, against the product and then the program.
    code = Code()
    p, s, b = code.load(0, 0, kind), code.load(2, 2, kind), code.load(1, 1, kind)
    y = code.binary(lib.SUB, code.binary(lib.MUL, p, s), b)
    code.store(code.compare(lib.MAX, y, code.const(0.125 + m)), kind, 0)
    code.store(p, lib.F32, 1)
    rng = np.random.default_rng(kind)
    a, w, bias, scale = (to_kind(rng.uniform(-1, 1, shape), kind) for shape in ((m, k), (k, n), n, m))
    places = [identity_place(m, n), row_broadcast(n), column_broadcast(m)]
    da, dw, db, ds = (lib.Buffer.of(x) for x in (a, w, bias, scale))
    inputs, size = [(db, n), (ds, m)], HOST[kind](0).itemsize
    product = lib.Buffer(m * n * size)
    lib.call("tc_matmul", kind, kind, lib.PLAIN, 0, m, k, n, da.ptr, dw.ptr, product.ptr)
    plain = [lib.Buffer(m * n * size), lib.Buffer(m * n * 4)]
    lib.fused(kind, code.code, places, [(product, m * n)] + inputs, [(o, m * n) for o in plain], m, n)
    want = (plain[0].download(HOST[kind], m * n), plain[1].download(np.float32, m * n))
    for _ in range(3):
        outs = [lib.Buffer(m * n * size), lib.Buffer(m * n * 4)]
        lib.matmul_epilogue(kind, code.code, places, da, dw, m, k, n, inputs, [(o, m * n) for o in outs])
        got = (outs[0].download(HOST[kind], m * n), outs[1].download(np.float32, m * n))
        for g, wt in zip(got, want):
            assert np.array_equal(g.view(np.uint8), wt.view(np.uint8))
