"""The reduction kernels' lane and row splits at the sizes where they change:
a few lanes a slice, a whole wave, a slice cut over blocks; columns narrower
than a word, narrower than a tile, tiles of 64 and of fewer lanes, runs of rows
and rows apart, several outer indexes a block, a depth split over blocks; and all
of them starting off 16 bytes.  Extremes and arg-reductions are exact, with NaNs, infinities and ties
among the values; sums, means and variances are within the bound of
tests/test_gpu_reduce.py of f64."""

import ctypes

import numpy as np
import pytest

from oracle import binding as oracle
from tensorcrate_amd import lib
from tensorcrate_amd.tensor import Tensor, TensorView, contiguous_strides
from tests.common import KINDS, KIND_NAMES, bits_equal, to_kind, widen
from tests.test_gpu_reduce import check_sum_like

pytestmark = pytest.mark.gpu

# (shape, folded axes).  Rows: every count of lanes from one to 64, with and
# without a part word, whole groups of words and parts of them.
ROWS = [([5, n], [1]) for n in (2, 3, 4, 7, 8, 9, 15, 16, 33, 63, 64, 65, 127, 130, 255, 513, 1023, 1024, 2049, 5000)]
# Enough rows that variances and arg-reductions take few lanes a row too; 125
# words of 16-bit elements are a whole round of some lanes only.
ROWS += [([9000, n], [1]) for n in (100, 257, 1000)]
ROWS += [([700, 37], [1]), ([3, 40, 61], [2]), ([1, 70001], [1]), ([3, 50011], [1]), ([2, 3, 30001], [1, 2])]
# Columns: narrower than any word, odd, a tile, tiles, with outer axes; depths
# within a group, of a few rounds, and split.
COLUMNS = [([d, c], [0]) for d in (2, 5, 33, 700) for c in (2, 3, 5, 8, 11, 16, 31, 64, 65, 257)]
COLUMNS += [([d, c], [0]) for d in (3, 4, 9, 17) for c in (3, 16, 33, 64)]
# Several outer indexes a block, and a last block of fewer: one group each and
# more, narrow rows and wide, with one column a lane and with words.
COLUMNS += [([o, d, c], [1]) for o, d, c in [(301, 3, 2), (301, 8, 3), (130, 33, 7), (97, 70, 5), (3000, 20, 10),
                                             (701, 6, 33), (2500, 50, 33), (53, 9, 64), (40, 17, 100), (9, 30, 130)]]
COLUMNS += [([9000, c], [0]) for c in (2, 7, 11, 40, 130)] + [([6, 77, 57], [1]), ([3, 300, 9], [1]), ([40, 9, 130], [0, 1])]
CASES = ROWS + COLUMNS


def views(values, kind, shape):
    """The array whole, and one element into a longer storage."""
    flat = to_kind(values, kind).reshape(-1)
    yield Tensor.from_numpy(flat.reshape(shape), kind).view()
    longer = np.concatenate([flat[:1], flat, flat[:3]])
    storage = Tensor.from_numpy(longer, kind).storage
    yield TensorView(storage, tuple(shape), contiguous_strides(shape), 1)


@pytest.mark.parametrize("kind", KINDS, ids=[KIND_NAMES[k] for k in KINDS])
def test_sums_means_and_variances(kind):
    for shape, axes in CASES:
        x = np.random.default_rng(sum(shape)).standard_normal(shape).astype(np.float32) + np.float32(0.5)
        for view in views(x, kind, shape):
            wide = widen(kind, to_kind(x, kind)).reshape(shape).astype(np.float64)
            depth = int(np.prod([shape[a] for a in axes]))
            fold = tuple(axes)
            scale = np.abs(wide).sum(fold).reshape(-1)
            got = widen(kind, view.sum_axes(axes).to_numpy()).reshape(-1)
            check_sum_like(got, wide.sum(fold).reshape(-1), scale, depth, kind, ("sum", shape, view.offset))
            got = widen(kind, view.mean_axes(axes).to_numpy()).reshape(-1)
            check_sum_like(got, wide.mean(fold).reshape(-1), scale / depth, depth, kind, ("mean", shape, view.offset))
            got = widen(kind, view.var_axes(axes).to_numpy()).reshape(-1)
            want = wide.var(fold).reshape(-1)
            spread = want + np.abs(wide).max(fold).reshape(-1) ** 2 / depth
            check_sum_like(got, want, spread, depth, kind, ("var", shape, view.offset))


@pytest.mark.parametrize("kind", KINDS, ids=[KIND_NAMES[k] for k in KINDS])
def test_extremes_and_arg_reductions_with_specials(kind):
    for shape, axes in CASES:
        rng = np.random.default_rng(sum(shape) + 1)
        x = rng.integers(-9, 9, shape).astype(np.float32)  # ties everywhere
        x.reshape(-1)[rng.integers(0, x.size, x.size // 9 + 1)] = np.nan
        x.reshape(-1)[rng.integers(0, x.size, 2)] = [np.inf, -np.inf]
        for view in views(x, kind, shape):
            host = view.storage.as_slice()
            for op, name in ((lib.RMAX, "max_axes"), (lib.RMIN, "min_axes")):
                want = oracle.reduce(kind, host, list(shape), view.offset, list(view.strides), axes, lib.FOLD, op)
                assert bits_equal(getattr(view, name)(axes).to_numpy(), want), (shape, axes, name, view.offset)
            if len(axes) > 1:
                continue
            for op, name in ((lib.RMAX, "argmax"), (lib.RMIN, "argmin")):
                want = oracle.arg_reduce(kind, host, list(shape), view.offset, list(view.strides), axes[0], op)
                got = getattr(view, name)(axes[0]).to_numpy()
                assert np.array_equal(got, want), (shape, axes, name, view.offset)


@pytest.mark.parametrize("columns", [1, 2, 5, 15, 16, 300])
def test_an_empty_fold_called_directly_gives_the_identity(columns):
    # Shape [0, columns] folded along axis 0, straight to the library: the
    # tensor layer answers empty folds itself.
    source, out = lib.Buffer(16), lib.Buffer(4 * columns)
    split = lib.split(0, [columns], [1], [0], [columns])
    for kind, op, want in ((lib.FOLD, lib.SUM, 0.0), (lib.FOLD, lib.RMAX, -np.inf), (lib.FOLD, lib.RMIN, np.inf)):
        lib.call("tc_reduce_axes", lib.F32, source.ptr, 0, ctypes.byref(split), kind, op, 0, out.ptr)
        assert np.all(out.download(np.float32, columns) == np.float32(want))


@pytest.mark.parametrize("depth", [2 ** 31 - 1, 2 ** 31 + 1, 2 ** 32 - 1000])
def test_depths_whose_steps_pass_32_bits(depth):
    # Two columns repeated: a lane's rows are 256 apart, eight in flight.
    view = Tensor.from_numpy(np.array([3.0, -2.0], np.float32)).broadcast_to([depth, 2])
    assert view.max_axes(0).to_numpy().tolist() == [3.0, -2.0]
