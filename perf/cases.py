"""The work this library's performance is measured on.

Each case is one pass through the entry points of ``libtchip`` (the C ABI of
``include/tchip.h``, and the C++ tape behind ``include/tchip_host.h``), called
as a binding calls them: operands, outputs and layout structs are laid out
once, and a pass is the calls alone.  The kinds are the paths a program over
this backend spends its time in:

- ``product``    ``Matrix::matmul`` in its forms (plain, and the transposed
                 forms the backward pass and layers stored out x in use),
                 f32 gradients accumulated or not;
- ``vector``     ``matvec`` and ``vecmat`` over one matrix;
- ``broadcast``  N-d broadcasting arithmetic and the layout copies after it:
                 x*y + z, its last two axes exchanged, a slice, a join;
- ``reduce``     every axis reduction and arg-reduction of one tensor;
- ``layer``      a dense layer's training step: relu(x w + b) forward; from
                 the gradient of x w + b backward, the gradients of w, of b
                 and of what the rectifier before gave as x; and (f32)
                 Adam's update, some steps into a training;
- ``norm``       the layer norm of every row, forward;
- ``network``    the training step of a small network on the C++ tape, read
                 back as a training loop that logs it does.

``exact`` gives the same results in 64 bits, from torch alone.
"""

import ctypes

import numpy as np
import torch

from tensorcrate_amd import lib
from tensorcrate_amd.optim import Adam

DTYPE = {"f32": lib.F32, "f16": lib.F16, "bf16": lib.BF16}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
FORM = {"plain": lib.PLAIN, "left": lib.LEFT, "right": lib.RIGHT}
RATE = 1e-3
STEPS = 20  # Adam's steps before the one a layer's pass takes
EPSILON = 1e-5  # of the layer norm


def listed():
    return [
        # A small square product, the size a first program tries; bound by
        # latency and by how many compute units get a tile.
        {"name": "product f32 512", "kind": "product", "dtype": "f32", "form": "plain", "accumulate": False,
         "m": 512, "k": 512, "n": 512},
        # A large dense product in a 16-bit type: the matrix cores' case.
        {"name": "product bf16 8192", "kind": "product", "dtype": "bf16", "form": "plain", "accumulate": False,
         "m": 8192, "k": 8192, "n": 8192},
        # Sizes that come from data, not from a tile: odd in every extent.
        {"name": "product bf16 odd", "kind": "product", "dtype": "bf16", "form": "plain", "accumulate": False,
         "m": 2047, "k": 1001, "n": 1531},
        # A batch of 16 rows through a layer stored out x in (inference on a
        # few samples): bound by reading the weights.
        {"name": "product f16 16 rows", "kind": "product", "dtype": "f16", "form": "right", "accumulate": False,
         "m": 16, "k": 4096, "n": 4096},
        # One sample through a layer, both ways.
        {"name": "matvec and vecmat f32", "kind": "vector", "dtype": "f32", "rows": 4096, "cols": 4096},
        # Broadcasting over a large activation and the layout copies after it.
        {"name": "broadcast f32 large", "kind": "broadcast", "dtype": "f32", "a": 256, "b": 512, "c": 512},
        # The same over a small odd one, where launches count.
        {"name": "broadcast bf16 odd", "kind": "broadcast", "dtype": "bf16", "a": 31, "b": 257, "c": 131},
        # Every reduction of a 32 MiB tensor.
        {"name": "reduce f32", "kind": "reduce", "dtype": "f32", "a": 64, "b": 128, "c": 1024},
        # The same of a 16-bit tensor with odd rows.
        {"name": "reduce bf16 odd", "kind": "reduce", "dtype": "bf16", "a": 150, "b": 77, "c": 513},
        # A dense layer's training step at the width of the tape's benchmark.
        {"name": "layer f32", "kind": "layer", "dtype": "f32", "m": 4096, "k": 1024, "n": 4096},
        # Layer norm of 16-bit activations, statistics in f32.
        {"name": "norm bf16", "kind": "norm", "dtype": "bf16", "rows": 8192, "cols": 1000},
        # A whole training step of a small network on the tape, ten outputs.
        {"name": "network", "kind": "network", "inputs": 100, "hidden": 256, "outputs": 10, "layers": 3,
         "batch": 64},
    ]


def _spread(rng, low, high):
    """A size between `low` and `high`, even over its logarithm; a third of
    them are rounded down to a multiple of 64, a third to one of 8, where
    they reach it, and a third stay as they fall."""
    size = int(low * ((high + 1) / low) ** rng.random())
    step = rng.choice((1, 8, 64))
    return min(high, size // step * step if size >= max(step, low + step) else size)


def draw(rng):
    kind = rng.choice(("product", "product", "product", "vector", "broadcast", "reduce", "layer", "norm", "network"))
    dtype = rng.choice(("f32", "f16", "bf16"))
    while True:
        if kind == "product":
            case = {"kind": kind, "dtype": dtype, "form": rng.choice(tuple(FORM)),
                    "accumulate": rng.random() < 0.25,
                    "m": _spread(rng, 1, 8192), "k": _spread(rng, 8, 8192), "n": _spread(rng, 1, 8192)}
        elif kind == "vector":
            case = {"kind": kind, "dtype": dtype, "rows": _spread(rng, 16, 8192), "cols": _spread(rng, 16, 8192)}
        elif kind in ("broadcast", "reduce"):
            case = {"kind": kind, "dtype": dtype, "a": _spread(rng, 2, 512), "b": _spread(rng, 8, 512),
                    "c": _spread(rng, 8, 2048)}
        elif kind == "layer":
            case = {"kind": kind, "dtype": dtype, "m": _spread(rng, 16, 4096), "k": _spread(rng, 16, 4096),
                    "n": _spread(rng, 16, 4096)}
        elif kind == "norm":
            case = {"kind": kind, "dtype": dtype, "rows": _spread(rng, 16, 16384), "cols": _spread(rng, 16, 8192)}
        else:
            case = {"kind": kind, "inputs": _spread(rng, 8, 512), "hidden": _spread(rng, 16, 512),
                    "outputs": _spread(rng, 2, 128), "layers": rng.randint(2, 3), "batch": _spread(rng, 8, 512)}
        need = work(case)
        rate = 100e9 if case.get("dtype", "f32") == "f32" else 1.2e12
        if need["flops"] <= rate and need["bytes"] <= 1.5e9:
            return case


# ---- operands ---------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(generator, shape, dtype, scale=1.0):
    return torch.randn(shape, generator=generator, device="cuda").mul_(scale).to(TORCH[dtype])


def _uniform(generator, shape, dtype, low, high):
    return torch.rand(shape, generator=generator, device="cuda").mul_(high - low).add_(low).to(TORCH[dtype])


def _empty(shape, dtype):
    return torch.empty(shape, device="cuda", dtype=TORCH[dtype])


class _Storage:
    """Device storage as ``lib``'s calls take it: something with a ``ptr``."""

    def __init__(self, tensor):
        self.ptr = tensor.data_ptr()


def _operands(*tensors):
    return lib._buffers([(_Storage(t), t.numel()) for t in tensors])


def _product_operands(case, seed):
    g = _generator(seed)
    m, k, n, form = case["m"], case["k"], case["n"], case["form"]
    a = _normal(g, (k, m) if form == "left" else (m, k), case["dtype"])
    b = _normal(g, (n, k) if form == "right" else (k, n), case["dtype"], k ** -0.5)
    out = "f32" if case["accumulate"] else case["dtype"]
    c = _normal(g, (m, n), out) if case["accumulate"] else _empty((m, n), out)
    return a, b, c, out


def _vector_operands(case, seed):
    g = _generator(seed)
    rows, cols, dtype = case["rows"], case["cols"], case["dtype"]
    return (_normal(g, (rows, cols), dtype, cols ** -0.5), _normal(g, (cols,), dtype), _normal(g, (rows,), dtype))


def _broadcast_operands(case, seed):
    g = _generator(seed)
    a, b, c, dtype = case["a"], case["b"], case["c"], case["dtype"]
    return (_normal(g, (a, b, c), dtype), _uniform(g, (1, b, 1), dtype, -1, 1), _uniform(g, (a, 1, c), dtype, -1, 1))


def _reduce_operands(case, seed):
    return _normal(_generator(seed), (case["a"], case["b"], case["c"]), case["dtype"])


def _layer_operands(case, seed):
    g = _generator(seed)
    m, k, n, dtype = case["m"], case["k"], case["n"], case["dtype"]
    return (_normal(g, (m, k), dtype).relu_(), _normal(g, (k, n), dtype, (2 / k) ** 0.5),
            _normal(g, (n,), dtype, 0.1), _normal(g, (m, n), dtype, m ** -0.5))


def _moments(case, seed):
    """Adam's first and second moments of w, then of b, as some steps leave them."""
    g = _generator(seed + 1)
    shapes = ((case["k"], case["n"]), (case["n"],))
    return [(_normal(g, shape, "f32", 0.3), _normal(g, shape, "f32").square_().mul_(1 - 0.999 ** STEPS))
            for shape in shapes]


def _norm_operands(case, seed):
    g = _generator(seed)
    return (_normal(g, (case["rows"], case["cols"]), case["dtype"], 2.0).add_(0.5),
            _uniform(g, (case["cols"],), case["dtype"], 0.5, 1.5))


def _network_operands(case, seed):
    """Weights and biases by layer, then inputs and targets, features x batch."""
    rng = np.random.default_rng(seed)
    widths = [case["inputs"]] + [case["hidden"]] * (case["layers"] - 1) + [case["outputs"]]
    weights = [rng.standard_normal((o, i), dtype=np.float32) * np.float32(np.sqrt(2.0 / i))
               for i, o in zip(widths, widths[1:])]
    biases = [rng.standard_normal(o, dtype=np.float32) * np.float32(0.1) for o in widths[1:]]
    x = rng.standard_normal((widths[0], case["batch"]), dtype=np.float32)
    y = rng.standard_normal((widths[-1], case["batch"]), dtype=np.float32)
    return widths, weights, biases, x, y


# ---- programs (instructions as `lib.fused` documents them) --------------------

LOAD, CONST, BINARY, UNARY, COMPARE, STORE = range(6)
SQRT = 13


def _relu_program(code):
    """max(input 0 + input 1, 0)."""
    return [(LOAD, 0, 0, 0, code, 0, 0.0), (LOAD, 1, 1, 1, code, 0, 0.0), (BINARY, lib.ADD, 2, 0, 1, 0, 0.0),
            (CONST, 0, 3, 0, 0, 0, 0.0), (COMPARE, lib.MAX, 4, 2, 3, 0, 0.0), (STORE, 0, 0, 4, code, 0, 0.0)]


def _relu_backward_program(code):
    """input 0 where input 1 > 0, else 0."""
    return [(LOAD, 0, 0, 0, code, 0, 0.0), (LOAD, 1, 1, 1, code, 0, 0.0), (CONST, 0, 2, 0, 0, 0, 0.0),
            (COMPARE, lib.GREATER, 3, 1, 2, 0, 0.0), (BINARY, lib.MUL, 4, 0, 3, 0, 0.0),
            (STORE, 0, 0, 4, code, 0, 0.0)]


def _norm_program(code, cols):
    """(x - mean) / sqrt(deviations / cols + epsilon) * gamma in f32, stored as `code`."""
    return [(LOAD, 0, 0, 0, code, 0, 0.0), (LOAD, 1, 1, 1, code, 0, 0.0), (LOAD, 2, 2, 2, lib.F32, 0, 0.0),
            (LOAD, 2, 3, 3, lib.F32, 0, 0.0), (CONST, 0, 4, 0, 0, 0, float(np.float32(1.0 / cols))),
            (BINARY, lib.MUL, 3, 3, 4, 0, 0.0), (CONST, 0, 4, 0, 0, 0, EPSILON), (BINARY, lib.ADD, 3, 3, 4, 0, 0.0),
            (UNARY, SQRT, 3, 3, 0, 0, 0.0), (BINARY, lib.SUB, 0, 0, 2, 0, 0.0), (BINARY, lib.DIV, 0, 0, 3, 0, 0.0),
            (BINARY, lib.MUL, 0, 0, 1, 0, 0.0), (STORE, 0, 0, 0, code, 0, 0.0)]


def _grid(rows, cols):
    return (0, 1, 1, [rows], [cols])


# ---- preparation: the calls of one pass, their arguments laid out ---------------


def prepare(case, seed):
    state = {"product": _prepare_product, "vector": _prepare_vector, "broadcast": _prepare_broadcast,
             "reduce": _prepare_reduce, "layer": _prepare_layer, "norm": _prepare_norm,
             "network": _prepare_network}[case["kind"]](case, seed)
    # The library runs on a stream of its own: what torch queued is done
    # before it reads it.
    torch.cuda.synchronize()
    return state


def _prepare_product(case, seed):
    a, b, c, out = _product_operands(case, seed)
    call = ("tc_matmul", (DTYPE[case["dtype"]], DTYPE[out], FORM[case["form"]], int(case["accumulate"]), case["m"],
                          case["k"], case["n"], a.data_ptr(), b.data_ptr(), c.data_ptr()))
    return {"calls": [call], "outputs": {"c": c}, "keep": (a, b)}


def _prepare_vector(case, seed):
    matrix, right, left = _vector_operands(case, seed)
    code, rows, cols = DTYPE[case["dtype"]], case["rows"], case["cols"]
    y, z = _empty(rows, case["dtype"]), _empty(cols, case["dtype"])
    calls = [("tc_matvec", (code, 0, rows, cols, matrix.data_ptr(), right.data_ptr(), y.data_ptr())),
             ("tc_vecmat", (code, rows, cols, left.data_ptr(), matrix.data_ptr(), z.data_ptr()))]
    return {"calls": calls, "outputs": {"matvec": y, "vecmat": z}, "keep": (matrix, right, left)}


def _prepare_broadcast(case, seed):
    x, y, z = _broadcast_operands(case, seed)
    a, b, c, dtype = case["a"], case["b"], case["c"], case["dtype"]
    code, width, n, half = DTYPE[dtype], x.element_size(), a * b * c, b // 2
    shape = (a, b, c)
    out = {"scaled": _empty(shape, dtype), "sum": _empty(shape, dtype), "exchanged": _empty((a, c, b), dtype),
           "middle": _empty((a, half, c), dtype), "joined": _empty((a, b, c), dtype)}
    whole, ptr = lib.strided(0, (b * c, c, 1)), {name: t.data_ptr() for name, t in out.items()}
    y_at, z_at = lib.strided(0, (0, 1, 0)), lib.strided(0, (c, 0, 1))
    exchanged, middle = lib.strided(0, (b * c, 1, c)), lib.strided((b - half) // 2 * c, (b * c, c, 1))
    # The second half of the rows first, then the first.
    regions = (lib.Region * 2)(
        lib.region(ptr["sum"], n, (a, b - half, c), half * c, (b * c, c, 1), 0, (b * c, c, 1)),
        lib.region(ptr["sum"], n, (a, half, c), 0, (b * c, c, 1), (b - half) * c, (b * c, c, 1)))
    calls = [
        ("tc_strided_binary", (code, lib.ARITHMETIC, lib.MUL, 3, lib.dims(shape), x.data_ptr(), n,
                               ctypes.byref(whole), y.data_ptr(), b, ctypes.byref(y_at), ptr["scaled"])),
        ("tc_strided_binary", (code, lib.ARITHMETIC, lib.ADD, 3, lib.dims(shape), ptr["scaled"], n,
                               ctypes.byref(whole), z.data_ptr(), a * c, ctypes.byref(z_at), ptr["sum"])),
        ("tc_strided_copy", (width, ptr["sum"], n, 3, lib.dims((a, c, b)), ctypes.byref(exchanged),
                             ptr["exchanged"])),
        ("tc_strided_copy", (width, ptr["sum"], n, 3, lib.dims((a, half, c)), ctypes.byref(middle), ptr["middle"])),
        ("tc_assemble", (width, ptr["joined"], n, regions, 2)),
    ]
    return {"calls": calls, "outputs": out, "keep": (x, y, z)}


# Name, folded axes, kind, op: the variance is the population's.
REDUCTIONS = [(f"{name} {axes}", axes, kind, op) for axes in ((2,), (0, 1))
              for name, kind, op in (("sum", lib.FOLD, lib.SUM), ("max", lib.FOLD, lib.RMAX),
                                     ("min", lib.FOLD, lib.RMIN), ("mean", lib.MEAN, 0), ("var", lib.VARIANCE, 0))]


def _split(shape, axes):
    strides = (shape[1] * shape[2], shape[2], 1)
    kept = [k for k in range(3) if k not in axes]
    return lib.split(0, [shape[k] for k in kept], [strides[k] for k in kept], [shape[k] for k in axes],
                     [strides[k] for k in axes])


def _prepare_reduce(case, seed):
    x = _reduce_operands(case, seed)
    shape, code = tuple(x.shape), DTYPE[case["dtype"]]
    out, calls = {}, []
    for name, axes, kind, op in REDUCTIONS:
        out[name] = _empty([shape[k] for k in range(3) if k not in axes], case["dtype"])
        split = _split(shape, axes)
        divisor = int(np.prod([shape[k] for k in axes])) if kind == lib.VARIANCE else 0
        calls.append(("tc_reduce_axes", (code, x.data_ptr(), x.numel(), ctypes.byref(split), kind, op, divisor,
                                         out[name].data_ptr())))
    for name, op in (("argmax", lib.RMAX), ("argmin", lib.RMIN)):
        out[name] = torch.empty((shape[0], shape[2]), device="cuda", dtype=torch.int32)
        split = _split(shape, (1,))
        calls.append(("tc_arg_reduce", (code, x.data_ptr(), x.numel(), ctypes.byref(split), op,
                                        out[name].data_ptr())))
    return {"calls": calls, "outputs": out, "keep": (x,)}


def _prepare_layer(case, seed):
    x, w, b, dz = _layer_operands(case, seed)
    m, k, n, dtype = case["m"], case["k"], case["n"], case["dtype"]
    code = DTYPE[dtype]
    y, through, dx = _empty((m, n), dtype), _empty((m, k), dtype), _empty((m, k), dtype)
    dw, db = _empty((k, n), "f32"), _empty(n, dtype)
    relu, backward = _relu_program(code), _relu_backward_program(code)
    relu_code, relu_places = lib._program(relu, [_grid(m, n), (0, 1, 0, [], [])])
    back_code, back_places = lib._program(backward, [_grid(m, k)] * 2)
    split = lib.split(0, [n], [1], [m], [n])
    calls = [
        ("tc_matmul_epilogue", (code, relu_code, len(relu), relu_places, 2, m, k, n, x.data_ptr(), w.data_ptr(),
                                *_operands(b), 1, *_operands(y), 1)),
        ("tc_matmul", (code, lib.F32, lib.LEFT, 0, k, m, n, x.data_ptr(), dz.data_ptr(), dw.data_ptr())),
        ("tc_reduce_axes", (code, dz.data_ptr(), m * n, ctypes.byref(split), lib.FOLD, lib.SUM, 0, db.data_ptr())),
        ("tc_matmul", (code, code, lib.RIGHT, 0, m, n, k, dz.data_ptr(), w.data_ptr(), through.data_ptr())),
        ("tc_fused", (code, back_code, len(backward), back_places, 2, *_operands(through, x), 2, *_operands(dx), 1,
                      m, k)),
    ]
    # A 16-bit layer's update runs on a 32-bit copy of its weights elsewhere.
    updates, moments = [], []
    outputs = {"y": y, "dx": dx, "dw": dw, "db": db}
    if dtype == "f32":
        moments = _moments(case, seed)
        for parameters, gradient, rows, (first, second) in ((w, dw, k, moments[0]), (b, db, 1, moments[1])):
            rule = Adam(RATE)
            rule.steps, rule.first, rule.second = STEPS, _Storage(first), _Storage(second)
            updates.append((rule, _Storage(parameters), _Storage(gradient), rows, n))
        outputs.update(w=w, b=b)
    return {"calls": calls, "updates": updates, "outputs": outputs, "keep": (x, dz, w, b, through, moments)}


def _prepare_norm(case, seed):
    x, gamma = _norm_operands(case, seed)
    rows, cols, code = case["rows"], case["cols"], DTYPE[case["dtype"]]
    out = _empty((rows, cols), case["dtype"])
    program = _norm_program(code, cols)
    encoded, places = lib._program(program, [_grid(rows, cols), (0, 1, 0, [], []), (0, 0, 1, [rows], [1])])
    _, whole = lib._program([], [_grid(rows, cols)])
    statistics = (lib.Statistic * 2)()
    for i, which in enumerate((lib.STAT_MEAN, lib.STAT_DEVIATIONS)):
        statistics[i].source, statistics[i].source_len, statistics[i].source_dtype = x.data_ptr(), rows * cols, code
        statistics[i].which, statistics[i].place = which, whole[0]
    call = ("tc_fused_with_statistics", (lib.F32, encoded, len(program), places, 3, *_operands(x, gamma), 2,
                                         *_operands(out), 1, rows, cols, statistics, 2))
    return {"calls": [call], "outputs": {"y": out}, "keep": (x, gamma)}


def _prepare_network(case, seed):
    widths, weights, biases, x, y = _network_operands(case, seed)
    return {"network": lib.Mlp(widths, case["batch"], weights, biases, x, y, RATE), "layers": case["layers"]}


# ---- one pass -----------------------------------------------------------------


def run(state):
    if "network" in state:
        network = state["network"]
        network.step()
        out = {"loss": network.loss()}
        for layer in range(state["layers"]):
            out[f"dw{layer}"], out[f"db{layer}"] = network.gradients(layer)
        return out
    for name, args in state["calls"]:
        lib.call(name, *args)
    for rule, parameters, gradient, rows, cols in state.get("updates", ()):
        rule.update(parameters, gradient, rows, cols)
    return state["outputs"]


# ---- what a pass cannot do without ----------------------------------------------


def work(case):
    size = 4 if case.get("dtype", "f32") == "f32" else 2
    kind = case["kind"]
    if kind == "product":
        m, k, n = case["m"], case["k"], case["n"]
        c = 8 if case["accumulate"] else size
        return {"bytes": size * (m * k + k * n) + c * m * n, "flops": 2.0 * m * k * n}
    if kind == "vector":
        rows, cols = case["rows"], case["cols"]
        # The matrix once for each of the two products.
        return {"bytes": size * 2 * (rows * cols + rows + cols), "flops": 4.0 * rows * cols}
    if kind == "broadcast":
        a, b, c = case["a"], case["b"], case["c"]
        n, half = a * b * c, a * (b // 2) * c
        # Product, sum, exchange and join read and write n; the slice half.
        return {"bytes": size * (8 * n + 2 * half + b + a * c), "flops": 2.0 * n}
    if kind == "reduce":
        a, b, c = case["a"], case["b"], case["c"]
        n = a * b * c
        return {"bytes": size * (12 * n + 5 * (a * b + c)) + 8 * a * c, "flops": 16.0 * n}
    if kind == "layer":
        m, k, n = case["m"], case["k"], case["n"]
        # The three products, the rectifier's pass, db, and the update's seven streams.
        moved = size * (6 * m * k + 2 * k * n + 4 * m * n) + 4 * k * n
        moved += 4 * 7 * (k * n + n) if size == 4 else 0
        return {"bytes": moved, "flops": 6.0 * m * k * n}
    if kind == "norm":
        return {"bytes": size * (2 * case["rows"] * case["cols"] + case["cols"]),
                "flops": 8.0 * case["rows"] * case["cols"]}
    widths = [case["inputs"]] + [case["hidden"]] * (case["layers"] - 1) + [case["outputs"]]
    batch = case["batch"]
    parameters = sum(i * o + o for i, o in zip(widths, widths[1:]))
    activations = sum(widths) * batch
    return {"bytes": 4.0 * (10 * parameters + 4 * activations),
            "flops": 6.0 * batch * sum(i * o for i, o in zip(widths, widths[1:]))}


def tolerance(case):
    """About four times what a pass was seen to be off the same in 64 bits,
    which two orders of the sums or one more rounding come to as well."""
    kind = case["kind"]
    if kind == "broadcast":
        return "exact"  # one rounding an operation, and copies
    if kind == "network" or case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 4e-4}
    return {"rel": 1e-3, "max": 8e-3} if case["dtype"] == "f16" else {"rel": 8e-3, "max": 6e-2}


# ---- the same in 64 bits ----------------------------------------------------------


def exact(case, seed):
    kind = case["kind"]
    if kind == "product":
        a, b, c, _ = _product_operands(case, seed)
        a, b = a.double(), b.double()
        value = (a.T.contiguous() if case["form"] == "left" else a) @ (b.T.contiguous() if case["form"] == "right" else b)
        return {"c": value + c.double() if case["accumulate"] else value}
    if kind == "vector":
        matrix, right, left = (t.double() for t in _vector_operands(case, seed))
        return {"matvec": (matrix * right).sum(1), "vecmat": (matrix * left[:, None]).sum(0)}
    if kind == "broadcast":
        x, y, z = (t.double() for t in _broadcast_operands(case, seed))
        scaled = x * y
        total = scaled + z
        b = case["b"]
        half = b // 2
        start = (b - half) // 2
        return {"scaled": scaled, "sum": total, "exchanged": total.permute(0, 2, 1).contiguous(),
                "middle": total[:, start:start + half].contiguous(),
                "joined": torch.cat((total[:, half:], total[:, :half]), 1)}
    if kind == "reduce":
        x = _reduce_operands(case, seed).double()
        fold = {"sum": lambda t, axes: t.sum(axes), "max": lambda t, axes: t.amax(axes),
                "min": lambda t, axes: t.amin(axes), "mean": lambda t, axes: t.mean(axes),
                "var": lambda t, axes: t.var(axes, correction=0)}
        out = {name: fold[name.split(" ")[0]](x, axes) for name, axes, _, _ in REDUCTIONS}
        return {**out, "argmax": None, "argmin": None}
    if kind == "layer":
        x, w, b, dz = (t.double() for t in _layer_operands(case, seed))
        dw, db = x.T.contiguous() @ dz, dz.sum(0)
        out = {"y": (x @ w + b).relu(), "dx": (dz @ w.T.contiguous()) * (x > 0), "dw": dw, "db": db}
        if case["dtype"] == "f32":
            (mw, vw), (mb, vb) = _moments(case, seed)
            out.update(w=_adam(w, dw, mw, vw), b=_adam(b, db, mb, vb))
        return out
    if kind == "norm":
        x, gamma = (t.double() for t in _norm_operands(case, seed))
        x = x - x.mean(1, keepdim=True)
        return {"y": x / (x.square().mean(1, keepdim=True) + EPSILON).sqrt() * gamma}
    return _exact_network(case, seed)


def _adam(p, g, first, second):
    """Adam's step after STEPS others, its decays as f32 holds them."""
    b1, b2 = float(np.float32(0.9)), float(np.float32(0.999))
    first = b1 * first.double() + (1 - b1) * g
    second = b2 * second.double() + (1 - b2) * g.square()
    correct = (second / (1 - b2 ** (STEPS + 1))).sqrt() + 1e-8
    return p - RATE * first / (1 - b1 ** (STEPS + 1)) / correct


def _exact_network(case, seed):
    _, weights, biases, x, y = _network_operands(case, seed)
    weights, biases = [torch.from_numpy(w).double() for w in weights], [torch.from_numpy(b).double() for b in biases]
    hidden, before = [torch.from_numpy(x).double()], []
    for layer, (w, b) in enumerate(zip(weights, biases)):
        before.append(w @ hidden[-1] + b[:, None])
        hidden.append(before[-1].relu() if layer + 1 < len(weights) else before[-1])
    residual = hidden[-1] - torch.from_numpy(y).double()
    out = {"loss": residual.square().mean()}
    d = 2 * residual / residual.numel()
    for layer in range(len(weights) - 1, -1, -1):
        dw, db = d @ hidden[layer].T, d.sum(1)
        out.update({f"dw{layer}": dw, f"db{layer}": db})
        if layer:
            d = (weights[layer].T @ d) * (before[layer - 1] > 0)
    return out
