"""Scratch that only makes a call faster is done without where there is no
memory for it: reductions then keep a depth whole, products read odd operands
where they are.

The library's own `tc_alloc` is answered by one that can refuse, ahead of it in
a child process's symbol order; the child's own storage comes from the
library's.  Values are small integers, so every sum is exact in any order."""

import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

REFUSING = """
#include <stddef.h>
static int (*real)(size_t, void**);
static int refusing, refused;
extern "C" {
void answer_with(void* alloc) { real = (int (*)(size_t, void**))alloc; }
void refuse(int on) { refusing = on; }
int times() { return refused; }
int tc_alloc(size_t bytes, void** out) {
    if (!refusing) return real(bytes, out);
    refused++;
    return 4;  // TC_OUT_OF_MEMORY
}
}
"""

CHILD = """
import ctypes, sys
import numpy as np
refusing = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
from tensorcrate_amd import lib
refusing.answer_with(ctypes.cast(lib.load().tc_alloc, ctypes.c_void_p))
rng = np.random.default_rng(0)

def without_memory(name, *args):
    before = refusing.times()
    refusing.refuse(1)
    lib.call(name, *args)
    refusing.refuse(0)
    assert refusing.times() > before, "nothing was refused"

for shape, axis in (((2, 1000001), 1), ((100003, 11), 0), ((60000, 300), 0)):
    x = rng.integers(-3, 4, shape).astype(np.float32)
    results = x.shape[1 - axis]
    source, out = lib.Buffer.of(x), lib.Buffer(4 * results)
    steps = [shape[1], 1]
    split = lib.split(0, [shape[1 - axis]], [steps[1 - axis]], [shape[axis]], [steps[axis]])
    without_memory("tc_reduce_axes", lib.F32, source.ptr, x.size, ctypes.byref(split), lib.FOLD, lib.SUM, 0, out.ptr)
    assert np.array_equal(out.download(np.float32, results), x.sum(axis, dtype=np.float64)), ("sum", shape)
    without_memory("tc_reduce_axes", lib.F32, source.ptr, x.size, ctypes.byref(split), lib.VARIANCE, 0, shape[axis],
                   out.ptr)
    assert np.allclose(out.download(np.float32, results), x.var(axis, dtype=np.float64), rtol=1e-5), ("var", shape)
    without_memory("tc_arg_reduce", lib.F32, source.ptr, x.size, ctypes.byref(split), lib.RMAX, out.ptr)
    assert np.array_equal(out.download(np.uint32, results), x.argmax(axis)), ("argmax", shape)

for m, k, n in ((1153, 1001, 1031), (257, 4097, 255)):
    a, b = rng.integers(-1, 2, (m, k)), rng.integers(-1, 2, (k, n))
    bits = [(x.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16) for x in (a, b)]  # bf16
    left, right, out = lib.Buffer.of(bits[0]), lib.Buffer.of(bits[1]), lib.Buffer(4 * m * n)
    without_memory("tc_matmul", lib.BF16, lib.F32, lib.PLAIN, 0, m, k, n, left.ptr, right.ptr, out.ptr)
    want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(out.download(np.float32, m * n).reshape(m, n), want), (m, k, n)
print("passed")
"""


def test_calls_do_without_scratch_there_is_no_memory_for(tmp_path):
    source, library = tmp_path / "refusing.cpp", tmp_path / "refusing.so"
    source.write_text(REFUSING)
    subprocess.run(["g++", "-shared", "-fPIC", str(source), "-o", str(library)], check=True, timeout=60)
    child = subprocess.run([sys.executable, "-c", CHILD, str(library)], capture_output=True, text=True, timeout=100,
                           cwd=Path(__file__).resolve().parent.parent)
    assert child.returncode == 0 and child.stdout.endswith("passed\n"), child.stdout + child.stderr
