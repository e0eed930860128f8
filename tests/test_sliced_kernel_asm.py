"""The register-fed product kernel's wait states, checked in its gfx950
assembly.

A matrix-core step needs two wait states after a vector instruction that wrote
one of its A or B registers.  The compiler counts them, except where the step
begins a basic block entered by falling through from the write; `settle`
(csrc/gemm_sliced.hpp) holds them there.  This compiles every instance that the
library launches, and ones with a program's epilogue as the runtime compiler
builds them, with the library's own flags and scans each in program order,
across labels, for a step that follows such a write too closely; without
`settle` it finds them.  Runs on the CPU: hipcc cross-compiles for gfx950."""

import re
import subprocess
from pathlib import Path

import pytest

from tensorcrate_amd import _build
from tests.test_four_wave_kernel_asm import registers

CSRC = Path(__file__).resolve().parent.parent / "tensorcrate_amd" / "csrc"
SHAPES = ("4, 4, 4, 1", "2, 2, 4, 1", "1, 1, 8, 4", "1, 1, 2, 1")
FORMS = ("true, false", "false, false", "true, true")
# A program's store of one element a lane's group, as the compiled epilogues
# hold it: a row's and a column's operand, two outputs.
PROGRAM = """template <int N> struct RowStore {
  static constexpr bool kProgram = true;
  static constexpr int kElems = N;
  float *out, *copy;
  const float *bias, *scale;
  __device__ __forceinline__ void group(const bool (&live)[N], const uint32_t (&row)[N], const uint32_t (&col)[N],
                                        uint32_t width, const float (&product)[N]) const {
    float x[N], y[N];
    for (int e = 0; e < N; e++) x[e] = live[e] ? bias[col[e]] : 0.0f, y[e] = live[e] ? scale[row[e]] : 0.0f;
    for (int e = 0; e < N; e++) {
      if (live[e]) out[row[e] * width + col[e]] = fmaxf(product[e] * y[e] + x[e], 0.0f), copy[row[e] * width + col[e]] = product[e];
    }
  }
};
"""


def instances(element):
    """(output type, forms and shape, store) of each instance."""
    outs = {element, "float"}
    found = [(out, f"{form}, {shape}", "PlainStore") for out in outs for form in FORMS for shape in SHAPES]
    # 16-bit operands along K are the ones copied for this kernel.
    if element != "float":
        found += [(out, f"{form}, {shape}", "PaddedStore") for out in outs for form in FORMS if form != FORMS[1]
                  for shape in SHAPES]
    return found + [(element, f"true, false, {shape}", f"RowStore<{4 * int(shape[0])}>") for shape in SHAPES]


def close_writes(assembly):
    """(steps seen, [a write and the step fewer than two wait states later])."""
    steps, found, last, position = 0, [], {}, 0
    for raw in assembly.split("\n"):
        line = raw.split(";")[0].strip()
        if line.startswith("_Z") and line.endswith(":"):
            last = {}
        if not line or line.startswith(".") or line.endswith(":"):
            continue
        parts = line.replace(",", " ").split()
        if parts[0] == "s_nop":
            position += int(parts[1], 0) + 1
            continue
        position += 1
        if parts[0].startswith("v_mfma"):
            steps += 1
            for token in parts[2:4]:
                for kind in ("v", "a"):
                    for r in registers(token, kind):
                        wrote = last.get((kind, r))
                        if wrote is not None and position - wrote[0] <= 2:
                            found.append(f"{wrote[1]!r} then {line!r}")
        elif parts[0].startswith("v_") and len(parts) > 1:
            for kind in ("v", "a"):
                for r in registers(parts[1], kind):
                    last[(kind, r)] = (position, line)
    return steps, found


@pytest.mark.parametrize("element", ["float", "bf16_t", "_Float16"])
def test_steps_stand_two_wait_states_after_their_operands(element, tmp_path):
    source = tmp_path / "sliced.hip"
    wanted = instances(element)
    source.write_text(f'#include <hip/hip_runtime.h>\n#include "gemm_sliced.hpp"\n{PROGRAM}namespace tc {{\n' + "".join(
        f"template __global__ void sliced_kernel<{element}, {out}, {shape}, {store}>(const {element}*, "
        f"const {element}*, {out}*, uint32_t, uint32_t, uint32_t, bool, {store});\n"
        for out, shape, store in wanted) + "}\n")
    target = tmp_path / "sliced.s"
    flags = [f for f in _build.HIP_FLAGS if f not in ("-fPIC", "-Wall")]
    subprocess.run([_build.hipcc(), *flags, f"-I{CSRC}", "--cuda-device-only", "-S", str(source), "-o", str(target)],
                   check=True, capture_output=True, timeout=600)
    text = target.read_text()
    steps, found = close_writes(text)
    assert steps > len(wanted) and not found, found[:5]
    assert text.count("amdhsa_private_segment_fixed_size 0") == len(wanted)
    assert not re.search(r"\.(sgpr|vgpr)_spill_count:\s*[1-9]", text)
