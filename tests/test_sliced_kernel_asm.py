"""The register-fed product kernel's wait states, checked in its gfx950
assembly.

A matrix-core step needs two wait states after a vector instruction that wrote
one of its A or B registers.  The compiler counts them, except where the step
begins a basic block entered by falling through from the write; `settle`
(csrc/gemm_sliced.hpp) holds them there.  This compiles the kernel's tiles in
every form with the library's own flags and scans each in program order, across
labels, for a step that follows such a write too closely; without `settle` it
finds them.  Runs on the CPU: hipcc cross-compiles for gfx950."""

import re
import subprocess
from pathlib import Path

import pytest

from tensorcrate_amd import _build
from tests.test_four_wave_kernel_asm import registers

CSRC = Path(__file__).resolve().parent.parent / "tensorcrate_amd" / "csrc"
SHAPES = ("4, 4, 4, 1", "2, 2, 4, 1", "1, 1, 8, 4")
FORMS = ("true, false", "false, false", "true, true")


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


@pytest.mark.parametrize("element", ["float", "tc::bf16_t"])
def test_steps_stand_two_wait_states_after_their_operands(element, tmp_path):
    source = tmp_path / "sliced.hip"
    source.write_text('#include <hip/hip_runtime.h>\n#include "gemm_sliced.hpp"\nnamespace tc {\n' + "".join(
        f"template __global__ void sliced_kernel<{element}, {element}, {form}, {shape}>(const {element}*, "
        f"const {element}*, {element}*, uint32_t, uint32_t, uint32_t, bool, PlainStore);\n"
        for form in FORMS for shape in SHAPES) + "}\n")
    target = tmp_path / "sliced.s"
    flags = [f for f in _build.HIP_FLAGS if f not in ("-fPIC", "-Wall")]
    subprocess.run([_build.hipcc(), *flags, f"-I{CSRC}", "--cuda-device-only", "-S", str(source), "-o", str(target)],
                   check=True, capture_output=True, timeout=600)
    text = target.read_text()
    steps, found = close_writes(text)
    assert steps > 9 and not found, found[:5]
    assert not re.search(r"\.(sgpr|vgpr)_spill_count:\s*[1-9]", text)
