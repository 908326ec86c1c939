"""Properties of the compiled kernels that no result shows, read from the code
objects built from this source: which loads the hardware bounds-checks, and in
which order loads that hide each other's latency go out."""
import os
import re
import subprocess

import pytest

import xpu_playground_amd as xpu

LLVM = "/opt/rocm/llvm/bin"


def assembly(code_object, kernel):
    out = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn",
                          f"--disassemble-symbols={kernel}", os.path.join(xpu.BUILD_DIR, code_object)],
                         capture_output=True, text=True, check=True).stdout
    return [line.split("//")[0].strip() for line in out.splitlines()]


@pytest.mark.parametrize("code_object", ["xpu_kernels.hsaco", "xpu_kernels_stamps.hsaco"])
def test_split_pv_loads_are_bounds_checked(code_object):
    """The P.V kernel asks for V rows past the context and relies on its buffer
    descriptor for them. The check covers the vector and the immediate offset
    only, so no load may carry a scalar one."""
    loads = [i for i in assembly(code_object, "xpu_q3_attn_pv") if i.startswith("buffer_load")]
    assert len(loads) >= 32  # four batches of eight
    for i in loads:
        m = re.fullmatch(r"buffer_load_dwordx4 v\[\d+:\d+\], v\d+, s\[\d+:\d+\], (\S+) offen( offset:\d+)?", i)
        assert m and m.group(1) == "0", i


def test_split_pv_asks_for_the_scores_before_v():
    """Loads return in order, so V rows asked for ahead of the scores would be
    waited for before the first exponential."""
    loads = [i.split()[0] for i in assembly("xpu_kernels.hsaco", "xpu_q3_attn_pv") if re.match(r"(global|buffer)_load", i)]
    # the partial maximum, four score vectors, the first half of the V ring
    assert loads[:21] == ["global_load_dword"] + ["global_load_dwordx4"] * 4 + ["buffer_load_dwordx4"] * 16
