"""Properties of the compiled kernels that no result shows, read from the code
objects built from this source: which loads the hardware bounds-checks, in which
order loads that hide each other's latency go out, and how many wavefronts
the registers leave room for."""
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


def vgprs(kernel):
    notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes",
                            os.path.join(xpu.BUILD_DIR, "xpu_kernels.hsaco")],
                           capture_output=True, text=True, check=True).stdout
    block = next(b for b in notes.split("  - .agpr_count:")[1:] if re.search(rf"\.symbol:\s+{kernel}\.kd", b))
    return int(re.search(r"\.vgpr_count:\s+(\d+)", block).group(1))


@pytest.mark.parametrize("kernel,waves", [
    ("xpu_q3_norm_gemv_r2", 4), ("xpu_q3_norm_gemv_swiglu_r2", 4), ("xpu_q3_norm_gemv_logits_r2", 4),
    ("xpu_q3_gemv_residual_r1", 6)])
def test_staged_decode_kernels_keep_their_wavefronts(kernel, waves):
    """Wavefronts per SIMD that 512 registers in steps of 8 allow the decode
    kernels of wide models, which stream their weights on that many."""
    assert 512 // ((vgprs(kernel) + 7) // 8 * 8) >= waves


def test_whole_batch_gemv_keeps_no_row_ends():
    """Rows of whole batches do not pay for ends loaded ahead (107 registers
    without them, 119 with)."""
    assert vgprs("xpu_gemv_bf16_r2u2_vec") < vgprs("xpu_gemv_bf16_r2u2_ends")
