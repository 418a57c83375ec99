"""What the compiler makes of the device code's cross-lane moves (no GPU needed: device code is compiled to assembly text).

A lane move that is folded into a reversed operation (v_subrev_*_dpp and its like) moves the lanes of the wrong operand on
the card: a - below(b) becomes below(a) - b.  No such instruction may come out of this repository's sources."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ml_dataflow_amd", "csrc")
REVERSED_WITH_LANE_MOVE = re.compile(r"\bv_\w*rev\w*_dpp\b")


def assembly(source, tmp_path):
    out = tmp_path / "out.s"
    subprocess.run(["/opt/rocm/bin/hipcc", "-O3", "--offload-arch=gfx950", "-Wno-inline-asm", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-I", CSRC, "-I", os.path.join(ROOT, "include"), "-S", "--cuda-device-only", "-o", str(out), str(source)],
                   check=True, capture_output=True)
    return out.read_text()


@pytest.mark.parametrize("difference", ["end - wave_lane_below(end, 0)", "2 * lane - wave_lane_below(end, 0)", "end - wave_lane_below(end, 7)",
                                        "lane < groups ? end - wave_lane_below(end, 0) : 0"])
def test_the_value_of_the_lane_below_is_not_folded_into_a_difference(tmp_path, difference):
    source = tmp_path / "difference.hip"
    source.write_text('#include "matmul/gemm_kernel.h"\n'
                      "__global__ void difference(const int * ends, int * rows, int groups) {\n"
                      "\tconst int lane = threadIdx.x & 63, end = lane < groups ? ends[lane] : 0;\n"
                      "\trows[lane] = %s;\n}\n" % difference)
    text = assembly(source, tmp_path)
    assert re.search(r"v_mov_b32_dpp .* wave_shr:1", text)
    assert not re.search(r"v_sub\w*_dpp", text)


def test_no_lane_move_in_a_reversed_operation_of_the_native_kernels(tmp_path):
    text = assembly(os.path.join(CSRC, "kernels", "hip_kernels.hip"), tmp_path)
    assert "_dpp" in text
    assert not REVERSED_WITH_LANE_MOVE.search(text)


def test_no_lane_move_in_a_reversed_operation_of_the_matmul_library(tmp_path):
    library = os.path.join(ROOT, "ml_dataflow_amd", "lib", "libamd_matmul.so")
    copy = tmp_path / "libamd_matmul.so"
    copy.write_bytes(open(library, "rb").read())
    objdump = "/opt/rocm/llvm/bin/llvm-objdump"
    subprocess.run([objdump, "--offloading", str(copy)], check=True, capture_output=True, cwd=str(tmp_path))
    objects = [f for f in os.listdir(tmp_path) if f.endswith("gfx950")]
    assert len(objects) == 1
    text = subprocess.run([objdump, "-d", str(tmp_path / objects[0])], check=True, capture_output=True, text=True).stdout
    assert "_dpp" in text
    assert not REVERSED_WITH_LANE_MOVE.search(text)


def test_six_work_groups_of_the_norms_backward_fit_a_compute_unit(tmp_path):
    """the number that its rule for few rows counts with (norm.hip): 512 registers a lane of a SIMD, four waves a work-group, one on each"""
    text = assembly(os.path.join(CSRC, "kernels", "hip_kernels.hip"), tmp_path)
    entry = next(e for e in text[text.index("amdhsa.kernels:"):].split("  - .agpr_count:") if ".symbol:         default_rms_norm_bwd_x_bf16_bf16_kernel.kd" in e)
    count = {name: int(re.search(r"\.%s: +(\d+)" % name, entry).group(1)) for name in ("vgpr_count", "vgpr_spill_count", "private_segment_fixed_size")}
    assert count["vgpr_count"] <= 80 and 512 // 80 == 6
    assert count["vgpr_spill_count"] == 0 and count["private_segment_fixed_size"] == 0
