"""Registers of the kernels whose launch shapes count on a number of waves a SIMD, from the code object's metadata of the built library's objects."""
import os
import re
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tensor_amd", "lib")
LLVM = "/opt/rocm/llvm/bin"


def kernels(name, tmp_path, kernel=None):
    """(template arguments, vector registers, spilled ones, bytes of static LDS) of the kernel's instances in <name>.o"""
    obj = os.path.join(LIB, name + ".o")
    if not os.path.exists(obj) or not os.path.isdir(LLVM):
        pytest.skip("no object of the build here")
    fat, code = str(tmp_path / "fat"), str(tmp_path / "code")
    subprocess.check_call([LLVM + "/llvm-objcopy", "--dump-section=.hip_fatbin=" + fat, obj, str(tmp_path / "copy")])
    subprocess.check_call([LLVM + "/clang-offload-bundler", "--unbundle", "--type=o", "--input=" + fat, "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--output=" + code])
    notes = subprocess.run([LLVM + "/llvm-readelf", "--notes", code], capture_output=True, text=True, check=True).stdout
    found = re.findall(r"\.group_segment_fixed_size:\s+(\d+)(?:(?!group_segment).)*?\.symbol:\s+_ZN4ohip\d+" + (kernel or name) +
                       r"_kernelI(\S+?)EEvP.*?\.vgpr_count:\s+(\d+)\s+\.vgpr_spill_count:\s+(\d+)", notes, re.S)
    return [([int(v) for v in re.findall(r"L[ib](\d+)E", args)], int(n), int(spilled), int(lds)) for lds, args, n, spilled in found]


def test_depthwise_and_pointwise_launch(tmp_path):
    """Five waves a SIMD with a 3x3 window, four with 5x5, with and without staged pixels (512 registers, allocated in eights)."""
    seen = kernels("conv_dwpw", tmp_path)
    assert len(seen) >= 92
    for args, registers, spilled, _ in seen:
        waves, taps = args[:2]
        assert waves in (4, 8) and taps in (9, 25)
        assert spilled == 0 and 512 // ((registers + 7) // 8 * 8) >= (5 if taps == 9 else 4), (args, registers)


def test_depthwise_launch_on_an_fp32_blob(tmp_path):
    """Three waves a SIMD, and no LDS but what the launch asks for by its waves: four waves' lines in each one-wave workgroup fill a compute unit with four waves."""
    seen = kernels("conv_dw_mfma", tmp_path, "conv_dw3x3_f32in")
    assert len(seen) >= 80
    for args, registers, spilled, lds in seen:
        assert lds == 0 and spilled == 0 and registers <= 168, (args, registers, spilled, lds)
