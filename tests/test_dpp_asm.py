"""The inline assembly of the extraction walk keeps its operands apart: an output that is written before the last
input is read must not share a register with that input, also where the caller passes the same values for both."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"

SOURCE = """
#include "extract.hip"
namespace qcs {
// the sums start as the shifted values themselves, one place further
template <bool PREV> __global__ void shift_alias_kernel(const float *in, float *out, float w)
{
    float x[4], a[4];
    for (int k = 0; k < 4; k++) x[k] = in[threadIdx.x + 64 * ((k + 1) & 3)];
    for (int k = 0; k < 4; k++) a[k] = x[(k + 1) & 3];
    fma_shifted<PREV>(a, x, w);
    for (int k = 0; k < 4; k++) out[threadIdx.x + 64 * k] = a[k];
}
template __global__ void shift_alias_kernel<true>(const float *, float *, float);
template __global__ void shift_alias_kernel<false>(const float *, float *, float);
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_shifted_multiply_adds_do_not_overwrite_their_inputs(tmp_path):
    src, asm = tmp_path / "alias.hip", tmp_path / "alias.s"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-fno-fast-math", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "--cuda-device-only", "-S", "-I", os.path.join(ROOT, "qc-storm_amd", "csrc"), str(src),
                    "-o", str(asm)], check=True, capture_output=True, timeout=300)
    kernels = re.findall(r"^\S*shift_alias_kernel\S*:.*?s_endpgm", asm.read_text(), re.S | re.M)
    assert len(kernels) == 2
    for body in kernels:
        ops = re.findall(r"v_fmac_f32_dpp (v\d+), (v\d+), (v\d+) wave_sh[rl]:1", body)
        assert len(ops) == 4
        written = set()
        for dst, shifted, weight in ops:
            assert shifted not in written and weight not in written, ops
            written.add(dst)
        assert len(written) == 4
