"""The assembly that the codebook's interleaved adds (cb_quads) are compiled to, on the CPU (the compiler alone)."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

# pairs of equal states, which the compiler can see
SOURCE = """
#include <hip/hip_runtime.h>
#include "ea_device.hpp"
using namespace ea;
template <int CB>
__global__ void same(const uint32_t* a, u4v* o) {
    uint32_t s[8];
    for (int i = 0; i < 8; ++i) s[i] = a[threadIdx.x + 64 * (i >> 1)];
    o[threadIdx.x] = cb_quads<CB>(s);
}
template __global__ void same<CB_MCG>(const uint32_t*, u4v*);
template __global__ void same<CB_3INST>(const uint32_t*, u4v*);
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_second_operands_outlive_the_first_adds(tmp_path):
    """The four first halves are written before the four second operands are read: none of those may have been given a
    register that a first add writes, not even where both states of a pair are one value."""
    src, out = tmp_path / "t.hip", tmp_path / "t.s"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "-O3", "--offload-arch=gfx950", "--cuda-device-only", "-std=c++17", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "expertatlas-glm5.3_amd", "csrc"), "-S", str(src), "-o", str(out)],
                   check=True, capture_output=True)
    blocks = re.findall(r"#ASMSTART(.*?)#ASMEND", out.read_text(), re.S)
    seen = 0
    for block in blocks:
        adds = re.findall(r"v_add_f16_sdwa (v\d+), (v\d+), (v\d+) dst_sel:WORD_([01])", block)
        if len(adds) != 8:
            continue
        seen += 1
        written = {d for d, _, _, half in adds if half == "0"}
        assert len(written) == 4
        for d, x, y, half in adds:
            if half == "1":
                assert d in written and x == y and x not in written, block
    assert seen == 2  # one block a codebook
