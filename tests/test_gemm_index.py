"""Host-side index rules of the GEMM kernels (csrc/kernels/gemm.hpp), compiled with g++.  CPU only."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

# every tile that a block may take, whole blocks of 32 rows past the end included: the low-rank
# columns it reads lie in X2's N / seg_n segments, and a tile inside N takes its own
SEGMENTS = """
#include "gemm.hpp"
#include <cstdio>
int main() {
    const int sizes[][2] = {{16464, 5488}, {16400, 16400}, {16416, 16}, {32, 16}, {192, 96}, {48, 0}, {16464, 0}};
    for (auto& [N, seg] : sizes)
        for (int row = 0; row < (N + 31) / 32 * 32; row += 16) {
            const int s = aic::hip::low_rank_segment(row, N, seg), segs = seg > 0 ? N / seg : 1;
            if (s < 0 || s >= segs || (row < N && seg > 0 && s != row / seg)) {
                std::printf("N %d seg %d row %d: segment %d\\n", N, seg, row, s);
                return 1;
            }
        }
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(os.path.join(ROCM, "include", "hip")),
                    reason="needs g++ and the HIP headers")
def test_low_rank_segments_stay_inside_x2(tmp_path):
    src, exe = tmp_path / "segments.cpp", tmp_path / "segments"
    src.write_text(SEGMENTS)
    p = subprocess.run(["g++", "-std=c++20", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"), "-I",
                        os.path.join(ROOT, "autonomousaicore_amd", "csrc", "kernels"), str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert p.returncode == 0, p.stderr
    p = subprocess.run([str(exe)], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout
