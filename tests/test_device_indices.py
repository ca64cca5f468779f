"""Index helpers that the kernels share with the host, compiled for the CPU and compared with 64-bit
arithmetic up to the largest grids that mpx_create takes (2^31 - 1 storage cells)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM_INCLUDE = "/opt/rocm/include"

pytestmark = pytest.mark.skipif(not (shutil.which("g++") and os.path.isdir(ROCM_INCLUDE)),
                                reason="needs g++ and the HIP headers")


def compile_and_run(tmp_path, body):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text("#include <hip/hip_runtime.h>\n#include <cstdio>\n#include <algorithm>\n"
                   '#include "mpx_types.h"\nusing namespace mpx;\n' + body)
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I", ROCM_INCLUDE, "-I",
                    os.path.join(ROOT, "mpulse_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], stdout=subprocess.PIPE, check=True, text=True).stdout


PSI = """
int main()
{
    // a wave's 64 consecutive y-z cells (rows of nz cells, pitch pz) at the ends of a block of `cells`
    const size_t blocks[] = {4096, 89478464, 433ull * 433 * 480, 1431655765, 0x7ffffffe};
    for (size_t cells : blocks)
        for (int nz : {1, 2, 30, 63, 64, 65, 478}) {
            const size_t pz = 32 + (nz + 1 + 31) / 32 * 32, span = 64 / nz * pz + pz;
            for (size_t c0 : {(size_t)32, (size_t)33, (size_t)95, cells / 2 + 7, cells - 1 - span}) {
                if (c0 + span >= cells) continue;
                for (int lane = 0; lane < 64; ++lane) {
                    const size_t c = c0 + lane / nz * pz + lane % nz;
                    const unsigned o = psi_ahead(c0, (unsigned)(c - c0));
                    const unsigned bytes = o * 16u;  // as the loads form it
                    if (bytes / 16u != o || psi_base(c0) + o != psi_at(c)) {
                        std::printf("cells %zu nz %d c0 %zu lane %d\\n", cells, nz, c0, lane);
                        return 0;
                    }
                }
            }
        }
    std::printf("ok\\n");
}
"""


def test_accumulator_address_of_a_wave(tmp_path):
    assert compile_and_run(tmp_path, PSI) == "ok\n"
