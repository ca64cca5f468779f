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


LAYERS = """
// the first and last cells of both faces of one dimension, by 64-bit arithmetic and by cpml_index
static int faces(int dim, const int n[3], int d)
{
    CpmlFace F[2]{};
    CpmlDim D{};
    for (int q = 0; q < 2; ++q) {  // 0: high side, 1: low
        F[q].dim = dim;
        for (int a = 0; a < 3; ++a) F[q].hi[a] = n[a] + 1;
        F[q].lo[dim] = q ? 1 : n[dim] + 1 - d;
        F[q].hi[dim] = F[q].lo[dim] + d - 1;
        F[q].n1 = F[q].hi[1] - F[q].lo[1] + 1;
        F[q].n2 = F[q].hi[2] - F[q].lo[2] + 1;
    }
    const long long cnt = (long long)(F[0].hi[0] - F[0].lo[0] + 1) * F[0].n1 * F[0].n2, block = (cnt + 63) / 64 * 64;
    if (cnt >= 1LL << 31) return 0;
    D.s0 = F[0].n1 * F[0].n2;
    D.s1 = F[0].n2;
    for (int q = 0; q < 2; ++q) set_face(D, q, F[q], q * block);
    for (int q = 0; q < 2; ++q)
        for (int corner = 0; corner < 8; ++corner) {
            int at[3];
            for (int a = 0; a < 3; ++a) at[a] = corner >> a & 1 ? F[q].hi[a] : F[q].lo[a];
            const long long want = q * block + ((long long)(at[0] - F[q].lo[0]) * F[q].n1 + at[1] - F[q].lo[1]) * F[q].n2 +
                                   at[2] - F[q].lo[2];
            if ((long long)cpml_index(D, q, at[0], at[1], at[2]) != want) return 0;
        }
    return 1;
}
int main()
{
    const int grids[][4] = {{24, 20, 28, 6}, {8, 8, 8, 8}, {512, 512, 512, 16}, {13, 11600, 11500, 8}, {13, 11500, 11600, 9},
                            {11600, 13, 11000, 8}, {11600, 11000, 13, 8}, {1, 30000, 20000, 1}, {1288, 1288, 1288, 700}};
    for (auto &g : grids)
        for (int dim = 0; dim < 3; ++dim)
            if (g[dim] >= g[3] && !faces(dim, g, g[3])) {
                std::printf("%d x %d x %d dim %d layers %d\\n", g[0], g[1], g[2], dim, g[3]);
                return 0;
            }
    std::printf("ok\\n");
}
"""


def test_layer_index_up_to_the_largest_faces(tmp_path):
    assert compile_and_run(tmp_path, LAYERS) == "ok\n"


STENCIL = """
int main()
{
    for (int n = 1; n <= 9; ++n)
        for (int d = 1; d <= 12; ++d)
            for (int dim = 0; dim < 3; ++dim)
                for (int isH = 0; isH < 2; ++isH)
                    for (int high = 0; high < 2; ++high) {
                        // the layer as border_extent places it: distance 1 from either end, the low H face 0
                        int N[3] = {5, 5, 5};
                        N[dim] = n;
                        CpmlFace f{};
                        f.dim = dim;
                        for (int a = 0; a < 3; ++a) f.hi[a] = N[a] + 1;
                        f.lo[dim] = high ? n + 1 - d : (isH ? 0 : 1);
                        f.hi[dim] = f.lo[dim] + d - 1;
                        const FaceCells c = face_cells(f, N, isH);
                        const int below = isH ? 0 : 1, above = isH ? 1 : 0;
                        bool good = c.lo[dim] <= c.hi[dim] && c.lo[dim] >= f.lo[dim] && c.hi[dim] <= f.hi[dim];
                        for (int a = 0; a < 3; ++a) {
                            good = good && c.lo[a] - (a == dim ? below : 0) >= 0 && c.hi[a] + (a == dim ? above : 0) <= N[a] + 1;
                            if (d <= n) good = good && c.lo[a] == f.lo[a] && c.hi[a] == f.hi[a];
                            // every cell the updates use (1 .. n; H from 0) that lies in the layer is kept
                            const int first = f.lo[a] > (isH ? 0 : 1) ? f.lo[a] : (isH ? 0 : 1);
                            const int last = f.hi[a] < N[a] ? f.hi[a] : N[a];
                            good = good && c.lo[a] <= first && c.hi[a] >= last;
                        }
                        if (!good) {
                            std::printf("n %d d %d dim %d H %d high %d\\n", n, d, dim, isH, high);
                            return 0;
                        }
                    }
    std::printf("ok\\n");
}
"""


def test_layer_thicker_than_the_box_keeps_its_stencil_inside(tmp_path):
    assert compile_and_run(tmp_path, STENCIL) == "ok\n"
