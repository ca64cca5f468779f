"""The block of device memory kept between adjoint calls: its bookkeeping on the CPU (the unit compiled
against a HIP stand-in with a fixed amount of memory), and on the GPU that it is given back, serves
grids of different sizes one after the other and calls from two threads."""
import ctypes as C
import os
import re
import shutil
import subprocess
import threading
import time

import numpy as np
import pytest

from mpulse_amd import abi, configs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "mpulse_amd", "csrc")

HIP = """
#pragma once
#include <cstdlib>
#include <map>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorInvalidValue = 1 };
inline std::map<void *, size_t> &live() { static std::map<void *, size_t> m; return m; }
inline size_t &held() { static size_t h = 0; return h; }
constexpr size_t TOTAL = 8000;
inline hipError_t hipMalloc(void **p, size_t n)
{
    if (held() + n > TOTAL) return hipErrorOutOfMemory;
    *p = std::malloc(1);
    live()[*p] = n;
    held() += n;
    return hipSuccess;
}
inline hipError_t hipFree(void *p)
{
    auto it = live().find(p);
    if (it == live().end()) return hipErrorInvalidValue;
    held() -= it->second;
    live().erase(it);
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipMemGetInfo(size_t *a, size_t *t) { *a = TOTAL - held(); *t = TOTAL; return hipSuccess; }
"""

MAIN = """
#include "mpx_memory.h"
#include <cstdio>
using namespace mpx;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\\n", __LINE__, #c); return 0; } } while (0)
int main()
{
    spare_solvers(1);
    size_t n = 900;
    void *a = spare_take(0, &n), *q = nullptr;
    CHECK(a && n == 900 && held() == 900);
    spare_give(0, a, n);
    CHECK(held() == 900);  // kept
    n = 500;
    void *b = spare_take(0, &n);
    CHECK(b == a && n == 900);  // taken again, whole
    size_t m = 500;
    void *c = spare_take(0, &m);
    CHECK(c && c != b && m == 500 && held() == 1400);  // a second call at the same time
    spare_give(0, b, n);
    spare_give(0, c, m);
    CHECK(held() == 500);  // one block a device
    n = 600;
    a = spare_take(0, &n);
    CHECK(a && n == 600 && held() == 600);  // too small a block goes
    spare_give(0, a, n);
    n = 1001;
    a = spare_take(0, &n);
    CHECK(a && n == 1001);
    spare_give(0, a, n);
    CHECK(held() == 0);  // past an eighth
    n = 1000;
    a = spare_take(1, &n);
    spare_give(1, a, n);
    CHECK(held() == 1000);
    CHECK(dev_malloc(&q, 7500) == hipSuccess && held() == 7500);  // a full GPU takes the kept block
    CHECK(dev_malloc(&a, 7500) == hipErrorOutOfMemory && held() == 7500);
    n = 2000;
    CHECK(!spare_take(0, &n));
    CHECK(hipFree(q) == hipSuccess);
    n = 700;
    a = spare_take(0, &n);
    spare_give(0, a, n);
    CHECK(spare_drop() && held() == 0 && !spare_drop());  // the release call
    n = 700;
    a = spare_take(0, &n);
    spare_give(0, a, n);
    spare_solvers(1);
    spare_solvers(-1);
    CHECK(held() == 700);
    n = 700;
    b = spare_take(0, &n);
    spare_solvers(-1);
    spare_give(0, b, n);
    CHECK(held() == 0);  // nothing is kept once the last solver is gone
    std::printf("ok\\n");
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="needs g++")
def test_bookkeeping(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", str(tmp_path), "-I", CSRC, str(tmp_path / "main.cpp"), "-x", "c++",
                    os.path.join(CSRC, "mpx_memory.hip"), "-o", str(tmp_path / "t")], check=True)
    assert subprocess.run([str(tmp_path / "t")], stdout=subprocess.PIPE, text=True).stdout == "ok\n"


def test_every_device_allocation_can_have_the_kept_block():
    for fn in os.listdir(CSRC):
        if fn.endswith((".hip", ".h")) and fn != "mpx_memory.hip":
            src = re.sub(r"//[^\n]*|/\*.*?\*/", "", open(os.path.join(CSRC, fn)).read(), flags=re.S)
            assert not re.search(r"\bhipMalloc\w*\s*\(", src), fn


def gradient(n, nz, seed=3, keep=None):
    """J, dJ/dEps and dJ/dchi of a small run; with keep the solver is appended there, still alive"""
    d, _ = configs.plrc_kerr_pulse(n, 3, 4.0, 3, 2e9, 0, d_src=5, nz=nz)
    d.factories[1].tshift = 2.0
    s = abi.Solver(d)
    rng = np.random.default_rng(seed)
    s.set("Ey", np.pad(rng.uniform(-0.5, 0.5, (n, n, nz)), 1, mode="wrap"))
    r = s.adjoint_grad(nz - 4, 1.0, 12, checkpoint_every=5)
    if keep is None:
        s.close()
    else:
        keep.append(s)
    return r


def same(a, b):
    return a[0] == b[0] and np.array_equal(a[1], b[1]) and a[2] == b[2]


@pytest.mark.gpu
def test_release_gives_the_block_back():
    abi.load()
    hip = C.CDLL("libamdhip64.so.7")  # the runtime the library links, by its soname: no second one

    def free():
        avail, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(avail), C.byref(total)) == 0
        return avail.value

    print("case: kept adjoint block, release", flush=True)
    keep = []
    gradient(24, 24, keep=keep)
    abi.release_memory()
    before = free()
    keep[0].adjoint_grad(20, 1.0, 200, checkpoint_every=100)  # over 100 states of 0.4 MB each
    kept = before - free()
    abi.release_memory()
    assert kept >= 1 << 25
    end = time.monotonic() + 20  # the driver reports freed memory up to a second late
    while free() < before and time.monotonic() < end:
        time.sleep(0.1)
    assert free() >= before
    keep[0].close()


@pytest.mark.gpu
def test_one_block_for_grids_of_different_sizes_and_threads():
    print("case: kept adjoint block, sizes and threads", flush=True)
    sizes = [(24, 30), (17, 21), (30, 40)]
    want = []
    for n, nz in sizes:  # each with a block of its own: the last solver takes it along
        want.append(gradient(n, nz))
    assert all(np.any(w[1]) and w[2] != 0 for w in want)
    keep = []
    for q in (2, 1, 0, 1, 2):  # the block of the largest serves the smaller ones
        assert same(gradient(*sizes[q], keep=keep), want[q]), sizes[q]
    got = [None] * 6

    def work(t):
        got[t] = gradient(*sizes[t % 3], keep=keep)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(6)]
    for pair in (threads[:2], threads[2:4], threads[4:]):
        for t in pair:
            t.start()
        for t in pair:
            t.join()
    for t in range(6):
        assert got[t] is not None and same(got[t], want[t % 3]), t
    for s in keep:
        s.close()
