"""Host paths of the library that need a failing allocation, on the CPU: the library as built, over
tests/fake_hip.cpp, which takes the place of the HIP runtime."""
import os
import subprocess

import pytest

from conftest import REPO

LIBDIR = os.path.join(REPO, "md-bench_amd", "lib")

TABLES = """
#include <cstdio>
#include "mdbench_driver.h"
#include "mdgfx950.h"
extern size_t g_budget, g_used;
extern int g_refused;
int main()
{
    mdb_config cfg;
    mdbDefaultConfig(&cfg);
    cfg.nx = cfg.ny = cfg.nz = 51;  // 530,604 atoms: lists with staging tables
    mdb_vl* s               = nullptr;
    if (mdbVLCreate(&cfg, &s)) return 1;
    const size_t full = g_used;
    g_budget = g_used + (1 << 20);  // less than the second position buffer
    computeForceFinalInitialGFX950(mdbVLParam(s), mdbVLAtom(s), mdbVLNeighbor(s), mdbVLStats(s));
    std::printf("%d %d %lld\\n", mdgfx950Status(), g_refused, (long long)g_used - (long long)full);
    // without tables left to give back the error stays an error
    g_budget = g_used;
    mdbVLAtom(s)->Nlocal *= 2;
    setupPbcGFX950(mdbVLAtom(s), mdbVLParam(s));
    std::printf("%d %d\\n", mdgfx950Status(), g_refused);
    mdbVLAtom(s)->Nlocal /= 2;
    mdbVLDestroy(s);
    std::printf("%lld\\n", (long long)g_used);
}
"""

THREADS = """
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>
namespace mdg {
void copy_to_device(void*, const void*, size_t);
void copy_from_device(void*, const void*, size_t);
}
static thread_local int g_news = -1;  // allocations of this thread left before one fails (-1: no limit)
void* operator new(size_t n)
{
    if (g_news == 0) throw std::bad_alloc();
    if (g_news > 0) g_news--;
    if (void* p = malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
int main()
{
    const size_t n = 17 << 20;  // nine chunks
    std::vector<unsigned char> a(n), b(n), c(n);
    for (size_t i = 0; i < n; i++)
        a[i] = (unsigned char)(i * 2654435761u >> 13);
    for (int news = 0; news < 4; news++) {
        g_news = news;
        mdg::copy_to_device(b.data(), a.data(), n);
        g_news = news;
        mdg::copy_from_device(c.data(), b.data(), n);
        g_news = -1;
        std::printf("%d\\n", a == b && a == c);
        b.assign(n, 0);
        c.assign(n, 0);
    }
}
"""


def _run(tmp_path, source):
    (tmp_path / "main.cpp").write_text(source)
    exe = str(tmp_path / "t")
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        "-I", os.path.join(REPO, "include"), str(tmp_path / "main.cpp"),
                        os.path.join(REPO, "tests", "fake_hip.cpp"), "-rdynamic", "-L", LIBDIR,
                        "-lmdgfx950", "-Wl,-rpath," + LIBDIR, "-Wl,--allow-shlib-undefined", "-pthread",
                        "-o", exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr[-3000:])
    return [line.split() for line in r.stdout.splitlines()]


def test_staging_tables_make_room_for_what_a_run_needs(tmp_path):
    """The tables of a large full list only save time: where the device has no room left for the second
    position buffer they go, and the call runs."""
    first, second, _ = _run(tmp_path, TABLES)
    status, refused, change = map(int, first)
    assert refused == 1
    assert status == 0  # MDG_ERR_CAPACITY (3) where the tables stay
    assert change < -100e6  # 123 MB of tables for 16 MB of positions
    assert [int(v) for v in second] == [3, 2]


def test_host_copies_without_memory_for_threads(tmp_path):
    """A copy whose threads cannot be started for want of memory is made by the calling thread."""
    assert _run(tmp_path, THREADS) == [["1"]] * 4
