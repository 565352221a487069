"""A pool's page-locked blocks (csrc/pinned.hpp), compiled for the host with an
allocator of the test's own: which block a request takes, what waiting inputs
may hold, and what happens when there is no more page-locked memory."""
import os
import subprocess

from conftest import PKG

PROGRAM = r"""
#include "pinned.hpp"
#include <cstdio>
#include <cstdlib>
static int left = 1 << 30, made = 0;
extern "C" hipError_t hipHostMalloc(void **p, size_t, unsigned)
{
    if (left <= 0) return hipErrorOutOfMemory;
    --left; ++made;
    *p = malloc(1);
    return hipSuccess;
}
extern "C" hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
extern "C" hipError_t hipGetLastError(void) { return hipSuccess; }
#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
int main()
{
    using mdpd::PinnedCache;
    const size_t MiB = 1 << 20;
    void *p, *q;
    size_t a, b;
    {   // a small request does not take a large block
        PinnedCache c;
        CHECK(c.get(30 * MiB, &p, a) == hipSuccess && a == 32 * MiB);
        c.put(p, a);
        CHECK(c.stage(60000, &q, b) && b == MiB && c.staged == MiB);
        CHECK(c.get(17 * MiB, &p, a) == hipSuccess && a == 32 * MiB && made == 2);
        c.put(p, a);
        c.unstage(b);
        c.put(q, b);
        // the result of a job (88 bytes a slot) reuses its input's block (44)
        CHECK(c.get(88 * 9216, &p, a) == hipSuccess && p == q && made == 2);
        c.put(p, a);
    }
    {   // classes: powers of two from 1 MiB
        const size_t want[][2] = {{1, MiB}, {MiB, MiB}, {MiB + 1, 2 * MiB}, {4 * MiB, 4 * MiB}, {5 * MiB, 8 * MiB}};
        for (auto &w : want) CHECK(PinnedCache::size_class(w[0]) == w[1]);
    }
    {   // waiting inputs never hold more than the limit, whatever their sizes
        PinnedCache c;
        void *held[1024];
        size_t n = 0, sum = 0;
        while (n < 1024 && c.stage(n % 3 ? 100 : 3 * MiB, &held[n], a)) { sum += a; ++n; }
        CHECK(n < 1024 && c.staged == sum && sum <= PinnedCache::MAX_STAGED);
        CHECK(c.staged + 4 * MiB > PinnedCache::MAX_STAGED);
        CHECK(!c.stage(4 * MiB, &q, b) && c.staged == sum);
        for (size_t k = 0; k < n; ++k) free(held[k]);
    }
    {   // no page-locked memory left: not staged, nothing charged
        PinnedCache c;
        left = 0;
        CHECK(!c.stage(100, &q, b) && c.staged == 0);
        CHECK(c.get(100, &q, b) != hipSuccess);
    }
    return 0;
}
"""


def test_pinned_blocks(tmp_path):
    src, exe = tmp_path / "blocks.cpp", tmp_path / "blocks"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(PKG, "csrc"),
                    "-I", "/opt/rocm/include", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
