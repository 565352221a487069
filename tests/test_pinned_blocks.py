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

# page-locked memory runs out at MEMORY bytes
FREE_BLOCKS = r"""
#include "pinned.hpp"
#include <cstdio>
#include <cstdlib>
#include <map>
static const size_t MEMORY = (size_t)6 << 30;
static size_t used = 0;
static std::map<void *, size_t> size;
extern "C" hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    if (used + n > MEMORY) return hipErrorOutOfMemory;
    used += n;
    size[*p = malloc(1)] = n;
    return hipSuccess;
}
extern "C" hipError_t hipHostFree(void *p)
{
    used -= size.at(p);
    size.erase(p);
    free(p);
    return hipSuccess;
}
extern "C" hipError_t hipGetLastError(void) { return hipSuccess; }
#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
int main()
{
    using mdpd::PinnedCache;
    const size_t MiB = 1 << 20;
    void *p[2048];
    size_t got;
    {   // sizes that drift: every class holds a GiB at its time, one by one
        PinnedCache c;
        for (size_t sz = MiB; sz <= 64 * MiB; sz *= 2) {
            const size_t n = 1024 * MiB / sz;
            for (size_t k = 0; k < n; ++k) CHECK(c.get(sz, &p[k], got) == hipSuccess && got == sz);
            CHECK(used <= PinnedCache::MAX_FREE + n * sz);
            for (size_t k = 0; k < n; ++k) c.put(p[k], sz);
            CHECK(c.free_bytes == used);
            for (size_t k = 0; k < n; ++k) CHECK(c.get(sz, &p[k], got) == hipSuccess);     // its own again
            CHECK(c.free_bytes + n * sz == used);
            for (size_t k = 0; k < n; ++k) c.put(p[k], sz);
        }
    }
    CHECK(used == 0 && size.empty());
    {   // no memory left but what larger free blocks hold
        PinnedCache c;
        for (size_t k = 0; k < 16; ++k) CHECK(c.get(128 * MiB, &p[k], got) == hipSuccess);
        for (size_t k = 0; k < 16; ++k) c.put(p[k], 128 * MiB);
        for (size_t k = 0; k < 1024; ++k) CHECK(c.get(4 * MiB, &p[k], got) == hipSuccess);
        CHECK(used == MEMORY && c.free_bytes == 2048 * MiB);
        void *q, *r;
        CHECK(c.get(3 * MiB, &q, got) == hipSuccess && used == MEMORY - 2044 * MiB && c.free_bytes == 0);
        for (size_t k = 0; k < 511; ++k) CHECK(c.get(4 * MiB, &p[1024 + k], got) == hipSuccess);
        CHECK(used == MEMORY && c.get(MiB, &r, got) != hipSuccess);
        for (size_t k = 0; k < 1535; ++k) c.put(p[k], 4 * MiB);
        c.put(q, 4 * MiB);
    }
    CHECK(used == 0 && size.empty());
    return 0;
}
"""


def test_free_pinned_blocks_are_bounded_and_given_back(tmp_path):
    run_program(tmp_path, FREE_BLOCKS)


def test_pinned_blocks(tmp_path):
    run_program(tmp_path, PROGRAM)


def run_program(tmp_path, program):
    src, exe = tmp_path / "blocks.cpp", tmp_path / "blocks"
    src.write_text(program)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(PKG, "csrc"),
                    "-I", "/opt/rocm/include", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
