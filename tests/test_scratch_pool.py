"""CPU tests of the library's device memory: the scratch that builds keep between
calls goes back when memory runs out, on request, and past its bound, and a build
refused in a capture leaves the capturing stream alone.  A small program stands in
for the HIP runtime (its symbols come before libamdhip64's): device memory is host
memory with a budget, kernels do nothing."""
import os
import subprocess
import tempfile

import pytest

import gchi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROG = r'''
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <dlfcn.h>
#include <map>
#include "gchi.h"

struct Dim3 { unsigned x, y, z; };
static std::map<void *, size_t> g_blocks;
static size_t g_used = 0, g_budget = (size_t)1 << 40;
static int g_error = 0, g_capturing = 0, g_waits = 0;

extern "C" {
int hipMalloc(void **p, size_t n) {
    if (g_used + n > g_budget) return g_error = 2;  // hipErrorOutOfMemory
    *p = calloc(n, 1);
    g_blocks[*p] = n;
    g_used += n;
    return 0;
}
int hipFree(void *p) {
    if (!p) return 0;
    g_used -= g_blocks.at(p);
    g_blocks.erase(p);
    free(p);
    return 0;
}
int hipGetLastError() { int e = g_error; g_error = 0; return e; }
const char *hipGetErrorString(int) { return "stub"; }
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipGetDeviceCount(int *n) { *n = 1; return 0; }
int hipSetDevice(int) { return 0; }
int hipDeviceGetAttribute(int *v, int, int) { *v = 256; return 0; }
int hipGetDevicePropertiesR0600(void *, int) { return 1; }
int hipFuncSetAttribute(const void *, int, int) { return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) { memcpy(d, s, n); return 0; }
int hipStreamSynchronize(void *) { g_waits++; return 0; }
int hipDeviceSynchronize() { return 0; }
int hipStreamIsCapturing(void *, int *st) { *st = g_capturing; return 0; }
int hipLaunchKernel(const void *, Dim3, Dim3, void **, size_t, void *) { return 0; }
int __hipPushCallConfiguration(Dim3, Dim3, size_t, void *) { return 0; }
int __hipPopCallConfiguration(Dim3 *, Dim3 *, size_t *, void **) { return 0; }
}

#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)

int main(int, char **argv) {
    void *h = dlopen(argv[1], RTLD_NOW);
    if (!h) { printf("%s\n", dlerror()); return 1; }
#define FN(name) auto *name##_ = (decltype(&name))dlsym(h, #name)
    FN(gchi_malloc);
    FN(gchi_free);
    FN(gchi_shard_build);
    FN(gchi_shard_destroy);
    FN(gchi_pr_plan_create);
    const int what = atoi(argv[2]);
    const uint32_t top = (1u << 20) - 1;  // vertex ids: about 20 bytes each of scratch, 8 of the handle
    gchi_shards *sh = nullptr;
    CHECK(gchi_shard_build_(nullptr, nullptr, 0, top, 2, &sh, nullptr) == GCHI_OK);
    gchi_shard_destroy_(sh);
    const size_t kept = g_used;
    CHECK(kept > (size_t)8 << 20);
    void *p = nullptr;
    if (what == 0) {  // gchi_malloc takes the kept bytes when there are no others
        g_budget = kept + 1000;
        CHECK(gchi_malloc_(&p, kept) == GCHI_OK);
        CHECK(g_used == kept && g_error == 0);
        CHECK(gchi_malloc_(&p, kept) == GCHI_ERR_HIP);  // now there are none
        CHECK(g_error == 0);                           // and no launch check finds that error later
    } else if (what == 1) {  // so does a handle, and its build's own scratch
        g_budget = (size_t)28 * (top / 2 + 1) + ((size_t)1 << 20);  // less than what is kept
        CHECK(gchi_shard_build_(nullptr, nullptr, 0, top / 2, 2, &sh, nullptr) == GCHI_OK);
        gchi_shard_destroy_(sh);
    } else if (what == 2) {  // on request
        FN(gchi_pool_trim);
        size_t n = 0;
        CHECK(gchi_pool_trim_ && gchi_pool_trim_(&n) == GCHI_OK && n == kept && g_used == 0);
        CHECK(gchi_pool_trim_(nullptr) == GCHI_OK);
        CHECK(gchi_shard_build_(nullptr, nullptr, 0, top, 2, &sh, nullptr) == GCHI_OK);
        gchi_shard_destroy_(sh);
        CHECK(g_used == kept);
    } else if (what == 3) {  // past the bound of 1 GiB
        CHECK(gchi_shard_build_(nullptr, nullptr, 0, 80 * (top + 1) - 1, 2, &sh, nullptr) == GCHI_OK);
        gchi_shard_destroy_(sh);
        CHECK(g_used <= (size_t)1 << 30);
    } else {  // refused while the stream captures, with no wait: that would end the capture
        uint32_t off[2] = {0, 0}, deg[1] = {0};
        gchi_dgraph g = {};
        g.nvertices = 1;
        g.in_off = off;
        g.in_src = deg;
        g.outdeg = deg;
        g_capturing = 1;
        g_waits = 0;
        for (int form = 0; form <= 4; form++) {
            gchi_pr_tune t = {form == 2 ? 256 : 0, 0, form, 0};
            gchi_pr_plan *plan = nullptr;
            CHECK(gchi_pr_plan_create_(&g, &t, &plan, nullptr) == GCHI_ERR_HIP);
        }
        CHECK(gchi_shard_build_(nullptr, nullptr, 0, top, 2, &sh, nullptr) == GCHI_ERR_HIP);
        CHECK(g_waits == 0);
        CHECK(g_used == kept);
    }
    puts("ok");
    return 0;
}
'''


@pytest.fixture(scope="module")
def prog():
    with tempfile.TemporaryDirectory(prefix="gchi_pool_") as d:
        src, exe = os.path.join(d, "pool.cpp"), os.path.join(d, "pool")
        with open(src, "w") as f:
            f.write(PROG)
        subprocess.run(["g++", "-std=c++17", "-O1", "-rdynamic", "-I" + os.path.join(ROOT, "include"), src, "-o", exe,
                        "-ldl"], check=True)
        yield exe


CASES = ["malloc", "handle", "trim", "bound", "capture"]


@pytest.mark.parametrize("what", range(len(CASES)), ids=CASES)
def test_scratch_against_stand_in(prog, what):
    run = subprocess.run([prog, gchi.LIB_PATH, str(what)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and run.stdout.strip() == "ok", run.stdout + run.stderr
