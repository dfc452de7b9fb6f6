"""The library's kept device memory over a device that the test plays: a few megabytes of memory, counted, with calls
that can be made to fail."""

import pytest

from test_host_kernels import _run

DEVICE = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include "pool.hip"
using namespace hipcstone;

static std::map<void*, size_t> g_held;
static size_t g_used = 0, g_limit = size_t(1) << 40;
static int g_frees = 0;
static bool g_refused = false; // as while the thread's stream is captured

extern "C" hipError_t hipMalloc(void** p, size_t n)
{
    *p = nullptr;
    if (g_refused) return hipErrorStreamCaptureUnsupported;
    if (g_used + n > g_limit) return hipErrorOutOfMemory;
    static uintptr_t next = 1 << 20;
    *p = reinterpret_cast<void*>(next);
    next += (n + 4095) / 4096 * 4096;
    g_held[*p] = n;
    g_used += n;
    return hipSuccess;
}
extern "C" hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { return hipMalloc(p, n); }
extern "C" hipError_t hipFree(void* p)
{
    if (g_refused) return hipErrorStreamCaptureUnsupported;
    if (!g_held.count(p)) { printf("free of memory that is not held\n"); exit(1); }
    g_used -= g_held[p];
    g_held.erase(p);
    ++g_frees;
    return hipSuccess;
}
extern "C" hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
extern "C" hipError_t hipGetLastError() { return hipSuccess; }
extern "C" hipError_t hipStreamCreate(hipStream_t*) { return hipErrorUnknown; }
extern "C" hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }

static void need(bool ok, const char* what)
{
    if (ok) return;
    printf("%s\n", what);
    exit(1);
}
static void* take(size_t n)
{
    void* p = nullptr;
    need(poolTake(&p, n) == hipSuccess, "take");
    return p;
}
constexpr size_t MB = size_t(1) << 20;
"""


@pytest.mark.parametrize("how", ["deviceMalloc(&p, 8 * MB)", "deviceMallocAsync(&p, 8 * MB, nullptr)", "poolTake(&p, 8 * MB)"])
def test_allocations_get_the_kept_blocks_back(tmp_path, how):
    """With 10 MB on the device and 6 of them kept, an allocation of 8 MB succeeds, whichever way it is made."""
    run = _run(tmp_path, "trim", DEVICE + r"""
int main()
{
    g_limit = 10 * MB;
    void *a = take(2 * MB), *b = take(4 * MB);
    poolGive(a);
    poolGive(b);
    need(g_used >= 6 * MB, "kept");
    void* p = nullptr;
    need(%s == hipSuccess && p, "no memory");
    need(g_held.size() == 1, "the kept blocks are given back");
    return 0;
}
""" % how)
    assert run.returncode == 0, run.stdout + run.stderr
