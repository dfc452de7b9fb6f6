"""The library's kept device memory over a device that the test plays: a few megabytes of memory, counted, with calls
that can be made to fail."""

import pytest

from test_host_kernels import _run

DEVICE = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include "host_util.hpp"
#include "pool.hip"
void hipcstone::setError(const std::string&) {}
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
static hipError_t g_query = hipSuccess;
static hipStreamCaptureStatus g_status = hipStreamCaptureStatusNone;
extern "C" hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s)
{
    *s = g_status;
    return g_query;
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
    need(poolTake(&p, &n) == hipSuccess, "take");
    return p;
}
constexpr size_t MB = size_t(1) << 20;
"""


@pytest.mark.parametrize("how", ["deviceMalloc(&p, 8 * MB)", "deviceMallocAsync(&p, 8 * MB, nullptr)",
                                 "poolTake(&p, &size)"])
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
    void* p     = nullptr;
    size_t size = 8 * MB;
    need(size && %s == hipSuccess && p, "no memory");
    need(g_held.size() == 1, "the kept blocks are given back");
    return 0;
}
""" % how)
    assert run.returncode == 0, run.stdout + run.stderr


def test_buffers_know_what_they_hold(tmp_path):
    """Buffers that take each other's blocks report what the device holds for them, and that is never much more than was
    asked for: an eighth of slack of the buffer's own, and the pool's rounding by at most another."""
    run = _run(tmp_path, "size", DEVICE + r"""
int main()
{
    PoolScope scope;
    DeviceBuf buf[6];
    size_t asked[6] = {};
    unsigned r      = 1;
    for (int step = 0; step < 4000; ++step)
    {
        r              = r * 1664525u + 1013904223u;
        DeviceBuf& b   = buf[r >> 8 & 3];
        const size_t n = size_t(1) << (10 + (r >> 12) % 16), more = (r >> 16) % 1000;
        if (r >> 28 & 1)
        {
            DeviceBuf empty;
            swap(empty, b);
            asked[&b - buf] = 0;
        }
        else if (n + n * more / 1000 > asked[&b - buf])
        {
            asked[&b - buf] = n + n * more / 1000;
            need(b.reserve(asked[&b - buf]) == HIPCSTONE_OK, "reserve");
        }
        scope.flush();
        size_t held = 0;
        for (DeviceBuf& o : buf)
        {
            const size_t n = asked[&o - buf];
            need(o.bytes >= n && (!o.ptr || g_held[o.ptr] == o.bytes), "a buffer does not know its size");
            // (what it was asked for last may be less than what it once grew to: then bytes stay)
            held += o.bytes;
        }
        need(held <= g_used, "more than the device holds");
    }
    // a block that was kept is not handed out for less than it was made for
    for (DeviceBuf& o : buf)
    {
        DeviceBuf empty;
        swap(empty, o);
    }
    scope.flush();
    poolTrim();
    for (int k = 0; k < 64; ++k)
    {
        const size_t big = (50 + k) * MB, small = 40 * MB;
        need(buf[0].reserve(big) == HIPCSTONE_OK, "reserve");
        {
            DeviceBuf empty;
            swap(empty, buf[0]);
        }
        scope.flush();
        need(buf[1].reserve(small) == HIPCSTONE_OK, "reserve");
        need(g_held[buf[1].ptr] <= small + small / 4 + small / 32, "a block much larger than asked for");
        {
            DeviceBuf empty;
            swap(empty, buf[1]);
        }
        scope.flush();
        poolTrim();
    }
    return 0;
}
""")
    assert run.returncode == 0, run.stdout + run.stderr


def test_memory_outlives_a_refused_free(tmp_path):
    """Where hipFree is refused (while a stream is captured) nothing is lost: blocks are freed at the next chance, a
    buffer keeps its memory, and an allocation that is refused too does not give the kept blocks away."""
    run = _run(tmp_path, "refused", DEVICE + r"""
int main()
{
    void *a = take(MB), *b = take(2 * MB), *c = take(4 * MB), *p = nullptr;
    DeviceBuf buf;
    need(buf.reserve(MB) == HIPCSTONE_OK, "reserve");
    void* before = buf.ptr;
    const size_t bytes = buf.bytes;
    poolGive(a);
    poolGive(b);
    g_refused = true;
    need(deviceMalloc(&p, MB) == hipErrorStreamCaptureUnsupported, "refused allocation");
    poolGive(c, false);
    need(buf.reserve(8 * MB) != HIPCSTONE_OK && buf.ptr == before && buf.bytes == bytes, "buffer without its memory");
    g_refused = false;
    need(g_held.size() == 4, "held");
    need(take(MB) == a, "the kept blocks are still kept");
    poolTrim();
    need(g_held.size() == 2 && g_held.count(a) && g_held.count(before), "everything else is freed");
    return 0;
}
""")
    assert run.returncode == 0, run.stdout + run.stderr


def test_no_allocation_where_a_capture_may_run(tmp_path):
    """Searches that can do without memory of their own take none while their stream is captured, nor where the runtime
    does not tell (it refuses the question for the null stream while another stream is captured); that is no error."""
    run = _run(tmp_path, "capture", DEVICE + r"""
int main()
{
    need(mayAllocate(nullptr), "no capture");
    g_status = hipStreamCaptureStatusActive;
    need(!mayAllocate(nullptr), "captured");
    g_status = hipStreamCaptureStatusNone;
    g_query  = hipErrorStreamCaptureImplicit;
    need(!mayAllocate(nullptr), "not told");
    return 0;
}
""")
    assert run.returncode == 0, run.stdout + run.stderr
