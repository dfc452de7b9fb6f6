// Device memory and streams kept for the next taker (host code only).
#include "runtime.hpp"

#include <algorithm>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace hipcstone
{

constexpr int kMaxDevices = 64;

namespace
{

struct PoolBlock
{
    void* ptr;
    size_t bytes;
    int device;
};

// never destroyed: threads may return memory while the process ends
struct Pool
{
    std::mutex m;
    std::unordered_map<void*, PoolBlock> taken;
    std::vector<PoolBlock> kept; // oldest first
    std::vector<PoolBlock> late; // to be freed: hipFree was refused (as while a stream is captured)
    size_t keptBytes[kMaxDevices] = {};
    std::vector<hipStream_t> streams[kMaxDevices];
};

Pool& pool()
{
    static Pool* p = new Pool;
    return *p;
}

// Block sizes are rounded up to steps of at most an eighth, so that blocks of similar sizes serve each other. Only blocks
// of the very size do (blocks up to half larger made neither sorts nor served bursts faster, and hold that much more).
size_t poolSize(size_t bytes)
{
    size_t step = 4096;
    while (step * 16 <= bytes)
        step *= 2;
    return (bytes + step - 1) / step * step;
}

thread_local PoolScope* t_scope = nullptr;

// frees the blocks, and the late ones with them; those that are refused (again) wait
void freeBlocks(std::vector<PoolBlock>& blocks)
{
    Pool& p = pool();
    {
        std::lock_guard<std::mutex> lock(p.m);
        blocks.insert(blocks.end(), p.late.begin(), p.late.end());
        p.late.clear();
    }
    for (const PoolBlock& b : blocks)
    {
        if (hipFree(b.ptr) == hipSuccess) continue;
        (void)hipGetLastError();
        std::lock_guard<std::mutex> lock(p.m);
        p.late.push_back(b);
    }
}

// once more with all kept blocks given back, where there was no memory
template<class Allocate>
hipError_t allocateOrTrim(Allocate allocate)
{
    hipError_t e = allocate();
    if (e != hipErrorOutOfMemory) return e;
    if (t_scope && !t_scope->freed.empty()) t_scope->flush(false);
    poolTrim();
    (void)hipGetLastError();
    return allocate();
}

} // namespace

hipError_t deviceMalloc(void** ptr, size_t bytes)
{
    return allocateOrTrim([&] { return hipMalloc(ptr, bytes); });
}

hipError_t deviceMallocAsync(void** ptr, size_t bytes, hipStream_t s)
{
    return allocateOrTrim([&] { return hipMallocAsync(ptr, bytes, s); });
}

bool mayAllocate(hipStream_t s)
{
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &status) == hipSuccess) return status == hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return false;
}

hipError_t poolTake(void** ptr, size_t* bytes)
{
    *ptr       = nullptr;
    int device = 0;
    if (hipError_t e = hipGetDevice(&device); e != hipSuccess) return e;
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    const size_t size = poolSize(*bytes);
    Pool& p           = pool();
    {
        std::lock_guard<std::mutex> lock(p.m);
        auto it = std::find_if(p.kept.begin(), p.kept.end(),
                               [&](const PoolBlock& b) { return b.device == device && b.bytes == size; });
        if (it != p.kept.end())
        {
            *ptr          = it->ptr;
            *bytes        = size;
            p.taken[*ptr] = *it;
            p.keptBytes[device] -= size;
            p.kept.erase(it);
            return hipSuccess;
        }
    }
    if (hipError_t e = deviceMalloc(ptr, size); e != hipSuccess) return e;
    std::lock_guard<std::mutex> lock(p.m);
    p.taken[*ptr] = PoolBlock{*ptr, size, device};
    *bytes        = size;
    return hipSuccess;
}

void poolGive(void* ptr, bool idle)
{
    if (!ptr) return;
    Pool& p = pool();
    std::vector<PoolBlock> out;
    {
        std::lock_guard<std::mutex> lock(p.m);
        auto it = p.taken.find(ptr);
        if (it == p.taken.end()) return;
        const PoolBlock b = it->second;
        p.taken.erase(it);
        if (!idle || b.bytes > kPoolBytes) { out.push_back(b); }
        else
        {
            p.kept.push_back(b);
            p.keptBytes[b.device] += b.bytes;
            for (size_t i = 0; p.keptBytes[b.device] > kPoolBytes; ++i)
            {
                if (p.kept[i].device != b.device) continue;
                p.keptBytes[b.device] -= p.kept[i].bytes;
                out.push_back(p.kept[i]);
                p.kept.erase(p.kept.begin() + ptrdiff_t(i--));
            }
        }
    }
    if (!out.empty()) freeBlocks(out);
}

void poolTrim()
{
    Pool& p = pool();
    std::vector<PoolBlock> out;
    {
        std::lock_guard<std::mutex> lock(p.m);
        out.swap(p.kept);
        for (size_t& b : p.keptBytes)
            b = 0;
    }
    freeBlocks(out);
}

hipError_t poolTakeStream(hipStream_t* s)
{
    int device = 0;
    if (hipError_t e = hipGetDevice(&device); e != hipSuccess) return e;
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    Pool& p = pool();
    {
        std::lock_guard<std::mutex> lock(p.m);
        auto& v = p.streams[device];
        if (!v.empty())
        {
            *s = v.back();
            v.pop_back();
            return hipSuccess;
        }
    }
    return hipStreamCreate(s);
}

void poolGiveStream(hipStream_t s)
{
    int device = 0;
    Pool& p    = pool();
    if (hipGetDevice(&device) == hipSuccess && device >= 0 && device < kMaxDevices)
    {
        std::lock_guard<std::mutex> lock(p.m);
        if (p.streams[device].size() < kPoolStreams)
        {
            p.streams[device].push_back(s);
            return;
        }
    }
    (void)hipStreamDestroy(s);
}

PoolScope* poolScope() { return t_scope; }

PoolScope::PoolScope()
    : outer(t_scope)
{
    t_scope = this;
}

PoolScope::~PoolScope()
{
    flush(false);
    t_scope = outer;
}

void PoolScope::flush(bool idle)
{
    for (void* p : freed)
        poolGive(p, idle);
    freed.clear();
}

} // namespace hipcstone
