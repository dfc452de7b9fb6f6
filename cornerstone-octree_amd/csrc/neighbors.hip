// a16: radius neighbor search with the per-particle semantics of the reference CPU path (findneighbors.hpp:77-177,
// traversal.hpp:26-69): the library's launches of the wave walk in hipcstone_nbwalk.hpp (which documents the
// semantics and the design), row-major or slot-major, plain or segmented (the batched clouds).
#include <limits>
#include <type_traits>

#include "common.hpp"
#include "hipcstone_nbwalk.hpp"
#include "runtime.hpp"

namespace hipcstone
{

// SlotMajor: the rows of 64 targets are stored slot-major (neighbor k of the l-th of them at k * 64 + l) instead of
// row-major (l * ngmax + k), so that a consumer with one thread per target reads each slot with one coalesced load.
// Segmented: many independent trees in one set of arrays (the batched clouds). Wave `group` then takes its targets
// [first, last) (at most 64, inside one cloud) and the index of its cloud's root node from the wave table
// (waves[3 g], waves[3 g + 1], cloud = waves[3 g + 2], root = roots[cloud]); rows and counts are indexed by the
// particle index itself (firstId = 0), and a child block may lie before its parent (the batched link places children
// by internal-node slot, not level by level), so only the bounds and depth guards and the step budget apply.
// Waves per workgroup: 4 by default; 2 and 8 are the other shapes the autotuner measures
// (hipcstone_set_neighbor_waves). Every wave owns its own targets, stack and leaf list, so the shape changes only
// how waves are grouped onto CUs (LDS per workgroup, scheduling granularity), never a result.
// targetsPerWave: 64, or fewer where that many waves would leave the device idle (kFullWaves).
//
// Vector and scalar issue bound it (no unit of memory is near its limit, the matrix cores are a sixth busy): the walk takes
// 2.25 of 6.2 ms, the chunks' set-up 1.0, the pair tests 1.45, the rows 1.5 (16.8M targets, 100 neighbors, fp32). The
// search of that size took 7.65 ms with the pair tests in vector code, one candidate of one leaf at a time (38.7K
// instructions a wave, now 25.0K); in fp64 at 2M, where nothing was compact either, 1.57 -> 0.90 ms.

// Minimum waves per SIMD the registers are allocated for. fp32: 5 waves 6.53 ms, 6 waves 6.20, where 5 vector registers go
// to memory, none of them in the inner loops (16.8M targets); the LDS holds no seventh wave. fp64, 300k uniform targets
// open / periodic: 4 and 5 waves (one allocation in open boxes) 201 / 282 and 200 / 254 us, 6 waves 217 / 274; 2M open:
// 904, 906, 999; 30k, which do not fill the device: 79, 79, 87. At 5 open fp64 walks spill nothing, periodic ones 5 vector
// and 49 to 58 scalar registers.
template<class T>
constexpr int kNbMinWavesPerEu = std::is_same_v<T, float> ? 6 : 5;

typedef uint32_t Row4 __attribute__((ext_vector_type(4), aligned(4)));

template<class T, bool AnyPbc, bool SlotMajor, bool Segmented, int kNbWaves>
__global__ __launch_bounds__(kNbWaves * kWave) __attribute__((amdgpu_waves_per_eu(kNbMinWavesPerEu<T>, 8)))
void findNeighborsKernel(
    const T* __restrict__ x, const T* __restrict__ y, const T* __restrict__ z, const T* __restrict__ h,
    uint32_t firstId, uint32_t lastId, typename BoxOf<T>::type box, const int32_t* __restrict__ childOffsets,
    const int32_t* __restrict__ internalToLeaf, const uint32_t* __restrict__ layout, const T* __restrict__ centers,
    const T* __restrict__ sizes, int32_t numNodes, float ext, uint32_t ngmax, uint32_t* __restrict__ neighbors,
    uint32_t* __restrict__ neighborsCount, uint32_t numBlocksPadded, uint32_t* __restrict__ faults,
    uint32_t targetsPerWave, const uint32_t* __restrict__ waves = nullptr, uint32_t numWaves = 0,
    const int32_t* __restrict__ roots = nullptr, const nbwalk::ChildGroup<T>* __restrict__ groups = nullptr)
{
    __shared__ nbwalk::Shared<T, kNbWaves> sh;
    const int lane       = laneId();
    const int w          = threadIdx.x / kWave;
    const uint32_t block = xcdContiguousBlock(blockIdx.x, numBlocksPadded);
    const uint32_t group = uniform(block * uint32_t(kNbWaves) + uint32_t(w));
    uint64_t first;
    int32_t root = 0;
    if constexpr (Segmented)
    {
        if (group >= numWaves) return;
        first  = uniform(waves[3 * group]);
        lastId = uniform(waves[3 * group + 1]);
        root   = uniform(roots[uniform(waves[3 * group + 2])]);
        if (root < 0 || root >= numNodes)
        {
            if (lane == 0) atomicOr(faults, HIPCSTONE_FAULT_MALFORMED_TREE);
            return;
        }
    }
    else
    {
        first = uint64_t(firstId) + uint64_t(group) * targetsPerWave;
        if (first >= lastId) return;
    }
    const uint32_t i = uint32_t(first) + uint32_t(lane);
    const bool valid = i < lastId && uint32_t(lane) < targetsPerWave;
    // the wave's rows: row-major, or slot-major in their group of 64 (which holds whole waves)
    const size_t row = Segmented ? size_t(first) : size_t(first) - firstId;
    uint32_t* rows   = neighbors;
    if (ngmax) rows += SlotMajor ? row / kWave * kWave * ngmax + row % kWave : row * ngmax;
    const nbwalk::Tree<T> tree{childOffsets, internalToLeaf, layout, centers, sizes, numNodes, ext, groups};
    const uint32_t count = nbwalk::walk<T, AnyPbc, Segmented, kNbWaves>(
        x, y, z, h, box, tree, root, first, valid, ngmax != 0, sh, w, faults,
        [&](uint32_t before, uint32_t hits, auto&& next) __attribute__((always_inline)) {
            // the row's next slots, four to a store; the last ones one by one
            uint32_t rest = min(hits, ngmax - min(before, ngmax));
            uint32_t slot = SlotMajor ? before * kWave + uint32_t(lane) : uint32_t(lane) * ngmax + before;
            while (rest != 0)
            {
                const uint32_t j0 = next(), j1 = next(), j2 = next(), j3 = next();
                uint32_t* row     = rows + slot;
                if constexpr (SlotMajor)
                {
                    row[0] = j0;
                    if (rest > 1) row[kWave] = j1;
                    if (rest > 2) row[2 * kWave] = j2;
                    if (rest > 3) row[3 * kWave] = j3;
                    slot += 4 * kWave;
                }
                else
                {
                    if (rest > 3) *reinterpret_cast<Row4*>(row) = Row4{j0, j1, j2, j3};
                    else
                    {
                        row[0] = j0;
                        if (rest > 1) row[1] = j1;
                        if (rest > 2) row[2] = j2;
                    }
                    slot += 4;
                }
                rest -= min(rest, 4u);
            }
        });
    if (valid) neighborsCount[i - firstId] = count;
}

// the segmented search of the batched clouds (row-major rows, open boxes): see findNeighborsKernel
template<class T>
hipcstone_status findNeighborsSegmented(hipStream_t s, const T* x, const T* y, const T* z, const T* h,
                                        const typename BoxOf<T>::type& box, const int32_t* childOffsets,
                                        const int32_t* internalToLeaf, const uint32_t* layout, const T* centers,
                                        const T* sizes, int32_t numNodesCap, uint32_t ngmax, uint32_t* neighbors,
                                        uint32_t* neighborsCount, const uint32_t* waves, uint32_t numWaves,
                                        const int32_t* roots, const nbwalk::ChildGroup<T>* groups)
{
    if (numWaves == 0) return HIPCSTONE_OK;
    if (ngmax > (1u << 20)) return invalid("findNeighbors: ngmax above 2^20");
    uint32_t* faults = faultWord();
    if (!faults) return HIPCSTONE_HIP_ERROR;
    auto launch = [&](auto wv) {
        constexpr int W = decltype(wv)::value;
        unsigned blocks = ceilDiv(size_t(numWaves), W);
        blocks          = (blocks + kXcds - 1) / kXcds * kXcds;
        findNeighborsKernel<T, false, false, true, W><<<blocks, W * kWave, 0, s>>>(
            x, y, z, h, 0u, 0u, box, childOffsets, internalToLeaf, layout, centers, sizes, numNodesCap, 1.0f, ngmax,
            neighbors, neighborsCount, blocks, faults, kWave, waves, numWaves, roots, groups);
    };
    switch (neighborWaves())
    {
    case 2: launch(std::integral_constant<int, 2>{}); break;
    case 8: launch(std::integral_constant<int, 8>{}); break;
    default: launch(std::integral_constant<int, 4>{}); break;
    }
    HC_CHECK_LAUNCH("findNeighborsKernel (segmented)");
    return HIPCSTONE_OK;
}

template hipcstone_status findNeighborsSegmented<float>(hipStream_t, const float*, const float*, const float*,
                                                        const float*, const BoxOf<float>::type&, const int32_t*,
                                                        const int32_t*, const uint32_t*, const float*, const float*,
                                                        int32_t, uint32_t, uint32_t*, uint32_t*, const uint32_t*,
                                                        uint32_t, const int32_t*, const nbwalk::ChildGroup<float>*);

// (a record is 128 bytes for either float type)
size_t neighborGroupsBytes(int32_t numNodes)
{
    static_assert(sizeof(nbwalk::ChildGroup<float>) == 128 && sizeof(nbwalk::ChildGroup<double>) == 128);
    return nbwalk::childGroupCount(numNodes) * sizeof(nbwalk::ChildGroup<double>);
}

template<class T>
static hipcstone_status buildChildGroups(hipStream_t s, const T* centers, const T* sizes, const int32_t* childOffsets,
                                         const int32_t* internalToLeaf, int32_t numNodes,
                                         nbwalk::ChildGroup<T>* groups)
{
    const uint32_t numGroups = uint32_t(nbwalk::childGroupCount(numNodes));
    if (numGroups == 0) return HIPCSTONE_OK;
    nbwalk::childGroupsKernel<T><<<(numGroups + 255) / 256, 256, 0, s>>>(centers, sizes, childOffsets, internalToLeaf,
                                                                          numNodes, numGroups, groups);
    HC_CHECK_LAUNCH("childGroupsKernel");
    return HIPCSTONE_OK;
}

// Targets of a wave: 64, halved down to 4 while that gives fewer waves than kFullWaves. A wave's time is its own chain of
// descents and chunks, so on an idle device more, smaller waves end sooner; on a full one they test more candidates.
// Measured with 64 / 32 / 16 / 8 targets a wave (Plummer clouds, ngmax 150, fp32, us): 1000 targets 164 / 144 / 120 / 105
// (4: 98), 16000: 588 / 528 / 460 / 432, 65000: 287 / 257 / 216 / 248, 131000: 184 / 155 / 187 / 248, 200000: 188 / 198 /
// 227 / 323; fp64 turns at the same sizes. So each half stops paying where the double of it fills 2048 waves, two for
// each SIMD. Below 4 targets another 1-5 %.
constexpr uint32_t kFullWaves = 2048;

static uint32_t targetsPerWave(uint32_t n)
{
    uint32_t t = kWave;
    while (t > 4 && n / t < kFullWaves)
        t /= 2;
    return t;
}

template<class T>
static hipcstone_status findNeighbors(hipcstone_stream s, const T* x, const T* y, const T* z, const T* h,
                                      uint32_t firstId, uint32_t lastId, const typename BoxOf<T>::type* box,
                                      const int32_t* childOffsets, const int32_t* parents,
                                      const int32_t* internalToLeaf, const uint32_t* layout, const T* centers,
                                      const T* sizes, int32_t numNodes, float ext, uint32_t ngmax,
                                      uint32_t* neighbors, uint32_t* neighborsCount, bool slotMajor,
                                      void* groupsWs = nullptr, size_t groupsWsBytes = 0)
{
    if (lastId <= firstId) return HIPCSTONE_OK;
    if (!x || !y || !z || !h || !box || !childOffsets || !parents || !internalToLeaf || !layout || !centers ||
        !sizes || !neighborsCount)
        return invalid("findNeighbors: null pointer");
    if (ngmax > 0 && !neighbors) return invalid("findNeighbors: neighbors is null with ngmax > 0");
    if (ngmax > (1u << 20)) return invalid("findNeighbors: ngmax above 2^20");
    if (numNodes <= 0) return invalid("findNeighbors: numNodes must be positive");
    const uint32_t perWave  = targetsPerWave(lastId - firstId);
    const size_t waveGroups = (size_t(lastId - firstId) + perWave - 1) / perWave;
    uint32_t* faults = faultWord();
    if (!faults) return HIPCSTONE_HIP_ERROR;
    bool anyPbc     = box->bnd[0] == HIPCSTONE_PERIODIC || box->bnd[1] == HIPCSTONE_PERIODIC ||
                  box->bnd[2] == HIPCSTONE_PERIODIC;
    // the walk goes through the compact child blocks, built here into the caller's workspace or into memory allocated
    // on the stream for this call; fp64 and periodic searches, which take no memory of their own elsewhere, do
    // without them (child by child) where there is none to be had: while a stream is captured, or at the limit
    void* owned                         = nullptr;
    const nbwalk::ChildGroup<T>* groups = nullptr;
    if (const size_t need = neighborGroupsBytes(numNodes))
    {
        constexpr bool kOptional = !std::is_same_v<T, float>;
        const bool optional      = kOptional || anyPbc;
        void* dst                = groupsWs && groupsWsBytes >= need ? groupsWs : nullptr;
        bool allocate            = !dst;
        if (allocate && optional) allocate = mayAllocate(stream(s));
        if (allocate)
        {
            const hipError_t e = deviceMallocAsync(&owned, need, stream(s));
            if (e != hipSuccess && !optional) return hipFail(e, "findNeighbors: child blocks");
            if (e != hipSuccess)
            {
                (void)hipGetLastError();
                owned = nullptr;
            }
            dst = owned;
        }
        if (dst)
        {
            auto* blocks = static_cast<nbwalk::ChildGroup<T>*>(dst);
            if (auto e = buildChildGroups<T>(stream(s), centers, sizes, childOffsets, internalToLeaf, numNodes, blocks))
            {
                if (owned) (void)hipFreeAsync(owned, stream(s));
                return e;
            }
            groups = blocks;
        }
    }
    auto shaped = [&](auto pbc, auto slots, auto wv) {
        constexpr int W = decltype(wv)::value;
        unsigned blocks = ceilDiv(waveGroups, W);
        blocks          = (blocks + kXcds - 1) / kXcds * kXcds; // whole rounds over the XCDs; extra groups exit
        findNeighborsKernel<T, decltype(pbc)::value, decltype(slots)::value, false, W>
            <<<blocks, W * kWave, 0, stream(s)>>>(x, y, z, h, firstId, lastId, *box, childOffsets, internalToLeaf,
                                                  layout, centers, sizes, numNodes, ext, ngmax, neighbors,
                                                  neighborsCount, blocks, faults, perWave, nullptr, 0u, nullptr, groups);
    };
    auto launch = [&](auto pbc, auto slots) {
        switch (neighborWaves())
        {
        case 2: shaped(pbc, slots, std::integral_constant<int, 2>{}); break;
        case 8: shaped(pbc, slots, std::integral_constant<int, 8>{}); break;
        default: shaped(pbc, slots, std::integral_constant<int, 4>{}); break;
        }
    };
    if (anyPbc && slotMajor) launch(std::true_type{}, std::true_type{});
    else if (anyPbc) launch(std::true_type{}, std::false_type{});
    else if (slotMajor) launch(std::false_type{}, std::true_type{});
    else launch(std::false_type{}, std::false_type{});
    hipError_t launched = hipGetLastError();
    if (owned) HC_CHECK(hipFreeAsync(owned, stream(s)));
    if (launched != hipSuccess) return hipFail(launched, "findNeighborsKernel");
    return HIPCSTONE_OK;
}

template<class T>
hipcstone_status findNeighborsWs(hipcstone_stream s, const T* x, const T* y, const T* z, const T* h, uint32_t firstId,
                                 uint32_t lastId, const typename BoxOf<T>::type* box, const int32_t* childOffsets,
                                 const int32_t* parents, const int32_t* internalToLeaf, const uint32_t* layout,
                                 const T* centers, const T* sizes, int32_t numNodes, float ext, uint32_t ngmax,
                                 uint32_t* neighbors, uint32_t* neighborsCount, void* groupsWs, size_t groupsWsBytes)
{
    return findNeighbors<T>(s, x, y, z, h, firstId, lastId, box, childOffsets, parents, internalToLeaf, layout,
                            centers, sizes, numNodes, ext, ngmax, neighbors, neighborsCount, false, groupsWs,
                            groupsWsBytes);
}

#define HIPCSTONE_INST_NEIGHBORS_WS(T)                                                                                 \
    template hipcstone_status findNeighborsWs<T>(                                                                      \
        hipcstone_stream, const T*, const T*, const T*, const T*, uint32_t, uint32_t, const BoxOf<T>::type*,           \
        const int32_t*, const int32_t*, const int32_t*, const uint32_t*, const T*, const T*, int32_t, float, uint32_t, \
        uint32_t*, uint32_t*, void*, size_t);
HIPCSTONE_INST_NEIGHBORS_WS(float)
HIPCSTONE_INST_NEIGHBORS_WS(double)

} // namespace hipcstone

using namespace hipcstone;

extern "C"
{

#define HIPCSTONE_DEF_NEIGHBORS(RS, T)                                                                                 \
    hipcstone_status hipcstone_find_neighbors_##RS(                                                                    \
        hipcstone_stream s, const T* x, const T* y, const T* z, const T* h, uint32_t first_id, uint32_t last_id,      \
        const hipcstone_box_##RS* box, const int32_t* child_offsets, const int32_t* parents,                          \
        const int32_t* internal_to_leaf, const uint32_t* layout, const T* centers, const T* sizes, int32_t num_nodes,  \
        float ext, uint32_t ngmax, uint32_t* neighbors, uint32_t* neighbors_count)                                     \
    {                                                                                                                  \
        return findNeighbors<T>(s, x, y, z, h, first_id, last_id, box, child_offsets, parents, internal_to_leaf,      \
                                layout, centers, sizes, num_nodes, ext, ngmax, neighbors, neighbors_count, false);     \
    }                                                                                                                  \
    hipcstone_status hipcstone_find_neighbors_slot_major_##RS(                                                         \
        hipcstone_stream s, const T* x, const T* y, const T* z, const T* h, uint32_t first_id, uint32_t last_id,      \
        const hipcstone_box_##RS* box, const int32_t* child_offsets, const int32_t* parents,                          \
        const int32_t* internal_to_leaf, const uint32_t* layout, const T* centers, const T* sizes, int32_t num_nodes,  \
        float ext, uint32_t ngmax, uint32_t* neighbors, uint32_t* neighbors_count)                                     \
    {                                                                                                                  \
        return findNeighbors<T>(s, x, y, z, h, first_id, last_id, box, child_offsets, parents, internal_to_leaf,      \
                                layout, centers, sizes, num_nodes, ext, ngmax, neighbors, neighbors_count, true);      \
    }

HIPCSTONE_DEF_NEIGHBORS(f32, float)
HIPCSTONE_DEF_NEIGHBORS(f64, double)

} // extern "C"
