/*
 * hipcstone neighbor walk: the device side of the radius neighbor search, for HIP C++ code built for gfx950.
 *
 * One wave64 walks the octree for up to 64 consecutive targets and hands each its neighbors. The library's search entry
 * points (hipcstone_find_neighbors_*, libhipcstone.so) launch it as is; hipcstone_ijloop.hpp instantiates it in the
 * caller's translation unit inside its fused interaction loop, which folds the neighbors as they come.
 *
 * Reference semantics (findneighbors.hpp:77-177, traversal.hpp:26-69, boxoverlap.hpp:217-250, util/array.hpp:237-240):
 * particle i visits node n iff every node on the root->n path passes
 *     norm2(minDistance(p_i, center_n, size_n)) < 4 h_i^2 * ext^2      (right-fold norm2, CPU minDistance order)
 * and at each visited leaf records j != i with  dx*dx + dy*dy + dz*dz < 4 h_i^2  (left fold), ascending j,
 * keeping the first ngmax and counting all.
 *
 * Design — one wave64 owns up to 64 consecutive targets (compact in space because they are SFC-ordered):
 *  * Walk: depth-first with an explicit per-wave stack, one entry per lane of a few vector registers (readlane and
 *    writelane at a uniform index), whose older half moves to LDS when it is full. Descending into a node evaluates its
 *    8 children at once, from the compact record of the block (ChildGroup: one wide scalar load, and 12 additions for
 *    the 8 distances), each with the ballot of lanes whose own predicate chain passed: a lane is tested at a child only
 *    if it passed the parent. Where a block has no such record the children's own centers and sizes are loaded.
 *    The visited leaf set of every lane is therefore exactly the CPU's, not the superset a group-box walk gives.
 *    Children are taken in order 0..7, so leaves come out in the CPU's visiting order (ascending SFC order).
 *  * Leaves and their lane masks go to a per-wave list. A full list becomes candidates: the listed leaves' particles
 *    one after another, in chunks of 64. Each chunk is tested against all 64 targets on the matrix cores and leaves
 *    every target one 64-bit word of hits, which then loses the candidates of leaves the target did not visit.
 *  * Hit words are kept in LDS for several chunks, then every lane takes its own target's hits out of its words in
 *    ascending order, four at a time, and hands them on (rows in memory, or a caller's fold over the neighbors).
 *  * Every loop is bounded: the walk by 2 * numNodes + 8 steps and the stack depth by the key's level count. A guard
 *    that fires ends the walk and ORs its HIPCSTONE_FAULT_* bit into the fault word.
 *
 * The pair test on the matrix cores. With coordinates relative to a center c near the wave's targets,
 *     D = |x_j - x_i|^2 - 4 h_i^2 = (|x_i|^2 - 4 h_i^2) + |x_j|^2 - 2 x_i . x_j
 * is one 16x16x4 fp32 product (x_j, y_j, z_j, |x_j|^2) . (-2 x_i, -2 y_i, -2 z_i, 1) accumulated onto the target's
 * constant: the sign of D is the test. D is not the reference's rounded distance, so the sign is taken only where
 * |D| >= E, with E an upper bound of the error of D and of the reference's own distance for every pair that matters:
 * with u = 2^-24, a = |x_i|, r = 2 h_i and S = 2 a + r, a pair with D near 0 has |x_j| <= a + r, so the roundings of
 * the relative coordinates (2 u r S), of |x_j|^2 and |x_i|^2 (7 u S^2), of the four accumulations (each of at most
 * (a + |x_j|)^2 + r^2 <= S^2 + r^2, counted with a whole ulp) and of the reference's distance (5 u r^2) stay below
 * 16 u (S^2 + r^2). E is 1e-6 (S^2 + r^2), more by 0.7 u S^2. A pair with |x_j| = a + r + d, d > 0, has D >= d^2 and an
 * error that is larger by at most 44 u S d + 22 u d^2: less than both together, so it never comes out at -E or below. E is
 * taken at the wave's largest target. A chunk with a |D| < E (about one wave in five has one at 100 neighbors) tests the
 * 16-candidate groups it occurs in again, in the reference's own operations. fp64 lengths are first multiplied by one
 * power of two for the whole wave, so the products do not depend on the unit of length; only waves whose largest length
 * is beyond 2^-48 to 2^60 (fp32, where the reference's own squares near the ends of the range) or 2^-100 to 2^101 (fp64)
 * do without the products and test each target against a chunk's 64 candidates at once. So every decision is the
 * reference's, bit for bit, for fp32 and fp64 alike.
 * A wave with a target whose 2h box leaves a periodic domain folds its candidates to their images nearest to c. While
 * S < L / 2 these are the reference's images for every pair that can be a hit, and the folded differences are off by at
 * most 2 u L per dimension, the reference's included, so E grows by 8 u r L; with a larger S the wave does without the
 * products, and a chunk with a particle outside the domain is tested again (the reference folds only for targets near
 * its faces).
 *
 * What bounds it is instruction issue: a wave of 64 targets with 100 neighbors takes 12.2K vector, 7.1K scalar and
 * 2.6K branch instructions, and 323 matrix products, which replace some 90K multiply-adds and compares by lane. Pair
 * tests one candidate at a time took 16.2K vector and 12.8K scalar instructions (16.8M targets: 7.65 ms, now 6.2).
 *
 * Everything that decides is evaluated in the reference's floating-point order; compile with -ffp-contract=off and
 * without packed fp32 ops (-Xclang -target-feature -Xclang -packed-fp32-ops).
 */
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <limits>
#include <type_traits>

#include "hipcstone.h"

namespace hipcstone
{

// ---- wave64 primitives ----

constexpr int kWave = 64;

__device__ inline uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }

// this lane's bit of a wave-uniform mask; the mask is used as a lane predicate as is (no per-lane shift and compare)
__device__ inline bool laneIn(uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

// number of set bits of mask below this lane
__device__ inline unsigned laneRank(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi(uint32_t(mask >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mask), 0u));
}

__device__ inline int laneId() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

__device__ inline int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline unsigned uniform(unsigned v) { return unsigned(__builtin_amdgcn_readfirstlane(int(v))); }

__device__ inline uint64_t uniform64(uint64_t v)
{
    uint32_t lo = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v))));
    uint32_t hi = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v >> 32))));
    return (uint64_t(hi) << 32) | lo;
}

// order LDS writes of some lanes before LDS reads of other lanes of the same wave
__device__ inline void waveSync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// XCD-aware work order: workgroups are dealt round-robin to the 8 XCDs (each with its own L2); remap so that each
// XCD walks one contiguous range of groups, whose neighbouring work items share tree nodes in its L2.
// numBlocksPadded is a multiple of kXcds.
constexpr uint32_t kXcds = 8;

__device__ inline uint32_t xcdContiguousBlock(uint32_t b, uint32_t numBlocksPadded)
{
    uint32_t perXcd = numBlocksPadded / kXcds;
    return (b % kXcds) * perXcd + b / kXcds;
}

template<class T>
struct BoxOf;
template<>
struct BoxOf<float>
{
    using type = hipcstone_box_f32;
};
template<>
struct BoxOf<double>
{
    using type = hipcstone_box_f64;
};

namespace nbwalk
{

constexpr int kLeafList = kWave;
// the walk's stack: 64 entries in registers, of which 32 at a time move to memory when they run out. A descent leaves
// at most 7 siblings per level behind and adds 8: 21 levels below the root need at most 155 entries.
constexpr int kSpillEntries = 32;
constexpr int kSpills       = 3;
// Chunks of 64 candidates whose hits are kept before they are taken out, and kept hit entries per target: as many as six
// waves per SIMD leave LDS for. With more kept hits the lanes' counts differ less and fewer turns are spent on the fullest
// lane, with more waves the latencies hide better: 16 chunks at 2 waves per SIMD took 13.0 ms, 10 at 3 9.9, 8 at 4 8.4.
constexpr int kChunks  = 5;
constexpr int kEntries = 13;

// Exponents of a wave's largest relative coordinate or radius for which the products decide: while the reference's own
// squares stay well inside fp32's range, and while an fp64 length as a float does. Squares of lengths below all of
// these are below kFarSq.
template<class T>
constexpr int kMinExponent = std::is_same_v<T, float> ? -48 : -100;
template<class T>
constexpr int kMaxExponent = std::is_same_v<T, float> ? 59 : 100;
constexpr float kFarSq     = 1.0e38f;

typedef float Float4 __attribute__((ext_vector_type(4)));

// wave-wide inclusive scans (row shifts, then the rows' last lanes broadcast into the rows above)
template<int Ctrl, int RowMask>
__device__ inline uint32_t dppOrZero(uint32_t v)
{
    return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), Ctrl, RowMask, 0xF, false));
}
template<class Op>
__device__ inline uint32_t waveScan(uint32_t v, Op op)
{
    v = op(v, dppOrZero<0x111, 0xF>(v)); // row_shr:1
    v = op(v, dppOrZero<0x112, 0xF>(v));
    v = op(v, dppOrZero<0x114, 0xF>(v));
    v = op(v, dppOrZero<0x118, 0xF>(v));
    v = op(v, dppOrZero<0x142, 0xA>(v)); // row_bcast:15 into rows 1 and 3
    return op(v, dppOrZero<0x143, 0xC>(v)); // row_bcast:31 into rows 2 and 3
}
__device__ inline uint32_t waveScanAdd(uint32_t v) { return waveScan(v, [](uint32_t a, uint32_t b) { return a + b; }); }
__device__ inline uint32_t waveScanMax(uint32_t v)
{
    return waveScan(v, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}

__device__ inline uint32_t readLane(uint32_t v, int l) { return uint32_t(__builtin_amdgcn_readlane(int(v), l)); }
__device__ inline float readLane(float v, int l)
{
    return __uint_as_float(uint32_t(__builtin_amdgcn_readlane(int(__float_as_uint(v)), l)));
}
__device__ inline double readLane(double v, int l)
{
    const uint64_t b = uint64_t(__double_as_longlong(v));
    return __longlong_as_double((long long)((uint64_t(readLane(uint32_t(b >> 32), l)) << 32) | readLane(uint32_t(b), l)));
}

// (a's rows 0, 1 and b's rows 0, 1), (a's rows 2, 3 and b's rows 2, 3), a row being 16 lanes
__device__ inline void swapHalves(uint32_t& a, uint32_t& b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a            = r[0];
    b            = r[1];
}
// a's odd rows exchanged with b's even rows
__device__ inline void swapRows(uint32_t& a, uint32_t& b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a            = r[0];
    b            = r[1];
}
// 4 x 4 transpose of registers and rows: row k of register q becomes row q of register k
__device__ inline void transposeRows(float (&f)[4])
{
    uint32_t v[4];
    for (int k = 0; k < 4; ++k)
        v[k] = __float_as_uint(f[k]);
    swapHalves(v[0], v[2]);
    swapHalves(v[1], v[3]);
    swapRows(v[0], v[1]);
    swapRows(v[2], v[3]);
    for (int k = 0; k < 4; ++k)
        f[k] = __uint_as_float(v[k]);
}

// index of the lowest set bit, 2^32 - 1 for zero (one instruction; the language's forms leave zero undefined or
// select a value for it)
__device__ inline uint32_t lowestBit(uint32_t v)
{
    uint32_t r;
    asm("v_ffbl_b32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// lo |= low half, hi |= high half of v in the lanes of the mask. Call where all lanes are active.
__device__ inline void orLanes(uint64_t mask, uint64_t v, uint32_t& lo, uint32_t& hi)
{
    asm volatile("s_mov_b64 exec, %2\n\tv_or_b32_e32 %0, %3, %0\n\tv_or_b32_e32 %1, %4, %1\n\ts_mov_b64 exec, -1"
        : "+v"(lo), "+v"(hi)
        : "s"(mask), "s"(uint32_t(v)), "s"(uint32_t(v >> 32)));
}

// v with lane l's value replaced by the wave-uniform x (l < 64), which has no clang builtin
__device__ int writeLaneI32(int x, int l, int v) __asm("llvm.amdgcn.writelane.i32");
__device__ inline uint32_t writeLane(uint32_t v, int l, uint32_t x) { return uint32_t(writeLaneI32(int(x), l, int(v))); }

// m[k] = lanes of `in` with v[k] < r: the compares run under `in`, which masks them for nothing. Call where all lanes
// are active.
__device__ inline void lessIn(uint64_t in, const float (&v)[8], float r, uint64_t (&m)[8])
{
    asm volatile("s_mov_b64 exec, %8\n\t"
        "v_cmp_lt_f32_e64 %0, %9, %17\n\tv_cmp_lt_f32_e64 %1, %10, %17\n\t"
        "v_cmp_lt_f32_e64 %2, %11, %17\n\tv_cmp_lt_f32_e64 %3, %12, %17\n\t"
        "v_cmp_lt_f32_e64 %4, %13, %17\n\tv_cmp_lt_f32_e64 %5, %14, %17\n\t"
        "v_cmp_lt_f32_e64 %6, %15, %17\n\tv_cmp_lt_f32_e64 %7, %16, %17\n\t"
        "s_mov_b64 exec, -1"
        : "=&s"(m[0]), "=&s"(m[1]), "=&s"(m[2]), "=&s"(m[3]), "=&s"(m[4]), "=&s"(m[5]), "=&s"(m[6]), "=&s"(m[7])
        : "s"(in), "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]), "v"(r));
}
__device__ inline void lessIn(uint64_t in, const double (&v)[8], double r, uint64_t (&m)[8])
{
    asm volatile("s_mov_b64 exec, %8\n\t"
        "v_cmp_lt_f64_e64 %0, %9, %17\n\tv_cmp_lt_f64_e64 %1, %10, %17\n\t"
        "v_cmp_lt_f64_e64 %2, %11, %17\n\tv_cmp_lt_f64_e64 %3, %12, %17\n\t"
        "v_cmp_lt_f64_e64 %4, %13, %17\n\tv_cmp_lt_f64_e64 %5, %14, %17\n\t"
        "v_cmp_lt_f64_e64 %6, %15, %17\n\tv_cmp_lt_f64_e64 %7, %16, %17\n\t"
        "s_mov_b64 exec, -1"
        : "=&s"(m[0]), "=&s"(m[1]), "=&s"(m[2]), "=&s"(m[3]), "=&s"(m[4]), "=&s"(m[5]), "=&s"(m[6]), "=&s"(m[7])
        : "s"(in), "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]), "v"(r));
}

// the structured buffer load of the LLVM AMDGPU back end (address = base + vindex * stride), which has no clang builtin:
// fp32 coordinates as buffers of 4-byte records take the particle index itself, with no 64-bit address arithmetic
__device__ float structBufferLoadF32(__amdgpu_buffer_rsrc_t rsrc, int vindex, int voffset, int soffset,
                                     int aux) __asm("llvm.amdgcn.struct.ptr.buffer.load.f32");

// dword 3 of an untyped, unswizzled buffer resource on gfx9-family targets (32-bit data format); with a stride in
// dword 1, accesses are range checked against the record count in dword 2 (none here)
constexpr int kBufferFlags = 0x00020000;

// the LDS of one walking wave
struct WaveShared
{
    uint32_t spilled[kSpills][3][kSpillEntries]; // stack entries that did not fit the registers
    uint32_t marks[kWave];                       // scratch of one chunk
    uint32_t cand[(kChunks + 1) * kWave];        // the kept chunks' candidates (particle indices), and the next one's
    float unit;                                  // fp64: the wave's unit of length in the products
    uint32_t entries[kEntries + 1][kWave];       // column l: target l's kept hits (see HitReader), then one without any
};

// LDS by its address
typedef __attribute__((address_space(3))) uint32_t LdsWord;
__device__ inline uint32_t ldsAddress(const void* p) { return uint32_t((__UINTPTR_TYPE__)(const LdsWord*)p); }
__device__ inline void ldsWrite(uint32_t address, uint32_t v) { *(LdsWord*)(__UINTPTR_TYPE__)address = v; }
struct Lds
{
    __device__ static inline uint32_t read(uint32_t address) { return *(const LdsWord*)(__UINTPTR_TYPE__)address; }
    __device__ static inline uint32_t lowest(uint32_t v) { return lowestBit(v); }
};

template<class T, int kNbWaves>
struct Shared
{
    WaveShared wave[kNbWaves];
};

// The 8 children of one internal node in a compact form. In each dimension geometric centers depend only on the node's
// integer box, so the children's centers take two values and their sizes one, and along the Hilbert curve (which all
// node boxes are decoded from) the children's octants follow one pattern up to the order of the axes: one axis changes
// with every second child (kFast), one with every fourth (kMiddle), one half way (kSlow). With the first child's
// center as each axis' first value, child k therefore lies at the second one where bit k of the axis' pattern is set.
// Along the Morton curve (a caller's own geometry) x is the slow axis, the others have patterns of their own.
// Record g describes the children [8 g + 1, 8 g + 9), the child block of some internal node.
//   v0, v1, s: the center of child 0, the other center and the size, for x, for the faster of y and z, and for the other
//   flags:     bit k set if child k is internal; kXFast, kXMiddle: x's pattern (neither: it is the slow axis); kZFaster:
//              z is faster than y; kMorton: the Morton curve's patterns; kGroupValid if every child matched bit for bit
//              (else the walk takes the children's own centers and sizes); kGroupOutside if an internal child's block
//              lies outside the tree or a leaf child has no leaf index, kGroupBackward if a block does not come after
//              its parent
//   link:      a leaf child's leaf index (internalToLeaf), an internal child's own child block (childOffsets)
template<class T>
struct alignas(128) ChildGroup
{
    T v0[3], v1[3], s[3];
    uint32_t flags;
    alignas(32) int32_t link[8];
};
typedef uint32_t Words16 __attribute__((ext_vector_type(16)));
typedef uint32_t Words8 __attribute__((ext_vector_type(8)));
typedef int32_t Links8 __attribute__((ext_vector_type(8)));
constexpr uint32_t kGroupValid = 0x80000000u, kGroupOutside = 0x40000000u, kGroupBackward = 0x20000000u;
constexpr uint32_t kXFast = 0x100u, kXMiddle = 0x200u, kZFaster = 0x400u, kMorton = 0x800u;
constexpr uint32_t kFast = 0x66u, kMiddle = 0x3Cu, kSlow = 0xF0u, kMortonFast = 0xAAu, kMortonMiddle = 0xCCu;

// the ChildGroup records of a tree with numNodes nodes: (numNodes - 1) / 8 of them (none for a root-only tree)
inline size_t childGroupCount(int32_t numNodes) { return numNodes > 8 ? size_t((numNodes - 1) / 8) : 0; }

// builds the ChildGroup records, one thread per block of 8 children [8 g + 1, 8 g + 9); a template so that every
// translation unit that launches it has its own copy
template<class T>
__global__ void childGroupsKernel(const T* __restrict__ centers, const T* __restrict__ sizes,
                                  const int32_t* __restrict__ childOffsets, const int32_t* __restrict__ internalToLeaf,
                                  int32_t numNodes, uint32_t numGroups, ChildGroup<T>* __restrict__ groups)
{
    using Bits = std::conditional_t<std::is_same_v<T, float>, uint32_t, uint64_t>;
    auto bits  = [](T v) { return __builtin_bit_cast(Bits, v); };
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= numGroups) return;
    const size_t co = size_t(g) * 8 + 1;
    bool same = true;
    T v0[3], v1[3], size[3];
    uint32_t pattern[3];
    for (int d = 0; d < 3; ++d)
    {
        const T a  = centers[co * 3 + d];
        const T s  = sizes[co * 3 + d];
        T b        = a;
        pattern[d] = 0;
        for (int k = 1; k < 8; ++k)
        {
            const T c = centers[(co + k) * 3 + d];
            if (bits(c) != bits(a))
            {
                if (pattern[d] == 0) b = c;
                same = same && bits(c) == bits(b);
                pattern[d] |= 1u << k;
            }
            same = same && bits(sizes[(co + k) * 3 + d]) == bits(s);
        }
        v0[d]   = a;
        v1[d]   = b;
        size[d] = s;
    }
    // the axes' order; an axis whose two centers round to one value goes with any pattern
    constexpr uint32_t kOrders[8][4] = {{kFast, kMiddle, kSlow, kXFast},   {kFast, kSlow, kMiddle, kXFast | kZFaster},
                                        {kMiddle, kFast, kSlow, kXMiddle}, {kMiddle, kSlow, kFast, kXMiddle | kZFaster},
                                        {kSlow, kFast, kMiddle, 0u},       {kSlow, kMiddle, kFast, kZFaster},
                                        {kSlow, kMortonFast, kMortonMiddle, kMorton},
                                        {kSlow, kMortonMiddle, kMortonFast, kMorton | kZFaster}};
    bool found     = false;
    uint32_t flags = 0;
    for (int o = 0; o < 8; ++o)
    {
        bool ok = true;
        for (int d = 0; d < 3; ++d)
            ok = ok && (pattern[d] == kOrders[o][d] || pattern[d] == 0);
        if (ok && !found)
        {
            found = true;
            flags = kOrders[o][3];
        }
    }
    ChildGroup<T> r{};
    const bool swapped = (flags & kZFaster) != 0;
    for (int d = 0; d < 3; ++d)
    {
        const int to = d == 0 || !swapped ? d : 3 - d;
        r.v0[to]     = v0[d];
        r.v1[to]     = v1[d];
        r.s[to]      = size[d];
    }
    for (int k = 0; k < 8; ++k)
    {
        const int32_t child = childOffsets[co + k];
        r.link[k]           = child != 0 ? child : internalToLeaf[co + k];
        if (r.link[k] < 0) flags |= kGroupOutside;
        if (child == 0) continue;
        flags |= 1u << k;
        if (child > numNodes - 8) flags |= kGroupOutside;
        if (child <= int32_t(co) + k) flags |= kGroupBackward;
    }
    if (same && found) flags |= kGroupValid;
    r.flags   = flags;
    groups[g] = r;
}

// a linked octree with its geometry and leaf layout (device pointers; centers and sizes as x,y,z triples). A kernel
// that walks should take these arrays (and x, y, z, h) as separate __restrict__ arguments and assemble the Tree
// itself: only then does the compiler know they are read-only and unaliased and fetch the wave-uniform node values
// with scalar loads (a Tree passed in as a kernel argument costs some 25 vector registers more)
template<class T>
struct Tree
{
    const int32_t* childOffsets;
    const int32_t* internalToLeaf;
    const uint32_t* layout;
    const T* centers;
    const T* sizes;
    int32_t numNodes;
    float ext;
    // optional: the child blocks in compact form, numbered by (first child - 1) / 8
    const ChildGroup<T>* groups = nullptr;
};

/*
 * A target's kept hits, in ascending order. They lie in its lane's column of WaveShared::entries, one entry per group of
 * 16 consecutive candidates that has any: bits 0-15 the hits, bits 16-31 the address of the group's first candidate
 * (in words of LDS). After them comes one without hits (noHits), which stays the current one when next() is called past
 * the last hit (by lanes that have fewer than others): its lowest bit is one of 16 to 31, so those calls read, and
 * return, one of the candidates.
 */
template<class Memory>
struct HitReader
{
    uint32_t at, end;    // addresses of the entry read ahead and of the last one, without hits
    uint32_t cur, ahead; // the entry being emptied, the one after it

    static constexpr uint32_t kEntryStep = kWave * sizeof(uint32_t);

    // candidates: the address (in words, not 0) of at least 32 of them
    __host__ __device__ static inline uint32_t noHits(uint32_t candidates) { return candidates << 16; }

    __host__ __device__ inline HitReader(uint32_t from, uint32_t last)
        : at(from + kEntryStep < last ? from + kEntryStep : last)
        , end(last)
        , cur(Memory::read(from))
        , ahead(Memory::read(at))
    {
    }

    __host__ __device__ inline uint32_t next()
    {
        const uint32_t j = Memory::read(((cur >> 16) + Memory::lowest(cur)) * 4u);
        cur &= cur - 1;
        if (uint16_t(cur) == 0)
        {
            cur   = ahead;
            at    = at + kEntryStep < end ? at + kEntryStep : end;
            ahead = Memory::read(at);
        }
        return j;
    }
};
using LdsHits = HitReader<Lds>;

/*
 * Walks the tree from `root` for the wave's targets first + lane (lanes with `valid` false take no part); returns this
 * lane's neighbor count (all neighbors). Whenever hits have been collected, consume(before, hits, next) is called from all
 * lanes: `before` and `hits` are the numbers of this target's neighbors handed on before and now, and next() returns the
 * latter one by one, in ascending order. consume is not called if `handOn` is false (only the counts are wanted).
 *
 * Segmented: the tree is one of many in the same arrays, children may lie before their parents (only the bounds
 * and depth guards and the step budget apply).
 * w is the wave's index in its workgroup (its part of `shared`). Call from all 64 lanes, with wave-uniform arguments
 * except `valid`.
 */
template<class T, bool AnyPbc, bool Segmented, int kNbWaves, class Consume>
__device__ __attribute__((always_inline)) inline uint32_t
walk(const T* __restrict__ x, const T* __restrict__ y, const T* __restrict__ z, const T* __restrict__ h,
     const typename BoxOf<T>::type& box, const Tree<T>& tree, int32_t root, uint64_t first, bool valid, bool handOn,
     Shared<T, kNbWaves>& shared, int w, uint32_t* faults, Consume&& consume)
{
    const int32_t* __restrict__ childOffsets   = tree.childOffsets;
    const int32_t* __restrict__ internalToLeaf = tree.internalToLeaf;
    const uint32_t* __restrict__ layout        = tree.layout;
    const T* __restrict__ centers              = tree.centers;
    const T* __restrict__ sizes                = tree.sizes;
    const int32_t numNodes                     = tree.numNodes;
    const ChildGroup<T>* __restrict__ groups   = tree.groups;
    WaveShared& sh = shared.wave[w];

    const int lane   = laneId();
    const uint32_t i = uint32_t(first) + uint32_t(lane);

    T xi = 0, yi = 0, zi = 0, hi = 0;
    if (valid)
    {
        xi = x[i];
        yi = y[i];
        zi = z[i];
        hi = h[i];
    }
    const T radiusSq0 = T(4.0) * hi * hi;
    const T cellR2    = radiusSq0 * T(tree.ext) * T(tree.ext);

    // periodic images only for particles whose 2h box leaves the domain (findneighbors.hpp:102-104)
    bool px = false, py = false, pz = false;
    if constexpr (AnyPbc)
    {
        T s2        = T(2) * hi;
        bool inside = (xi - s2) >= box.lim[0] && (yi - s2) >= box.lim[2] && (zi - s2) >= box.lim[4] &&
                      (xi + s2) <= box.lim[1] && (yi + s2) <= box.lim[3] && (zi + s2) <= box.lim[5];
        px          = !inside && box.bnd[0] == HIPCSTONE_PERIODIC;
        py          = !inside && box.bnd[1] == HIPCSTONE_PERIODIC;
        pz          = !inside && box.bnd[2] == HIPCSTONE_PERIODIC;
    }
    auto fold = [&](T d, bool p, int dim) -> T {
        if constexpr (AnyPbc) { return p ? d - box.len[dim] * rint(d * box.ilen[dim]) : d; }
        else { return d; }
    };

    // minDistance + right-fold norm2 against a node given by its center and half size
    auto nodeDist2 = [&](T c0, T c1, T c2, T s0, T s1, T s2) -> T {
        // the reference's d += |d|; d *= 0.5 is exactly max(d, +0) for finite d (2d and the halving are exact,
        // and d + |d| is +0 for d <= 0)
        T d0 = fmax(fabs(fold(c0 - xi, px, 0)) - s0, T(0));
        T d1 = fmax(fabs(fold(c1 - yi, py, 1)) - s1, T(0));
        T d2 = fmax(fabs(fold(c2 - zi, pz, 2)) - s2, T(0));
        return d0 * d0 + (d1 * d1 + d2 * d2);
    };

    // the pair test in the reference's operations (with radiusSq0, which the rare callers compute anew)
    auto close = [&](T xj, T yj, T zj, T radiusSq) -> bool {
        T xx = fold(xj - xi, px, 0);
        T yy = fold(yj - yi, py, 1);
        T zz = fold(zj - zi, pz, 2);
        return xx * xx + yy * yy + zz * zz < radiusSq;
    };

    const T* rc             = centers + size_t(root) * 3;
    const T* rsz            = sizes + size_t(root) * 3;
    const uint64_t rootMask = ballot(valid & (nodeDist2(rc[0], rc[1], rc[2], rsz[0], rsz[1], rsz[2]) < cellR2));
    if (rootMask == 0) return 0;
    const bool inRoot = laneIn(rootMask);

    // ---- operands of the matrix-core pair test (see the top of this file). The center is the mean of four targets
    //      spread over the wave's; lanes without a target stand at the first one's place and get a constant that
    //      keeps D far above zero.
    const int laneF = __builtin_ctzll(rootMask);
    const int laneL = 63 - __builtin_clzll(rootMask);
    auto middle     = [&](T p) -> T {
        const T q = inRoot ? p : readLane(p, laneF);
        T s       = 0;
#pragma unroll
        for (int k = 1; k < 8; k += 2)
            s += readLane(q, laneF + (laneL - laneF) * k / 8);
        return readLane(s * T(0.25), 0); // (held in scalar registers)
    };
    const T cx = middle(xi), cy = middle(yi), cz = middle(zi);
    float tgt[4];
    Float4 tgtConst[4]; // per 16 targets: the constant of target lane % 16, in every register of the accumulator
    float errBound;
    bool allExact;
    [[maybe_unused]] bool images = false; // some target's neighbors are looked for across a periodic face
    [[maybe_unused]] const uint32_t unitAt = ldsAddress(&sh.unit);
    // fp64: what lengths are multiplied by for the products, a power of two that brings the largest to [1, 2)
    [[maybe_unused]] float unit = 1.0f;
    auto inUnits                = [&](float length) {
        if constexpr (std::is_same_v<T, float>) { return length; }
        else { return length * unit; }
    };
    {
        float xr        = inRoot ? float(xi - cx) : 0.0f;
        float yr        = inRoot ? float(yi - cy) : 0.0f;
        float zr        = inRoot ? float(zi - cz) : 0.0f;
        const float big = fmaxf(fmaxf(fabsf(xr), fabsf(yr)), fmaxf(fabsf(zr), inRoot ? fabsf(float(T(2) * hi)) : 0.0f));
        // (non-negative floats order as their bit patterns)
        const int exponent = int(readLane(waveScanMax(__float_as_uint(big)), kWave - 1) >> 23) - 127;
        allExact           = exponent < kMinExponent<T> || exponent > kMaxExponent<T>;
        if constexpr (!std::is_same_v<T, float>)
        {
            // (read back for each chunk: a register that holds it all along costs fp64 2 to 4 %)
            unit    = __uint_as_float(uint32_t(127 - exponent) << 23);
            ldsWrite(unitAt, __float_as_uint(unit));
        }
        xr                 = inUnits(xr);
        yr                 = inUnits(yr);
        zr                 = inUnits(zr);
        const float a2  = xr * xr + yr * yr + zr * zr;
        float r2        = 0.0f;
        if constexpr (std::is_same_v<T, float>) { r2 = inRoot ? radiusSq0 : 0.0f; }
        else { r2 = inRoot ? float(radiusSq0 * T(unit) * T(unit)) : 0.0f; }
        const float s   = 2.0f * __builtin_amdgcn_sqrtf(a2) + __builtin_amdgcn_sqrtf(r2);
        const float s2r = inRoot ? s * s + r2 : 0.0f;
        const float most = __uint_as_float(readLane(waveScanMax(__float_as_uint(s2r)), kWave - 1));
        errBound         = readLane(1.0e-6f * most, 0); // 16 u (S^2 + r^2), rounded up
        allExact         = allExact || !(most < kFarSq); // (a coordinate that is not a number)
        if constexpr (AnyPbc)
        {
            images = ballot(px | py | pz) != 0;
            if (images)
            {
                const float mostR2 = __uint_as_float(readLane(waveScanMax(__float_as_uint(r2)), kWave - 1));
                float longest      = 0.0f;
                for (int d = 0; d < 3; ++d)
                {
                    if (box.bnd[d] != HIPCSTONE_PERIODIC) continue;
                    const float len = inUnits(float(box.len[d]));
                    longest         = fmaxf(longest, len);
                    allExact        = allExact || !(sqrtf(most) < 0.4999f * len);
                }
                // (u of the coordinates' own type: fp64 ones are folded in fp64)
                constexpr float kFold = std::is_same_v<T, float> ? 5.0e-7f : 1.0e-15f;
                errBound = readLane(errBound + kFold * sqrtf(mostR2) * longest, 0);
                allExact = allExact || !(errBound <= 1.0e-6f * kFarSq);
            }
        }
        float c0[4];
        c0[0] = c0[1] = c0[2] = c0[3] = inRoot ? a2 - r2 : kFarSq;
        transposeRows(c0);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            tgtConst[t] = Float4{c0[t], c0[t], c0[t], c0[t]};
        tgt[0] = -2.0f * xr;
        tgt[1] = -2.0f * yr;
        tgt[2] = -2.0f * zr;
        tgt[3] = 1.0f;
        transposeRows(tgt);
    }
    // the candidate (of a chunk of 64) whose position this lane loads: with rows 4 g + r of the q-th product being
    // candidates 16 g + 4 q + r, the 16 results a lane gets for one target are 16 consecutive candidates; in their order
    // where the products are not used
    const int loadPos = allExact ? lane : 16 * ((lane & 15) >> 2) + 4 * (lane >> 4) + (lane & 3);
    // byte selector that joins the even rows' low or the odd rows' high halves of two words
    const uint32_t halfSel = (lane & 16) ? 0x07060302u : 0x05040100u;

    uint32_t total   = 0; // neighbors of this lane's target so far
    uint32_t handed  = 0; // those of them handed on
    int numChunks    = 0; // kept chunks
    uint32_t slot    = 0; // the next chunk's place in sh.cand, a ring
    // the place of this lane's next entry
    const uint32_t entriesAt = ldsAddress(&sh.entries[0][0]);
    uint32_t entryEnd        = entriesAt + uint32_t(lane) * 4u;
    const uint32_t candAt = ldsAddress(sh.cand) / 4u;
    static_assert(offsetof(WaveShared, cand) > 0); // (so candAt is not 0, see HitReader)

    auto handOver = [&]() __attribute__((always_inline)) {
        ldsWrite(entryEnd, LdsHits::noHits(candAt));
        waveSync();
        if (handOn)
        {
            LdsHits hits(entriesAt + uint32_t(lane) * 4u, entryEnd);
            consume(handed, total - handed, [&]() __attribute__((always_inline)) { return hits.next(); });
        }
        waveSync();
        handed    = total;
        numChunks = 0;
        entryEnd  = entriesAt + uint32_t(lane) * 4u;
    };

    [[maybe_unused]] __amdgpu_buffer_rsrc_t xRes, yRes, zRes;
    if constexpr (std::is_same_v<T, float>)
    {
        xRes = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(x), 4, -1, kBufferFlags);
        yRes = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(y), 4, -1, kBufferFlags);
        zRes = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(z), 4, -1, kBufferFlags);
    }

    // ---- leaves to be tested, in visiting order: entry e in lane e (the leaf and the lanes that visit it)
    uint32_t listLeaf = 0, listLo = 0, listHi = 0;
    int listCount   = 0;
    auto appendLeaf = [&](int32_t leafIdx, uint64_t m) __attribute__((always_inline)) {
        listLeaf = writeLane(listLeaf, listCount, uint32_t(leafIdx));
        listLo   = writeLane(listLo, listCount, uint32_t(m));
        listHi   = writeLane(listHi, listCount, uint32_t(m >> 32));
        ++listCount;
        // (keeps the compiler from merging this tail with the stack's, which would put both counts into memory)
        asm volatile("; listed");
    };

    // ---- the listed leaves' particles become candidates, 64 at a time, and are tested; `last`: nothing follows
    auto drain = [&](bool last) __attribute__((always_inline)) {
        uint32_t jb = 0, cnt = 0;
        if (lane < listCount)
        {
            jb  = layout[int32_t(listLeaf)];
            cnt = layout[int32_t(listLeaf) + 1] - jb;
        }
        // leaves without particles leave the list
        const uint64_t filled = ballot(cnt != 0);
        if (filled != (listCount == kWave ? ~uint64_t(0) : (uint64_t(1) << listCount) - 1))
        {
            const uint32_t numFilled = uint32_t(__builtin_popcountll(filled));
            const int to = int((cnt != 0 ? laneRank(filled) : numFilled + laneRank(~filled)) << 2);
            jb           = uint32_t(__builtin_amdgcn_ds_permute(to, int(jb)));
            cnt          = uint32_t(__builtin_amdgcn_ds_permute(to, int(cnt)));
            listLo       = uint32_t(__builtin_amdgcn_ds_permute(to, int(listLo)));
            listHi       = uint32_t(__builtin_amdgcn_ds_permute(to, int(listHi)));
        }
        const uint32_t upTo = waveScanAdd(cnt);
        const uint32_t off  = upTo - cnt; // the leaf's first position among the candidates
        const uint32_t num  = readLane(upTo, kWave - 1);

        // a chunk's candidates and, in the order of the matrix operand's rows, their positions; read one chunk ahead
        uint32_t nextEntry = 0, nextJ = 0;
        uint32_t started   = 0; // list entries that start before the chunk's end
        T nextX = 0, nextY = 0, nextZ = 0;
        auto fetch = [&](uint32_t at) __attribute__((always_inline)) {
            // list entry of each position: the entries that start in this chunk mark their first position; a position
            // belongs to the last entry that starts at or before it
            const uint32_t start = off - at;
            sh.marks[lane]       = 0;
            waveSync();
            if (cnt != 0 && start < uint32_t(kWave)) sh.marks[start] = 1;
            waveSync();
            const uint64_t starts = ballot(sh.marks[lane] != 0);
            nextEntry = __builtin_amdgcn_mbcnt_hi(
                uint32_t(starts >> 33), __builtin_amdgcn_mbcnt_lo(uint32_t(starts >> 1),
                                                                  started + (uint32_t(starts) & 1u) - 1u));
            started += uint32_t(__builtin_popcountll(starts));
            // positions past the last repeat the last candidate (their hits are masked out)
            const uint32_t p = min(at + uint32_t(lane), num - 1u);
            nextJ            = p + uint32_t(__builtin_amdgcn_ds_bpermute(int(nextEntry << 2), int(jb - off)));
            uint32_t* cand   = sh.cand + slot * kWave;
            cand[lane]       = nextJ;
            waveSync();
            const uint32_t jl = cand[loadPos];
            if constexpr (std::is_same_v<T, float>)
            {
                nextX = structBufferLoadF32(xRes, int(jl), 0, 0, 0);
                nextY = structBufferLoadF32(yRes, int(jl), 0, 0, 0);
                nextZ = structBufferLoadF32(zRes, int(jl), 0, 0, 0);
            }
            else
            {
                nextX = x[jl];
                nextY = y[jl];
                nextZ = z[jl];
            }
        };
        if (num != 0) fetch(0);
        for (uint32_t at = 0;; at += kWave)
        {
            const bool more = at < num;
            if (more)
            {
                const uint32_t entry    = nextEntry;
                const uint32_t j        = nextJ;
                const T xj = nextX, yj = nextY, zj = nextZ;
                const uint32_t lastLeaf = started - 1u;
                const uint32_t group    = candAt + slot * kWave; // of the chunk's first 16 candidates
                slot                    = slot == uint32_t(kChunks) ? 0u : slot + 1u;
                if (at + kWave < num) fetch(at + kWave);

                const uint32_t inChunk = num - at < uint32_t(kWave) ? num - at : uint32_t(kWave);
                const uint64_t present = ~uint64_t(0) >> (kWave - inChunk);
                // the candidates this lane's target visited, leaf by leaf
                uint32_t seenLo = 0, seenHi = 0;
                for (uint32_t e = readLane(entry, 0); e <= lastLeaf; ++e)
                {
                    const uint64_t range = ballot(entry == e) & present;
                    const uint64_t lanes = (uint64_t(readLane(listHi, e)) << 32) | readLane(listLo, e);
                    orLanes(lanes, range, seenLo, seenHi);
                }
                // a target is not its own neighbor
                const uint64_t own = ballot(j - uint32_t(first) < uint32_t(kWave)) & present;
                if (own != 0)
                {
                    sh.marks[lane] = kWave;
                    waveSync();
                    if (laneIn(own)) sh.marks[j - uint32_t(first)] = uint32_t(lane);
                    waveSync();
                    const uint32_t self = sh.marks[lane];
                    if (self < 32u) seenLo &= ~(1u << self);
                    else if (self < 64u) seenHi &= ~(1u << (self - 32u));
                }
                const uint64_t active = ballot((seenLo | seenHi) != 0);

                uint32_t lo = 0, hw = 0;
                // (where the compiler places this costs: as unlikely 0.5 % less at 16.8M in open boxes, 1.2 % more in the
                // segmented walk and 15 % more in periodic fp64 steps)
                if (__builtin_expect(allExact, AnyPbc || Segmented ? allExact : 0))
                {
                    // target by target against the chunk's 64 candidates (in their order, see loadPos), in the
                    // reference's operations
                    const T hAgain       = valid ? h[i] : T(0);
                    const T radiusSq     = T(4.0) * hAgain * hAgain;
                    const uint64_t folds = AnyPbc ? ballot(px | py | pz) : 0;
                    for (uint64_t rest = active; rest != 0; rest &= rest - 1)
                    {
                        const int t = __builtin_ctzll(rest);
                        T ax = xj - readLane(xi, t), ay = yj - readLane(yi, t), az = zj - readLane(zi, t);
                        if (AnyPbc && (folds >> t & 1))
                        {
                            ax = fold(ax, box.bnd[0] == HIPCSTONE_PERIODIC, 0);
                            ay = fold(ay, box.bnd[1] == HIPCSTONE_PERIODIC, 1);
                            az = fold(az, box.bnd[2] == HIPCSTONE_PERIODIC, 2);
                        }
                        const uint64_t hits = ballot(ax * ax + ay * ay + az * az < readLane(radiusSq, t));
                        lo                  = writeLane(lo, t, uint32_t(hits));
                        hw                  = writeLane(hw, t, uint32_t(hits >> 32));
                    }
                }
                else
                {
                    // D of 4 x 16 candidates and 4 x 16 targets: per 16 targets four products, whose signs are shifted
                    // into one word (bit s of its half: candidate 16 (lane / 16) + s)
                    float cnd[4];
                    T dx = xj - cx, dy = yj - cy, dz = zj - cz;
                    bool outside = false;
                    if constexpr (AnyPbc)
                    {
                        if (images)
                        {
                            const bool bx = box.bnd[0] == HIPCSTONE_PERIODIC, by = box.bnd[1] == HIPCSTONE_PERIODIC,
                                       bz = box.bnd[2] == HIPCSTONE_PERIODIC;
                            dx      = fold(dx, bx, 0);
                            dy      = fold(dy, by, 1);
                            dz      = fold(dz, bz, 2);
                            outside = (bx && !(xj >= box.lim[0] && xj <= box.lim[1])) ||
                                      (by && !(yj >= box.lim[2] && yj <= box.lim[3])) ||
                                      (bz && !(zj >= box.lim[4] && zj <= box.lim[5]));
                        }
                    }
                    if constexpr (!std::is_same_v<T, float>) { unit = __uint_as_float(Lds::read(unitAt)); }
                    cnd[0]          = inUnits(float(dx));
                    cnd[1]          = inUnits(float(dy));
                    cnd[2]          = inUnits(float(dz));
                    cnd[3]          = __builtin_fmaf(cnd[2], cnd[2], __builtin_fmaf(cnd[1], cnd[1], cnd[0] * cnd[0]));
                    const bool far  = !(cnd[3] < kFarSq); // or not a number
                    transposeRows(cnd);
                    float least = std::numeric_limits<float>::max();
                    auto tile   = [&](uint32_t bits, int t) __attribute__((always_inline)) -> uint32_t {
                        if ((uint32_t(active >> (16 * t)) & 0xFFFFu) == 0) return bits << 16;
                        Float4 d[4];
#pragma unroll
                        for (int q = 3; q >= 0; --q)
                            d[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(cnd[q], tgt[t], tgtConst[t], 0, 0, 0);
#pragma unroll
                        for (int q = 3; q >= 0; --q)
                        {
#pragma unroll
                            for (int r = 3; r >= 0; --r)
                                bits = __builtin_amdgcn_alignbit(bits, __float_as_uint(d[q][r]), 31);
                            least = fminf(fminf(least, fabsf(d[q][0])), fabsf(d[q][1]));
                            least = fminf(fminf(least, fabsf(d[q][2])), fabsf(d[q][3]));
                        }
                        return bits;
                    };
                    uint32_t b01 = 0, b23 = 0;
                    b01 = tile(b01, 1);
                    b01 = tile(b01, 0);
                    b23 = tile(b23, 3);
                    b23 = tile(b23, 2);
                    // row k of a lane's targets gets its 16 bits from all four rows: candidates [0, 32) and [32, 64)
                    swapHalves(b01, b23);
                    uint32_t o01 = b01, o23 = b23;
                    swapRows(b01, o01);
                    swapRows(b23, o23);
                    lo = __builtin_amdgcn_perm(o01, b01, halfSel);
                    hw = __builtin_amdgcn_perm(o23, b23, halfSel);

                    uint64_t unsure = ballot(least < errBound);
                    if (ballot(far || outside) != 0) unsure = ~uint64_t(0);
                    if (unsure != 0)
                    {
                        // the 16-candidate groups with a pair too close to call, in the reference's operations
                        const T hAgain   = valid ? h[i] : T(0);
                        const T radiusSq = T(4.0) * hAgain * hAgain;
#pragma unroll 1
                        for (int g = 0; g < 4; ++g)
                        {
                            if ((uint32_t(unsure >> (16 * g)) & 0xFFFFu) == 0) continue;
                            uint32_t bits = 0;
#pragma unroll 1
                            for (int s = 0; s < 16; ++s)
                            {
                                const int from = 16 * (s >> 2) + 4 * g + (s & 3);
                                bits |= uint32_t(close(readLane(xj, from), readLane(yj, from), readLane(zj, from), radiusSq))
                                        << s;
                            }
                            const uint32_t shift = 16u * (g & 1);
                            uint32_t& word       = g < 2 ? lo : hw;
                            word                 = (word & ~(0xFFFFu << shift)) | (bits << shift);
                        }
                    }
                }
                lo &= seenLo;
                hw &= seenHi;
                total += uint32_t(__builtin_popcount(lo)) + uint32_t(__builtin_popcount(hw));
                // an entry for each group of 16 with hits: every group's is written, only those with hits stay
                auto append = [&](uint32_t entry) {
                    ldsWrite(entryEnd, entry);
                    entryEnd += uint16_t(entry) != 0 ? LdsHits::kEntryStep : 0u;
                };
                append((group << 16) | (lo & 0xFFFFu));
                append(((group + 16u) << 16) | (lo >> 16));
                append(((group + 32u) << 16) | (hw & 0xFFFFu));
                append(((group + 48u) << 16) | (hw >> 16));
                ++numChunks;
            }
            // a full set of chunks, or a column without room for another chunk's entries, goes out; at the end the rest
            const bool full = numChunks == kChunks ||
                              ballot(entryEnd >= entriesAt + (kEntries - 3) * LdsHits::kEntryStep) != 0;
            if (more ? full : last && numChunks != 0) handOver();
            if (!more) break;
        }
        listCount = 0;
        waveSync();
    };

    // ---- the walk's stack, entry e in lane e: a leaf (its complement) or an internal node's child block, and the lanes
    //      that passed it
    uint32_t stackLink = 0, stackLo = 0, stackHi = 0;
    int stackCount = 0, spills = 0;
    uint32_t fault = 0; // a guard that fires ends the walk: the counts and what was handed on are then incomplete
    auto push = [&](int32_t link, uint64_t m) __attribute__((always_inline)) {
        stackLink = writeLane(stackLink, stackCount, uint32_t(link));
        stackLo   = writeLane(stackLo, stackCount, uint32_t(m));
        stackHi   = writeLane(stackHi, stackCount, uint32_t(m >> 32));
        ++stackCount;
    };
    auto inTree = [&](int32_t block) { return block > 0 && block <= numNodes - 8; };

    // the 8 children [co, co + 8) of a node that the lanes `pm` passed: leaves that come before every internal child go
    // to the list, the rest that some lane passes onto the stack, first child on top
    auto descend = [&](int32_t co, uint64_t pm) __attribute__((always_inline)) {
        uint64_t mk[8]; // the lanes that pass child k
        Links8 link;
        uint32_t flags = 0;
        if (groups != nullptr && ((co - 1) & 7) == 0)
        {
            // the whole record with a few wide scalar loads, issued together
            const ChildGroup<T>* __restrict__ g = groups + (uint32_t(co - 1) >> 3);
            const Words16 head                  = *reinterpret_cast<const Words16*>(g);
            link                                = *reinterpret_cast<const Links8*>(g->link);
            T geo[9];
            if constexpr (std::is_same_v<T, float>)
            {
                asm volatile("" ::"s"(link)); // (waits for both loads here, not for one after the other)
#pragma unroll
                for (int k = 0; k < 9; ++k)
                    geo[k] = __uint_as_float(head[k]);
                flags = head[9];
            }
            else
            {
                const Words8 more = *reinterpret_cast<const Words8*>(reinterpret_cast<const char*>(g) + sizeof(head));
                asm volatile("" ::"s"(link), "s"(more));
#pragma unroll
                for (int k = 0; k < 9; ++k)
                {
                    const uint32_t lo = k < 8 ? head[2 * k % 16] : more[0];
                    const uint32_t hw = k < 8 ? head[(2 * k + 1) % 16] : more[1];
                    geo[k]            = __longlong_as_double((long long)((uint64_t(hw) << 32) | lo));
                }
                flags = more[2];
            }
            // two distance terms per lane and axis, 8 sums of them: nodeDist2 of the 8 children bit for bit
            auto term = [&](T c, T half, T p, bool pbc, T len, T ilen) {
                T d = c - p;
                if constexpr (AnyPbc) { d = pbc ? d - len * rint(d * ilen) : d; }
                d = fmax(fabs(d) - half, T(0));
                return d * d;
            };
            const bool zy = flags & kZFaster;
            const T pa = zy ? zi : yi, pb = zy ? yi : zi;
            const bool wa = AnyPbc && (zy ? pz : py), wb = AnyPbc && (zy ? py : pz);
            const T la = zy ? box.len[2] : box.len[1], lb = zy ? box.len[1] : box.len[2];
            const T ia = zy ? box.ilen[2] : box.ilen[1], ib = zy ? box.ilen[1] : box.ilen[2];
            const T tx[2] = {term(geo[0], geo[6], xi, px, box.len[0], box.ilen[0]),
                             term(geo[3], geo[6], xi, px, box.len[0], box.ilen[0])};
            const T ta[2] = {term(geo[1], geo[7], pa, wa, la, ia), term(geo[4], geo[7], pa, wa, la, ia)};
            const T tb[2] = {term(geo[2], geo[8], pb, wb, lb, ib), term(geo[5], geo[8], pb, wb, lb, ib)};
            const T tab[2][2] = {{ta[0] + tb[0], ta[0] + tb[1]}, {ta[1] + tb[0], ta[1] + tb[1]}};
            auto compare = [&](uint32_t patX, uint32_t patA, uint32_t patB) __attribute__((always_inline)) {
                T d2[8];
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    d2[k] = tx[(patX >> k) & 1] + tab[(patA >> k) & 1][(patB >> k) & 1];
                lessIn(pm, d2, cellR2, mk);
            };
            if (flags & kXFast) compare(kFast, kMiddle, kSlow);
            else if (flags & kXMiddle) compare(kMiddle, kFast, kSlow);
            // (the hint keeps this out of the way of the reference's own geometry, 0.4 % of a search of 16.8M)
            else if (__builtin_expect((flags & kMorton) != 0, 0)) compare(kSlow, kMortonFast, kMortonMiddle);
            else compare(kSlow, kFast, kMiddle);
        }
        if (!(flags & kGroupValid))
        {
            // children in no such form: from their own centers and sizes
            flags = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k)
            {
                const T* c        = centers + (size_t(co) + k) * 3;
                const T* sz       = sizes + (size_t(co) + k) * 3;
                mk[k]             = ballot(nodeDist2(c[0], c[1], c[2], sz[0], sz[1], sz[2]) < cellR2) & pm;
                const int32_t block = childOffsets[co + k];
                if constexpr (!AnyPbc && !std::is_same_v<T, float>)
                {
                    // (without branches the loads go out together: captured fp64 searches, which have no compact blocks,
                    // 250 -> 237 us at 100k targets and 100 neighbors, 206 -> 179 at 200k and 12. Elsewhere it costs
                    // registers of the whole walk: periodic fp64 255 -> 331 us, 16.8M fp32 5.87 -> 6.08 ms.)
                    const int32_t leaf = internalToLeaf[co + k];
                    link[k]            = block != 0 ? block : leaf;
                    flags |= block != 0 ? 1u << k : 0u;
                    flags |= block != 0 && !inTree(block) ? kGroupOutside : 0u;
                    flags |= block != 0 && block <= co + k ? kGroupBackward : 0u;
                }
                else
                {
                    link[k] = block != 0 ? block : internalToLeaf[co + k];
                    if (block == 0) continue;
                    flags |= 1u << k;
                    if (!inTree(block)) flags |= kGroupOutside;
                    if (block <= co + k) flags |= kGroupBackward;
                }
            }
        }
        if (flags & (Segmented ? kGroupOutside : kGroupOutside | kGroupBackward))
        {
            fault = HIPCSTONE_FAULT_MALFORMED_TREE;
            return;
        }
        bool inner = false; // met an internal child
#pragma unroll
        for (int k = 0; k < 8; ++k)
        {
            if (inner || mk[k] == 0) continue;
            if (flags & (1u << k)) { inner = true; }
            else
            {
                appendLeaf(link[k], mk[k]);
                mk[k] = 0;
            }
        }
        if (!inner) return;
#pragma unroll
        for (int k = 7; k >= 0; --k)
        {
            if (mk[k] != 0) push(flags & (1u << k) ? link[k] : ~link[k], mk[k]);
        }
    };

    // root (traversal.hpp:35-45)
    const int32_t rootChild = uniform(childOffsets[root]);
    if (rootChild == 0) { appendLeaf(uniform(internalToLeaf[root]), rootMask); }
    else if (!inTree(rootChild)) { fault = HIPCSTONE_FAULT_MALFORMED_TREE; }
    else { push(rootChild, rootMask); }
    // a 32-bit budget (saturated) of nodes taken from the stack, so that the test is a scalar compare
    const uint64_t budget = 2 * uint64_t(uint32_t(numNodes)) + 8;
    uint32_t stepsLeft    = budget > 0xFFFFFFFFu ? 0xFFFFFFFFu : uint32_t(budget);
    while (true)
    {
        bool done = fault != 0;
        if (stackCount == 0)
        {
            if (spills == 0) { done = true; }
            else
            {
                // (lanes from kSpillEntries on keep what they have: the count says which entries are live)
                --spills;
                if (lane < kSpillEntries)
                {
                    stackLink = sh.spilled[spills][0][lane];
                    stackLo   = sh.spilled[spills][1][lane];
                    stackHi   = sh.spilled[spills][2][lane];
                }
                stackCount = kSpillEntries;
            }
        }
        if (done || listCount > kLeafList - 9)
        {
            drain(done);
            if (done) break;
        }
        --stackCount;
        const int32_t link = int32_t(readLane(stackLink, stackCount));
        const uint64_t m   = (uint64_t(readLane(stackHi, stackCount)) << 32) | readLane(stackLo, stackCount);
        if (link < 0)
        {
            appendLeaf(~link, m);
            continue;
        }
        if (stepsLeft == 0) fault = HIPCSTONE_FAULT_WALK_BUDGET;
        --stepsLeft;
        if (stackCount > kWave - 8)
        {
            if (spills == kSpills) { fault = HIPCSTONE_FAULT_MALFORMED_TREE; }
            else
            {
                if (lane < kSpillEntries)
                {
                    sh.spilled[spills][0][lane] = stackLink;
                    sh.spilled[spills][1][lane] = stackLo;
                    sh.spilled[spills][2][lane] = stackHi;
                }
                waveSync();
                ++spills;
                const int from = ((lane + kSpillEntries) & (kWave - 1)) << 2;
                stackLink      = uint32_t(__builtin_amdgcn_ds_bpermute(from, int(stackLink)));
                stackLo        = uint32_t(__builtin_amdgcn_ds_bpermute(from, int(stackLo)));
                stackHi        = uint32_t(__builtin_amdgcn_ds_bpermute(from, int(stackHi)));
                stackCount -= kSpillEntries;
            }
        }
        if (link == 0) fault = HIPCSTONE_FAULT_MALFORMED_TREE;
        if (fault == 0) descend(link, m);
    }
    if (fault != 0 && lane == 0) atomicOr(faults, fault);
    return total;
}

} // namespace nbwalk
} // namespace hipcstone
