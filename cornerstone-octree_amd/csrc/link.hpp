// The steps of the internal-tree link around its sort, per thread. They are plain index arithmetic, so the host can run
// them too.
//
// The sort's output is taken as it comes: a look-back that gives up (reported through the fault word, which is read only
// after these kernels) leaves entries unwritten or written twice. Every step keeps to its arrays for any order and
// level, and whatever they hold, the results lead no later kernel out of its arrays or round in a circle: indices lie in
// [0, numNodes), a child block lies in the tree after its parent, a parent before its children, and a node without
// children has the index of a leaf.
#pragma once

#include "common.hpp"

namespace hipcstone
{

// the arrays of one link; in a kernel, plain pointers
template<class K>
struct LinkArrays
{
    const uint32_t* order; // the sorted entries' nodes
    const uint32_t* level; // and levels
    const K* unsortedPrefixes;
    K* prefixes;
    int32_t* childOffsets;
    int32_t* parents;
    int32_t* levelRange;
    int32_t* internalToLeaf;
    int32_t* leafToInternal;
    int32_t numNodes, numInternal;
};

// What placeNode and linkNode overwrite where the order is one. By the threads [0, 256 n) with 256 n >= numLeaves.
template<class K, class Arrays>
__host__ __device__ inline void presetLink(int32_t t, const Arrays& a)
{
    constexpr int L = int(maxLevel<K>());
    if (t <= L + 1) a.levelRange[t] = a.numNodes;
    if (t < a.numNodes - a.numInternal) a.leafToInternal[a.numInternal + t] = 0;
    if (t < a.numInternal)
    {
        a.leafToInternal[t] = 0;
        a.parents[t]        = 0;
    }
}

// createUnsortedLayout (octree.hpp:77-100): leaf t is node t + numInternal of the unsorted layout and, when it and the
// next leaf share a prefix of whole octal digits, creates internal node (t + binaryKeyWeight) / 7. Besides the unsorted
// prefixes, every leaf emits its nodes' levels in creation order: entry 2 t the internal node's (255 when t creates
// none), entry 2 t + 1 its own. Within one level, creation order is key order (keys ascend with t, and a level holds no
// node twice), so a stable sort of these entries by level alone gives the level-major, key-ordered node order that
// sorting the prefixes gives (a level's prefixes are exactly the ones with their placeholder bit at 3 * level).
template<class K, class Keys, class Prefixes, class Words>
__host__ __device__ inline void createNodes(int32_t t, const Keys& leaves, int32_t numInternal, int32_t numLeaves,
                                            const Prefixes& unsortedPrefixes, const Words& level, const Words& node)
{
    K key                             = leaves[t];
    K next                            = leaves[t + 1];
    unsigned leafLevel                = treeLevel(K(next - key));
    unsortedPrefixes[t + numInternal] = encodePlaceholderBit(key, int(3 * leafLevel));
    level[2 * t + 1]                  = leafLevel;
    node[2 * t + 1]                   = uint32_t(t + numInternal);
    unsigned prefixLength             = unsigned(commonPrefix(key, next));
    if (prefixLength % 3 == 0 && t < numLeaves - 1)
    {
        int32_t octIndex           = (t + binaryKeyWeight(key, prefixLength / 3)) / 7;
        unsortedPrefixes[octIndex] = encodePlaceholderBit(key, int(prefixLength));
        level[2 * t]               = prefixLength / 3;
        node[2 * t]                = uint32_t(octIndex);
    }
    else
    {
        level[2 * t] = 255u;
        node[2 * t]  = ~0u;
    }
}

// Sorted entry i < numNodes: prefixes[i] = unsorted prefix of node order[i]; leafToInternal[order[i]] = i;
// internalToLeaf[i] = order[i] - numInternal for leaves (octree.hpp:176-185; linkNode does the inner nodes);
// childOffsets[i] = 0 for linkNode; levelRange (getLevelRangeCpu, octree.hpp:151-160): the first node index of every level
// from the places where the level changes; the levels after the last one keep numNodes
template<class K, class Arrays>
__host__ __device__ inline void placeNode(int32_t i, const Arrays& a)
{
    constexpr uint32_t L = maxLevel<K>();
    const uint32_t o     = a.order[i];
    const bool known     = o < uint32_t(a.numNodes);
    a.childOffsets[i]    = 0;
    a.prefixes[i]        = known ? a.unsortedPrefixes[o] : K(1); // (the root's)
    a.internalToLeaf[i]  = known && o >= uint32_t(a.numInternal) ? int32_t(o) - a.numInternal : 0;
    if (known) a.leafToInternal[o] = i;
    const uint32_t here = a.level[i] < L ? a.level[i] : L;
    uint32_t from       = 0; // the first level without a place so far
    if (i > 0) from = (a.level[i - 1] < L ? a.level[i - 1] : L) + 1;
    for (uint32_t l = from; l <= here; ++l)
        a.levelRange[l] = i;
}

// first index of [lo, hi) whose value is not below v, lo where the range is empty
template<class K, class Array>
__host__ __device__ inline int32_t lowerBoundIdx(const Array& a, int32_t lo, int32_t hi, K v)
{
    int32_t count = hi - lo;
    while (count > 0)
    {
        int32_t step = count / 2;
        int32_t it   = lo + step;
        if (a[it] < v)
        {
            lo = it + 1;
            count -= step + 1;
        }
        else
            count = step;
    }
    return lo;
}

// Internal node i of the unsorted layout finds its children: linkTreeCpu (octree.hpp:114-148). Only with children does it
// get its negative internalToLeaf, so a node without any always names a leaf. Blocks of children start
// at 8 k + 1 (level by level, all nodes but the root come in eights).
template<class K, class Arrays>
__host__ __device__ inline void linkNode(int32_t i, const Arrays& a)
{
    const int32_t idxA          = a.leafToInternal[i];
    const K prefix              = a.prefixes[idxA];
    const unsigned prefixLength = decodePrefixLength(prefix);
    const unsigned level        = prefixLength / 3;
    if (level >= maxLevel<K>()) return;
    const K nodeKey        = decodePlaceholderBit(prefix);
    const K childPrefix    = encodePlaceholderBit(nodeKey, int(prefixLength) + 3);
    const int32_t lo       = a.levelRange[level + 1];
    const int32_t hi       = a.levelRange[level + 2];
    const int32_t childIdx = lowerBoundIdx(a.prefixes, lo, hi, childPrefix);
    if (childIdx < hi && childIdx > idxA && childIdx % 8 == 1 && childIdx <= a.numNodes - 8 &&
        childPrefix == a.prefixes[childIdx])
    {
        a.childOffsets[idxA]          = childIdx;
        a.internalToLeaf[idxA]        = i - a.numInternal;
        a.parents[(childIdx - 1) / 8] = idxA;
    }
}

} // namespace hipcstone
