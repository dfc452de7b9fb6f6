"""Parts of the kernels that are plain arithmetic, compiled for the host and run there."""

import os
import subprocess

from conftest import ROOT

HIPCC = "/opt/rocm/bin/hipcc"


def _run(tmp_path, name, source):
    src, exe = tmp_path / f"{name}.hip", tmp_path / name
    src.write_text(source)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-std=c++20", "-O1", "-ffp-contract=off", "-Wno-everything",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "cornerstone-octree_amd", "csrc"),
                    "-o", str(exe), str(src)], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True)


HITS = r"""
#include <cstddef>
#include <cstdio>
#include <random>
#include <vector>
#include "hipcstone_nbwalk.hpp"
using namespace hipcstone::nbwalk;

// one wave's memory; every read has to be of a word of it that was written
static std::vector<int64_t> words;
static uint32_t base;
static int bad = 0;
struct Checked
{
    static uint32_t read(uint32_t address)
    {
        const uint64_t w = (uint64_t(address) - base) / 4;
        if (address < base || address % 4 != 0 || w >= words.size() || words[w] < 0)
        {
            if (!bad++) printf("read of address %u, wave's memory [%u, %zu)\n", address, base, base + 4 * words.size());
            return 0;
        }
        return uint32_t(words[w]);
    }
    static uint32_t lowest(uint32_t v) { return v ? uint32_t(__builtin_ctz(v)) : ~0u; }
};

int main()
{
    std::mt19937 rng(5);
    const uint32_t candOff = offsetof(WaveShared, cand) / 4, entryOff = offsetof(WaveShared, entries) / 4;
    // the waves of a workgroup, the first one's memory at address 0
    for (uint32_t wave = 0; wave < 8; ++wave)
        for (int numEntries = 0; numEntries <= kEntries; ++numEntries)
            for (uint32_t lane : {0u, 17u, 63u})
            {
                base = wave * uint32_t(sizeof(WaveShared));
                words.assign(sizeof(WaveShared) / 4, -1);
                const uint32_t candAt = base / 4 + candOff, from = base + 4 * (entryOff + lane);
                for (uint32_t c = 0; c < (kChunks + 1) * 64; ++c)
                    words[candOff + c] = 1000 + c;
                std::vector<uint32_t> want;
                uint32_t end = from;
                for (int e = 0; e < numEntries; ++e, end += HitReader<Checked>::kEntryStep)
                {
                    const uint32_t group = 16 * e, hits = e % 3 == 0 ? 0x8000u : 1 + rng() % 0xFFFF;
                    words[(end - base) / 4] = ((candAt + group) << 16) | hits;
                    for (uint32_t b = 0; b < 16; ++b)
                        if (hits >> b & 1) want.push_back(1000 + group + b);
                }
                words[(end - base) / 4] = HitReader<Checked>::noHits(candAt);
                HitReader<Checked> reader(from, end);
                for (uint32_t w : want)
                    if (const uint32_t j = reader.next(); j != w)
                    {
                        printf("entries %d: %u instead of %u\n", numEntries, j, w);
                        return 1;
                    }
                for (int past = 0; past < 40; ++past)
                    if (const uint32_t j = reader.next(); j < 1000 || j >= 1000 + (kChunks + 1) * 64)
                    {
                        printf("past the end: %u\n", j);
                        return 1;
                    }
            }
    return bad != 0;
}
"""


def test_hit_reader_stays_inside_its_wave(tmp_path):
    """A target's hits come out in order, and reading on past the last one (lanes with fewer hits than others do) reads
    only words of the wave's own memory that were written."""
    run = _run(tmp_path, "hits", HITS)
    assert run.returncode == 0, run.stdout + run.stderr


LINK = r"""
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <numeric>
#include <random>
#include <vector>
#include "link.hpp"
using namespace hipcstone;

template<class V>
struct Checked
{
    std::vector<V> v;
    const char* name;
    V& operator[](int64_t i) const
    {
        if (i < 0 || i >= int64_t(v.size()))
        {
            printf("%s[%lld] of %zu\n", name, (long long)i, v.size());
            exit(1);
        }
        return const_cast<V&>(v[size_t(i)]);
    }
};

template<class K>
struct Arrays
{
    Checked<uint32_t> order, level;
    Checked<K> unsortedPrefixes, prefixes;
    Checked<int32_t> childOffsets, parents, levelRange, internalToLeaf, leafToInternal;
    int32_t numNodes, numInternal;
};

static void need(bool ok, const char* what)
{
    if (ok) return;
    printf("%s\n", what);
    exit(1);
}

template<class K>
void check(int splits, int numWrong, uint32_t anything, uint32_t seed)
{
    std::mt19937 rng(seed);
    std::vector<K> leaves{K(0), nodeRange<K>(0)};
    for (int s = 0; s < splits; ++s)
    {
        const size_t i = s < 12 ? leaves.size() / 3 : rng() % (leaves.size() - 1);
        const K step   = (leaves[i + 1] - leaves[i]) / 8;
        if (step == 0) continue;
        K kids[7];
        for (int k = 0; k < 7; ++k)
            kids[k] = leaves[i] + K(k + 1) * step;
        leaves.insert(leaves.begin() + i + 1, kids, kids + 7);
    }
    const int32_t numLeaves = int32_t(leaves.size()) - 1, I = (numLeaves - 1) / 7, N = numLeaves + I;
    constexpr int L         = int(maxLevel<K>());
    const int32_t junk      = int32_t(0x80000000u + rng() % 1000);
    Checked<K> keys{leaves, "leaves"};
    Checked<uint32_t> level{std::vector<uint32_t>(2 * numLeaves), "level"}, node{level.v, "node"};
    Arrays<K> a{{std::vector<uint32_t>(N), "order"}, {std::vector<uint32_t>(N), "sorted level"},
                {std::vector<K>(N), "unsortedPrefixes"}, {std::vector<K>(N, ~K(0)), "prefixes"},
                {std::vector<int32_t>(N, junk), "childOffsets"}, {std::vector<int32_t>(I, junk), "parents"},
                {std::vector<int32_t>(L + 2, junk), "levelRange"}, {std::vector<int32_t>(N, junk), "internalToLeaf"},
                {std::vector<int32_t>(N, junk), "leafToInternal"}, N, I};
    for (int t = 0; t < (numLeaves + 255) / 256 * 256; ++t)
    {
        presetLink<K>(t, a);
        if (t < numLeaves) createNodes<K>(t, keys, I, numLeaves, a.unsortedPrefixes, level, node);
    }
    std::vector<uint32_t> by(2 * numLeaves);
    std::iota(by.begin(), by.end(), 0u);
    std::stable_sort(by.begin(), by.end(), [&](uint32_t p, uint32_t q) { return level[p] < level[q]; });
    for (int32_t i = 0; i < N; ++i)
    {
        a.order[i] = node[by[i]];
        a.level[i] = level[by[i]];
    }
    // entries that the sort did not write
    for (int w = 0; w < numWrong; ++w)
    {
        const int32_t i = int32_t(rng() % N);
        a.order[i]      = rng() & anything;
        a.level[i]      = rng() & anything;
    }
    std::vector<int32_t> threads(N);
    std::iota(threads.begin(), threads.end(), 0);
    std::shuffle(threads.begin(), threads.end(), rng);
    for (int32_t i : threads)
        placeNode<K>(i, a);
    for (int32_t i : threads)
        if (i < I) linkNode<K>(i, a);

    for (int l = 0; l <= L + 1; ++l)
        need(a.levelRange[l] >= 0 && a.levelRange[l] <= N, "level range outside the tree");
    for (int32_t b = 0; b < I; ++b)
        need(a.parents[b] >= 0 && a.parents[b] < 8 * b + 1, "parent not before its children");
    int32_t children = 0;
    for (int32_t i = 0; i < N; ++i)
    {
        const int32_t c = a.childOffsets[i];
        need(c == 0 || (c > i && c <= N - 8 && c % 8 == 1), "child block");
        need(a.leafToInternal[i] >= 0 && a.leafToInternal[i] < N, "leafToInternal");
        need(a.internalToLeaf[i] >= (c ? -I : 0) && a.internalToLeaf[i] < numLeaves, "internalToLeaf");
        need(a.prefixes[i] != 0 && decodePrefixLength(a.prefixes[i]) <= 3u * L, "prefix");
        children += c != 0;
        if (numWrong) continue;
        // the tree itself
        const unsigned len = decodePrefixLength(a.prefixes[i]);
        const K key        = decodePlaceholderBit(a.prefixes[i]);
        need(a.levelRange[len / 3] <= i && i < a.levelRange[len / 3 + 1], "level");
        need((c != 0) == (a.internalToLeaf[i] < 0), "inner nodes have children");
        need(a.leafToInternal[a.internalToLeaf[i] + I] == i, "inverse");
        if (c == 0) need(leaves[a.internalToLeaf[i]] == key, "leaf's key");
        for (int k = 0; c != 0 && k < 8; ++k)
        {
            need(decodePrefixLength(a.prefixes[c + k]) == len + 3, "child's level");
            need(decodePlaceholderBit(a.prefixes[c + k]) == K(key + K(k) * nodeRange<K>(len / 3 + 1)), "child's key");
            need(a.parents[(c + k - 1) / 8] == i, "child's parent");
        }
    }
    if (!numWrong) need(children == I, "all inner nodes have children");
}

int main()
{
    uint32_t seed = 0;
    for (int splits : {0, 1, 2, 9, 40, 400})
        for (int wrong : {0, 1, 5, 100, 4000})
            for (uint32_t anything : {~0u, 0x800001FFu, 0xFFu, 0x1Fu})
            {
                check<uint32_t>(splits, wrong, anything, ++seed);
                check<uint64_t>(splits, wrong, anything, ++seed);
            }
    return 0;
}
"""


def test_link_of_any_order(tmp_path):
    """The internal-tree link around its sort: right for the sorted entries, and for an order and levels with anything
    in them (a sort that gave up and left entries unwritten) every access stays inside its array and every result
    inside the tree."""
    run = _run(tmp_path, "link", LINK)
    assert run.returncode == 0, run.stdout + run.stderr
