"""Parts of the neighbor walk that are plain arithmetic, compiled for the host and run there."""

import os
import subprocess

from conftest import ROOT

HIPCC = "/opt/rocm/bin/hipcc"


def _run(tmp_path, name, source):
    src, exe = tmp_path / f"{name}.hip", tmp_path / name
    src.write_text(source)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-std=c++20", "-O1", "-ffp-contract=off", "-Wno-everything",
                    "-I", os.path.join(ROOT, "include"), "-o", str(exe), str(src)], check=True)
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
