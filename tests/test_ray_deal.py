"""How a ray batch is dealt to the wavefronts of a traversal launch
(csrc/rt_deal.h, the rules that trace.hip launches with and rt_device.h runs),
walked on the CPU: every ray belongs to one place, a batch of up to 8192 rays
starts on lanes of its own at once, and no wavefront hands out rays that it
has not claimed."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <algorithm>
#include <cstdio>
#include <vector>
#include "rt_deal.h"
using namespace rt;

// Turns of the slowest wavefront when all of them claim from their own stripe
// one after the other.
static uint32_t turns(uint32_t n, const RayDeal &d)
{
    const uint32_t waves = d.blocks * kWavesPerBlock, width = deal_width(n, waves), per = waves / kStripes;
    uint32_t wlog = 0, worst = 0;
    while ((2u << wlog) <= per) ++wlog;
    for (uint32_t j = 0; j < kStripes; ++j) {
        const uint32_t items = deal_count(n, d.lc, j);
        std::vector<uint32_t> got;
        for (uint32_t b = j; b < d.blocks; b += kStripes)
            for (uint32_t w = 0; w < kWavesPerBlock; ++w)
                if (!deal_leaves(width, (b / kStripes) * kWavesPerBlock + w, items)) got.push_back(0);
        if (items && got.empty()) return 1000;  // nobody at home
        for (uint32_t left = items, at = 0; left; at = (at + 1) % got.size()) {
            const uint32_t c = std::min(left, deal_claim(left, wlog, width));
            got[at] += (c + width - 1) / width;
            worst = std::max(worst, got[at]);
            left -= c;
        }
    }
    return worst;
}

int main()
{
    const uint32_t most = 4096;
    std::vector<uint32_t> ns;
    for (uint32_t n = 1; n <= 9000; ++n) ns.push_back(n);
    for (uint32_t n = 9001; n < 3000000; n += n / 7) ns.push_back(n);
    for (uint32_t n : {1u << 14, (1u << 17) - 1, 1u << 17, 1u << 20, 0xffffffffu}) ns.push_back(n);
    for (uint32_t n : ns) {
        const RayDeal d = ray_deal(n, most);
        if (d.blocks < 1 || d.blocks > most || (n <= 131072 && d.blocks > 1024)) return printf("%u: %u blocks\n", n, d.blocks), 1;
        uint64_t sum = 0;
        for (uint32_t j = 0; j < kStripes; ++j) sum += deal_count(n, d.lc, j);
        if (sum != n) return printf("%u: the stripes hold %llu\n", n, (unsigned long long)sum), 1;
        if (n <= 300000) {
            std::vector<char> seen(n, 0);
            for (uint32_t j = 0; j < kStripes; ++j)
                for (uint32_t o = 0; o < deal_count(n, d.lc, j); ++o) {
                    const uint32_t r = deal_ray(d.lc, j, o);
                    if (r >= n || seen[r]++) return printf("%u: ray %u\n", n, r), 1;
                }
        }
        if (n <= 8192 && turns(n, d) != 1) return printf("%u: %u turns (lc %u, %u blocks)\n", n, turns(n, d), d.lc, d.blocks), 1;
        const uint32_t width = deal_width(n, d.blocks * kWavesPerBlock);
        if (deal_refill(width) < 1 || deal_claim(1, 0, width) < 1) return printf("%u: width %u\n", n, width), 1;
    }
    // a few workgroups only (all rays still have a wavefront)
    for (uint32_t n : {1u, 70u, 1000u, 100000u})
        if (ray_deal(n, 3).blocks > 3 || ray_deal(n, 3).blocks < 1) return printf("%u\n", n), 1;
    return 0;
}
"""


def test_small_batches_start_at_once(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "deal.cpp", tmp_path / "deal"
    src.write_text(SRC)
    inc = os.path.join(ROOT, "2023_render_engine_amd", "csrc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", inc, "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
