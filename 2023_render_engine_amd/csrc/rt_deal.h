// rt_deal.h -- how the persistent traversal launches deal their items to
// wavefronts: plain integer rules shared by the host (launch sizes) and the
// kernels (rt_device.h), free of HIP so that a CPU test can walk them.
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define RT_HD __host__ __device__ __forceinline__
#else
#define RT_HD inline
#endif

namespace rt {

// Work striping of the persistent kernels and the wavefront queues: work is
// cut into kStripes stripes whose counters sit kCtrStride u32 words (one
// 128-byte line) apart, so device atomics spread over 64 addresses.
constexpr uint32_t kStripes = 64;
constexpr uint32_t kCtrStride = 32;
constexpr uint32_t kClaimWords = kStripes * kCtrStride;  // one striped counter set

// Tuning constants of the claims (build-time, -D overridable).
#ifndef RT_REFILL_LANES
#define RT_REFILL_LANES 16
#endif
#ifndef RT_CLAIM_CHUNK
#define RT_CLAIM_CHUNK 128
#endif
#ifndef RT_CLAIM_MIN
#define RT_CLAIM_MIN 64
#endif
constexpr uint32_t kRefillLanes = RT_REFILL_LANES;  // refill a wavefront when at least this many of 64 lanes are idle
constexpr uint32_t kClaimChunk = RT_CLAIM_CHUNK;
constexpr uint32_t kClaimMin = RT_CLAIM_MIN;
static_assert(kClaimMin >= 1 && kClaimMin <= kClaimChunk, "claim sizes run from kClaimMin to kClaimChunk");

// A launch with fewer items than kWidthWaves full wavefronts (two per SIMD)
// takes them with fewer lanes of more wavefronts, down to kMinWidth: a small
// launch is as long as its slowest wavefront, and a wavefront runs through the
// node and leaf work of all its rays in turn.  8192 rays against 4096
// triangles, closest and any hit: 248 us with 64 lanes, 224 with 16, 214 with
// 4; cached 960x540 frames 7.28 and 7.03 ms with 64 and 4.
constexpr uint32_t kWidthWaves = 2048, kMinWidth = 4;
constexpr uint32_t kWavesPerBlock = 2;  // of the traversal kernels

// Lanes of a wavefront that take items, in a launch of `waves` wavefronts.
RT_HD uint32_t deal_width(uint32_t total, uint32_t waves)
{
    if (waves > kWidthWaves) waves = kWidthWaves;
    uint32_t width = 64;
    while (width > kMinWidth && total <= (width >> 1) * waves) width >>= 1;
    return width;
}

// Whether the nth wavefront at home on a stripe of n items leaves at once: in
// a narrow launch it does when the ones before it take all of the stripe's
// items in one turn.
RT_HD bool deal_leaves(uint32_t width, uint32_t nth, uint32_t n) { return width < 64u && nth * width >= n; }

// Idle lanes (of `width`) that start a refill: at least one, or a wavefront
// without an idle lane would hand out items that nobody claimed.
RT_HD uint32_t deal_refill(uint32_t width) { return (width * kRefillLanes) >> 6; }
static_assert((kMinWidth * kRefillLanes) >> 6 >= 1, "kRefillLanes of 64 lanes is at least one of kMinWidth lanes");

// Items of the next claim: `left` items of the stripe over its 2^wlog
// wavefronts, between kClaimMin (what a narrow wavefront can start at once,
// if that is less) and kClaimChunk.
RT_HD uint32_t deal_claim(uint32_t left, uint32_t wlog, uint32_t width)
{
    const uint32_t k = left >> wlog, least = width < kClaimMin ? width : kClaimMin;
    return k < least ? least : (k > kClaimChunk ? kClaimChunk : k);
}

// A ray batch: dealt to the stripes in chunks of 2^lc consecutive rays (chunk
// c to stripe c % kStripes), so every stripe holds a sample of the whole
// batch and the stripes take about equally long.
struct RayDeal {
    uint32_t lc, blocks;
};

// Rays of stripe j.
RT_HD uint32_t deal_count(uint32_t n, uint32_t lc, uint32_t j)
{
    const uint32_t nfull = n >> lc, rem = n & ((1u << lc) - 1u), last = nfull & (kStripes - 1u);
    uint32_t k = ((nfull / kStripes) + (j < last ? 1u : 0u)) << lc;
    if (rem && j == last) k += rem;
    return k;
}

// Ray `off` of stripe j.
RT_HD uint32_t deal_ray(uint32_t lc, uint32_t j, uint32_t off)
{
    return ((off >> lc) * kStripes + j) * (1u << lc) + (off & ((1u << lc) - 1u));
}

// Chunks and workgroups of a launch of n rays, on a chip that holds `most`
// workgroups.  From 2^14 rays on a chunk is 64 rays, from 2^18 on n / 2048, up
// to 4096.  Below, chunks shrink down to kMinWidth rays, so that every stripe
// gets four or more while there are that many, and every stripe has the
// wavefronts that start all of its rays at once with kMinWidth lanes each.
// Closest hits of 64, 256, 1000 and 2048 rays against 4096 triangles: 103, 108,
// 111 and 129 us; with chunks of 64 rays at every size, whose few stripes' few
// wavefronts took them with four lanes, 347, 458, 295 and 163; with 64 lanes
// per wavefront 128, 140, 140 and 161.
inline RayDeal ray_deal(uint32_t n, uint32_t most)
{
    RayDeal d{2, 0};
    while (d.lc < 6 && ((uint64_t)512 << d.lc) <= n) ++d.lc;
    if (d.lc == 6)
        while (d.lc < 12 && ((uint64_t)2048 << d.lc) <= n) ++d.lc;
    constexpr uint64_t kLanes = kWavesPerBlock * kMinWidth;
    const uint64_t chunks = ((uint64_t)n + (1u << d.lc) - 1) >> d.lc;
    uint64_t blocks = chunks;  // one chunk per stripe, or none
    if (chunks > kStripes || d.lc > 2) {
        // (a power of two per stripe, so that a claim's share is what one wavefront starts)
        const uint64_t rays = ((chunks + kStripes - 1) / kStripes) << d.lc;  // of the fullest stripe
        for (blocks = kStripes; blocks / kStripes * kLanes < rays; blocks *= 2) {
        }
    }
    // kWidthWaves wavefronts take up to 64 rays each in one turn; more rays are
    // taken by as many wavefronts as the chip holds
    if (n <= kWidthWaves * 64u && blocks > kWidthWaves / kWavesPerBlock) blocks = kWidthWaves / kWavesPerBlock;
    d.blocks = (uint32_t)(blocks < most ? blocks : most);
    if (d.blocks == 0) d.blocks = 1;
    return d;
}

}  // namespace rt
