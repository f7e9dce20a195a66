// cache.hip -- online-trained neural radiance cache for gfx950.
//
// Model: a multiresolution hash-grid encoding of position (Mueller et al.,
// "Instant Neural Graphics Primitives with a Multiresolution Hash Encoding",
// SIGGRAPH 2022: L levels, 2^log2T entries of 2 BF16 features per level,
// trilinear interpolation, spatial hash x*1 ^ y*2654435761 ^ z*805459861)
// concatenated with the surface normal, view direction and roughness, then a
// bias-free MLP 64 -> 64 -> 64 -> 64 -> 64 -> 3 with ReLU on the hidden
// layers, trained online with Adam on a relative L2 loss (the loss of
// Mueller et al., "Real-time Neural Radiance Caching for Path Tracing",
// SIGGRAPH 2021).  The reference renderer has no counterpart (its learned
// component is a per-shape polynomial regression,
// sampling/ShapeLightDistribution.cu:20-345).
//
// Matmuls run on the matrix cores: v_mfma_f32_16x16x16_bf16 (BF16 inputs,
// FP32 accumulation).  One wavefront takes a 16-row strip through all layers
// in registers, forward (k_infer) and back (k_train_rows); only what the
// weight gradient reads (k_wgrad) is written to memory, as BF16.  Master
// weights, Adam moments and gradients are FP32.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include <hipcub/device/device_radix_sort.hpp>

#include "rt_cache.h"

namespace rt {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float f)
{
    // round to nearest even (no NaN inputs here)
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// Wavefront MFMA: D[16x16] += A[16xK] B[Kx16].  Lane l supplies
// A[l%16][k0 + 4(l/16) + 0..3] and B[k0 + 4(l/16) + 0..3][l%16]; D comes back
// as D[4(l/16) + r][l%16], r = 0..3.
__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------------
// hash-grid encoding
// ---------------------------------------------------------------------
__device__ __forceinline__ uint32_t grid_index(const CacheDev &c, uint32_t l, uint32_t x, uint32_t y, uint32_t z)
{
    const uint32_t res1 = c.res[l] + 1;
    if (c.dense[l]) return x + res1 * (y + res1 * z);
    return (x * 1u ^ y * 2654435761u ^ z * 805459861u) & (c.table_size - 1u);
}

// position -> level coordinates; writes the 8 corner indices and weights
__device__ __forceinline__ void grid_corners(const CacheDev &c, uint32_t l, float px, float py, float pz,
                                             uint32_t idx[8], float w[8])
{
    const float r = (float)c.res[l];
    const float x = px * r, y = py * r, z = pz * r;
    const float fx0 = floorf(x), fy0 = floorf(y), fz0 = floorf(z);
    const uint32_t x0 = (uint32_t)fx0, y0 = (uint32_t)fy0, z0 = (uint32_t)fz0;
    const float fx = x - fx0, fy = y - fy0, fz = z - fz0;
    const uint32_t rmax = c.res[l];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const uint32_t dx = k & 1, dy = (k >> 1) & 1, dz = (k >> 2) & 1;
        const uint32_t xi = min(x0 + dx, rmax), yi = min(y0 + dy, rmax), zi = min(z0 + dz, rmax);
        idx[k] = grid_index(c, l, xi, yi, zi);
        w[k] = (dx ? fx : 1 - fx) * (dy ? fy : 1 - fy) * (dz ? fz : 1 - fz);
    }
}

__device__ __forceinline__ void normalise_pos(const CacheDev &c, const float *q, float &px, float &py, float &pz)
{
    px = fminf(fmaxf((q[0] - c.lo[0]) * c.inv_ext[0], 0.0f), 1.0f);
    py = fminf(fmaxf((q[1] - c.lo[1]) * c.inv_ext[1], 0.0f), 1.0f);
    pz = fminf(fmaxf((q[2] - c.lo[2]) * c.inv_ext[2], 0.0f), 1.0f);
}

// ---------------------------------------------------------------------
// weight gradients of all layers: dW[64][NOUT] += X^T dY over all rows, one
// layer per blockIdx.y.  A workgroup stages 64-row chunks of X and dY in LDS,
// wave w accumulates dW rows 16w..16w+15 in registers and adds them to the
// FP32 gradient once at the end.  A staged row takes 72 elements: the 2-byte
// reads of four rows 4 apart then fall into different banks.
// ---------------------------------------------------------------------
constexpr uint32_t kWgradStride = 72;
// Blocks per layer: 65,536 rows take 8 chunks each.  With 256 or 512 a call
// took 17 us longer: more chunks at a time, but each block ends in 4096 atomics
// on the same 16 KB.
constexpr uint32_t kWgradBlocks = 128;

template <int NOUT>
__device__ __forceinline__ void wgrad_layer(const uint16_t *__restrict__ X, const uint16_t *__restrict__ dY, uint32_t n,
                                            float *__restrict__ dW, uint16_t *sX, uint16_t *sD)
{
    const uint32_t lane = __lane_id();
    const uint32_t wave = threadIdx.x / 64;
    const uint32_t li = lane & 15, lq = lane >> 4;
    f32x4 acc[NOUT / 16];
#pragma unroll
    for (int t = 0; t < NOUT / 16; ++t) acc[t] = f32x4{0, 0, 0, 0};
    const uint32_t chunks = (n + 63) / 64;
    for (uint32_t ch = blockIdx.x; ch < chunks; ch += gridDim.x) {
        const uint32_t r0 = ch * 64;
        // stage (zero rows past n)
        for (uint32_t e = threadIdx.x; e < 64 * kCacheWidth / 8; e += 256) {
            const uint32_t r = e / (kCacheWidth / 8), c8 = e % (kCacheWidth / 8);
            uint4 v = {0, 0, 0, 0};
            if (r0 + r < n) v = *(const uint4 *)(X + (size_t)(r0 + r) * kCacheWidth + c8 * 8);
            *(uint4 *)(sX + r * kWgradStride + c8 * 8) = v;
        }
        for (uint32_t e = threadIdx.x; e < 64 * NOUT / 8; e += 256) {
            const uint32_t r = e / (NOUT / 8), c8 = e % (NOUT / 8);
            uint4 v = {0, 0, 0, 0};
            if (r0 + r < n) v = *(const uint4 *)(dY + (size_t)(r0 + r) * NOUT + c8 * 8);
            *(uint4 *)(sD + r * kWgradStride + c8 * 8) = v;
        }
        __syncthreads();
        // dW[16w + i][j] += sum_m X[m][16w + i] dY[m][j]; A[i][m] = X[m][16w+i], B[m][j] = dY[m][j]
#pragma unroll
        for (int m0 = 0; m0 < 64; m0 += 16) {
            bf16x4 a;
#pragma unroll
            for (int q = 0; q < 4; ++q) a[q] = (short)sX[(m0 + 4 * lq + q) * kWgradStride + 16 * wave + li];
#pragma unroll
            for (int t = 0; t < NOUT / 16; ++t) {
                bf16x4 b;
#pragma unroll
                for (int q = 0; q < 4; ++q) b[q] = (short)sD[(m0 + 4 * lq + q) * kWgradStride + t * 16 + li];
                acc[t] = mfma16(a, b, acc[t]);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < NOUT / 16; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t wr = 16 * wave + 4 * lq + r, wc = t * 16 + li;
            atomicAdd(&dW[wr * NOUT + wc], acc[t][r]);
        }
}

__global__ __launch_bounds__(256) void k_wgrad(CacheDev c, CacheWork w, uint32_t n, const uint32_t *__restrict__ n_dev)
{
    __shared__ uint16_t sX[64 * kWgradStride], sD[64 * kWgradStride];
    if (n_dev) n = min(n, *n_dev);
    const uint32_t l = blockIdx.y;
    if (l + 1 < kCacheLayers)
        wgrad_layer<kCacheWidth>(w.act[l], w.dact[l], n, c.grad + kCacheLayerOffset(l), sX, sD);
    else
        wgrad_layer<kCacheOut>(w.act[l], w.dy16, n, c.grad + kCacheLayerOffset(l), sX, sD);
}

// Morton key of each sample's normalised position (10 bits per axis; rows
// past the count get the largest key and sort last), and its index.
__global__ __launch_bounds__(256) void k_sample_morton(CacheDev c, const float *__restrict__ in, uint32_t n,
                                                       const uint32_t *__restrict__ n_dev, uint32_t *__restrict__ key,
                                                       uint32_t *__restrict__ idx)
{
    const uint32_t count = n_dev ? min(n, *n_dev) : n;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        uint32_t k = 0xffffffffu;
        if (i < count) {
            float p[3];
            normalise_pos(c, in + (size_t)i * kCacheInStride, p[0], p[1], p[2]);
            k = 0;
            for (int a = 0; a < 3; ++a) {
                uint32_t q = (uint32_t)fminf(p[a] * 1024.0f, 1023.0f);
                q &= 1023u;
                q = (q | (q << 16)) & 0x030000FFu;
                q = (q | (q << 8)) & 0x0300F00Fu;
                q = (q | (q << 4)) & 0x030C30C3u;
                q = (q | (q << 2)) & 0x09249249u;
                k |= q << (2 - a);
            }
        }
        key[i] = k;
        idx[i] = i;
    }
}

// hash-grid gradient: scatter the features' gradients through the trilinear
// weights.  Block (level l, run jb) takes the samples at positions jb*256 ..
// +255 of the batch's Morton order, so its lanes sit close together in space
// and share grid cells on all but the finest levels.  Their 8 corner updates
// are first merged in an LDS table keyed by pairs of cells 2k, 2k + 1 (open
// addressing, 2048 slots for at most 2048 distinct pairs, so a probe always
// ends): on a surface-sampled batch that is 2.4x fewer atomics overall and
// 50-130x fewer on the coarse levels, where one atomic per corner serialised
// on a few thousand addresses.
//
// What bounds it: the requests of the device-scope atomics.  A pair's four
// sums are added by four neighbouring lanes, whose words lie in one cache
// line, so they are one request; corners one x apart are mostly a pair (in a
// hashed level where x is even).  65,536 uniform samples, 16 levels of 2^15
// entries: 194 us, against 387 us keyed by single cells, one lane adding a
// cell's two features in turn and the gradients read from rows of 256 B.
constexpr uint32_t kGridPairs = 2048;
constexpr uint32_t kGridEmpty = 0xffffffffu;

__global__ __launch_bounds__(256) void k_grid_bwd(CacheDev c, const float *__restrict__ in, uint32_t n,
                                                  const uint32_t *__restrict__ n_dev, uint32_t runs,
                                                  const uint32_t *__restrict__ order, const float2 *__restrict__ dfeat,
                                                  uint32_t rows, float *__restrict__ dgrid)
{
    __shared__ uint32_t skey[kGridPairs];
    __shared__ float sv[kGridPairs * 4];
    const uint32_t count = n_dev ? min(n, *n_dev) : n;
    const uint32_t l = blockIdx.x / runs, jb = blockIdx.x - l * runs;
    if (l >= c.levels || jb * 256 >= count) return;  // whole block: before any barrier
    for (uint32_t t = threadIdx.x; t < kGridPairs; t += 256) skey[t] = kGridEmpty;
    for (uint32_t t = threadIdx.x; t < kGridPairs; t += 256) ((float4 *)sv)[t] = make_float4(0, 0, 0, 0);
    __syncthreads();
    const uint32_t j = jb * 256 + threadIdx.x;
    if (j < count) {
        const uint32_t i = order[j];
        const float2 g = dfeat[(size_t)l * rows + i];
        if (g.x != 0.0f || g.y != 0.0f) {
            float px, py, pz;
            normalise_pos(c, in + (size_t)i * kCacheInStride, px, py, pz);
            uint32_t idx[8];
            float w[8];
            grid_corners(c, l, px, py, pz, idx, w);
            uint32_t h = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint32_t pair = idx[k] >> 1;
                if (!(k & 1) || pair != idx[k - 1] >> 1) {
                    h = (pair * 2654435761u) >> 21;  // 11 bits
                    for (;;) {
                        const uint32_t prev = atomicCAS(&skey[h], kGridEmpty, pair);
                        if (prev == kGridEmpty || prev == pair) break;
                        h = (h + 1) & (kGridPairs - 1);
                    }
                }
                float *v = sv + 4 * h + 2 * (idx[k] & 1u);
                atomicAdd(v, w[k] * g.x);
                atomicAdd(v + 1, w[k] * g.y);
            }
        }
    }
    __syncthreads();
    float *tab = dgrid + (size_t)l * c.table_size * 2;
    for (uint32_t t = threadIdx.x; t < kGridPairs * 4; t += 256) {
        const float v = sv[t];
        if (v != 0.0f) atomicAdd(&tab[4 * (size_t)skey[t >> 2] + (t & 3u)], v);
    }
}

// Adam (Kingma & Ba 2015) on FP32 master weights; refreshes the BF16 copies.
// For the MLP it also writes the transposed forward copy.
__global__ __launch_bounds__(256) void k_adam(float *__restrict__ w, float *__restrict__ g, float *__restrict__ m,
                                              float *__restrict__ v, uint32_t count, float lr, float b1, float b2,
                                              float eps, float bc1, float bc2, uint16_t *__restrict__ wbf,
                                              uint16_t *__restrict__ wbf_t, uint32_t mlp)
{
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < count; i += gridDim.x * 256) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1 - b1) * gi;
        const float vi = b2 * v[i] + (1 - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        const float wi = w[i] - lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
        w[i] = wi;
        g[i] = 0.0f;
        const uint16_t h = f2bf(wi);
        wbf[i] = h;
        if (mlp) {
            // layer l: W stored [64][nout] at offset kCacheLayerOffset(l); the
            // transposed copy [nout][64] at the same offset in wbf_t
            uint32_t l = 0, off = 0, nout = kCacheWidth;
            while (l + 1 < kCacheLayers && i >= off + kCacheWidth * nout) {
                off += kCacheWidth * nout;
                ++l;
                nout = (l + 1 == kCacheLayers) ? kCacheOut : kCacheWidth;
            }
            const uint32_t k = (i - off) / nout, j = (i - off) % nout;
            wbf_t[off + j * kCacheWidth + k] = h;
        }
    }
}

__global__ __launch_bounds__(256) void k_fill(float *__restrict__ p, uint32_t count, float value)
{
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < count; i += gridDim.x * 256) p[i] = value;
}

// ---------------------------------------------------------------------
// Inference in one kernel: encoding and all five layers of a 16-row strip in
// the registers of one wavefront.
//
// Each layer is computed transposed, Y^T = W^T X^T.  v_mfma_f32_16x16x16
// returns D[m][n] with n = l % 16 and m = 4 (l / 16) + r in lane l, register
// r, and takes B[k][n] with k = 4 (l / 16) + 0..3 from lane l: with n the row
// and m (then k) the feature, a layer's result is the next layer's operand in
// the same lane, and only ReLU and rounding to BF16 stand between them.  So
// lane l holds features 16t + 4 (l / 16) + 0..3 of row l % 16: of the encoding
// that is two grid levels per tile, and the four lanes of a row share its
// 8 x levels gathers.
//
// What bounds it: the gathers.  A pair of corners one x apart lies in one
// 8-byte word of a dense level, and of a hashed one when x is even, so a
// level takes 4 loads, or 8 where x is odd, instead of 8.  One wavefront
// needs 68 matrix instructions per strip; the weights (34 KB, in fragment
// order) come through LDS and stay in registers (228 in all, two wavefronts per
// SIMD; read from LDS for every strip, at five per SIMD, the kernel takes 432
// to 480 us).  1,000,003 queries, 16 levels of 2^19 entries: 390 us, against
// 1350 us in seven kernels per 65,536 rows with the activations in memory.  A
// row makes 61 requests to the L2, of which 18 miss; 2.3 GB come from beyond it.
// ---------------------------------------------------------------------
constexpr uint32_t kXcds = 8;
constexpr int kCacheFrags = 16 * 4 + 4;  // A fragments of W^T: four 64 x 64 layers, one 16 x 64

typedef uint32_t u32x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// Two floats rounded to nearest even, packed (the first in the low half).
__device__ __forceinline__ uint32_t pack_bf16(float a, float b)
{
    const bf2 v = __builtin_convertvector((f32x2){a, b}, bf2);
    return __builtin_bit_cast(uint32_t, v);
}

// Fragment f of W^T for lane l: out 16o + l % 16, inputs 16k + 4 (l / 16) + 0..3.
__device__ __forceinline__ void load_weight_frags(const CacheDev &c, uint2 *frags)
{
    for (uint32_t e = threadIdx.x; e < kCacheFrags * 64; e += blockDim.x) {
        const uint32_t f = e >> 6, l = e & 63u;
        const uint32_t layer = f >> 4, o = f < 64 ? (f >> 2) & 3u : 0u, k = f & 3u;
        frags[e] = *(const uint2 *)(c.w_t + kCacheLayerOffset(layer) + (16 * o + (l & 15u)) * kCacheWidth + 16 * k +
                                    4 * (l >> 4));
    }
}

// Trilinear features of grid level `lev` (resolution res) at p.
__device__ __forceinline__ f32x2 grid_feature(const CacheDev &c, uint32_t lev, uint32_t res, bool dense, float px,
                                              float py, float pz)
{
    const float r = (float)res;
    const float x = px * r, y = py * r, z = pz * r;
    const float fx0 = floorf(x), fy0 = floorf(y), fz0 = floorf(z);
    const uint32_t x0 = (uint32_t)fx0, y0 = (uint32_t)fy0, z0 = (uint32_t)fz0;
    const float fx = x - fx0, fy = y - fy0, fz = z - fz0;
    const uint32_t x1 = min(x0 + 1, res), mask = c.table_size - 1u;
    const uint32_t *tab = (const uint32_t *)c.grid_bf16 + (size_t)lev * c.table_size;
    uint32_t i0[4], i1[4], at[4], v0[4], v1[4];
    bool second = false;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t yi = min(y0 + (k & 1), res), zi = min(z0 + (k >> 1), res);
        if (dense) {
            const uint32_t row = (res + 1) * (yi + (res + 1) * zi);
            i0[k] = row + x0;
            i1[k] = row + x1;
            at[k] = min(i0[k], c.table_size - 2u);  // the pair stays inside the level
        } else {
            const uint32_t h = yi * 2654435761u ^ zi * 805459861u;
            i0[k] = (x0 ^ h) & mask;
            i1[k] = (x1 ^ h) & mask;
            at[k] = i0[k] & ~1u;
        }
        second = second || i1[k] - at[k] > 1u;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const u32x2u v = *(const u32x2u *)(tab + at[k]);
        v0[k] = i0[k] == at[k] ? v.x : v.y;
        v1[k] = i1[k] == at[k] ? v.x : v.y;
    }
    if (second) {
#pragma unroll
        for (int k = 0; k < 4; ++k) v1[k] = tab[i1[k]];
    }
    float f0 = 0, f1 = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float wy = (k & 1) ? fy : 1 - fy, wz = (k >> 1) ? fz : 1 - fz;
        const float w0 = (1 - fx) * wy * wz, w1 = fx * wy * wz;
        f0 += w0 * bf2f((uint16_t)(v0[k] & 0xffffu));
        f1 += w0 * bf2f((uint16_t)(v0[k] >> 16));
        f0 += w1 * bf2f((uint16_t)(v1[k] & 0xffffu));
        f1 += w1 * bf2f((uint16_t)(v1[k] >> 16));
    }
    return {f0, f1};
}

// The grid levels of a lane and their parameters: tile t, pair e is level
// 8t + 2 (l / 16) + e.
struct LaneLevels {
    uint32_t res[4];
    uint32_t dense;  // bit 2t + e
};

__device__ __forceinline__ LaneLevels lane_levels(const CacheDev &c, uint32_t q)
{
    LaneLevels ll{{1, 1, 1, 1}, 0};
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t lev = 8 * (i >> 1) + 2 * q + (i & 1u);
        for (uint32_t l = 0; l < c.levels; ++l)
            if (l == lev) {
                ll.res[i] = c.res[l];
                ll.dense |= (c.dense[l] ? 1u : 0u) << i;
            }
    }
    return ll;
}

// The encoding of the strip's row l % 16: features 16t + 4 (l / 16) + 0..3 in x[t].
__device__ __forceinline__ void encode_strip(const CacheDev &c, const LaneLevels &ll, const float *__restrict__ rec,
                                             uint32_t q, bf16x4 x[4])
{
    float px, py, pz;
    normalise_pos(c, rec, px, py, pz);
    // feature 2 levels + j: normal, view direction, roughness, the constant 1, zeros
    auto other = [&](uint32_t j) {
        const float v = rec[3 + min(j, 6u)];
        return j < 7u ? v : (j == 7u ? 1.0f : 0.0f);
    };
#pragma unroll
    for (uint32_t t = 0; t < 4; ++t) {
        uint32_t w[2];
#pragma unroll
        for (uint32_t e = 0; e < 2; ++e) {
            const uint32_t lev = 8 * t + 2 * q + e;
            f32x2 f;
            if (t < 2 && lev < c.levels) {
                const uint32_t i = 2 * (t & 1u) + e;
                f = grid_feature(c, lev, ll.res[i], (ll.dense >> i) & 1u, px, py, pz);
            } else {
                const uint32_t j = 2 * (lev - c.levels);
                f = {other(j), other(j + 1)};
            }
            w[e] = pack_bf16(f.x, f.y);
        }
        x[t] = __builtin_bit_cast(bf16x4, make_uint2(w[0], w[1]));
    }
}

// One hidden layer in registers: x (features of a row) -> ReLU(W^T x).
__device__ __forceinline__ void hidden_layer(const uint2 *frags, uint32_t layer, uint32_t lane, bf16x4 x[4])
{
    f32x4 acc[4];
#pragma unroll
    for (int o = 0; o < 4; ++o) {
        acc[o] = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < 4; ++k)
            acc[o] = mfma16(__builtin_bit_cast(bf16x4, frags[(layer * 16 + o * 4 + k) * 64 + lane]), x[k], acc[o]);
    }
#pragma unroll
    for (int o = 0; o < 4; ++o)
        x[o] = __builtin_bit_cast(bf16x4, make_uint2(pack_bf16(fmaxf(acc[o][0], 0.0f), fmaxf(acc[o][1], 0.0f)),
                                                     pack_bf16(fmaxf(acc[o][2], 0.0f), fmaxf(acc[o][3], 0.0f))));
}

// The output layer: outputs 4 (l / 16) + r of row l % 16.
__device__ __forceinline__ f32x4 output_layer(const uint2 *frags, uint32_t lane, const bf16x4 x[4])
{
    f32x4 y{0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 4; ++k) y = mfma16(__builtin_bit_cast(bf16x4, frags[(64 + k) * 64 + lane]), x[k], y);
    return y;
}

__global__ __launch_bounds__(256) void k_infer(CacheDev c, const float *__restrict__ in, uint32_t n,
                                               const uint32_t *__restrict__ n_dev, float *__restrict__ rgb)
{
    __shared__ uint2 frags[kCacheFrags * 64];
    if (n_dev) n = min(n, *n_dev);
    // an eighth of the strips for each eighth of the blocks (see cache_infer)
    const uint32_t strips = (n + 15) / 16, part = (strips + kXcds - 1) / kXcds;
    const uint32_t lo = (blockIdx.x % kXcds) * part, hi = min(lo + part, strips);
    if (lo + blockIdx.x / kXcds * 4 >= hi) return;  // whole block: before the barrier
    load_weight_frags(c, frags);
    __syncthreads();
    const uint32_t lane = __lane_id(), wave = threadIdx.x / 64, q = lane >> 4;
    const LaneLevels ll = lane_levels(c, q);
    for (uint32_t s = lo + blockIdx.x / kXcds * 4 + wave; s < hi; s += gridDim.x / kXcds * 4) {
        const uint32_t row = s * 16 + (lane & 15u);
        bf16x4 x[4];
        encode_strip(c, ll, in + (size_t)min(row, n - 1) * kCacheInStride, q, x);
#pragma unroll
        for (uint32_t l = 0; l + 1 < kCacheLayers; ++l) hidden_layer(frags, l, lane, x);
        const f32x4 y = output_layer(frags, lane, x);
        if (q == 0 && row < n) {
            rgb[(size_t)row * 3] = fmaxf(y[0], 0.0f);
            rgb[(size_t)row * 3 + 1] = fmaxf(y[1], 0.0f);
            rgb[(size_t)row * 3 + 2] = fmaxf(y[2], 0.0f);
        }
    }
}

// ---------------------------------------------------------------------
// Training: encoding, forward, loss and data gradients of a 16-row strip in
// one wavefront, in k_infer's layout.  The backward products are transposed the
// same way, dX^T = W dY^T, with W (in x out) as the A operand.  The loss is the
// relative L2 loss of Mueller et al. 2021: l = (y - t)^2 / (sg(y)^2 + 0.01),
// mean over rows and the 3 channels (with n_dev the count, and so the mean's
// scale, comes from device memory).  What the weight gradient needs goes to
// memory as BF16: every layer's input act[l] and its masked output gradient
// dact[l] (dy16 for the output layer); the encoding's gradient as FP32, one
// float2 per level and row.
//
// Both weight layouts (70 KB) stay in LDS: a wavefront has one or two strips
// of a batch, so registers would only be filled once or twice.  65,536 rows:
// 74 us (bound by its chain of gathers, products and stores at two wavefronts
// per SIMD), against 159 us in twelve kernels; with k_wgrad 100 us against 247.
// ---------------------------------------------------------------------
__device__ __forceinline__ void load_backward_frags(const CacheDev &c, uint2 *frags)
{
    for (uint32_t e = threadIdx.x; e < kCacheFrags * 64; e += blockDim.x) {
        const uint32_t f = e >> 6, l = e & 63u;
        const uint32_t layer = f >> 4, o = f < 64 ? (f >> 2) & 3u : f & 3u, k = f < 64 ? f & 3u : 0u;
        const uint32_t nout = f < 64 ? kCacheWidth : kCacheOut;
        frags[e] = *(const uint2 *)(c.w + kCacheLayerOffset(layer) + (16 * o + (l & 15u)) * nout + 16 * k + 4 * (l >> 4));
    }
}

__device__ __forceinline__ bf16x4 pack4(const f32x4 &v)
{
    return __builtin_bit_cast(bf16x4, make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])));
}

// v where the activation a is positive, else 0.
__device__ __forceinline__ f32x4 relu_mask(f32x4 v, bf16x4 a)
{
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (!(bf2f((uint16_t)a[r]) > 0.0f)) v[r] = 0.0f;
    return v;
}

__device__ __forceinline__ void store_strip(uint16_t *dst, uint32_t row, uint32_t q, const bf16x4 x[4])
{
#pragma unroll
    for (int t = 0; t < 4; ++t) *(bf16x4 *)(dst + (size_t)row * kCacheWidth + 16 * t + 4 * q) = x[t];
}

__global__ __launch_bounds__(256) void k_train_rows(CacheDev c, CacheWork w, const float *__restrict__ in,
                                                    const float *__restrict__ target, uint32_t n,
                                                    const uint32_t *__restrict__ n_dev, float scale,
                                                    float *__restrict__ loss)
{
    __shared__ uint2 fw[kCacheFrags * 64], bw[kCacheFrags * 64];
    if (n_dev) {
        n = min(n, *n_dev);
        scale = n ? 1.0f / (3.0f * (float)n) : 0.0f;
    }
    const uint32_t strips = (n + 15) / 16;
    if (blockIdx.x * 4 >= strips) return;  // whole block: before the barrier
    load_weight_frags(c, fw);
    load_backward_frags(c, bw);
    __syncthreads();
    const uint32_t lane = __lane_id(), wave = threadIdx.x / 64, q = lane >> 4;
    const LaneLevels ll = lane_levels(c, q);
    float lsum = 0;
    for (uint32_t s = blockIdx.x * 4 + wave; s < strips; s += gridDim.x * 4) {
        uint32_t at = lane;
        asm volatile("" : "+v"(at));  // the fragments are read for every strip
        const uint32_t row = s * 16 + (lane & 15u);
        const bool valid = row < n;
        bf16x4 a[kCacheLayers][4];
        encode_strip(c, ll, in + (size_t)min(row, n - 1) * kCacheInStride, q, a[0]);
        if (valid) store_strip(w.act[0], row, q, a[0]);
#pragma unroll
        for (uint32_t l = 0; l + 1 < kCacheLayers; ++l) {
#pragma unroll
            for (int t = 0; t < 4; ++t) a[l + 1][t] = a[l][t];
            hidden_layer(fw, l, at, a[l + 1]);
            if (valid) store_strip(w.act[l + 1], row, q, a[l + 1]);
        }
        const f32x4 y = output_layer(fw, at, a[kCacheLayers - 1]);
        f32x4 g{0, 0, 0, 0};
        if (q == 0 && valid) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const float t = target[(size_t)row * 3 + k];
                const float den = y[k] * y[k] + 0.01f;
                const float d = y[k] - t;
                lsum += d * d / den;
                g[k] = 2.0f * d / den * scale;
            }
        }
        const bf16x4 dy = pack4(g);
        if (valid) *(bf16x4 *)(w.dy16 + (size_t)row * kCacheOut + 4 * q) = dy;
        bf16x4 d[4];
#pragma unroll
        for (int o = 0; o < 4; ++o)
            d[o] = pack4(relu_mask(mfma16(__builtin_bit_cast(bf16x4, bw[(64 + o) * 64 + at]), dy, f32x4{0, 0, 0, 0}),
                                   a[kCacheLayers - 1][o]));
#pragma unroll
        for (int l = (int)kCacheLayers - 2; l >= 0; --l) {
            if (valid) store_strip(w.dact[l], row, q, d);
            f32x4 acc[4];
#pragma unroll
            for (int o = 0; o < (l ? 4 : 2); ++o) {
                acc[o] = f32x4{0, 0, 0, 0};
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    acc[o] = mfma16(__builtin_bit_cast(bf16x4, bw[(l * 16 + o * 4 + k) * 64 + at]), d[k], acc[o]);
            }
            if (l) {
#pragma unroll
                for (int o = 0; o < 4; ++o) d[o] = pack4(relu_mask(acc[o], a[l][o]));
            } else if (valid) {
                // features 16o + 4q + 0..3 are levels 8o + 2q and the next
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) {
                    const uint32_t lev = 8 * (i >> 1) + 2 * q + (i & 1u);
                    if (lev < c.levels)
                        w.dfeat[(size_t)lev * w.rows + row] = make_float2(acc[i >> 1][2 * (i & 1u)], acc[i >> 1][2 * (i & 1u) + 1]);
                }
            }
        }
    }
    // wavefront reduction, one atomic per wavefront
    for (int off = 32; off > 0; off >>= 1) lsum += __shfl_down(lsum, off);
    if (lane == 0 && loss) atomicAdd(loss, lsum);
}

// ---------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------
static dim3 grid_for(uint32_t work, uint32_t per_block, uint32_t cap = 4096)
{
    uint32_t b = (work + per_block - 1) / per_block;
    if (b < 1) b = 1;
    if (b > cap) b = cap;
    return dim3(b);
}

hipError_t cache_infer(const CacheDev &c, const float *in, uint32_t n, float *rgb, hipStream_t s,
                       const uint32_t *n_dev)
{
    if (n == 0) return hipSuccess;
    // Four wavefronts of 16 rows per block, two blocks per CU.  Blocks go to the
    // eight XCDs in turn, and each XCD takes one contiguous eighth of the rows:
    // rows in image order then touch an eighth of the grid's cells, which the
    // XCD's own L2 holds.
    const uint32_t blocks = std::min((n + 63) / 64, 512u);
    hipLaunchKernelGGL(k_infer, dim3((blocks + kXcds - 1) / kXcds * kXcds), dim3(256), 0, s, c, in, n, n_dev, rgb);
    return hipGetLastError();
}

hipError_t cache_backward(const CacheDev &c, const CacheWork &w, const float *in, const float *target, uint32_t n,
                          float *loss, hipStream_t s, const uint32_t *n_dev)
{
    if (n == 0) return hipSuccess;
    const dim3 blk(256);
    // four strips of 16 rows per block and turn, two blocks per CU
    hipLaunchKernelGGL(k_train_rows, grid_for((n + 15) / 16, 4, 512), blk, 0, s, c, w, in, target, n, n_dev,
                       1.0f / (3.0f * (float)n), loss);
    hipLaunchKernelGGL(k_wgrad, dim3(grid_for((n + 63) / 64, 1, kWgradBlocks).x, kCacheLayers), blk, 0, s, c, w, n, n_dev);
    // the grid gradient in Morton order of the samples' positions
    hipLaunchKernelGGL(k_sample_morton, grid_for(n, 256), blk, 0, s, c, in, n, n_dev, w.skey[0], w.sidx[0]);
    size_t tb = w.sort_bytes;
    hipError_t e = hipcub::DeviceRadixSort::SortPairs(w.sort_tmp, tb, w.skey[0], w.skey[1], w.sidx[0], w.sidx[1], (int)n, 0, 32,
                                           s);
    if (e != hipSuccess) return e;
    const uint32_t runs = (n + 255) / 256;
    hipLaunchKernelGGL(k_grid_bwd, dim3(runs * c.levels), blk, 0, s, c, in, n, n_dev, runs, w.sidx[1], w.dfeat,
                       w.rows, c.grid_grad);
    return hipGetLastError();
}

size_t cache_sort_bytes(uint32_t rows)
{
    size_t b = 0;
    if (hipcub::DeviceRadixSort::SortPairs(nullptr, b, (const uint32_t *)nullptr, (uint32_t *)nullptr,
                                           (const uint32_t *)nullptr, (uint32_t *)nullptr, (int)rows, 0, 32) !=
        hipSuccess)
        return 0;
    return b;
}

hipError_t cache_adam(const CacheDev &c, const CacheOptsDev &o, uint32_t step, hipStream_t s)
{
    const float bc1 = 1.0f - powf(o.beta1, (float)step);
    const float bc2 = 1.0f - powf(o.beta2, (float)step);
    const dim3 blk(256);
    hipLaunchKernelGGL(k_adam, grid_for(kCacheParams, 256), blk, 0, s, c.w32, c.grad, c.m, c.v, kCacheParams, o.lr,
                       o.beta1, o.beta2, o.eps, bc1, bc2, c.w, c.w_t, 1u);
    const uint32_t gp = c.levels * c.table_size * 2;
    hipLaunchKernelGGL(k_adam, grid_for(gp, 256), blk, 0, s, c.grid32, c.grid_grad, c.grid_m, c.grid_v, gp, o.lr,
                       o.beta1, o.beta2, o.eps, bc1, bc2, (uint16_t *)c.grid_bf16, (uint16_t *)nullptr, 0u);
    return hipGetLastError();
}

hipError_t cache_fill(float *p, uint32_t count, float value, hipStream_t s)
{
    if (count == 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill, grid_for(count, 256), dim3(256), 0, s, p, count, value);
    return hipGetLastError();
}

}  // namespace rt
