// bvh_gpu.hip -- the BVH built on the GPU from device-resident triangles, in
// the layouts the traversal kernels read (rt_internal.h: Node2, Node4, Tri3).
//
// The reference builds its tree on the GPU from Morton codes of the
// triangles (cuda_libraries/BVH.cu:136-151, 314-341: codes, a sort, leaves
// initialised in parallel, then pairing).  This builder follows the same
// idea with a linear-time radix tree:
//   1. triangle boxes, and the bounds of their centres (k_tri_boxes per
//      block, k_bounds over the blocks: no contended atomics);
//   2. 30-bit Morton codes of the centres in those bounds, sorted with the
//      triangle index as the value (rocPRIM radix sort);
//   3. Karras' binary radix tree over the sorted codes (k_radix_tree: each
//      internal node finds its range and split from the common prefixes of
//      its neighbours; equal codes are split by index);
//   4. boxes and SAH costs bottom-up in passes (k_node_pass: a node is
//      computed once both children were computed by an earlier launch, so
//      nothing is read across work-groups within a launch and no
//      device-scope fence is needed -- on this GPU each such fence writes
//      back the XCD's L2); a subtree of at most max_leaf triangles becomes
//      a leaf when that is no dearer by the SAH;
//   5. the kept internal nodes are numbered by a prefix sum and written as
//      Node2 records with both child boxes (k_emit_node2), and the
//      triangles as Tri3 records in code order plus the degenerate
//      sentinel (k_emit_tris);
//   6. for the four-wide layout, the Node2 tree is collapsed level by level
//      (k_collapse4_count, a prefix sum, k_collapse4): each wide node opens
//      its largest-area internal child until it has four, as the host
//      collapse does, and quantizes the boxes outward; nodes are numbered
//      breadth-first.
// Every step is deterministic: the same input gives the same records.
// The tree is worse than the host's binned SAH (its SAH cost is reported),
// and it is built in milliseconds.
#include <hip/hip_runtime.h>
#include <hipcub/device/device_radix_sort.hpp>
#include <hipcub/device/device_scan.hpp>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <string>
#include <vector>

#include "rt_bvh_gpu.h"
#include "rt_internal.h"

namespace rt {

namespace {

constexpr int kBB = 256;  // block size of the build kernels

__device__ inline uint32_t ord(float f)
{
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ inline float unord(uint32_t u) { return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u); }

__device__ inline uint32_t spread10(uint32_t v)
{
    v &= 1023u;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// Per triangle: its box (6 floats: lo xyz, hi xyz).  Each block reduces
// its triangles' bounds into part[block * 12 ..] as ordered ints: [0..2] /
// [3..5] the min / max of the centres, [6..8] / [9..11] the min / max of the
// boxes (k_bounds finishes the reduction).  Indices out of range or
// non-finite coordinates set *bad.
__global__ __launch_bounds__(kBB) void k_tri_boxes(const float *xyz, uint32_t nv, const uint32_t *idx, uint32_t nt,
                                                   float *tbox, uint32_t *part, uint32_t *bad)
{
    __shared__ uint32_t smin[6][kBB], smax[6][kBB];
    const uint32_t t = blockIdx.x * kBB + threadIdx.x;
    uint32_t mn[6], mx[6];
    for (int a = 0; a < 6; ++a) { mn[a] = 0xffffffffu; mx[a] = 0u; }
    if (t < nt) {
        float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        bool ok = true;
        for (int k = 0; k < 3; ++k) {
            uint32_t v = idx[3 * (size_t)t + k];
            if (v >= nv) { ok = false; v = 0; }
            for (int a = 0; a < 3; ++a) {
                const float c = xyz[3 * (size_t)v + a];
                if (!isfinite(c)) ok = false;
                lo[a] = fminf(lo[a], c);
                hi[a] = fmaxf(hi[a], c);
            }
        }
        if (!ok) atomicOr(bad, 1u);
        for (int a = 0; a < 3; ++a) {
            tbox[6 * (size_t)t + a] = lo[a];
            tbox[6 * (size_t)t + 3 + a] = hi[a];
            if (ok) {
                mn[a] = mx[a] = ord(0.5f * lo[a] + 0.5f * hi[a]);
                mn[3 + a] = ord(lo[a]);
                mx[3 + a] = ord(hi[a]);
            }
        }
    }
    for (int a = 0; a < 6; ++a) { smin[a][threadIdx.x] = mn[a]; smax[a][threadIdx.x] = mx[a]; }
    __syncthreads();
    for (int s = kBB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            for (int a = 0; a < 6; ++a) {
                smin[a][threadIdx.x] = min(smin[a][threadIdx.x], smin[a][threadIdx.x + s]);
                smax[a][threadIdx.x] = max(smax[a][threadIdx.x], smax[a][threadIdx.x + s]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 12) {
        const uint32_t j = threadIdx.x, a = j % 3, q = j / 3;  // q: centre min, centre max, box min, box max
        const uint32_t v = (q & 1u) ? smax[(q >> 1) * 3 + a][0] : smin[(q >> 1) * 3 + a][0];
        part[(size_t)blockIdx.x * 12 + j] = v;
    }
}

// One block: the per-block bounds of k_tri_boxes into cb[0..11].
__global__ __launch_bounds__(kBB) void k_bounds(const uint32_t *part, uint32_t nblocks, uint32_t *cb)
{
    __shared__ uint32_t red[12][kBB];
    uint32_t v[12];
    for (int j = 0; j < 12; ++j) v[j] = ((j / 3) & 1) ? 0u : 0xffffffffu;
    for (uint32_t b = threadIdx.x; b < nblocks; b += kBB)
        for (int j = 0; j < 12; ++j) {
            const uint32_t x = part[(size_t)b * 12 + j];
            v[j] = ((j / 3) & 1) ? max(v[j], x) : min(v[j], x);
        }
    for (int j = 0; j < 12; ++j) red[j][threadIdx.x] = v[j];
    __syncthreads();
    for (int st = kBB / 2; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st)
            for (int j = 0; j < 12; ++j) {
                const uint32_t x = red[j][threadIdx.x + st];
                red[j][threadIdx.x] = ((j / 3) & 1) ? max(red[j][threadIdx.x], x) : min(red[j][threadIdx.x], x);
            }
        __syncthreads();
    }
    if (threadIdx.x < 12) cb[threadIdx.x] = red[threadIdx.x][0];
}

// Outward padding of every child box, the host build's rule: 2^-19 of
// (scene diagonal + largest |coordinate|) per side, so the FP32 slab test is
// conservative with respect to the watertight triangle test.
__host__ __device__ inline float box_pad(const float lo[3], const float hi[3])
{
    double diag = 0.0, amax = 0.0;
    for (int k = 0; k < 3; ++k) {
        diag += ((double)hi[k] - lo[k]) * ((double)hi[k] - lo[k]);
        const double m = fabs((double)lo[k]) > fabs((double)hi[k]) ? fabs((double)lo[k]) : fabs((double)hi[k]);
        amax = amax > m ? amax : m;
    }
    return (float)((sqrt(diag) + amax) * ldexp(1.0, -19));
}

__device__ inline float scene_pad(const uint32_t *cb)
{
    float lo[3], hi[3];
    for (int a = 0; a < 3; ++a) { lo[a] = unord(cb[6 + a]); hi[a] = unord(cb[9 + a]); }
    return box_pad(lo, hi);
}

__global__ __launch_bounds__(kBB) void k_morton(const float *tbox, uint32_t nt, const uint32_t *cb, uint32_t *key,
                                                uint32_t *val)
{
    const uint32_t t = blockIdx.x * kBB + threadIdx.x;
    if (t >= nt) return;
    uint32_t q[3];
    for (int a = 0; a < 3; ++a) {
        const float lo = unord(cb[a]), hi = unord(cb[3 + a]);
        const float c = 0.5f * tbox[6 * (size_t)t + a] + 0.5f * tbox[6 * (size_t)t + 3 + a];
        const float ext = hi - lo;
        float u = ext > 0.0f ? (c - lo) / ext * 1024.0f : 0.0f;
        u = u > 0.0f ? (u < 1023.0f ? u : 1023.0f) : 0.0f;  // NaN -> 0
        q[a] = (uint32_t)u;
    }
    key[t] = spread10(q[0]) << 2 | spread10(q[1]) << 1 | spread10(q[2]);
    val[t] = t;
}

// Common-prefix length of sorted codes i and j (equal codes: 32 + the
// common prefix of the indices); -1 outside [0, n).
__device__ inline int prefix(const uint32_t *key, int64_t n, int64_t i, int64_t j)
{
    if (j < 0 || j >= n) return -1;
    const uint32_t a = key[i], b = key[j];
    if (a != b) return __clz(a ^ b);
    return 32 + __clz((uint32_t)i ^ (uint32_t)j);
}

// encode_leaf of rt_internal.h for device code: ~(first << 3 | count - 1).
__device__ inline int32_t leaf_ref(uint32_t first, uint32_t count)
{
    return (int32_t)~((first << kLeafCountBits) | (count - 1u));
}

// Child reference: internal node c, or leaf (sorted position) c | kLeafBit.
constexpr uint32_t kLeafBit = 0x80000000u;
constexpr uint32_t kNotReady = 0xffffffffu;  // pass index of a node not computed yet

__global__ __launch_bounds__(kBB) void k_radix_tree(const uint32_t *key, uint32_t n, uint32_t *child, uint32_t *lo,
                                                    uint32_t *hi, uint32_t *parent)
{
    const int64_t i = (int64_t)blockIdx.x * kBB + threadIdx.x;
    const int64_t N = n;
    if (i >= N - 1) return;
    const int d = prefix(key, N, i, i + 1) - prefix(key, N, i, i - 1) >= 0 ? 1 : -1;
    const int dmin = prefix(key, N, i, i - d);
    int64_t lmax = 2;
    while (prefix(key, N, i, i + lmax * d) > dmin) lmax <<= 1;
    int64_t l = 0;
    for (int64_t t = lmax >> 1; t >= 1; t >>= 1)
        if (prefix(key, N, i, i + (l + t) * d) > dmin) l += t;
    const int64_t j = i + l * d;
    const int dnode = prefix(key, N, i, j);
    int64_t s = 0;
    for (int64_t div = 2;; div <<= 1) {
        const int64_t t = (l + div - 1) / div;
        if (prefix(key, N, i, i + (s + t) * d) > dnode) s += t;
        if (t <= 1) break;
    }
    const int64_t g = i + s * d + (d < 0 ? -1 : 0);
    const uint32_t a = (uint32_t)(i < j ? i : j), b = (uint32_t)(i < j ? j : i);
    const uint32_t c0 = (a == (uint32_t)g) ? ((uint32_t)g | kLeafBit) : (uint32_t)g;
    const uint32_t c1 = (b == (uint32_t)g + 1) ? ((uint32_t)(g + 1) | kLeafBit) : (uint32_t)(g + 1);
    child[2 * i] = c0;
    child[2 * i + 1] = c1;
    lo[i] = a;
    hi[i] = b;
    // parents: internal nodes at [0, n-1), leaves at [n-1, 2n-1)
    parent[(c0 & kLeafBit) ? (N - 1 + (c0 & ~kLeafBit)) : c0] = (uint32_t)i;
    parent[(c1 & kLeafBit) ? (N - 1 + (c1 & ~kLeafBit)) : c1] = (uint32_t)i;
}

__device__ inline double area6(const float b[6])
{
    double d[3];
    for (int a = 0; a < 3; ++a) d[a] = fmax(0.0, (double)b[3 + a] - (double)b[a]);
    return 2.0 * (d[0] * d[1] + d[1] * d[2] + d[2] * d[0]);
}

// A subtree's box, SAH cost and kept height.
struct NodeVal {
    float box[6];
    double cost;
    uint32_t height, leaf;
};

__device__ inline NodeVal leaf_val(const float *b)
{
    NodeVal v;
    for (int j = 0; j < 6; ++j) v.box[j] = b[j];
    v.cost = area6(v.box);
    v.height = 0;
    v.leaf = 0;
    return v;
}

// An internal node from its children: its box (their union), its SAH cost
// (cost of a triangle test 1, of a node visit trav_cost, per unit of area)
// and its choice: a node over at most max_leaf triangles becomes a leaf when
// (triangles x area) does not exceed (trav_cost x area + its children's
// costs); and the height of the kept tree below it (0 for a node that became
// a leaf).  The root (i = 0) never becomes a leaf.
__device__ inline NodeVal node_val(uint32_t i, uint32_t size, const NodeVal &c0, const NodeVal &c1, uint32_t max_leaf,
                                   double trav_cost)
{
    NodeVal v;
    for (int a = 0; a < 3; ++a) {
        v.box[a] = fminf(c0.box[a], c1.box[a]);
        v.box[3 + a] = fmaxf(c0.box[3 + a], c1.box[3 + a]);
    }
    const double area = area6(v.box);
    const double split = trav_cost * area + c0.cost + c1.cost;
    const double as_leaf = (double)size * area;
    const bool leaf = i != 0 && size <= max_leaf && as_leaf <= split;
    v.cost = leaf ? as_leaf : split;
    v.height = leaf ? 0u : 1u + (c0.height > c1.height ? c0.height : c1.height);
    v.leaf = leaf ? 1u : 0u;
    return v;
}

// Bottom-up boxes and SAH costs, in two parts.  A block takes kRun
// consecutive leaves and every internal node whose range lies inside them (a
// radix-tree node's own number is one end of its range, so these nodes are
// numbered within the run), and computes them in LDS, round by round, each
// node once its children are done.  The nodes whose range crosses the end of a
// run -- a few thousand above 1M triangles -- go onto a list for k_node_pass.
// At 2^20 triangles: 63 us here (bound by the reads and writes of ~90 B per
// triangle) and 24 passes of 4.9 us over the list, launch-bound, in place of
// 32 passes over every node with a look from the host after each 8.
constexpr uint32_t kRun = 512;
struct RunLds {
    float lbox[kRun][6], nbox[kRun][6];
    double cost[kRun];
    uint8_t height[kRun], leaf[kRun], done[kRun];
    uint32_t ntop, top0;
};

__global__ __launch_bounds__(kBB) void k_node_runs(const uint32_t *child, const uint32_t *lo, const uint32_t *hi,
                                                   const float *tbox, const uint32_t *val, uint32_t n,
                                                   uint32_t max_leaf, double trav_cost, float *nbox, double *cost,
                                                   uint32_t *height, uint32_t *leafc, uint32_t *ready, uint32_t *top,
                                                   uint32_t *ntop)
{
    __shared__ RunLds r;
    constexpr uint32_t kPer = kRun / kBB;
    const uint32_t b0 = blockIdx.x * kRun, b1 = min(b0 + kRun, n);  // leaves [b0, b1)
    uint32_t c0[kPer], c1[kPer], size[kPer];
    bool mine[kPer];
    if (threadIdx.x == 0) r.ntop = 0;
    for (uint32_t k = 0; k < kPer; ++k) {
        const uint32_t t = threadIdx.x + k * kBB, i = b0 + t;
        r.done[t] = 0;
        mine[k] = false;
        if (i < b1) {
            const float *src = tbox + 6 * (size_t)val[i];
            for (int j = 0; j < 6; ++j) r.lbox[t][j] = src[j];
        }
        if (i < n - 1) {
            const uint32_t l = lo[i], h = hi[i];
            mine[k] = l >= b0 && h < b1;
            c0[k] = child[2 * (size_t)i];
            c1[k] = child[2 * (size_t)i + 1];
            size[k] = h - l + 1;
        }
    }
    __syncthreads();
    uint32_t at[kPer];
    for (uint32_t k = 0; k < kPer; ++k) {
        const uint32_t i = b0 + threadIdx.x + k * kBB;
        at[k] = 0;
        if (i < n - 1 && !mine[k]) at[k] = atomicAdd(&r.ntop, 1u);
    }
    auto of = [&](uint32_t c) {
        const uint32_t t = (c & ~kLeafBit) - b0;
        if (c & kLeafBit) return leaf_val(r.lbox[t]);
        NodeVal v;
        for (int j = 0; j < 6; ++j) v.box[j] = r.nbox[t][j];
        v.cost = r.cost[t];
        v.height = r.height[t];
        v.leaf = r.leaf[t];
        return v;
    };
    auto is_done = [&](uint32_t c) { return (c & kLeafBit) || r.done[(c & ~kLeafBit) - b0]; };
    bool left[kPer];
    for (uint32_t k = 0; k < kPer; ++k) left[k] = mine[k];
    for (;;) {
        // every turn finishes at least the lowest nodes left, so the loop ends
        bool now[kPer], any = false;
        for (uint32_t k = 0; k < kPer; ++k) {
            now[k] = left[k] && is_done(c0[k]) && is_done(c1[k]);
            any = any || left[k];
        }
        if (!__syncthreads_or(any)) break;
        for (uint32_t k = 0; k < kPer; ++k) {
            if (!now[k]) continue;
            const uint32_t t = threadIdx.x + k * kBB;
            const NodeVal v = node_val(b0 + t, size[k], of(c0[k]), of(c1[k]), max_leaf, trav_cost);
            for (int j = 0; j < 6; ++j) r.nbox[t][j] = v.box[j];
            r.cost[t] = v.cost;
            r.height[t] = (uint8_t)v.height;
            r.leaf[t] = (uint8_t)v.leaf;
            left[k] = false;
        }
        __syncthreads();
        for (uint32_t k = 0; k < kPer; ++k)
            if (now[k]) r.done[threadIdx.x + k * kBB] = 1;
        __syncthreads();
    }
    if (threadIdx.x == 0) r.top0 = r.ntop ? atomicAdd(ntop, r.ntop) : 0u;
    __syncthreads();
    for (uint32_t k = 0; k < kPer; ++k) {
        const uint32_t t = threadIdx.x + k * kBB, i = b0 + t;
        if (i >= n - 1) continue;
        if (mine[k]) {
            for (int j = 0; j < 6; ++j) nbox[6 * (size_t)i + j] = r.nbox[t][j];
            cost[i] = r.cost[t];
            height[i] = r.height[t];
            leafc[i] = r.leaf[t];
            ready[i] = 0;
        } else {
            ready[i] = kNotReady;
            top[r.top0 + at[k]] = i;
        }
    }
}

// The nodes of the list, in passes: pass p computes every one whose children
// are leaves or were computed earlier (ready[c] < p).  All it reads was
// written by earlier launches, so no fence or coherent load is needed.
__global__ __launch_bounds__(kBB) void k_node_pass(const uint32_t *child, const uint32_t *lo, const uint32_t *hi,
                                                   const float *tbox, const uint32_t *val, const uint32_t *top,
                                                   const uint32_t *ntop, uint32_t pass, uint32_t max_leaf,
                                                   double trav_cost, float *nbox, double *cost, uint32_t *height,
                                                   uint32_t *leafc, uint32_t *ready)
{
    const uint32_t m = *ntop;
    for (uint32_t t = blockIdx.x * kBB + threadIdx.x; t < m; t += gridDim.x * kBB) {
        const uint32_t i = top[t];
        if (ready[i] != kNotReady) continue;
        const uint32_t c[2] = {child[2 * (size_t)i], child[2 * (size_t)i + 1]};
        bool ok = true;
        for (int k = 0; k < 2; ++k)
            if (!(c[k] & kLeafBit) && !(ready[c[k]] < pass)) ok = false;
        if (!ok) continue;
        auto of = [&](uint32_t ch) {
            if (ch & kLeafBit) return leaf_val(tbox + 6 * (size_t)val[ch & ~kLeafBit]);
            NodeVal v;
            for (int j = 0; j < 6; ++j) v.box[j] = nbox[6 * (size_t)ch + j];
            v.cost = cost[ch];
            v.height = height[ch];
            v.leaf = leafc[ch];
            return v;
        };
        const NodeVal v = node_val(i, hi[i] - lo[i] + 1, of(c[0]), of(c[1]), max_leaf, trav_cost);
        for (int j = 0; j < 6; ++j) nbox[6 * (size_t)i + j] = v.box[j];
        cost[i] = v.cost;
        height[i] = v.height;
        leafc[i] = v.leaf;
        ready[i] = pass;
    }
}

// Kept internal nodes: the root, and every node neither of whose own
// choice nor any ancestor's choice was a leaf (only nodes over at most
// max_leaf triangles choose; the walk up stops at the first larger one).
__global__ __launch_bounds__(kBB) void k_keep(const uint32_t *lo, const uint32_t *hi, const uint32_t *parent,
                                              const uint32_t *leafc, uint32_t n, uint32_t max_leaf, uint32_t *keep)
{
    const uint32_t i = blockIdx.x * kBB + threadIdx.x;
    if (i >= n - 1) return;
    uint32_t k = 1;
    if (i != 0) {
        if (leafc[i]) {
            k = 0;
        } else {
            for (uint32_t p = parent[i]; p != 0 && hi[p] - lo[p] + 1 <= max_leaf; p = parent[p])
                if (leafc[p]) { k = 0; break; }
        }
    }
    keep[i] = k;
}

// Node2 record of each kept node, its children as node indices or leaf
// ranges and their boxes padded outward; SAH terms (1.2 * area of an
// internal node, count * area of a leaf, unpadded, as the host build sums
// them) added per block into *sah.
__global__ __launch_bounds__(kBB) void k_emit_node2(const uint32_t *child, const uint32_t *lo, const uint32_t *hi,
                                                    const uint32_t *keep, const uint32_t *newidx, const float *tbox,
                                                    const uint32_t *val, const float *nbox, uint32_t n,
                                                    const uint32_t *cb, Node2 *nodes, double *sah)
{
    __shared__ double part[kBB];
    double acc = 0.0;
    const float pad = scene_pad(cb);
    for (uint32_t i = blockIdx.x * kBB + threadIdx.x; i < n - 1; i += gridDim.x * kBB) {
        if (!keep[i]) continue;
        Node2 nd{};
        float bx[2][6];
        for (int c = 0; c < 2; ++c) {
            const uint32_t ch = child[2 * i + c];
            int32_t ref;
            if (ch & kLeafBit) {
                const uint32_t pos = ch & ~kLeafBit;
                const float *src = tbox + 6 * (size_t)val[pos];
                for (int k = 0; k < 6; ++k) bx[c][k] = src[k];
                ref = leaf_ref(pos, 1);
                acc += area6(bx[c]);
            } else {
                for (int k = 0; k < 6; ++k) bx[c][k] = nbox[6 * (size_t)ch + k];
                if (keep[ch]) {
                    ref = (int32_t)newidx[ch];
                } else {
                    ref = leaf_ref(lo[ch], hi[ch] - lo[ch] + 1);
                    acc += (double)(hi[ch] - lo[ch] + 1) * area6(bx[c]);
                }
            }
            nd.child[c] = ref;
            for (int a = 0; a < 3; ++a) { bx[c][a] -= pad; bx[c][3 + a] += pad; }
        }
        nd.f[0] = bx[0][0]; nd.f[1] = bx[0][3]; nd.f[2] = bx[0][1]; nd.f[3] = bx[0][4];
        nd.f[4] = bx[1][0]; nd.f[5] = bx[1][3]; nd.f[6] = bx[1][1]; nd.f[7] = bx[1][4];
        nd.f[8] = bx[0][2]; nd.f[9] = bx[0][5]; nd.f[10] = bx[1][2]; nd.f[11] = bx[1][5];
        nodes[newidx[i]] = nd;
        float own[6];
        for (int k = 0; k < 6; ++k) own[k] = nbox[6 * (size_t)i + k];
        acc += 1.2 * area6(own);
    }
    part[threadIdx.x] = acc;
    __syncthreads();
    for (int s = kBB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0 && part[0] != 0.0) atomicAdd(sah, part[0]);
}

// Triangles in code order (leaf order) and the degenerate sentinel after
// them.  An index past the vertices (the build then fails) reads vertex 0.
__global__ __launch_bounds__(kBB) void k_emit_tris(const float *xyz, uint32_t nv, const uint32_t *idx,
                                                   const uint32_t *val, uint32_t n, Tri3 *tris)
{
    const uint32_t k = blockIdx.x * kBB + threadIdx.x;
    if (k > n) return;
    Tri3 t{};
    if (k == n) {
        t.id = -1;
    } else {
        const uint32_t tri = val[k];
        const float *v[3];
        for (int c = 0; c < 3; ++c) {
            const uint32_t vi = idx[3 * (size_t)tri + c];
            v[c] = xyz + 3 * (size_t)(vi < nv ? vi : 0u);
        }
        for (int a = 0; a < 3; ++a) { t.v0[a] = v[0][a]; t.v1[a] = v[1][a]; t.v2[a] = v[2][a]; }
        t.id = (int32_t)tri;
    }
    tris[k] = t;
}

// ---- four-wide collapse (bvh_build.cpp's Collapser, level by level) ----
struct Kid {
    float lo[3], hi[3];
    int32_t ref;
};

__device__ inline double kid_area(const Kid &k)
{
    double d[3];
    for (int a = 0; a < 3; ++a) d[a] = fmax(0.0, (double)k.hi[a] - (double)k.lo[a]);
    return 2.0 * (d[0] * d[1] + d[1] * d[2] + d[2] * d[0]);
}

__device__ inline void node2_kids(const Node2 &n, Kid &k0, Kid &k1)
{
    k0.lo[0] = n.f[0]; k0.hi[0] = n.f[1]; k0.lo[1] = n.f[2]; k0.hi[1] = n.f[3]; k0.lo[2] = n.f[8]; k0.hi[2] = n.f[9];
    k1.lo[0] = n.f[4]; k1.hi[0] = n.f[5]; k1.lo[1] = n.f[6]; k1.hi[1] = n.f[7]; k1.lo[2] = n.f[10]; k1.hi[2] = n.f[11];
    k0.ref = n.child[0];
    k1.ref = n.child[1];
}

// Smallest e >= -126 with 255 * 2^e >= extent: with extent = m * 2^k, m in
// [0.5, 1), 2^(k - 8) is enough up to m = 255/256 and 2^(k - 9) never is.
__device__ inline int scale_exponent(double extent)
{
    if (!(extent > 0.0)) return -126;
    int k;
    const double m = frexp(extent, &k);
    return max(-126, k - 8 + (m > 255.0 / 256.0 ? 1 : 0));
}

// The kids of a wide node: its two-wide node's two children, then the
// internal kid of largest surface area is opened (replaced by its two
// children) until there are four or none is internal.  Returns how many.
// Every index is a constant after unrolling, so the kids stay in registers:
// indexed by the kid opened they lay in 128 bytes of scratch memory, and the
// levels of 2^20 triangles took 0.42 ms against 0.24.
__device__ inline uint32_t open_kids(const Node2 *n2, uint32_t src, Kid kids[4])
{
    node2_kids(n2[src], kids[0], kids[1]);
    kids[2] = kids[3] = Kid{};
    kids[2].ref = kids[3].ref = -1;
    uint32_t nk = 2;
#pragma unroll
    for (int m = 2; m < 4; ++m) {
        int best = -1;
        int32_t ref = -1;
        double best_area = -1.0;
#pragma unroll
        for (int i = 0; i < m; ++i) {
            const double area = kid_area(kids[i]);
            if (kids[i].ref >= 0 && area > best_area) {
                best_area = area;
                best = i;
                ref = kids[i].ref;
            }
        }
        if (best < 0) break;
        Kid a;
        node2_kids(n2[ref], a, kids[m]);
#pragma unroll
        for (int i = 0; i < m; ++i)
            if (i == best) kids[i] = a;
        nk = m + 1;
    }
    return nk;
}

// The collapse's levels.  A level's figures are written on the device by the
// level before it, so the levels are launched one after the other without a
// look from the host; levels past the last find nothing to do.  At 2^20
// triangles (12 levels) this takes 0.24 ms, where a scan's launches, two
// copies and a wait per level took 1.3; the small levels are launch-bound
// (4-5 us each), the large ones wait on the gathers of two-wide nodes.
struct Level {
    uint32_t nfront, base;  // frontier entries, and the first one's wide node
};

// The frontier entries of a block of a level: contiguous, whole tiles.
__device__ inline void level_share(uint32_t nfront, uint32_t &f0, uint32_t &f1)
{
    const uint32_t tiles = (nfront + kBB - 1) / kBB, per = (tiles + gridDim.x - 1) / gridDim.x;
    f0 = min(blockIdx.x * per * kBB, nfront);
    f1 = min(f0 + per * kBB, nfront);
}

// One level, first pass: internal kids per frontier entry and per block.
__global__ __launch_bounds__(kBB) void k_collapse4_count(const Node2 *n2, const uint2 *front, const Level *level,
                                                         uint32_t *cnt, uint32_t *bsum)
{
    __shared__ uint32_t red[kBB];
    uint32_t f0, f1, sum = 0;
    level_share(level->nfront, f0, f1);
    for (uint32_t f = f0 + threadIdx.x; f < f1; f += kBB) {
        Kid kids[4];
        open_kids(n2, front[f].x, kids);
        uint32_t ni = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) ni += kids[i].ref >= 0 ? 1u : 0u;
        cnt[f] = ni;
        sum += ni;
    }
    red[threadIdx.x] = sum;
    __syncthreads();
    for (int s = kBB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) bsum[blockIdx.x] = red[0];
}

__device__ void collapse_entry(const Node2 *n2, const uint2 *front, uint32_t f, uint32_t nfront, uint32_t q,
                               uint32_t base, uint32_t sentinel, Node4 *n4, uint2 *next, uint32_t &need);

// One level, second pass: the entries' offsets from the blocks' sums and a
// prefix sum per tile; the last block writes the next level's figures.
__global__ __launch_bounds__(kBB) void k_collapse4(const Node2 *n2, const uint2 *front, Level *level,
                                                   const uint32_t *cnt, const uint32_t *bsum, uint32_t sentinel,
                                                   Node4 *n4, uint2 *next, uint32_t *need)
{
    __shared__ uint32_t sc[kBB];
    const Level lv = *level;
    uint32_t before = 0;
    for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kBB) before += bsum[b];
    sc[threadIdx.x] = before;
    __syncthreads();
    for (int s = kBB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sc[threadIdx.x] += sc[threadIdx.x + s];
        __syncthreads();
    }
    uint32_t off = sc[0], most = 0;
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        level[1].nfront = off + bsum[blockIdx.x];
        level[1].base = lv.base + lv.nfront;
    }
    uint32_t f0, f1;
    level_share(lv.nfront, f0, f1);
    for (uint32_t t0 = f0; t0 < f1; t0 += kBB) {
        const uint32_t f = t0 + threadIdx.x;
        const uint32_t mine = f < f1 ? cnt[f] : 0u;
        __syncthreads();
        sc[threadIdx.x] = mine;
        __syncthreads();
        for (int s = 1; s < kBB; s <<= 1) {
            const uint32_t v = (int)threadIdx.x >= s ? sc[threadIdx.x - s] : 0u;
            __syncthreads();
            sc[threadIdx.x] += v;
            __syncthreads();
        }
        if (f < f1) collapse_entry(n2, front, f, lv.nfront, off + sc[threadIdx.x] - mine, lv.base, sentinel, n4, next, most);
        off += sc[kBB - 1];
    }
    for (int o = 32; o > 0; o >>= 1) most = max(most, (uint32_t)__shfl_xor((int)most, o));
    if ((threadIdx.x & 63u) == 0 && most) atomicMax(need, most);
}

// Frontier entry f (two-wide node, pending entries above it) becomes wide
// node base + f; its internal kids, in slot order, become next-level entries
// q, q + 1, ... and wide nodes base + nfront + q + j.  The numbering is
// breadth-first and does not depend on scheduling.  The four-wide traversal
// holds at most (pending above) + kids - 1 entries at a node, so the deepest
// such sum is its stack bound (need), the host collapse's figure.
__device__ void collapse_entry(const Node2 *n2, const uint2 *front, uint32_t f, uint32_t nfront, uint32_t q,
                               uint32_t base, uint32_t sentinel, Node4 *n4, uint2 *next, uint32_t &need)
{
    const uint2 fe = front[f];
    Kid kids[4];
    const uint32_t nk = open_kids(n2, fe.x, kids);
    const uint32_t pending = fe.y + nk - 1u;
    need = max(need, pending);
    int32_t refs[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        refs[i] = i < nk ? kids[i].ref : leaf_ref(sentinel, 1);
        if (kids[i].ref >= 0) {
            next[q] = make_uint2((uint32_t)kids[i].ref, pending);
            refs[i] = (int32_t)(base + nfront + q);
            ++q;
        }
    }
    Node4 n{};
    uint32_t meta = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float p = kids[0].lo[a];
#pragma unroll
        for (uint32_t i = 1; i < 4; ++i)
            if (i < nk) p = fminf(p, kids[i].lo[a]);
        double ext = 0.0;
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
            if (i < nk) ext = fmax(ext, (double)kids[i].hi[a] - (double)p);
        const int e = min(scale_exponent(ext), kMaxScaleExp);
        const double sc = ldexp(1.0, e), inv = ldexp(1.0, -e);  // x * inv is x / sc exactly
        n.origin[a] = ext > 255.0 * sc ? __builtin_nanf("") : p;
        meta |= (uint32_t)(e + 127) << (8 * a);
        uint32_t qlo = 0, qhi = 0;
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            if (i >= nk) {
                qlo |= 255u << (8 * i);
                continue;
            }
            double l = floor(((double)kids[i].lo[a] - (double)p) * inv);
            double h = ceil(((double)kids[i].hi[a] - (double)p) * inv);
            l = fmin(fmax(l, 0.0), 255.0);
            h = fmin(fmax(h, 0.0), 255.0);
            while (l > 0.0 && (double)p + l * sc > (double)kids[i].lo[a]) l -= 1.0;
            while (h < 255.0 && (double)p + h * sc < (double)kids[i].hi[a]) h += 1.0;
            qlo |= (uint32_t)l << (8 * i);
            qhi |= (uint32_t)h << (8 * i);
        }
        n.q[2 * a] = qlo;
        n.q[2 * a + 1] = qhi;
    }
    meta |= (uint32_t)((1u << nk) - 1u) << 24;
    n.meta = meta;
    for (int i = 0; i < 4; ++i) n.child[i] = refs[i];
    n4[base + f] = n;
}

// What the host reads back from a build: gathered, so that it is one copy.
struct BuildInfo {
    uint32_t nodes, bad, height;
    float root_box[6];
};

__global__ void k_build_info(const uint32_t *last_idx, const uint32_t *last_keep, const uint32_t *bad,
                             const uint32_t *height, const float *nbox, BuildInfo *out)
{
    if (threadIdx.x != 0) return;
    BuildInfo in;
    in.nodes = *last_idx + *last_keep;
    in.bad = *bad;
    in.height = *height;
    for (int j = 0; j < 6; ++j) in.root_box[j] = nbox[j];
    *out = in;
}

constexpr uint32_t kLevels = 16, kMaxLevels = 64;
constexpr unsigned kCollapseBlocks = 512;
constexpr unsigned kEmitBlocks = 1024;  // each ends in one atomic on the SAH sum
struct CollapseState {
    Level level[kMaxLevels + 1];
    uint32_t need;
};

// The root's frontier entry and the level table's start.
__global__ void k_collapse4_begin(uint2 *front, CollapseState *st)
{
    for (uint32_t l = threadIdx.x; l <= kMaxLevels; l += blockDim.x) st->level[l] = Level{l == 0 ? 1u : 0u, 0u};
    if (threadIdx.x == 0) {
        front[0] = make_uint2(0u, 0u);
        st->need = 0;
    }
}

struct BuildReadback {
    uint32_t root_ready;
    BuildInfo info;
    double sah;
    CollapseState collapse;
};
static_assert(sizeof(BuildReadback) <= BvhBuildSpace::kPinned, "the pinned block holds every read-back");

unsigned blocks(uint64_t n) { return (unsigned)std::max<uint64_t>(1, (n + kBB - 1) / kBB); }

}  // namespace

hipError_t build_bvh_device(const float *xyz, uint32_t nv, const uint32_t *idx, uint32_t nt, const rt_bvh_opts &o,
                            hipStream_t s, BvhBuildSpace &space, size_t extra, DeviceBvhBuild &out, std::string &err)
{
    const auto t0 = std::chrono::steady_clock::now();
    out = DeviceBvhBuild{};
    const uint32_t max_leaf = o.max_leaf ? o.max_leaf : 4;  // 1..kMaxLeafCount, checked by the caller
    const bool wide = o.width != 2;
    hipError_t e = hipSuccess;
    auto fail = [&](hipError_t x, const char *what) {
        err = std::string("rt_bvh_build_device: ") + what + ": " + hipGetErrorString(x);
        return x;
    };
    // outputs: `nodes` two-wide nodes, as many wide nodes (each takes at least
    // one two-wide node of its own), triangles + sentinel and the caller's
    // `extra` bytes, in one allocation
    auto allocate = [&](uint32_t nodes) {
        const size_t o4 = (size_t)nodes * sizeof(Node2), ot = o4 + (wide ? (size_t)nodes * sizeof(Node4) : 0);
        const size_t ox = (ot + ((size_t)nt + 1) * sizeof(Tri3) + 255) & ~(size_t)255;
        char *m = nullptr;
        const hipError_t x = hipMalloc(&m, ox + extra);
        if (x != hipSuccess) return x;
        out.nodes2 = (Node2 *)m;
        out.nodes4 = wide ? (Node4 *)(m + o4) : nullptr;
        out.tris = (Tri3 *)(m + ot);
        out.extra = m + ox;
        return x;
    };
    struct Trim {
        BvhBuildSpace &space;
        hipStream_t s;
        ~Trim() { space.trim(s); }
    } trim{space, s};
    out.num_tris = nt;
    if ((e = space.reserve_pinned()) != hipSuccess) return fail(e, "pinned read-back");
    BuildReadback &rb = *(BuildReadback *)space.pinned;
    rb = BuildReadback{};
    if (nt <= 1) {
        // one node on the host: the triangle (if any) and the sentinel
        std::vector<float> v(9, 0.0f);
        uint32_t ii[3] = {0, 0, 0};
        if (nt == 1) {
            if ((e = hipMemcpyAsync(ii, idx, 12, hipMemcpyDeviceToHost, s)) != hipSuccess ||
                (e = hipStreamSynchronize(s)) != hipSuccess)
                return fail(e, "input");
            for (int c = 0; c < 3; ++c) {
                if (ii[c] >= nv) { err = "rt_bvh_build_device: triangle index out of range"; return hipErrorInvalidValue; }
                if ((e = hipMemcpyAsync(&v[3 * c], xyz + 3 * (size_t)ii[c], 12, hipMemcpyDeviceToHost, s)) !=
                    hipSuccess)
                    return fail(e, "input");
            }
            if ((e = hipStreamSynchronize(s)) != hipSuccess) return fail(e, "input");
            for (float x : v)
                if (!std::isfinite(x)) { err = "rt_bvh_build_device: non-finite coordinate"; return hipErrorInvalidValue; }
        }
        Node2 root{};
        Tri3 tr[2]{};
        tr[0].id = nt ? 0 : -1;
        for (int a = 0; a < 3; ++a) { tr[0].v0[a] = v[a]; tr[0].v1[a] = v[3 + a]; tr[0].v2[a] = v[6 + a]; }
        tr[1].id = -1;
        float lo[3], hi[3];
        for (int a = 0; a < 3; ++a) {
            lo[a] = std::min({v[a], v[3 + a], v[6 + a]});
            hi[a] = std::max({v[a], v[3 + a], v[6 + a]});
        }
        double area = 0.0;
        if (nt == 1) {
            const double d[3] = {(double)hi[0] - lo[0], (double)hi[1] - lo[1], (double)hi[2] - lo[2]};
            area = d[0] * d[1] + d[1] * d[2] + d[2] * d[0];
            const float pad = box_pad(lo, hi);
            for (int a = 0; a < 3; ++a) { lo[a] -= pad; hi[a] += pad; }
        } else {
            for (int a = 0; a < 3; ++a) lo[a] = hi[a] = 0.0f;
        }
        root.f[0] = lo[0]; root.f[1] = hi[0]; root.f[2] = lo[1]; root.f[3] = hi[1]; root.f[8] = lo[2]; root.f[9] = hi[2];
        root.child[0] = encode_leaf(nt ? 0u : nt, 1);
        root.child[1] = encode_leaf(nt, 1);
        if ((e = allocate(1)) != hipSuccess) return fail(e, "tree");
        if ((e = hipMemcpyAsync(out.nodes2, &root, sizeof root, hipMemcpyHostToDevice, s)) != hipSuccess ||
            (e = hipMemcpyAsync(out.tris, tr + (nt ? 0 : 1), (nt + 1) * sizeof(Tri3), hipMemcpyHostToDevice, s)) !=
                hipSuccess ||
            (e = hipStreamSynchronize(s)) != hipSuccess)
            return fail(e, "upload");
        out.num_nodes2 = 1;
        out.num_leaves = nt;
        out.max_depth = 1;
        out.sah_cost = area > 0.0 ? 1.0 : 0.0;
    } else {
        const size_t N = nt;
        const size_t nb = blocks(N);
        size_t off = 0;
        auto take = [&](size_t bytes) { size_t r = off; off += (bytes + 255) & ~(size_t)255; return r; };
        const size_t o_tbox = take(N * 24), o_cb = take(16 * 4), o_part = take(nb * 48), o_key = take(N * 4),
                     o_key2 = take(N * 4), o_val = take(N * 4), o_val2 = take(N * 4), o_child = take(2 * N * 4),
                     o_lo = take(N * 4), o_hi = take(N * 4), o_parent = take(2 * N * 4), o_nbox = take(N * 24),
                     o_cost = take(N * 8), o_height = take(N * 4), o_leafc = take(N * 4), o_ready = take(N * 4),
                     o_keep = take(N * 4), o_new = take(N * 4), o_top = take(N * 4);
        size_t sort_bytes = 0, scan_bytes = 0;
        if ((e = hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, (const uint32_t *)nullptr, (uint32_t *)nullptr,
                                                    (const uint32_t *)nullptr, (uint32_t *)nullptr, (int)N, 0, 30, s)) !=
                hipSuccess ||
            (e = hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, (const uint32_t *)nullptr, (uint32_t *)nullptr,
                                                  (int)(N - 1), s)) != hipSuccess)
            return fail(e, "sizing");
        const size_t o_tmp = take(std::max(sort_bytes, scan_bytes));
        if ((e = space.reserve(off, s)) != hipSuccess) return fail(e, "work space");
        char *b = (char *)space.dev;
        float *tbox = (float *)(b + o_tbox), *nbox = (float *)(b + o_nbox);
        // cb: centre and box bounds (12 words), the bad-input flag, then the
        // SAH sum (a double at word 14); word 13 the length of the top list
        uint32_t *cb = (uint32_t *)(b + o_cb), *bad = cb + 12, *ntop = cb + 13, *top = (uint32_t *)(b + o_top);
        double *sah = (double *)(cb + 14), *cost = (double *)(b + o_cost);
        uint32_t *part = (uint32_t *)(b + o_part), *key = (uint32_t *)(b + o_key), *key2 = (uint32_t *)(b + o_key2),
                 *val = (uint32_t *)(b + o_val), *val2 = (uint32_t *)(b + o_val2), *child = (uint32_t *)(b + o_child),
                 *lo = (uint32_t *)(b + o_lo), *hi = (uint32_t *)(b + o_hi), *parent = (uint32_t *)(b + o_parent),
                 *height = (uint32_t *)(b + o_height), *leafc = (uint32_t *)(b + o_leafc),
                 *ready = (uint32_t *)(b + o_ready), *keep = (uint32_t *)(b + o_keep), *newidx = (uint32_t *)(b + o_new);
        if ((e = hipMemsetAsync(cb, 0, 16 * 4, s)) != hipSuccess) return fail(e, "clear");
        const double trav_cost = o.trav_cost > 0 ? o.trav_cost : 1.2f;
        hipLaunchKernelGGL(k_tri_boxes, dim3(nb), dim3(kBB), 0, s, xyz, nv, idx, nt, tbox, part, bad);
        hipLaunchKernelGGL(k_bounds, dim3(1), dim3(kBB), 0, s, part, (uint32_t)nb, cb);
        hipLaunchKernelGGL(k_morton, dim3(nb), dim3(kBB), 0, s, tbox, nt, cb, key, val);
        if ((e = hipGetLastError()) != hipSuccess) return fail(e, "boxes");
        if ((e = hipcub::DeviceRadixSort::SortPairs(b + o_tmp, sort_bytes, key, key2, val, val2, (int)N, 0, 30, s)) !=
            hipSuccess)
            return fail(e, "sort");
        hipLaunchKernelGGL(k_radix_tree, dim3(blocks(N - 1)), dim3(kBB), 0, s, key2, nt, child, lo, hi, parent);
        if ((e = hipGetLastError()) != hipSuccess) return fail(e, "radix tree");
        hipLaunchKernelGGL(k_node_runs, dim3((unsigned)((N + kRun - 1) / kRun)), dim3(kBB), 0, s, child, lo, hi, tbox,
                           val2, nt, max_leaf, trav_cost, nbox, cost, height, leafc, ready, top, ntop);
        // passes over the rest until the root is done: its `ready` word is read
        // back after 24 and then every 8 (a look costs as much as 6 passes).  A radix tree of 30-bit codes split further by 32-bit positions
        // is at most 62 high
        uint32_t pass = 0;
        rb.root_ready = nt > kRun ? kNotReady : 0u;
        while (rb.root_ready == kNotReady) {
            if (pass >= 64) {
                err = "rt_bvh_build_device: radix tree higher than 64 levels";
                return hipErrorUnknown;
            }
            for (int k = pass ? 8 : 24; k > 0; --k) {
                ++pass;
                hipLaunchKernelGGL(k_node_pass, dim3(std::min(blocks(N), 64u)), dim3(kBB), 0, s, child, lo, hi, tbox,
                                   val2, top, ntop, pass, max_leaf, trav_cost, nbox, cost, height, leafc, ready);
            }
            if ((e = hipGetLastError()) != hipSuccess ||
                (e = hipMemcpyAsync(&rb.root_ready, ready, 4, hipMemcpyDeviceToHost, s)) != hipSuccess ||
                (e = hipStreamSynchronize(s)) != hipSuccess)
                return fail(e, "boxes");
        }
        hipLaunchKernelGGL(k_keep, dim3(blocks(N - 1)), dim3(kBB), 0, s, lo, hi, parent, leafc, nt, max_leaf, keep);
        if ((e = hipGetLastError()) != hipSuccess) return fail(e, "collapse");
        if ((e = hipcub::DeviceScan::ExclusiveSum(b + o_tmp, scan_bytes, keep, newidx, (int)(N - 1), s)) != hipSuccess)
            return fail(e, "scan");
        hipLaunchKernelGGL(k_build_info, dim3(1), dim3(64), 0, s, newidx + (N - 2), keep + (N - 2), bad, height, nbox,
                           (BuildInfo *)(b + o_part));
        if ((e = hipGetLastError()) != hipSuccess ||
            (e = hipMemcpyAsync(&rb.info, b + o_part, sizeof(BuildInfo), hipMemcpyDeviceToHost, s)) != hipSuccess ||
            (e = hipStreamSynchronize(s)) != hipSuccess)
            return fail(e, "read-back");
        const BuildInfo &in = rb.info;
        if (in.bad) { err = "rt_bvh_build_device: triangle index out of range or non-finite coordinate"; return hipErrorInvalidValue; }
        out.num_nodes2 = in.nodes;
        out.max_depth = in.height;
        if ((e = allocate(in.nodes)) != hipSuccess) return fail(e, "tree");
        hipLaunchKernelGGL(k_emit_node2, dim3(std::min(blocks(N - 1), kEmitBlocks)), dim3(kBB), 0, s, child, lo, hi, keep, newidx, tbox, val2,
                           nbox, nt, cb, out.nodes2, sah);
        hipLaunchKernelGGL(k_emit_tris, dim3(blocks(N + 1)), dim3(kBB), 0, s, xyz, nv, idx, val2, nt, out.tris);
        if ((e = hipGetLastError()) != hipSuccess ||
            (e = hipMemcpyAsync(&rb.sah, sah, 8, hipMemcpyDeviceToHost, s)) != hipSuccess)
            return fail(e, "emit");
        // a binary tree of m kept nodes has m + 1 leaves
        out.num_leaves = out.num_nodes2 + 1;
    }
    if (wide) {
        // level by level from the root, breadth-first numbering, kLevels of them
        // (each is two launches) before a look at how far it went, and no more
        // than the kept two-wide tree has (a wide level takes one or more of
        // them); num_nodes2 bounds any level's frontier
        const uint32_t cap4 = out.num_nodes2;
        const unsigned grid = std::min(blocks(cap4), kCollapseBlocks);
        size_t off = 0;
        auto take = [&](size_t bytes) { size_t r = off; off += (bytes + 255) & ~(size_t)255; return r; };
        // (the build's own arrays are not read any more)
        const size_t o_f0 = take((size_t)cap4 * 8), o_f1 = take((size_t)cap4 * 8), o_cnt = take((size_t)cap4 * 4),
                     o_bsum = take(kCollapseBlocks * 4), o_lev = take(sizeof(CollapseState));
        if ((e = space.reserve(off, s)) != hipSuccess) return fail(e, "frontier");
        char *b = (char *)space.dev;
        uint2 *front[2] = {(uint2 *)(b + o_f0), (uint2 *)(b + o_f1)};
        uint32_t *cnt = (uint32_t *)(b + o_cnt), *bsum = (uint32_t *)(b + o_bsum);
        CollapseState *st = (CollapseState *)(b + o_lev);
        hipLaunchKernelGGL(k_collapse4_begin, dim3(1), dim3(64), 0, s, front[0], st);
        uint32_t level = 0;
        for (bool more = true; more;) {
            const uint32_t upto = std::min({level + kLevels, out.max_depth, kMaxLevels});
            if (level >= upto) {
                err = "rt_bvh_build_device: four-wide tree deeper than its two-wide tree can be";
                return hipErrorUnknown;
            }
            for (; level < upto; ++level) {
                const uint32_t cur = level & 1u;
                hipLaunchKernelGGL(k_collapse4_count, dim3(grid), dim3(kBB), 0, s, out.nodes2, front[cur],
                                   st->level + level, cnt, bsum);
                hipLaunchKernelGGL(k_collapse4, dim3(grid), dim3(kBB), 0, s, out.nodes2, front[cur], st->level + level,
                                   cnt, bsum, out.num_tris, out.nodes4, front[cur ^ 1u], &st->need);
            }
            if ((e = hipGetLastError()) != hipSuccess ||
                (e = hipMemcpyAsync(&rb.collapse, st, sizeof(CollapseState), hipMemcpyDeviceToHost, s)) != hipSuccess ||
                (e = hipStreamSynchronize(s)) != hipSuccess)
                return fail(e, "collapse");
            more = rb.collapse.level[level].nfront != 0;
        }
        uint32_t depth = 0;
        while (depth < level && rb.collapse.level[depth].nfront != 0) ++depth;
        out.num_nodes4 = rb.collapse.level[depth].base;
        out.depth4 = depth;
        out.max_stack4 = rb.collapse.need;
    }
    if (!wide && (e = hipStreamSynchronize(s)) != hipSuccess) return fail(e, "emit");
    if (nt > 1) {
        double d[3];
        for (int a = 0; a < 3; ++a)
            d[a] = std::max(0.0, (double)rb.info.root_box[3 + a] - (double)rb.info.root_box[a]);
        const double ra = 2.0 * (d[0] * d[1] + d[1] * d[2] + d[2] * d[0]);
        out.sah_cost = ra > 0 ? rb.sah / ra : 0.0;
    }
    out.build_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return hipSuccess;
}

namespace {
__global__ __launch_bounds__(kBB) void k_set_flags(Tri3 *tris, uint32_t n, const uint8_t *flags)
{
    const uint32_t k = blockIdx.x * kBB + threadIdx.x;
    if (k >= n) return;
    tris[k].flags = flags[tris[k].id] ? 1u : 0u;
}
}  // namespace

hipError_t set_transparent_device(Tri3 *tris, uint32_t n, const uint8_t *flags, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_set_flags, dim3(blocks(n)), dim3(kBB), 0, s, tris, n, flags);
    return hipGetLastError();
}

hipError_t BvhBuildSpace::reserve(size_t bytes, hipStream_t s)
{
    if (bytes <= cap) return hipSuccess;
    if (dev) {
        hipError_t e = hipStreamSynchronize(s);
        if (e != hipSuccess) return e;
        (void)hipFree(dev);
        dev = nullptr;
        cap = 0;
    }
    hipError_t e = hipMalloc(&dev, bytes);
    if (e != hipSuccess) dev = nullptr;
    else cap = bytes;
    return e;
}

hipError_t BvhBuildSpace::reserve_pinned()
{
    if (pinned) return hipSuccess;
    hipError_t e = hipHostMalloc(&pinned, kPinned, hipHostMallocDefault);
    if (e != hipSuccess) pinned = nullptr;
    return e;
}

void BvhBuildSpace::trim(hipStream_t s)
{
    if (cap <= kKeep) return;
    (void)hipStreamSynchronize(s);
    (void)hipFree(dev);
    dev = nullptr;
    cap = 0;
}

void BvhBuildSpace::release()
{
    if (dev) (void)hipFree(dev);
    if (pinned) (void)hipHostFree(pinned);
    dev = pinned = nullptr;
    cap = 0;
}

void free_bvh_device(DeviceBvhBuild &b)
{
    if (b.nodes2) (void)hipFree(b.nodes2);  // the whole tree's allocation
    b.nodes2 = nullptr;
    b.nodes4 = nullptr;
    b.tris = nullptr;
    b.extra = nullptr;
}

}  // namespace rt
