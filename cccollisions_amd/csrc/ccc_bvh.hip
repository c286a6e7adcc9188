// BVH construction for gfx950: leaf (swept) boxes + Morton codes, a stable LDS radix
// sort of (code, triangle id), the Karras radix tree and a bottom-up refit.
// Morton modes (per context): the reference's (infinite scene box: every code is 0, so the
// sort is the identity and is skipped), or a scene box fitted to the leaf boxes with 30-bit
// (10 bits per axis) or 63-bit (21 bits per axis) codes.
// Output is the reference wire format (src/build_bvh.cu:309-378):
//   bboxes [B, 2n-1, 6] (min xyz, max xyz), tree [B, 2n-1, 4] int64 (parent, left, right,
//   id), internal rows 0..n-2 (row 0 = root), leaf rows n-1..2n-2 in sorted order.
#include <float.h>

#include "ccc_geom.h"
#include "ccc_internal.h"

namespace ccc {

constexpr int kSortThreads = 256;
constexpr int kSortRounds = 8;
constexpr int kSortTile = kSortThreads * kSortRounds;

template <typename T> struct Lim;
template <> struct Lim<double> { static constexpr double max() { return DBL_MAX; } };
template <> struct Lim<float> { static constexpr float max() { return FLT_MAX; } };

// Spread the low 10 bits of v to every third bit (bit k -> bit 3k).
__device__ __forceinline__ uint32_t spread_bits10(uint32_t v) {
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// bvh.cu:54-62: each normalised coordinate is scaled by 1024, clamped to [0, 1023] with
// fmin/fmax (NaN -> 0) and truncated; code = x-bits * 4 + y-bits * 2 + z-bits.
__device__ __forceinline__ uint32_t morton30(double x, double y, double z) {
    x = fmin(fmax(x * 1024.0, 0.0), 1023.0);
    y = fmin(fmax(y * 1024.0, 0.0), 1023.0);
    z = fmin(fmax(z * 1024.0, 0.0), 1023.0);
    return spread_bits10((uint32_t)x) * 4u + spread_bits10((uint32_t)y) * 2u + spread_bits10((uint32_t)z);
}
__device__ __forceinline__ uint32_t morton30(float x, float y, float z) {
    x = fminf(fmaxf(x * 1024.0f, 0.0f), 1023.0f);
    y = fminf(fmaxf(y * 1024.0f, 0.0f), 1023.0f);
    z = fminf(fmaxf(z * 1024.0f, 0.0f), 1023.0f);
    return spread_bits10((uint32_t)x) * 4u + spread_bits10((uint32_t)y) * 2u + spread_bits10((uint32_t)z);
}

// 63-bit codes (not in the reference): 21 bits per axis, the same quantisation (scale by
// 2^21, clamp to [0, 2^21 - 1] with fmin/fmax, truncate) and interleave order.
__device__ __forceinline__ uint64_t spread_bits21(uint64_t v) {
    v &= 0x1fffffull;
    v = (v | (v << 32)) & 0x001f00000000ffffull;
    v = (v | (v << 16)) & 0x001f0000ff0000ffull;
    v = (v | (v << 8)) & 0x100f00f00f00f00full;
    v = (v | (v << 4)) & 0x10c30c30c30c30c3ull;
    v = (v | (v << 2)) & 0x1249249249249249ull;
    return v;
}
__device__ __forceinline__ uint64_t morton63(double x, double y, double z) {
    x = fmin(fmax(x * 2097152.0, 0.0), 2097151.0);
    y = fmin(fmax(y * 2097152.0, 0.0), 2097151.0);
    z = fmin(fmax(z * 2097152.0, 0.0), 2097151.0);
    return spread_bits21((uint64_t)x) * 4u + spread_bits21((uint64_t)y) * 2u + spread_bits21((uint64_t)z);
}
__device__ __forceinline__ uint64_t morton63(float x, float y, float z) {
    x = fminf(fmaxf(x * 2097152.0f, 0.0f), 2097151.0f);
    y = fminf(fmaxf(y * 2097152.0f, 0.0f), 2097151.0f);
    z = fminf(fmaxf(z * 2097152.0f, 0.0f), 2097151.0f);
    return spread_bits21((uint64_t)x) * 4u + spread_bits21((uint64_t)y) * 2u + spread_bits21((uint64_t)z);
}

// The box of triangle gi (build_bvh.cu:212-219, :452-460): of t0, or of t0 and t1 (MOTION).
template <typename T, bool MOTION>
__device__ __forceinline__ Box<T> leaf_box(const T *__restrict__ t0, const T *__restrict__ t1, int64_t gi, V3<T> *cent) {
    const T *a = t0 + 9 * gi;
    V3<T> a0 = ld3(a), a1 = ld3(a + 3), a2 = ld3(a + 6);
    Box<T> bx = tri_box(a0, a1, a2);
    V3<T> c = mk((a0.x + a1.x + a2.x) / (T)3.0, (a0.y + a1.y + a2.y) / (T)3.0, (a0.z + a1.z + a2.z) / (T)3.0);
    if (MOTION) {
        const T *b = t1 + 9 * gi;
        V3<T> b0 = ld3(b), b1 = ld3(b + 3), b2 = ld3(b + 6);
        bx = unite(bx, tri_box(b0, b1, b2));
        V3<T> c2 = mk((b0.x + b1.x + b2.x) / (T)3.0, (b0.y + b1.y + b2.y) / (T)3.0, (b0.z + b1.z + b2.z) / (T)3.0);
        c = mk((c.x + c2.x) / (T)2.0, (c.y + c2.y) / (T)2.0, (c.z + c2.z) / (T)2.0);
    }
    if (cent) *cent = c;
    return bx;
}

// Fitted modes: leaf boxes, the triangle ids in input order and the centroids the Morton
// codes are computed from (build_bvh.cu:26-71).
// The reference's scene box is the union of all leaf boxes with the reduction's initial
// value AABB<T>() = [-MAX, +MAX] (build_bvh.cu:243-244, :505-506; aabb.cu:25-33); min/max
// against +-MAX leave that initial value unchanged whatever the boxes are, so the scene box
// is [-MAX, +MAX], every normalised centroid is ~0.5 * 2^-1023 or smaller and every code is
// 0: the stable sort then keeps the input order, and the compat mode needs neither codes nor
// a sort (k_index_leaves).
template <typename T, bool MOTION>
__global__ void k_leaf_boxes(const T *__restrict__ t0, const T *__restrict__ t1, int64_t total,
                             int64_t n, T *__restrict__ boxes, T *__restrict__ cent,
                             int32_t *__restrict__ ids) {
    int64_t gi = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gi >= total) return;
    V3<T> c;
    const Box<T> bx = leaf_box<T, MOTION>(t0, t1, gi, &c);
    T *o = boxes + 6 * gi;
    o[0] = bx.mn.x; o[1] = bx.mn.y; o[2] = bx.mn.z; o[3] = bx.mx.x; o[4] = bx.mx.y; o[5] = bx.mx.z;
    T *q = cent + 3 * gi;
    q[0] = c.x; q[1] = c.y; q[2] = c.z;
    ids[gi] = (int32_t)(gi % n);
}

// Fitted scene box of each batch element: the union of its leaf boxes (min / max are exact
// and order-independent, NaN coordinates are ignored as by the leaf boxes' fmin / fmax).
// Stage 1: each block of element b reduces a strided share of its leaves to one box.
constexpr int kSceneBlocks = 64;
template <typename T>
__global__ __launch_bounds__(256) void k_scene_partial(const T *__restrict__ boxes_all, int64_t n, T *__restrict__ part_all) {
    __shared__ T red[6][256];
    const int b = blockIdx.y, tid = threadIdx.x;
    const T *boxes = boxes_all + (int64_t)b * n * 6;
    // the empty box (+inf, -inf) is the identity of the union
    const T inf = (T)INFINITY;
    T acc[6] = {inf, inf, inf, -inf, -inf, -inf};
    for (int64_t i = (int64_t)blockIdx.x * 256 + tid; i < n; i += (int64_t)gridDim.x * 256) {
        const T *p = boxes + 6 * i;
#pragma unroll
        for (int k = 0; k < 3; ++k) { acc[k] = tmin(acc[k], p[k]); acc[k + 3] = tmax(acc[k + 3], p[k + 3]); }
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) red[k][tid] = acc[k];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (tid < w) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                red[k][tid] = tmin(red[k][tid], red[k][tid + w]);
                red[k + 3][tid] = tmax(red[k + 3][tid], red[k + 3][tid + w]);
            }
        }
        __syncthreads();
    }
    if (tid < 6) part_all[((int64_t)b * gridDim.x + blockIdx.x) * 6 + tid] = red[tid][0];
}

// Stage 2 and the codes: one block per batch element unions the partial boxes, then every
// leaf's centroid is normalised by the scene box and quantised (bvh.cu:54-62; NaN -> 0).
template <typename T, typename K>
__global__ __launch_bounds__(256) void k_codes(const T *__restrict__ part_all, int nparts, const T *__restrict__ cent_all,
                                               int64_t n, K *__restrict__ codes_all) {
    __shared__ T scene[6];
    const int b = blockIdx.y;
    if (threadIdx.x < 6) {
        const int k = threadIdx.x;
        const T *p = part_all + (int64_t)b * nparts * 6;
        T v = p[k];
        for (int j = 1; j < nparts; ++j) v = k < 3 ? tmin(v, p[6 * j + k]) : tmax(v, p[6 * j + k]);
        scene[k] = v;
    }
    __syncthreads();
    const V3<T> smin = mk(scene[0], scene[1], scene[2]), smax = mk(scene[3], scene[4], scene[5]);
    const T *cent = cent_all + (int64_t)b * n * 3;
    K *codes = codes_all + (int64_t)b * n;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const T *c = cent + 3 * i;
        const T x = (c[0] - smin.x) / (smax.x - smin.x);
        const T y = (c[1] - smin.y) / (smax.y - smin.y);
        const T z = (c[2] - smin.z) / (smax.z - smin.z);
        if (sizeof(K) == 8) codes[i] = (K)morton63(x, y, z);
        else codes[i] = (K)morton30(x, y, z);
    }
}

// ---- stable LSD radix sort of (code, id), 8 bits per pass --------------------------------
// Pass = per-tile digit histogram -> per-element exclusive scan (digit-major) -> stable
// scatter.  The scatter ranks keys inside a wave with a ballot multisplit (8 ballots give
// the lanes holding the same digit) and across the block's four waves with LDS counters.

template <typename K>
__global__ __launch_bounds__(kSortThreads) void k_sort_hist(const K *__restrict__ keys, int64_t n, int shift,
                                                            uint32_t *__restrict__ hist, int nb) {
    __shared__ uint32_t h[256];
    const int b = blockIdx.y, blk = blockIdx.x, tid = threadIdx.x;
    h[tid] = 0;
    __syncthreads();
    const K *k = keys + (int64_t)b * n;
    for (int r = 0; r < kSortRounds; ++r) {
        int64_t i = (int64_t)blk * kSortTile + r * kSortThreads + tid;
        if (i < n) atomicAdd(&h[(uint32_t)(k[i] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[((int64_t)b * 256 + tid) * nb + blk] = h[tid];
}

// Exclusive scan of one element's [256][nb] histogram, one block of 1024 threads.
__global__ __launch_bounds__(1024) void k_sort_scan(uint32_t *__restrict__ hist, int nb) {
    __shared__ uint32_t part[1024];
    const int tid = threadIdx.x;
    uint32_t *h = hist + (int64_t)blockIdx.x * 256 * nb;
    const int64_t total = (int64_t)256 * nb;
    const int64_t chunk = (total + 1023) / 1024;
    const int64_t lo = tid * chunk, hi = lo + chunk < total ? lo + chunk : total;
    uint32_t s = 0;
    for (int64_t i = lo; i < hi; ++i) s += h[i];
    part[tid] = s;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        uint32_t v = tid >= off ? part[tid - off] : 0u;
        __syncthreads();
        part[tid] += v;
        __syncthreads();
    }
    uint32_t run = part[tid] - s;
    for (int64_t i = lo; i < hi; ++i) {
        uint32_t v = h[i];
        h[i] = run;
        run += v;
    }
}

template <typename K>
__global__ __launch_bounds__(kSortThreads) void k_sort_scatter(const K *__restrict__ kin, const int32_t *__restrict__ vin,
                                                               K *__restrict__ kout, int32_t *__restrict__ vout,
                                                               int64_t n, int shift, const uint32_t *__restrict__ hist, int nb) {
    __shared__ uint32_t run[256];
    __shared__ uint32_t gbase[256];
    __shared__ uint32_t wcnt[kSortThreads / 64][256];
    const int b = blockIdx.y, blk = blockIdx.x, tid = threadIdx.x, w = tid >> 6;
    const int64_t off = (int64_t)b * n;
    gbase[tid] = hist[((int64_t)b * 256 + tid) * nb + blk];
    run[tid] = 0;
    for (int r = 0; r < kSortRounds; ++r) {
#pragma unroll
        for (int q = 0; q < kSortThreads / 64; ++q) wcnt[q][tid] = 0;
        __syncthreads();
        const int64_t i = (int64_t)blk * kSortTile + r * kSortThreads + tid;
        const bool valid = i < n;
        const K key = valid ? kin[off + i] : (K)0;
        const int32_t val = valid ? vin[off + i] : 0;
        const uint32_t d = (uint32_t)(key >> shift) & 255u;
        unsigned long long peers = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            unsigned long long bb = __ballot((d >> bit) & 1u);
            peers &= ((d >> bit) & 1u) ? bb : ~bb;
        }
        const unsigned rank = lanes_below(peers);
        if (valid && rank == 0) wcnt[w][d] = (uint32_t)__popcll(peers);
        __syncthreads();
        {
            uint32_t base = run[tid], acc = 0;
#pragma unroll
            for (int q = 0; q < kSortThreads / 64; ++q) {
                uint32_t c = wcnt[q][tid];
                wcnt[q][tid] = base + acc;
                acc += c;
            }
            run[tid] = base + acc;
        }
        __syncthreads();
        if (valid) {
            const int64_t dst = (int64_t)gbase[d] + wcnt[w][d] + rank;
            kout[off + dst] = key;
            vout[off + dst] = val;
        }
        __syncthreads();
    }
}

// ---- Karras radix tree ----------------------------------------------------------------------
// bvh.cu:70-89 LongestCommonPrefix: -1 outside [0, n-1]; equal codes extend the prefix with
// the ids' common prefix (32 + clz(id_i ^ id_j) for 32-bit keys, 64 + ... for 64-bit ones).
template <typename K> __device__ __forceinline__ int clz_key(K x);
template <> __device__ __forceinline__ int clz_key<uint32_t>(uint32_t x) { return __clz((int)x); }
template <> __device__ __forceinline__ int clz_key<uint64_t>(uint64_t x) { return __clzll((long long)x); }

template <typename K>
__device__ __forceinline__ int lcp_delta(const K *codes, const int32_t *ids, int64_t n, int64_t i, int64_t j) {
    if (j < 0 || j > n - 1) return -1;
    const K a = codes[i], c = codes[j];
    if (a != c) return clz_key<K>(a ^ c);
    return 8 * (int)sizeof(K) + __clz((int)((uint32_t)ids[i] ^ (uint32_t)ids[j]));
}

// Karras 2012, Algorithm 1 (what build_bvh.cu:74-143 computes): node i finds its range
// direction, the far end j by exponential + binary search and the split by binary search.
// Writes left/right/self of row i and the parent field of both children's rows.
template <typename K>
__global__ void k_karras(const K *__restrict__ codes_all, const int32_t *__restrict__ ids_all, int64_t n,
                         int64_t *__restrict__ tree_all, int2 *__restrict__ range_all) {
    const int b = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const K *codes = codes_all + (int64_t)b * n;
    const int32_t *ids = ids_all + (int64_t)b * n;
    int64_t *tree = tree_all + (int64_t)b * (2 * n - 1) * 4;
    int2 *range = range_all + (int64_t)b * (n - 1);
    const int d = (lcp_delta(codes, ids, n, i, i + 1) - lcp_delta(codes, ids, n, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = lcp_delta(codes, ids, n, i, i - d);
    int64_t lmax = 2;
    while (lcp_delta(codes, ids, n, i, i + lmax * d) > dmin) lmax *= 2;
    int64_t l = 0;
    for (int64_t t = lmax / 2; t >= 1; t /= 2)
        if (lcp_delta(codes, ids, n, i, i + (l + t) * d) > dmin) l += t;
    const int64_t j = i + l * d;
    const int dnode = lcp_delta(codes, ids, n, i, j);
    int64_t s = 0;
    for (int64_t div = 2;; div *= 2) {
        const int64_t t = (l + div - 1) / div;
        if (lcp_delta(codes, ids, n, i, i + (s + t) * d) > dnode) s += t;
        if (t <= 1) break;
    }
    const int64_t g = i + s * d + (d < 0 ? -1 : 0);
    const int64_t lo = i < j ? i : j, hi = i < j ? j : i;
    const int64_t left = (lo == g) ? (n - 1 + g) : g;
    const int64_t right = (hi == g + 1) ? (n - 1 + g + 1) : (g + 1);
    tree[4 * i + 1] = left;
    tree[4 * i + 2] = right;
    tree[4 * i + 3] = -1;
    if (i == 0) tree[0] = -1;
    tree[4 * left + 0] = i;
    tree[4 * right + 0] = i;
    range[i] = make_int2((int)lo, (int)hi);
}

// ---- node boxes -----------------------------------------------------------------------------
// The reference computes them by an atomic bottom-up climb (build_bvh.cu:145-209).  Every
// internal node of the Karras tree covers a contiguous range [lo, hi] of sorted leaf
// positions, so its box is the union of the leaf boxes of that range; min / max are exact and
// order-independent, so any grouping gives the climb's result, with no atomics or fences.
// Positions are grouped in chunks of 64, one per lane of a wave, whose unions come from lane
// exchanges.  (One thread per chunk, walking its 64 boxes one after the other, was bound by
// the latency of that chain: 12-22 us per level, and as much again for the nodes' own walks.)
constexpr int kChunkLevels = 5;      // 64^5 = 2^30 > 2^28 leaves

// Writes the boxes of the nodes that end at this level: `box` is the union over lane's leaf
// or chunk, unit `c` of `count` units of 2^shift leaves each; a unit's node is the one whose
// aligned block starts at its first leaf (c even) or ends at its last (c odd).  Lanes past
// the end hold a copy of the last unit's box, which changes no union.  Returns the union of
// the wave's 64 units.
template <typename T>
__device__ __forceinline__ BoxReg<T> index_nodes_of_wave(BoxReg<T> box, int64_t c, int64_t count, int shift, int64_t n, T *bb) {
    const int64_t i = (c & 1) ? ((c + 1) << shift) - 1 : c << shift;
    // unit 0's node is the root, which the top level writes
    const int k = c > 0 ? index_node_level(c) : kChunkBits + 1;
    const bool mine = c < count && i < n - 1;
    BoxReg<T> out = box;
#pragma unroll
    for (int l = 1; l <= kChunkBits; ++l) {
        box_join_xor(box, 1 << (l - 1));
        if (k == l) out = box;
    }
    if (mine && c == 0 && count <= kChunk) store_box(bb, box);
    else if (mine && k <= kChunkBits) store_box(bb + 6 * i, out);
    return box;
}

// Compat mode, first level: leaf boxes, leaf rows, the tree's internal rows (wire layout of
// build_bvh.cu:309-378), the boxes of all nodes of up to 64 leaves and each chunk's box, one
// wave per chunk, in one launch.  Bound by its reads and writes (226 B per fp64 triangle with
// motion); it stands in for five launches (boxes, tree, rows, chunks, nodes) that took 60-110
// us per build, nearly all of it latency, from 450 to 130k triangles.
template <typename T, bool MOTION>
__global__ __launch_bounds__(256) void k_index_leaves(const T *__restrict__ t0, const T *__restrict__ t1, int64_t n,
                                                      T *__restrict__ bboxes_all, int64_t *__restrict__ tree_all,
                                                      T *__restrict__ chunk_all, int64_t chunk_stride) {
    const int b = blockIdx.y;
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if ((p & ~(int64_t)(kChunk - 1)) >= n) return;      // the whole wave is past the end
    const int64_t rows = 2 * n - 1;
    T *bb = bboxes_all + (int64_t)b * rows * 6;
    int64_t *tree = tree_all + (int64_t)b * rows * 4;
    const Box<T> bx = leaf_box<T, MOTION>(t0, t1, (int64_t)b * n + (p < n ? p : n - 1), (V3<T> *)nullptr);
    const BoxReg<T> box{{bx.mn.x, bx.mn.y, bx.mn.z, bx.mx.x, bx.mx.y, bx.mx.z}};
    if (p < n) {
        const int64_t row = n - 1 + p;
        store_box(bb + 6 * row, box);
        if (n == 1) tree[4 * row] = -1;
        tree[4 * row + 1] = -1;
        tree[4 * row + 2] = -1;
        tree[4 * row + 3] = p;
    }
    if (p < n - 1) {
        int64_t left, right;
        index_node_row(p, n, left, right);
        if (p == 0) tree[0] = -1;
        tree[4 * p + 1] = left;
        tree[4 * p + 2] = right;
        tree[4 * p + 3] = -1;
        tree[4 * left] = p;
        tree[4 * right] = p;
    }
    if (n == 1) return;
    const BoxReg<T> all = index_nodes_of_wave(box, p, n, 0, n, bb);
    if (chunk_all && (threadIdx.x & 63) == 0) store_box(chunk_all + (int64_t)b * chunk_stride + 6 * (p >> kChunkBits), all);
}

// Compat mode, further levels: `count` units of 2^shift leaves, one per lane.
template <typename T>
__global__ __launch_bounds__(256) void k_index_nodes(const T *__restrict__ src_all, int64_t src_stride, int64_t count, int shift, int64_t n,
                                                     T *__restrict__ bboxes_all, T *__restrict__ dst_all, int64_t dst_stride) {
    const int b = blockIdx.y;
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if ((c & ~(int64_t)(kChunk - 1)) >= count) return;
    const BoxReg<T> box = load_box(src_all + (int64_t)b * src_stride + 6 * (c < count ? c : count - 1));
    const BoxReg<T> all = index_nodes_of_wave(box, c, count, shift, n, bboxes_all + (int64_t)b * (2 * n - 1) * 6);
    if (dst_all && (threadIdx.x & 63) == 0) store_box(dst_all + (int64_t)b * dst_stride + 6 * (c >> kChunkBits), all);
}

// Fitted modes: leaf rows in sorted order (the box of triangle ids[p] and (-1, -1, id)), each
// chunk's box and the boxes of the nodes whose range lies within a chunk, one wave per chunk.
// For those, level l of a table in LDS holds the unions over [p, p + 2^l), one coordinate at a
// time; a range is the union of the two table entries that cover it.
template <typename T>
__global__ __launch_bounds__(256) void k_sorted_leaves(const T *__restrict__ boxes_all, const int32_t *__restrict__ ids_all, int64_t n,
                                                       const int2 *__restrict__ range_all, T *__restrict__ bboxes_all,
                                                       int64_t *__restrict__ tree_all, T *__restrict__ chunk_all, int64_t chunk_stride) {
    __shared__ T s_tab[256 / kChunk][kChunkBits][kChunk];
    const int b = blockIdx.y, lane = threadIdx.x & 63;
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, first = p - lane;
    if (first >= n) return;
    const int64_t rows = 2 * n - 1, at = p < n ? p : n - 1;
    T *bb = bboxes_all + (int64_t)b * rows * 6;
    int64_t *tree = tree_all + (int64_t)b * rows * 4;
    T(*tab)[kChunk] = s_tab[threadIdx.x >> 6];
    const int32_t id = ids_all[(int64_t)b * n + at];
    const BoxReg<T> box = load_box(boxes_all + ((int64_t)b * n + id) * 6);
    if (p < n) {
        const int64_t row = n - 1 + p;
        store_box(bb + 6 * row, box);
        if (n == 1) tree[4 * row] = -1;
        tree[4 * row + 1] = -1;
        tree[4 * row + 2] = -1;
        tree[4 * row + 3] = id;
    }
    int lo = 0, hi = 0;
    bool mine = false;
    if (p < n - 1) {
        const int2 r = range_all[(int64_t)b * (n - 1) + p];
        mine = r.x >= first && r.y < first + kChunk;
        if (mine) { lo = (int)(r.x - first); hi = (int)(r.y - first); }
    }
    const int level = 31 - __clz(hi - lo + 1);      // 2^level <= length; at most 6: the whole chunk
    const int l = level < kChunkBits ? level : kChunkBits - 1;
    BoxReg<T> out, all;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        T v = box.v[k];
#pragma unroll
        for (int j = 0; j < kChunkBits; ++j) {
            tab[j][lane] = v;
            const T w = __shfl_down(v, 1 << j, 64);      // past the wave's end: the lane's own value
            v = k < 3 ? tmin(v, w) : tmax(v, w);
        }
        all.v[k] = v;                                    // lane 0: the union of all 64
        wave_sync();
        const T u = tab[l][lo], w = tab[l][hi + 1 - (1 << l)];
        out.v[k] = k < 3 ? tmin(u, w) : tmax(u, w);
        wave_sync();
    }
    if (mine) store_box(bb + 6 * p, out);
    if (chunk_all && lane == 0) store_box(chunk_all + (int64_t)b * chunk_stride + 6 * (p >> kChunkBits), all);
}

// chunk level L box c = union of the (at most 64) level L-1 boxes 64c .. 64c+63, one per lane.
template <typename T>
__global__ __launch_bounds__(256) void k_chunk_boxes(const T *__restrict__ src_all, int64_t src_stride, int64_t src_count,
                                                     T *__restrict__ dst_all, int64_t dst_stride) {
    const int b = blockIdx.y;
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if ((c & ~(int64_t)(kChunk - 1)) >= src_count) return;
    BoxReg<T> box = load_box(src_all + (int64_t)b * src_stride + 6 * (c < src_count ? c : src_count - 1));
#pragma unroll
    for (int d = 1; d < kChunk; d <<= 1) box_join_xor(box, d);
    if ((threadIdx.x & 63) == 0) store_box(dst_all + (int64_t)b * dst_stride + 6 * (c >> kChunkBits), box);
}

struct ChunkLevels {
    const void *box[kChunkLevels + 1];   // [0]: leaf boxes (bboxes leaf rows), [L]: level L chunks
    int64_t stride[kChunkLevels + 1];    // elements between batch elements
    int levels;                          // chunk levels in use
};

// Fitted modes: the nodes whose range crosses a chunk boundary (a few percent), each by its
// whole wave: at every level the units at both ends that no unit of the next level covers
// (at most 63 each, one per lane), until the rest lies within 64 units.
template <typename T>
__global__ __launch_bounds__(256) void k_cross_nodes(const int2 *__restrict__ range_all, int64_t n, ChunkLevels lv, T *__restrict__ bboxes_all) {
    const int b = blockIdx.y, lane = threadIdx.x & 63;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int2 r = make_int2(0, 0);
    if (i < n - 1) r = range_all[(int64_t)b * (n - 1) + i];
    unsigned long long todo = __ballot((r.x >> kChunkBits) != (r.y >> kChunkBits));
    T *bb = bboxes_all + (int64_t)b * (2 * n - 1) * 6;
    while (todo) {
        const int who = __ffsll((long long)todo) - 1;
        todo &= todo - 1;
        int64_t lo = __shfl(r.x, who, 64), hi = __shfl(r.y, who, 64);
        const int64_t node = i - lane + who;
        BoxReg<T> acc = load_box((const T *)lv.box[0] + (int64_t)b * lv.stride[0] + 6 * lo);
        for (int L = 0; lo <= hi; ++L) {
            const T *src = (const T *)lv.box[L] + (int64_t)b * lv.stride[L];
            if (L == lv.levels || hi - lo < kChunk) {
                // lanes past the end take the last unit again
                for (int64_t u = lo; u <= hi; u += kChunk) box_join(acc, load_box(src + 6 * (u + lane <= hi ? u + lane : hi)));
                break;
            }
            const int64_t up = (lo + kChunk - 1) >> kChunkBits, down = ((hi + 1) >> kChunkBits) - 1;   // whole units above
            const int64_t head = (up << kChunkBits) - 1, tail = (down + 1) << kChunkBits;             // units lo..head, tail..hi
            if (lo <= head) box_join(acc, load_box(src + 6 * (lo + lane <= head ? lo + lane : head)));
            if (tail <= hi) box_join(acc, load_box(src + 6 * (tail + lane <= hi ? tail + lane : hi)));
            lo = up;
            hi = down;
        }
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) box_join_xor(acc, d);
        if (lane == 0) store_box(bb + 6 * node, acc);
    }
}

// Stable LSD radix sort of B rows of n (key, id) pairs, 8 bits per pass over the key's width;
// returns which buffers hold the result.
template <typename K>
static ccc_status radix_sort(K *&ka, K *&kb, int32_t *&va, int32_t *&vb, int64_t B, int64_t n, int bits, uint32_t *hist,
                             hipStream_t s) {
    const int nb = (int)((n + kSortTile - 1) / kSortTile);
    for (int shift = 0; shift < bits; shift += 8) {
        hipLaunchKernelGGL((k_sort_hist<K>), dim3(nb, B), dim3(kSortThreads), 0, s, ka, n, shift, hist, nb);
        hipLaunchKernelGGL(k_sort_scan, dim3(B), dim3(1024), 0, s, hist, nb);
        hipLaunchKernelGGL((k_sort_scatter<K>), dim3(nb, B), dim3(kSortThreads), 0, s, ka, va, kb, vb, n, shift, hist, nb);
        CCC_LAUNCH_CHECK("radix sort");
        K *tk = ka; ka = kb; kb = tk;
        int32_t *tv = va; va = vb; vb = tv;
    }
    return CCC_OK;
}

template <typename T>
static ccc_status build(ccc_context *ctx, const T *t0, const T *t1, int64_t B, int64_t n, int morton, T *bboxes, int64_t *tree,
                        hipStream_t s, void *arena, size_t arena_bytes) {
    Workspace ws(ctx, s, arena, arena_bytes);
    KernelTimer tm(ctx, s);
    const int64_t total = B * n;
    const int nb = (int)((n + kSortTile - 1) / kSortTile);
    const bool fit = morton != CCC_MORTON_COMPAT;
    const size_t ksz = morton == CCC_MORTON_63 ? 8 : 4;
    T *boxes = fit ? ws.get_as<T>(total * 6) : nullptr;
    int32_t *va = fit ? ws.get_as<int32_t>(total) : nullptr;
    T *cent = fit ? ws.get_as<T>(total * 3) : nullptr;
    T *part = fit ? ws.get_as<T>((size_t)B * kSceneBlocks * 6) : nullptr;
    void *ka = fit ? ws.get(total * ksz) : nullptr;
    void *kb = fit ? ws.get(total * ksz) : nullptr;
    int32_t *vb = fit ? ws.get_as<int32_t>(total) : nullptr;
    uint32_t *hist = fit ? ws.get_as<uint32_t>((size_t)B * 256 * nb) : nullptr;
    int2 *range = fit ? ws.get_as<int2>((size_t)B * (n > 1 ? n - 1 : 1)) : nullptr;
    ChunkLevels lv{};
    lv.box[0] = bboxes + (size_t)6 * (n - 1);
    lv.stride[0] = (2 * n - 1) * 6;
    int64_t count = n;
    while (lv.levels < kChunkLevels && count > kChunk) {
        count = (count + kChunk - 1) / kChunk;
        ++lv.levels;
        lv.box[lv.levels] = ws.get_as<T>((size_t)B * count * 6);
        lv.stride[lv.levels] = count * 6;
    }
    if (ws.failed()) return CCC_ERR_NO_MEMORY;
    T *chunk1 = lv.levels > 0 ? (T *)lv.box[1] : nullptr;

    if (!fit) {
        // every code is 0 and the stable sort keeps the input order: the index tree
        tm.begin("bvh_leaves");
        if (t1) hipLaunchKernelGGL((k_index_leaves<T, true>), dim3(grid_for(n, 256), B), dim3(256), 0, s, t0, t1, n, bboxes, tree, chunk1, lv.stride[1]);
        else hipLaunchKernelGGL((k_index_leaves<T, false>), dim3(grid_for(n, 256), B), dim3(256), 0, s, t0, t1, n, bboxes, tree, chunk1, lv.stride[1]);
        tm.end();
        CCC_LAUNCH_CHECK("k_index_leaves");
        tm.begin("bvh_refit");
        int64_t units = n;
        for (int L = 1; L <= lv.levels; ++L) {
            units = (units + kChunk - 1) / kChunk;
            T *dst = L < lv.levels ? (T *)lv.box[L + 1] : nullptr;
            hipLaunchKernelGGL((k_index_nodes<T>), dim3(grid_for(units, 256), B), dim3(256), 0, s, (const T *)lv.box[L], lv.stride[L], units,
                               kChunkBits * L, n, bboxes, dst, L < lv.levels ? lv.stride[L + 1] : 0);
        }
        tm.end();
        CCC_LAUNCH_CHECK("node boxes");
        return CCC_OK;
    }

    tm.begin("bvh_leaves");
    if (t1) hipLaunchKernelGGL((k_leaf_boxes<T, true>), dim3(grid_for(total, 256)), dim3(256), 0, s, t0, t1, total, n, boxes, cent, va);
    else hipLaunchKernelGGL((k_leaf_boxes<T, false>), dim3(grid_for(total, 256)), dim3(256), 0, s, t0, t1, total, n, boxes, cent, va);
    tm.end();
    CCC_LAUNCH_CHECK("k_leaf_boxes");
    {
        tm.begin("bvh_sort");
        const unsigned gparts = (unsigned)std::min<int64_t>(kSceneBlocks, (n + 255) / 256);
        hipLaunchKernelGGL((k_scene_partial<T>), dim3(gparts, B), dim3(256), 0, s, boxes, n, part);
        const unsigned gc = (unsigned)std::min<int64_t>(1024, (n + 255) / 256);
        if (ksz == 8) {
            hipLaunchKernelGGL((k_codes<T, uint64_t>), dim3(gc, B), dim3(256), 0, s, part, (int)gparts, cent, n, (uint64_t *)ka);
            CCC_LAUNCH_CHECK("morton codes");
            uint64_t *a = (uint64_t *)ka, *b = (uint64_t *)kb;
            ccc_status st = radix_sort<uint64_t>(a, b, va, vb, B, n, 64, hist, s);
            if (st != CCC_OK) return st;
            ka = a;
        } else {
            hipLaunchKernelGGL((k_codes<T, uint32_t>), dim3(gc, B), dim3(256), 0, s, part, (int)gparts, cent, n, (uint32_t *)ka);
            CCC_LAUNCH_CHECK("morton codes");
            uint32_t *a = (uint32_t *)ka, *b = (uint32_t *)kb;
            ccc_status st = radix_sort<uint32_t>(a, b, va, vb, B, n, 32, hist, s);
            if (st != CCC_OK) return st;
            ka = a;
        }
        tm.end();
    }
    if (n > 1) {
        tm.begin("bvh_karras");
        if (ksz == 8) hipLaunchKernelGGL((k_karras<uint64_t>), dim3(grid_for(n - 1, 256), B), dim3(256), 0, s, (const uint64_t *)ka, va, n, tree, range);
        else hipLaunchKernelGGL((k_karras<uint32_t>), dim3(grid_for(n - 1, 256), B), dim3(256), 0, s, (const uint32_t *)ka, va, n, tree, range);
        tm.end();
        CCC_LAUNCH_CHECK("k_karras");
    }
    tm.begin("bvh_refit");
    hipLaunchKernelGGL((k_sorted_leaves<T>), dim3(grid_for(n, 256), B), dim3(256), 0, s, boxes, va, n, range, bboxes, tree, chunk1, lv.stride[1]);
    int64_t src_count = n;
    for (int L = 2; L <= lv.levels; ++L) {
        src_count = (src_count + kChunk - 1) / kChunk;
        hipLaunchKernelGGL((k_chunk_boxes<T>), dim3(grid_for(src_count, 256), B), dim3(256), 0, s, (const T *)lv.box[L - 1],
                           lv.stride[L - 1], src_count, (T *)lv.box[L], lv.stride[L]);
    }
    if (lv.levels > 0) hipLaunchKernelGGL((k_cross_nodes<T>), dim3(grid_for(n - 1, 256), B), dim3(256), 0, s, range, n, lv, bboxes);
    tm.end();
    CCC_LAUNCH_CHECK("node boxes");
    return CCC_OK;
}

ccc_status build_bvh_device(ccc_context *ctx, const void *t0, const void *t1, int64_t B, int64_t n, int32_t dtype, int morton,
                            void *bboxes, int64_t *tree, hipStream_t s, void *arena, size_t arena_bytes) {
    if (morton != CCC_MORTON_COMPAT && morton != CCC_MORTON_30 && morton != CCC_MORTON_63) return bad_arg("unknown Morton mode");
    if (dtype == CCC_FLOAT64)
        return build<double>(ctx, (const double *)t0, (const double *)t1, B, n, morton, (double *)bboxes, tree, s, arena, arena_bytes);
    if (dtype == CCC_FLOAT32)
        return build<float>(ctx, (const float *)t0, (const float *)t1, B, n, morton, (float *)bboxes, tree, s, arena, arena_bytes);
    return bad_arg("dtype must be CCC_FLOAT32 or CCC_FLOAT64");
}

size_t build_bvh_arena_bytes(int64_t B, int64_t n, int32_t dtype, int morton) {
    auto r = [](size_t b) { return ((b ? b : 256) + 255) & ~(size_t)255; };
    const size_t esz = dtype == CCC_FLOAT64 ? 8 : 4, total = (size_t)(B * n);
    const bool fit = morton != CCC_MORTON_COMPAT;
    const size_t ksz = morton == CCC_MORTON_63 ? 8 : 4;
    const int nb = (int)((n + kSortTile - 1) / kSortTile);
    size_t tot = 0;
    if (fit) {
        tot += r(esz * total * 6) + r(4 * total) + r(esz * total * 3) + r(esz * B * kSceneBlocks * 6) + 2 * r(ksz * total) + r(4 * total) +
               r(4 * (size_t)B * 256 * nb);
        tot += r(sizeof(int2) * B * (n > 1 ? n - 1 : 1));
    }
    int64_t count = n;
    for (int levels = 0; levels < kChunkLevels && count > kChunk; ++levels) {
        count = (count + kChunk - 1) / kChunk;
        tot += r(esz * B * count * 6);
    }
    return tot;
}

static ccc_status build_entry(ccc_context *ctx, const void *t0, const void *t1, int64_t B, int64_t n, int32_t dtype,
                              void *bboxes, int64_t *tree, void *stream) {
    clear_error();
    if (!ctx) return bad_arg("context is NULL");
    if (B < 0 || n < 1) return bad_arg("need batch >= 0 and n >= 1 triangles");
    if (n > (int64_t)INT32_MAX / 2) return bad_arg("too many triangles");
    if (B == 0) return CCC_OK;
    if (!t0 || !bboxes || !tree) return bad_arg("NULL tensor pointer");
    CCC_HIP_TRY(hipSetDevice(ctx->device));
    return build_bvh_device(ctx, t0, t1, B, n, dtype, ctx->morton, bboxes, tree, (hipStream_t)stream);
}

}  // namespace ccc

extern "C" {

ccc_status ccc_bvh(ccc_context *ctx, const void *triangles, int64_t batch, int64_t n, int32_t dtype, void *bboxes,
                   int64_t *tree, void *stream) {
    return ccc::build_entry(ctx, triangles, nullptr, batch, n, dtype, bboxes, tree, stream);
}

ccc_status ccc_bvh_motion(ccc_context *ctx, const void *triangles, const void *triangles_next, int64_t batch, int64_t n,
                          int32_t dtype, void *bboxes, int64_t *tree, void *stream) {
    if (!triangles_next) {
        ccc::set_error("triangles_next is NULL");
        return CCC_ERR_BAD_ARG;
    }
    return ccc::build_entry(ctx, triangles, triangles_next, batch, n, dtype, bboxes, tree, stream);
}

}  // extern "C"
