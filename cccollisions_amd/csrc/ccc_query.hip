// Queries over the BVH wire format for gfx950: preparation, candidate pairs, the 15-way
// sub-primitive box filter, the fused CCD (coefficients -> cubic -> filter -> collision or
// impulse) kernel, static proximity, static triangle-triangle SAT and impulses from
// collision lists.
//
// Pipeline of one query call (all batch elements at once, batch index = blockIdx.y):
//   k_prep: is the tree the index tree, boxes of the chunks of 64 leaf positions and of the
//   groups of 16 queries, vertex records -> k_pairs: each group against the chunks behind it,
//   exact leaf tests -> candidate pairs -> k_items: per pair the 15-bit sub-primitive mask and
//   its items, by kind in tiles of 64 -> k_ccd: the narrow phase and the impulse sums.
// Any other tree (another builder's, a fitted one given back to a stateless call) takes the
// checked walk of GeneralTree instead of k_pairs; the static queries share the pairs and take
// k_subprim / k_proximity / k_sat.
#include <float.h>
#include <limits.h>

#include <algorithm>

#include "ccc_geom.h"
#include "ccc_internal.h"

namespace ccc {

constexpr int kThreads = 256;
constexpr int kTravThreads = 64;   // one wave per traversal block (128: 20.2 ms per step, 64: 18.7)
// Pending subtrees per lane (LDS).  A four-wide visit (two binary levels) pushes at most
// three entries, so with start points kFrontierDepth = 7 levels down the short stack covers
// the balanced trees built here (index radix trees, ceil(log2 N) + 1 deep) up to 2^22
// leaves; a traversal that overflows it runs again with the deep one.
constexpr int kStackShort = 24;
constexpr int kStackDeep = 32;
constexpr int kStage = 512;       // staged pairs per wave before a flush
// queries start from the subtrees this deep below the root (measured when every query walked:
// k_traverse per pass on the 130k cloth at depth 6 2.85 ms, 7 2.02 ms, 8 2.60 ms)
constexpr int kFrontierDepth = 7;
constexpr int kFrontier = 1 << kFrontierDepth;

// Workgroups are dispatched to the eight XCDs round-robin by workgroup ID, and each XCD has
// its own L2.  Persistent kernels walk their tiles with CCC_FOR_TILES, which gives the
// workgroups of one XCD one contiguous range of tiles (neighbouring tiles read the same
// triangles); their grids are a multiple of kXcds.
constexpr int kXcds = 8;
#define CCC_FOR_TILES(tile, T)                                                                          \
    for (int64_t tile##_k = blockIdx.x / kXcds, tile##_per = ((T) + kXcds - 1) / kXcds,                 \
                 tile = (int64_t)(blockIdx.x % kXcds) * tile##_per + tile##_k;                          \
         tile##_k < tile##_per && tile < (T);                                                           \
         tile##_k += gridDim.x / kXcds, tile = (int64_t)(blockIdx.x % kXcds) * tile##_per + tile##_k)

struct alignas(16) TNode {
    float4 a;  // L.min.x, L.min.y, L.min.z, L.max.x
    float4 b;  // L.max.y, L.max.z, R.min.x, R.min.y
    float4 c;  // R.min.z, R.max.x, R.max.y, R.max.z
    int4 d;    // left ref, right ref, rightmost leaf position of left / right child
};               // ref >= 0: internal row; ref < 0: leaf at position ~ref

__device__ __forceinline__ float f32_down(double v) {
    float f = (float)v;
    if ((double)f > v) f = nextafterf(f, -INFINITY);
    return nextafterf(f, -INFINITY);
}
__device__ __forceinline__ float f32_up(double v) {
    float f = (float)v;
    if ((double)f < v) f = nextafterf(f, INFINITY);
    return nextafterf(f, INFINITY);
}

__device__ __forceinline__ int64_t pack_item(int64_t x, int64_t y, int type) {
    return (int64_t)(((uint64_t)x << 32) | ((uint64_t)y << 4) | (uint64_t)type);
}
__device__ __forceinline__ void unpack_item(int64_t it, int64_t &x, int64_t &y, int &type) {
    uint64_t u = (uint64_t)it;
    x = (int64_t)(u >> 32);
    y = (int64_t)((u & 0xffffffffull) >> 4);
    type = (int)(u & 15ull);
}

// Block-wide reservation of `cnt` (< 16) consecutive slots per thread with one atomic.
// Every thread of the block (of NT threads) must call it.
template <int NT = kThreads>
__device__ __forceinline__ unsigned long long block_reserve(unsigned long long *counter, unsigned cnt) {
    __shared__ unsigned long long s_wave[NT / 64];
    __shared__ unsigned long long s_base;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    unsigned long long b0 = __ballot(cnt & 1u), b1 = __ballot(cnt & 2u), b2 = __ballot(cnt & 4u), b3 = __ballot(cnt & 8u);
    unsigned below = lanes_below(b0) + 2u * lanes_below(b1) + 4u * lanes_below(b2) + 8u * lanes_below(b3);
    unsigned long long wt = (unsigned long long)__popcll(b0) + 2ull * __popcll(b1) + 4ull * __popcll(b2) + 8ull * __popcll(b3);
    if (lane == 0) s_wave[w] = wt;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long tot = 0;
        for (int q = 0; q < NT / 64; ++q) {
            unsigned long long v = s_wave[q];
            s_wave[q] = tot;
            tot += v;
        }
        s_base = tot ? atomicAdd(counter, tot) : 0ull;
    }
    __syncthreads();
    unsigned long long r = s_base + s_wave[w] + below;
    __syncthreads();
    return r;
}

__device__ __forceinline__ void block_add(unsigned long long *counter, unsigned long long v) {
    __shared__ unsigned long long s_sum;
    if (threadIdx.x == 0) s_sum = 0;
    __syncthreads();
    if (v) atomicAdd(&s_sum, v);
    __syncthreads();
    if (threadIdx.x == 0 && s_sum) atomicAdd(counter, s_sum);
}

// ---- tree preparation -------------------------------------------------------------------

// Checks that `tree` is a binary tree over n leaves in the wire format.  Violations set
// DEV_BAD_TREE; nothing else reads an index before it has been range-checked here.
__global__ void k_check_tree(const int64_t *__restrict__ tree_all, int64_t n, int *__restrict__ claims_all,
                             DevCounters *__restrict__ ctr) {
    const int b = blockIdx.y;
    const int64_t rows = 2 * n - 1;
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    const int64_t *tree = tree_all + (int64_t)b * rows * 4;
    int *claims = claims_all + (int64_t)b * n;
    const int64_t p = tree[4 * r], l = tree[4 * r + 1], rr = tree[4 * r + 2], id = tree[4 * r + 3];
    bool ok = true;
    if (n == 1) {
        ok = p == -1 && l == -1 && rr == -1 && id == 0;
    } else if (r < n - 1) {
        ok = l >= 1 && l < rows && rr >= 1 && rr < rows && l != rr;
        if (ok) ok = tree[4 * l] == r && tree[4 * rr] == r;
        ok = ok && (r == 0 ? p == -1 : (p >= 0 && p < n - 1));
    } else {
        ok = l == -1 && rr == -1 && id >= 0 && id < n && p >= 0 && p < n - 1;
        if (ok) ok = atomicAdd(&claims[id], 1) == 0;
    }
    if (ok && n > 1 && r != 0) ok = tree[4 * p + 1] == r || tree[4 * p + 2] == r;
    if (!ok) atomicOr(&ctr[b].flags, DEV_BAD_TREE);
}

// Rightmost leaf position under every internal node (build_bvh.cu:707-743): bottom-up
// climb, the second thread to arrive at a node combines its children.  Bounded by n steps
// (a longer climb can only come from a cycle, reported as DEV_BAD_TREE).
// Rightmost leaf position of every internal node (build_bvh.cu:707-741 set_rightmost_nodes:
// rightmost = the larger of the children's rightmost leaves, compared by leaf address).  Trees whose subtrees cover contiguous
// ordered leaf ranges -- every tree bvh / bvh_motion builds -- take the walk below; any
// other tree falls back to an atomic bottom-up climb.
//
// Walk: lo / hi of a node = position of the leaf reached by following left / right
// children (at most 64 steps).
__global__ void k_ranges(const int64_t *__restrict__ tree_all, int64_t n, int *__restrict__ lo_all, int *__restrict__ rm_all,
                         DevCounters *__restrict__ ctr) {
    const int b = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    if (ctr[b].flags & DEV_BAD_TREE) return;
    const int64_t *tree = tree_all + (int64_t)b * (2 * n - 1) * 4;
    int64_t c = i, d = i;
    for (int step = 0; c < n - 1 || d < n - 1; ++step) {
        if (step >= 64) {
            atomicOr(&ctr[b].flags, DEV_UNORDERED);
            return;
        }
        if (c < n - 1) c = tree[4 * c + 1];
        if (d < n - 1) d = tree[4 * d + 2];
    }
    lo_all[(int64_t)b * (n - 1) + i] = (int)(c - (n - 1));
    rm_all[(int64_t)b * (n - 1) + i] = (int)(d - (n - 1));
}

// The walk's hi is the subtree maximum only if, at every node, the left child's range ends
// right before the right child's begins.
__global__ void k_order_check(const int64_t *__restrict__ tree_all, int64_t n, const int *__restrict__ lo_all,
                              const int *__restrict__ rm_all, DevCounters *__restrict__ ctr) {
    const int b = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    if (ctr[b].flags & (DEV_BAD_TREE | DEV_UNORDERED)) return;
    const int64_t *tree = tree_all + (int64_t)b * (2 * n - 1) * 4;
    const int *lo = lo_all + (int64_t)b * (n - 1);
    const int *rm = rm_all + (int64_t)b * (n - 1);
    const int64_t l = tree[4 * i + 1], r = tree[4 * i + 2];
    const int hl = l >= n - 1 ? (int)(l - (n - 1)) : rm[l];
    const int lr = r >= n - 1 ? (int)(r - (n - 1)) : lo[r];
    if (hl + 1 != lr) atomicOr(&ctr[b].flags, DEV_UNORDERED);
}

// Climb for the remaining trees: the second thread to reach a node combines its children.
// The counters are k_check_tree's claims, one per leaf id and each 1 in a valid tree.
__global__ void k_rightmost(const int64_t *__restrict__ tree_all, int64_t n, int *__restrict__ counters_all,
                            int *__restrict__ rm_all, DevCounters *__restrict__ ctr) {
    const int b = blockIdx.y;
    const int64_t pos = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (pos >= n || n < 2) return;
    if ((ctr[b].flags & DEV_BAD_TREE) || !(ctr[b].flags & DEV_UNORDERED)) return;
    const int64_t rows = 2 * n - 1;
    const int64_t *tree = tree_all + (int64_t)b * rows * 4;
    int *counters = counters_all + (int64_t)b * n;
    int *rm = rm_all + (int64_t)b * (n - 1);
    int64_t cur = tree[4 * (n - 1 + pos)];
    for (int64_t step = 0; cur >= 0; ++step) {
        if (step > n) { atomicOr(&ctr[b].flags, DEV_BAD_TREE); return; }
        __threadfence();
        const int old = __hip_atomic_fetch_add(&counters[cur], 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (old == 1) return;
        __threadfence();
        const int64_t l = tree[4 * cur + 1], r = tree[4 * cur + 2];
        const int a = l >= n - 1 ? (int)(l - (n - 1)) : __hip_atomic_load(&rm[l], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int c = r >= n - 1 ? (int)(r - (n - 1)) : __hip_atomic_load(&rm[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(&rm[cur], a > c ? a : c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        cur = tree[4 * cur];
    }
}

// One 64-byte traversal node per internal row: both children's boxes in fp32, rounded
// outward, grown by the threshold and by one more float ulp on each side, so that the
// fp32 test passes whenever the reference's fp64 test passes for either orientation.
template <typename T>
__global__ void k_nodes(const T *__restrict__ bb_all, const int64_t *__restrict__ tree_all, const int *__restrict__ rm_all,
                        int64_t n, double thr, TNode *__restrict__ nodes_all, const DevCounters *__restrict__ ctr) {
    const int b = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    if (ctr[b].flags & DEV_BAD_TREE) return;
    const int64_t rows = 2 * n - 1;
    const T *bb = bb_all + (int64_t)b * rows * 6;
    const int64_t *tree = tree_all + (int64_t)b * rows * 4;
    const int *rm = rm_all + (int64_t)b * (n - 1);
    const int64_t l = tree[4 * i + 1], r = tree[4 * i + 2];
    float lo[6], ro[6];
    const T *lb = bb + 6 * l, *rb = bb + 6 * r;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        lo[k] = f32_down((double)lb[k] - thr);
        lo[k + 3] = f32_up((double)lb[k + 3] + thr);
        ro[k] = f32_down((double)rb[k] - thr);
        ro[k + 3] = f32_up((double)rb[k + 3] + thr);
    }
    TNode nd;
    nd.a = make_float4(lo[0], lo[1], lo[2], lo[3]);
    nd.b = make_float4(lo[4], lo[5], ro[0], ro[1]);
    nd.c = make_float4(ro[2], ro[3], ro[4], ro[5]);
    const int lref = l >= n - 1 ? ~(int)(l - (n - 1)) : (int)l;
    const int rref = r >= n - 1 ? ~(int)(r - (n - 1)) : (int)r;
    const int lrm = l >= n - 1 ? (int)(l - (n - 1)) : rm[l];
    const int rrm = r >= n - 1 ? (int)(r - (n - 1)) : rm[r];
    nd.d = make_int4(lref, rref, lrm, rrm);
    nodes_all[(int64_t)b * (n - 1) + i] = nd;
}

// Four-wide view of the binary tree for the traversal.  For internal row i: the up to four
// grandchildren of i, left to right (a child that is a leaf stands for itself), with their
// TNode fp32 boxes as structure of arrays, refs and rightmost leaf positions; unused entries
// (at the end) have a NaN box and rightmost INT_MIN.  Testing a grandchild's box without its
// parent's prunes nothing that matters when boxes contain their children's (the traversal's
// assumption throughout: it starts below the root, and its node tests are conservative fp32):
// a pair needs the leaf's exact box to overlap the query.  One node is 128 bytes, one cache
// line.
struct alignas(16) QNode {
    float4 mnx, mny, mnz, mxx, mxy, mxz;
    int4 ref;   // >= 0 internal row, < 0 leaf at position ~ref
    int4 rm;    // rightmost leaf position; INT_MIN: unused entry
};

// side 0 / 1 of a TNode: box, ref and rightmost leaf of that child
__device__ __forceinline__ void tnode_child(const TNode &nd, int side, float *mn, float *mx, int &ref, int &rm) {
    if (side == 0) {
        mn[0] = nd.a.x; mn[1] = nd.a.y; mn[2] = nd.a.z; mx[0] = nd.a.w; mx[1] = nd.b.x; mx[2] = nd.b.y;
        ref = nd.d.x; rm = nd.d.z;
    } else {
        mn[0] = nd.b.z; mn[1] = nd.b.w; mn[2] = nd.c.x; mx[0] = nd.c.y; mx[1] = nd.c.z; mx[2] = nd.c.w;
        ref = nd.d.y; rm = nd.d.w;
    }
}

struct QEntry {
    float mn[3], mx[3];
    int ref, rm;
};

__global__ void k_qnodes(const TNode *__restrict__ nodes_all, int64_t n, QNode *__restrict__ q_all,
                         const DevCounters *__restrict__ ctr) {
    const int b = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    if (ctr[b].flags & DEV_BAD_TREE) return;
    const TNode *nodes = nodes_all + (int64_t)b * (n - 1);
    const TNode nd = nodes[i];
    QEntry none;    // unused entry: a NaN box fails every comparison
#pragma unroll
    for (int a = 0; a < 3; ++a) { none.mn[a] = NAN; none.mx[a] = NAN; }
    none.ref = 0;
    none.rm = INT_MIN;
    // side s of row i -> its entries g[s][0], g[s][1] (g[s][1] unused when the child is a leaf)
    QEntry g[2][2];
    bool internal[2];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        QEntry c;
        tnode_child(nd, side, c.mn, c.mx, c.ref, c.rm);
        internal[side] = c.ref >= 0;
        if (internal[side]) {
            const TNode cn = nodes[c.ref];
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2) tnode_child(cn, s2, g[side][s2].mn, g[side][s2].mx, g[side][s2].ref, g[side][s2].rm);
        } else {
            g[side][0] = c;
            g[side][1] = none;
        }
    }
    // left to right, unused entries last
    const QEntry e0 = g[0][0];
    const QEntry e1 = internal[0] ? g[0][1] : g[1][0];
    const QEntry e2 = internal[0] ? g[1][0] : (internal[1] ? g[1][1] : none);
    const QEntry e3 = internal[0] && internal[1] ? g[1][1] : none;
    QNode q;
    q.mnx = make_float4(e0.mn[0], e1.mn[0], e2.mn[0], e3.mn[0]);
    q.mny = make_float4(e0.mn[1], e1.mn[1], e2.mn[1], e3.mn[1]);
    q.mnz = make_float4(e0.mn[2], e1.mn[2], e2.mn[2], e3.mn[2]);
    q.mxx = make_float4(e0.mx[0], e1.mx[0], e2.mx[0], e3.mx[0]);
    q.mxy = make_float4(e0.mx[1], e1.mx[1], e2.mx[1], e3.mx[1]);
    q.mxz = make_float4(e0.mx[2], e1.mx[2], e2.mx[2], e3.mx[2]);
    q.ref = make_int4(e0.ref, e1.ref, e2.ref, e3.ref);
    q.rm = make_int4(e0.rm, e1.rm, e2.rm, e3.rm);
    q_all[(int64_t)b * (n - 1) + i] = q;
}

// Leaf record by position: the leaf box rounded inward to fp32 and the leaf's triangle id.
// A query box that overlaps the inward box overlaps the exact box (fp rounding is monotone,
// so fl(inward.max + thr) <= fl(max + thr) and fl(inward.min - thr) >= fl(min - thr)); only
// when the inward test fails does the traversal read the exact box from `bboxes`.
struct alignas(32) LeafRec {
    float mn[3], mx[3];
    int id, pad;
};

template <typename T>
__global__ void k_leaf_recs(const T *__restrict__ bb_all, const int64_t *__restrict__ tree_all, int64_t n,
                            LeafRec *__restrict__ recs_all, const DevCounters *__restrict__ ctr) {
    const int b = blockIdx.y;
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    if (ctr[b].flags & DEV_BAD_TREE) return;
    const int64_t rows = 2 * n - 1, row = n - 1 + p;
    const T *bx = bb_all + (int64_t)b * rows * 6 + 6 * row;
    LeafRec r;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        r.mn[k] = f32_up((double)bx[k]);
        r.mx[k] = f32_down((double)bx[k + 3]);
    }
    r.id = (int)tree_all[(int64_t)b * rows * 4 + 4 * row + 3];
    r.pad = 0;
    recs_all[(int64_t)b * n + p] = r;
}

template <typename T> __device__ __forceinline__ bool overlap_inward(const Box<T> &q, const LeafRec &r, T thr) {
    return (q.mn.x <= ((T)r.mx[0] + thr)) && (q.mx.x >= ((T)r.mn[0] - thr)) && (q.mn.y <= ((T)r.mx[1] + thr)) &&
           (q.mx.y >= ((T)r.mn[1] - thr)) && (q.mn.z <= ((T)r.mx[2] + thr)) && (q.mx.z >= ((T)r.mn[2] - thr));
}

// Start points of the traversal: the subtrees kFrontierDepth levels below the root, each
// with its fp32 box grown outward by the threshold (as in TNode) and its rightmost leaf.  Slot
// i follows the path of the bits of i from the root (1 = right); a leaf reached above that
// depth stands for itself in the slot of its leftmost path, and the other slots below it are
// empty (a NaN box: no query enters them).
// A query runs one traversal per start point, so the launch has kFrontier times as many
// lanes.
struct Frontier {
    int count;               // slots in use: kFrontier, or 0 (no traversal)
    int ref[kFrontier];      // internal node index, or ~leaf position
    int rightmost[kFrontier];
    float box[kFrontier][6];
};

template <typename T>
__global__ __launch_bounds__(kFrontier) void k_frontier(const T *__restrict__ bb_all, const int64_t *__restrict__ tree_all,
                                                      const int *__restrict__ rm_all, int64_t n, double thr, Frontier *__restrict__ fr_all, const DevCounters *__restrict__ ctr) {
    const int b = blockIdx.x, i = threadIdx.x;     // one thread per slot
    Frontier &f = fr_all[b];
    if (n < 2 || (ctr[b].flags & DEV_BAD_TREE)) {
        if (i == 0) f.count = 0;
        return;
    }
    if (i == 0) f.count = kFrontier;
    const int64_t rows = 2 * n - 1;
    const T *bb = bb_all + (int64_t)b * rows * 6;
    const int64_t *tree = tree_all + (int64_t)b * rows * 4;
    const int *rm = rm_all + (int64_t)b * (n - 1);
    int ref = 0;            // the root row
    bool used = true;
    for (int level = 0; level < kFrontierDepth; ++level) {
        if (ref < 0) {      // a leaf above the frontier depth: only its leftmost slot keeps it
            used = (i & ((1 << (kFrontierDepth - level)) - 1)) == 0;
            break;
        }
        const int64_t c = tree[4 * ref + 1 + ((i >> (kFrontierDepth - 1 - level)) & 1)];
        ref = c >= n - 1 ? ~(int)(c - (n - 1)) : (int)c;
    }
    f.ref[i] = ref;
    if (!used) {
        f.rightmost[i] = 0;
        for (int k = 0; k < 6; ++k) f.box[i][k] = NAN;
        return;
    }
    const int64_t row = ref >= 0 ? ref : n - 1 + (int64_t)(~ref);
    f.rightmost[i] = ref >= 0 ? rm[ref] : ~ref;
    for (int k = 0; k < 3; ++k) {
        f.box[i][k] = f32_down((double)bb[6 * row + k] - thr);
        f.box[i][k + 3] = f32_up((double)bb[6 * row + k + 3] + thr);
    }
}

// fp32 box of each block of kTravThreads query leaves (the union of the lanes' outward-
// rounded query boxes; empty past the last leaf), so that a traversal block whose queries
// cannot enter its start point ends before it starts.
template <typename T>
__global__ __launch_bounds__(kTravThreads) void k_qblock_boxes(const T *__restrict__ bb_all, int64_t n, int nqb,
                                                               float *__restrict__ qbox_all, const DevCounters *__restrict__ ctr) {
    const int b = blockIdx.y;
    const int64_t p = (int64_t)blockIdx.x * kTravThreads + threadIdx.x;
    float v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    if (p < n && !(ctr[b].flags & DEV_BAD_TREE)) {
        const T *q = bb_all + (int64_t)b * (2 * n - 1) * 6 + 6 * (n - 1 + p);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            v[k] = f32_down((double)q[k]);
            v[k + 3] = f32_up((double)q[k + 3]);
        }
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            v[k] = fminf(v[k], __shfl_xor(v[k], d, 64));
            v[k + 3] = fmaxf(v[k + 3], __shfl_xor(v[k + 3], d, 64));
        }
    }
    static_assert(kTravThreads == 64, "one wave per query block");
    if (threadIdx.x == 0) {
        float *o = qbox_all + ((int64_t)b * nqb + blockIdx.x) * 6;
#pragma unroll
        for (int k = 0; k < 6; ++k) o[k] = v[k];
    }
}

// ---- traversal ----------------------------------------------------------------------------
// collisions_static.cu:10-120 (ordering on) and collisions_continuous.cu:127-230,
// :1079-1100 (PARTIAL: ordering off, queries with to_check[position]).  A leaf child is
// reported after the reference's exact test checkOverlap(query box, leaf box, threshold) on
// the boxes stored in `bboxes`; the pair is (min id, max id).  The walk runs over the
// four-wide nodes (QNode): each visit tests up to four grandchildren, which halves the
// dependent node reads of a query against the binary nodes.
template <typename T, bool PARTIAL, int DEPTH>
__global__ __launch_bounds__(kTravThreads) void k_traverse(const T *__restrict__ bb_all, const int64_t *__restrict__ tree_all,
                                                           const QNode *__restrict__ qnodes_all,
                                                           const LeafRec *__restrict__ recs_all, int64_t n, T thr,
                                                           const uint8_t *__restrict__ to_check_all,
                                                           int2 *__restrict__ pairs_all, int64_t cap,
                                                           DevCounters *__restrict__ ctr_all, const Frontier *__restrict__ fr_all,
                                                           const float *__restrict__ qbox_all) {
    // Pending right children: with the short stack as 16-bit offsets from the start point's
    // node (a subtree's nodes lie close together in the trees built here; a farther node
    // ends the traversal like an overflow, and the call runs again with the deep stack).
    using StackT = typename std::conditional<(DEPTH < kStackDeep), short, int>::type;
    __shared__ StackT stack[DEPTH][kTravThreads];
    constexpr int kStageCap = kStage + 128;   // an iteration that would overflow it flushes first
    __shared__ int stage[kTravThreads / 64][kStageCap];                             // the other triangle of each pair
    __shared__ int lqid[kTravThreads / 64][64];                                     // each lane's query triangle
    __shared__ unsigned short stag[kTravThreads / 64][kStageCap];                  // lane << 10 | rank within the lane
    __shared__ int loff[kTravThreads / 64][64];                         // a flush's offset of each lane
    __shared__ int fill[kTravThreads / 64];
    const int b = blockIdx.y, tid = threadIdx.x, w = tid >> 6;
    const int64_t rows = 2 * n - 1;
    const T *bb = bb_all + (int64_t)b * rows * 6;
    const int64_t *tree = tree_all + (int64_t)b * rows * 4;
    const QNode *qnodes = qnodes_all + (int64_t)b * (n - 1);
    const LeafRec *recs = recs_all + (int64_t)b * n;
    DevCounters *ctr = ctr_all + b;
    int2 *pairs = pairs_all + (int64_t)b * cap;

    // block -> (start point s, query block); query blocks in XCD-contiguous order (the
    // query-block count nqb is a multiple of kXcds)
    const int nqb = gridDim.x / kFrontier;
    const int s = blockIdx.x / nqb, local = blockIdx.x % nqb;
    const int64_t qblock = (int64_t)(local % kXcds) * (nqb / kXcds) + local / kXcds;
    const int64_t p = qblock * blockDim.x + tid;
    const Frontier &fr = fr_all[b];
    {
        // the whole block ends here when none of its queries can enter the start point (the
        // same box and rightmost tests as each lane's below, on the block's union box)
        const float *qb = qbox_all + ((int64_t)b * nqb + qblock) * 6;
        bool dead = s >= fr.count;
        if (!dead) {
            const float *fb = fr.box[s];
            dead = !(qb[0] <= fb[3] && qb[3] >= fb[0] && qb[1] <= fb[4] && qb[4] >= fb[1] && qb[2] <= fb[5] && qb[5] >= fb[2]);
            if (!PARTIAL) dead = dead || fr.rightmost[s] <= (int)(qblock * kTravThreads);
        }
        if (dead) return;
    }
    if ((tid & 63) == 0) fill[w] = 0;
    __syncthreads();
    bool active = p < n && n > 1 && !(ctr->flags & DEV_BAD_TREE) && s < fr.count;
    if (PARTIAL && active) active = to_check_all[(int64_t)b * n + p] != 0;
    const uint8_t *to_check = PARTIAL ? to_check_all + (int64_t)b * n : nullptr;

    // Query setup (inactive lanes: no query; they stay in the loop below as idle lanes).
    Box<T> q{};
    int qid = 0;
    float qx0 = 0, qy0 = 0, qz0 = 0, qx1 = 0, qy1 = 0, qz1 = 0;
    bool alive = false;
    if (active) {
        const int64_t qrow = n - 1 + p;
        q = ld_box(bb + 6 * qrow);
        qid = recs[p].id;
        qx0 = f32_down((double)q.mn.x); qy0 = f32_down((double)q.mn.y); qz0 = f32_down((double)q.mn.z);
        qx1 = f32_up((double)q.mx.x); qy1 = f32_up((double)q.mx.y); qz1 = f32_up((double)q.mx.z);
        // the start point itself: box and rightmost tests as for a child
        const float *fb = fr.box[s];
        alive = qx0 <= fb[3] && qx1 >= fb[0] && qy0 <= fb[4] && qy1 >= fb[1] && qz0 <= fb[5] && qz1 >= fb[2];
        if (!PARTIAL) alive = alive && fr.rightmost[s] > (int)p;
    }
    const int lane = tid & 63;
    const int sbase = fr.ref[s];
    int sp = 0, node = sbase;
    int mine = 0;   // pairs this lane has staged since the last flush
    // Writes the wave's nf staged pairs grouped by lane (lane order, each lane's pairs in the
    // order found), so that the pair list keeps one query's pairs together.  Full wave.
    auto flush_stage = [&](int nf) {
        int incl = mine;    // inclusive scan of `mine` over the wave
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(incl, d, 64);
            if (lane >= d) incl += v;
        }
        loff[w][lane] = incl - mine;
        lqid[w][lane] = qid;
        unsigned long long base = 0;
        if (lane == 0) base = atomicAdd(&ctr->cand, (unsigned long long)nf);
        base = readfirstlane_u64(base);
        for (int j = lane; j < nf; j += 64) {
            const unsigned t = stag[w][j];
            const unsigned long long d = base + (unsigned long long)(loff[w][t >> 10] + (int)(t & 1023u));
            if (d < (unsigned long long)cap) {
                const int qq = lqid[w][t >> 10], oo = stage[w][j];
                pairs[d] = make_int2(min(qq, oo), max(qq, oo));
            }
        }
        mine = 0;
    };
    // a pending subtree onto the stack; an overflow (or, with 16-bit entries, a node too far
    // from the start node) ends this lane and flags the call for the deep stack
    auto push = [&](int ref) {
        const int v = sizeof(StackT) < sizeof(int) ? ref - sbase : ref;
        const bool fits = sizeof(StackT) == sizeof(int) || (v >= -32768 && v <= 32767);
        if (sp >= DEPTH || !fits) { atomicOr(&ctr->flags, DEV_STACK); alive = false; }
        else stack[sp++][tid] = (StackT)v;
    };
    while (__any(alive)) {
        int o0 = -1, o1 = -1, o2 = -1, o3 = -1;     // pairs found in this iteration
        int r0 = 0, r1 = 0, r2 = 0, r3 = 0;         // children (entries) that may be descended into
        unsigned im = 0;                            // bit k: descend into r_k
        if (alive) {
            {
                QNode qn;
                if (node >= 0) {
                    qn = qnodes[node];
                } else {
                    // a start point that is a leaf: entry 0 is the leaf, with an unbounded box
                    qn.mnx = make_float4(-INFINITY, NAN, NAN, NAN);
                    qn.mxx = make_float4(INFINITY, NAN, NAN, NAN);
                    qn.mny = qn.mnx; qn.mnz = qn.mnx; qn.mxy = qn.mxx; qn.mxz = qn.mxx;
                    qn.ref = make_int4(node, 0, 0, 0);
                    qn.rm = make_int4(~node, INT_MIN, INT_MIN, INT_MIN);
                }
                const float mnx[4] = {qn.mnx.x, qn.mnx.y, qn.mnx.z, qn.mnx.w}, mxx[4] = {qn.mxx.x, qn.mxx.y, qn.mxx.z, qn.mxx.w};
                const float mny[4] = {qn.mny.x, qn.mny.y, qn.mny.z, qn.mny.w}, mxy[4] = {qn.mxy.x, qn.mxy.y, qn.mxy.z, qn.mxy.w};
                const float mnz[4] = {qn.mnz.x, qn.mnz.y, qn.mnz.z, qn.mnz.w}, mxz[4] = {qn.mxz.x, qn.mxz.y, qn.mxz.z, qn.mxz.w};
                const int rf[4] = {qn.ref.x, qn.ref.y, qn.ref.z, qn.ref.w}, rmv[4] = {qn.rm.x, qn.rm.y, qn.rm.z, qn.rm.w};
                int oid[4];
                bool leaf[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    bool hit = qx0 <= mxx[k] && qx1 >= mnx[k] && qy0 <= mxy[k] && qy1 >= mny[k] && qz0 <= mxz[k] && qz1 >= mnz[k];
                    if (!PARTIAL) hit = hit && rmv[k] > (int)p;
                    leaf[k] = hit && rf[k] < 0;
                    if (hit && rf[k] >= 0) im |= 1u << k;
                }
                // The four leaf records are requested before the first is tested, so that
                // their loads are in flight together (record 0 stands in for entries that are
                // not hit leaves: no branch around the loads).  A leaf whose inward-rounded
                // record does not decide is tested on its exact box from `bboxes`, under a
                // wave-uniform branch with every lane loading a valid row: with that fallback
                // in a lane-divergent branch per leaf, the compiler lost the record's id in
                // the lanes that took it (their pairs were dropped).
                LeafRec lr[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) lr[k] = recs[leaf[k] ? ~rf[k] : 0];
                bool ov[4];
                bool need = false;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    ov[k] = leaf[k] && overlap_inward(q, lr[k], thr);
                    need = need || (leaf[k] && !ov[k]);
                }
                if (__any(need)) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const bool nk = leaf[k] && !ov[k];
                        const Box<T> eb = ld_box(bb + 6 * (n - 1 + (int64_t)(nk ? ~rf[k] : 0)));
                        ov[k] = ov[k] || (nk && overlap(q, eb, thr));
                    }
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int id = lr[k].id;
                    oid[k] = ov[k] && (!PARTIAL || !to_check[id] || qid < id) ? id : -1;
                }
                o0 = oid[0]; o1 = oid[1]; o2 = oid[2]; o3 = oid[3];
                r0 = rf[0]; r1 = rf[1]; r2 = rf[2]; r3 = rf[3];
            }
        }
        // stage this iteration's pairs in the wave's LDS buffer (tagged with lane and rank)
        {
            const unsigned c = (o0 >= 0 ? 1u : 0u) + (o1 >= 0 ? 1u : 0u) + (o2 >= 0 ? 1u : 0u) + (o3 >= 0 ? 1u : 0u);
            const unsigned long long b0 = __ballot(c & 1u), b1 = __ballot(c & 2u), b2 = __ballot(c & 4u);
            const unsigned below = lanes_below(b0) + 2u * lanes_below(b1) + 4u * lanes_below(b2);
            const unsigned tot = (unsigned)__popcll(b0) + 2u * (unsigned)__popcll(b1) + 4u * (unsigned)__popcll(b2);
            if (tot) {
                int f = fill[w];
                if (f + (int)tot > kStageCap) {     // would not fit: write out what is staged first
                    flush_stage(f);
                    f = 0;
                }
                int pos = f + (int)below;
                const unsigned lane_tag = (unsigned)lane << 10;
                if (o0 >= 0) { stage[w][pos] = o0; stag[w][pos++] = (unsigned short)(lane_tag | mine++); }
                if (o1 >= 0) { stage[w][pos] = o1; stag[w][pos++] = (unsigned short)(lane_tag | mine++); }
                if (o2 >= 0) { stage[w][pos] = o2; stag[w][pos++] = (unsigned short)(lane_tag | mine++); }
                if (o3 >= 0) { stage[w][pos] = o3; stag[w][pos] = (unsigned short)(lane_tag | mine++); }
                const int nf = f + (int)tot;
                if (nf >= kStage) {
                    flush_stage(nf);
                    if (lane == 0) fill[w] = 0;
                } else {
                    if (lane == 0) fill[w] = nf;
                }
            }
        }
        if (alive) {
            if (im == 0) {
                if (sp == 0) alive = false;
                else node = sizeof(StackT) < sizeof(int) ? sbase + (int)stack[--sp][tid] : (int)stack[--sp][tid];
            } else {
                // descend into the leftmost; the others wait on the stack, right to left, so
                // that the next one to the right comes off first
                const int lo = __ffs(im) - 1;
                node = lo == 0 ? r0 : lo == 1 ? r1 : lo == 2 ? r2 : r3;
                if ((im & 8u) && lo != 3) push(r3);
                if (alive && (im & 4u) && lo != 2) push(r2);
                if (alive && (im & 2u) && lo != 1) push(r1);
            }
        }
    }
    // final flush of the wave's staged pairs
    {
        const int f = fill[w];
        if (f > 0) flush_stage(f);
    }
}

// ---- candidate pairs of an index tree -------------------------------------------------------
// A traversal reports the pairs (p, l) of leaf positions, l > p, whose exact boxes overlap
// (collisions_static.cu:10-120, collisions_continuous.cu:127-230, :1079-1100); which tree it
// walks does not matter as long as node boxes contain their leaves'.  For the trees whose
// leaves are in index or Morton order (the index tree, and the resident simulation's fitted
// trees), positions are therefore grouped in chunks of 64 instead: a wave takes a group of
// queries, tests the group's union box against 64 chunks at a time (one per lane), the leaves
// of each hit chunk against it (one per lane), and the leaves that are left against the
// queries.  There is no per-lane walk and no stack: the walk (k_traverse) spent 560 lane
// instructions per pair that it found, on dependent node reads.  Traversal per pass, walk ->
// chunks: 130k cloth (5.9e7 pairs) 1,770 -> 390 us, packed 12 meshes (1.4e8 pairs) 9,300 ->
// 1,000 us, shuffled 32k 500 -> 63 us, garment 122k 220 -> 130 us, 33k f32 144 -> 38 us.

// The answer of k_prep's tree check is a word per batch element (`foreign`): every wave of
// k_pairs reads it, so it lies apart from the counters that they reserve pairs on.

constexpr int kPairQ = 16;        // queries per wave of k_pairs, each held by 64 / kPairQ lanes

// The union of a group's kPairQ boxes as two boxes: those of the queries up to and after the
// place where splitting the sequence gives the smallest extents, when that is much smaller
// than the union of all.  Consecutive triangles are neighbours except where a row of the mesh
// or one of its parts ends; the union over such a place spans everything between, and the few
// waves that hold one would take many times as long as the others (with single boxes 400 us
// instead of 144 on the 122k garment scene, 1,075 instead of 395 on the 130k cloth).
// A partial query's groups leave out the triangles that are not checked (empty boxes): with one
// in a hundred checked at random, 1M unordered triangles take 47 ms, 490 with whole groups (a walk per lane 392).
template <typename T> __device__ __forceinline__ float box_extent(const BoxReg<T> &a) {
    const float e = (float)(a.v[3] - a.v[0]) + (float)(a.v[4] - a.v[1]) + (float)(a.v[5] - a.v[2]);
    return e < 0.0f ? 0.0f : e;      // an empty box
}
template <typename T> __device__ __forceinline__ void split_union(const BoxReg<T> &q, int qi, BoxReg<T> &ua, BoxReg<T> &ub) {
    BoxReg<T> pre = q, suf = q;      // of the queries 0..qi and qi..kPairQ - 1
#pragma unroll
    for (int d = 1; d < kPairQ; d <<= 1) {
        // a lane without a source gets its own value back: joining it changes nothing
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            pre.v[k] = tmin(pre.v[k], __shfl_up(pre.v[k], d, kPairQ));
            pre.v[k + 3] = tmax(pre.v[k + 3], __shfl_up(pre.v[k + 3], d, kPairQ));
            suf.v[k] = tmin(suf.v[k], __shfl_down(suf.v[k], d, kPairQ));
            suf.v[k + 3] = tmax(suf.v[k + 3], __shfl_down(suf.v[k + 3], d, kPairQ));
        }
    }
    const float whole = __shfl(box_extent(pre), kPairQ - 1, kPairQ);
    float cost = box_extent(pre) + __shfl_down(box_extent(suf), 1, kPairQ);
    if (!(cost <= 3.0e38f) || qi == kPairQ - 1) cost = 3.0e38f;      // no split here (NaN included)
    float best = cost;
#pragma unroll
    for (int d = 1; d < kPairQ; d <<= 1) best = fminf(best, __shfl_xor(best, d, kPairQ));
    // the wave holds 64 / kPairQ groups: of the ballot only the lane's own group's bits
    const unsigned lowest = (unsigned)(__ballot(cost == best) >> (threadIdx.x & 63 & ~(kPairQ - 1))) & ((1u << kPairQ) - 1u);
    const int at = best < 0.75f * whole ? __ffs(lowest) - 1 : kPairQ - 1;
    const int from = at == kPairQ - 1 ? 0 : at + 1;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        ua.v[k] = __shfl(pre.v[k], at, kPairQ);
        ub.v[k] = __shfl(suf.v[k], from, kPairQ);
    }
}

// First launch of a query: (1) does the tree equal the index tree?  Any other tree sets
// `foreign` and goes through the checked general path; (2) the box of each chunk of 64 leaf
// positions and the two unions of each query group; (3) the vertex records (when tv is given).
// Blocks of 256 threads, partitioned by blockIdx.x: rows, leaves, corners.
template <typename T>
__global__ __launch_bounds__(256) void k_prep(const T *__restrict__ bb_all, const int64_t *__restrict__ tree_all, int64_t n, unsigned row_blocks,
                                              unsigned leaf_blocks, const uint8_t *__restrict__ to_check_all,
                                              T *__restrict__ chunk_all, T *__restrict__ group_all,
                                              const T *__restrict__ t0_all,
                                              const T *__restrict__ t1_all, T *__restrict__ tv_all, unsigned *__restrict__ foreign) {
    const int b = blockIdx.y;
    const int64_t rows = 2 * n - 1;
    if (blockIdx.x < row_blocks) {
        const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
        if (r >= rows) return;
        const int64_t *tree = tree_all + (int64_t)b * rows * 4;
        const int64_t l = tree[4 * r + 1], rr = tree[4 * r + 2];
        bool ok = r != 0 || tree[0] == -1;
        if (r < n - 1) {
            int64_t left, right;
            index_node_row(r, n, left, right);
            ok = ok && l == left && rr == right && tree[4 * left] == r && tree[4 * right] == r;
        } else {
            ok = ok && l == -1 && rr == -1 && tree[4 * r + 3] == r - (n - 1);
        }
        if (!ok) foreign[b] = 1u;
    } else if (blockIdx.x < row_blocks + leaf_blocks) {
        const int64_t p = (int64_t)(blockIdx.x - row_blocks) * 256 + threadIdx.x;
        if ((p & ~(int64_t)(kChunk - 1)) >= n) return;
        const int64_t nc = (n + kChunk - 1) >> kChunkBits;
        const int64_t at = p < n ? p : n - 1;
        const bool skip = to_check_all && !to_check_all[(int64_t)b * n + at];
        BoxReg<T> leaf = load_box(bb_all + ((int64_t)b * rows + (n - 1) + at) * 6);
        BoxReg<T> box = leaf;
#pragma unroll
        for (int d = 1; d < kChunk; d <<= 1) box_join_xor(box, d);
        if ((threadIdx.x & 63) == 0) store_box(chunk_all + ((int64_t)b * nc + (p >> kChunkBits)) * 6, box);
        // the two unions of each query group
        const int qi = threadIdx.x & (kPairQ - 1);
        if (skip) leaf = BoxReg<T>{{(T)INFINITY, (T)INFINITY, (T)INFINITY, -(T)INFINITY, -(T)INFINITY, -(T)INFINITY}};
        BoxReg<T> ua, ub;
        split_union(leaf, qi, ua, ub);
        if (qi == 0) {
            T *g = group_all + ((int64_t)b * nc * (kChunk / kPairQ) + p / kPairQ) * 12;
            store_box(g, ua);
            store_box(g + 6, ub);
        }
    } else {
        const int64_t i = (int64_t)(blockIdx.x - row_blocks - leaf_blocks) * 256 + threadIdx.x;
        if (i >= 3 * n) return;
        const T *a = t0_all + ((int64_t)b * 3 * n + i) * 3, *c = t1_all + ((int64_t)b * 3 * n + i) * 3;
        VRec<T> r;
        r.a[0] = a[0]; r.a[1] = a[1]; r.a[2] = a[2];
        r.a[3] = c[0] - a[0]; r.a[4] = c[1] - a[1]; r.a[5] = c[2] - a[2];
        reinterpret_cast<VRec<T> *>(tv_all)[(int64_t)b * 3 * n + i] = r;
    }
}

// Boxes of 64 chunks each, for meshes of more than kSuperFrom chunks.
template <typename T>
__global__ __launch_bounds__(256) void k_super_boxes(const T *__restrict__ chunk_all, int64_t nc, T *__restrict__ super_all) {
    const int b = blockIdx.y;
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if ((c & ~(int64_t)(kChunk - 1)) >= nc) return;
    BoxReg<T> box = load_box(chunk_all + ((int64_t)b * nc + (c < nc ? c : nc - 1)) * 6);
#pragma unroll
    for (int d = 1; d < kChunk; d <<= 1) box_join_xor(box, d);
    if ((threadIdx.x & 63) == 0) store_box(super_all + ((int64_t)b * ((nc + kChunk - 1) >> kChunkBits) + (c >> kChunkBits)) * 6, box);
}
// Testing every chunk costs each query chunk nc / 64 wave steps: up to 64 steps (262k
// triangles) that is far less than its leaf tests.
constexpr int64_t kSuperFrom = 4096;

constexpr int kPairEnt = 512;    // (leaf, query mask) entries per wave before a flush
constexpr int kPairWaves = 8;     // waves per block; their last entries share one reservation
constexpr int kPairSub = 64 / kPairQ;

// The reference's checkOverlap(q, other, thr) term by term (aabb.cu:101-111), with the other
// box already moved by the threshold.  Rounding is monotone, so a box that contains another's
// passes whenever that one does.
template <typename T> __device__ __forceinline__ bool box_hits(const BoxReg<T> &q, const BoxReg<T> &o) {
    return (q.v[0] <= o.v[3]) & (q.v[3] >= o.v[0]) & (q.v[1] <= o.v[4]) & (q.v[4] >= o.v[1]) & (q.v[2] <= o.v[5]) & (q.v[5] >= o.v[2]);
}
// A box moved outward by the threshold, as checkOverlap moves it (aabb.cu:101-111).
template <typename T> __device__ __forceinline__ void box_grow(BoxReg<T> &o, T thr) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        o.v[k] = o.v[k] - thr;
        o.v[k + 3] = o.v[k + 3] + thr;
    }
}

static_assert(kPairQ < 32, "a group's lanes as bits of a word");

// One wave per (group of kPairQ queries, split): split s of `splits` takes every splits-th
// chunk, so that small meshes fill the chip too.  The chunks that the group's union box meets
// are visited one after the other (the next one's boxes already on their way); the leaves that
// it meets gather in a list in LDS, from which each step takes four, one per 16 lanes, against
// the 16 queries.  16 queries rather than 64: consecutive triangles are a strip of the mesh,
// and a shorter strip's union box meets fewer leaves (1.7e8 leaf tests against 5.1e8 on the
// 130k cloth, of which 5.9e7 are pairs).  A step is about 14 vector instructions and 26 LDS
// cycles for 64 tests.  Results are kept as (leaf, mask of the queries) until kPairEnt - 64
// entries are there; then one reservation and one run of coalesced stores writes the pairs,
// grouped by leaf.  A reservation is a returning atomic on one device address (6-12 ns each,
// whatever the number of waves), so there are few of them.
// Tried and slower: 64 queries against leaf boxes read by scalar loads, and against boxes
// broadcast from LDS one leaf at a time (1,570 and 1,150 us on the 130k cloth, both bound by
// the latency of that one read per leaf).
// leaf_ids: the tree (its id column) when position and triangle id differ, else NULL.
template <typename T, bool PARTIAL>
__global__ __launch_bounds__(64 * kPairWaves) void k_pairs(const T *__restrict__ bb_all, const int64_t *__restrict__ leaf_ids, int64_t n, T thr,
                                                           const T *__restrict__ chunk_all, const T *__restrict__ super_all,
                                                           const T *__restrict__ group_all, int splits,
                                                           const uint8_t *__restrict__ to_check_all, const int32_t *__restrict__ mesh_end,
                                                           int2 *__restrict__ pairs_all, int64_t cap, const unsigned *__restrict__ foreign_all,
                                                           DevCounters *__restrict__ ctr_all) {
    struct alignas(16) SBox { BoxReg<T> box; };
    constexpr int kList = kChunk + kPairSub;      // a visit's leaves and fewer than a step's left over
    __shared__ SBox s_boxes[kPairWaves][kList];
    __shared__ int s_leafs[kPairWaves][kList];             // position
    __shared__ int s_idss[kPairWaves][PARTIAL ? kList : 1];    // id | (to_check << 31)
    __shared__ uint32_t s_ents[kPairWaves][kPairEnt];          // (position - ebase) << kPairQ | mask of the queries
    __shared__ unsigned long long s_base[kPairWaves];
    const int b = blockIdx.y, lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int qi = lane & (kPairQ - 1), sub = lane / kPairQ;
    SBox *s_box = s_boxes[w];
    int *s_leaf = s_leafs[w], *s_id = s_idss[w];
    uint32_t *s_ent = s_ents[w];
    DevCounters *ctr = ctr_all + b;
    if (foreign_all && foreign_all[b]) {
        if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(&ctr->flags, DEV_FOREIGN);
        return;
    }
    const int64_t rows = 2 * n - 1;
    const unsigned nq = (unsigned)((n + kPairQ - 1) / kPairQ), task = blockIdx.x * kPairWaves + w;
    const unsigned qg = task % nq, split = task / nq;      // split >= splits: an idle wave
    const int64_t nc = (n + kChunk - 1) >> kChunkBits;
    const T *bb = bb_all + ((int64_t)b * rows + (n - 1)) * 6;          // leaf rows
    const int64_t *ids = leaf_ids ? leaf_ids + ((int64_t)b * rows + (n - 1)) * 4 + 3 : nullptr;
    const T *chunks = chunk_all + (int64_t)b * nc * 6;
    const T *supers = super_all ? super_all + (int64_t)b * ((nc + kChunk - 1) >> kChunkBits) * 6 : nullptr;
    int2 *pairs = pairs_all + (int64_t)b * cap;
    const uint8_t *to_check = PARTIAL ? to_check_all + (int64_t)b * n : nullptr;

    const int last = (int)n - 1, p0 = (int)qg * kPairQ, p = p0 + qi, pc = p < last ? p : last;
    bool active = p <= last && split < (unsigned)splits;
    if (PARTIAL) active = active && to_check[pc] != 0;
    const bool any = __any(active);
    const BoxReg<T> q = load_box(bb + 6 * (int64_t)pc);
    const int qid = ids ? (int)ids[4 * (int64_t)pc] : pc;
    // the group's unions are the same for the whole wave: scalar loads, scalar operands
    using ConstT = const __attribute__((address_space(4))) T;
    ConstT *group = (ConstT *)(uintptr_t)(group_all + ((int64_t)b * nc * (kChunk / kPairQ) + qg) * 12);
    BoxReg<T> ua, ub;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        ua.v[k] = group[k];
        ub.v[k] = group[6 + k];
    }
    auto meets = [&](const BoxReg<T> &o) { return box_hits(ua, o) | box_hits(ub, o); };
    // packed meshes: leaves from lim on belong to later meshes (lim does not decrease with p)
    const int lim = mesh_end ? mesh_end[pc] : (int)n;
    const int lend = mesh_end ? mesh_end[p0 + kPairQ - 1 < last ? p0 + kPairQ - 1 : last] : (int)n;
    const int64_t cend = any ? ((int64_t)lend + kChunk - 1) >> kChunkBits : 0;
    const int64_t first = PARTIAL ? 0 : (int64_t)(p0 >> kChunkBits);
    int nent = 0, cnt = 0, ebase = 0;
    unsigned total = 0;

    // one step: the leaf of a list entry against this lane's query
    auto test = [&](const BoxReg<T> &o, int l, int id, bool valid) {
        bool h = valid & active & box_hits(q, o);
        if (PARTIAL) h = h & ((id >= 0) | (qid < (id & 0x7fffffff)));   // collisions_continuous.cu:1090: the lower id of two checked ones
        else h = h & (l > p);
        if (mesh_end) h = h & (l < lim);
        const unsigned long long m = __ballot(h);
        total += (unsigned)__popcll(m);
        if (qi == 0) s_ent[nent + sub] = ((uint32_t)(l - ebase) << kPairQ) | ((uint32_t)(m >> (sub * kPairQ)) & ((1u << kPairQ) - 1));
        nent += kPairSub;
    };
    auto step = [&](int e, bool valid) { test(s_box[e].box, s_leaf[e], PARTIAL ? s_id[e] : 0, valid); };
    // two steps, all their reads in flight together
    auto step2 = [&](int e) {
        const BoxReg<T> o0 = s_box[e].box, o1 = s_box[e - kPairSub].box;
        const int l0 = s_leaf[e], l1 = s_leaf[e - kPairSub], i0 = PARTIAL ? s_id[e] : 0, i1 = PARTIAL ? s_id[e - kPairSub] : 0;
        test(o0, l0, i0, true);
        test(o1, l1, i1, true);
    };
    // writes the entries' pairs from slot `base` on, four entries at a time
    auto emit = [&](unsigned long long base) {
#pragma unroll 2
        for (int e = 0; e < nent; e += kPairSub) {
            const uint32_t en = s_ent[e + sub];
            const bool on = ((en >> qi) & 1u) != 0u;
            const unsigned long long m = __ballot(on), d = base + lanes_below(m);
            if (on && d < (unsigned long long)cap) {
                const int l = ebase + (int)(en >> kPairQ), lid = ids ? (int)ids[4 * (int64_t)l] : l;
                pairs[d] = make_int2(min(qid, lid), max(qid, lid));
            }
            base += (unsigned long long)__popcll(m);
        }
    };
    auto flush = [&]() {
        wave_sync();
        unsigned long long base = 0;
        if (lane == 0) base = atomicAdd(&ctr->cand, (unsigned long long)total);
        emit(readfirstlane_u64(base));
        wave_sync();
        nent = 0;
        total = 0;
    };
    // the leaves left over, fewer than a step's
    auto finish_list = [&]() {
        if (cnt > 0) step(sub < cnt ? sub : 0, sub < cnt);
        cnt = 0;
    };

    for (int64_t c0 = splits == 1 ? first & ~(int64_t)(kChunk - 1) : first; c0 < cend; c0 += (int64_t)kChunk * splits) {
        if (supers && splits == 1) {
            BoxReg<T> sb = load_box(supers + 6 * (c0 >> kChunkBits));
            box_grow(sb, thr);
            if (!meets(sb)) continue;
        }
        const int64_t mine = c0 + split + (int64_t)lane * splits;
        BoxReg<T> cb = load_box(chunks + 6 * (mine < cend ? mine : cend - 1));
        box_grow(cb, thr);
        unsigned long long hit = __ballot(mine >= first && mine < cend && meets(cb));
        // the boxes of the next chunk are loaded while this one's leaves are tested
        auto next_leaf = [&](BoxReg<T> &box) -> int {
            const int k = __ffsll((long long)hit) - 1;
            hit &= hit - 1;
            const int l = (int)((c0 + split + (int64_t)k * splits) << kChunkBits) + lane;
            box = load_box(bb + 6 * (int64_t)(l < last ? l : last));
            return l;
        };
        BoxReg<T> nb;
        int nl = -1;
        if (hit) nl = next_leaf(nb);
        while (nl >= 0) {
            BoxReg<T> lb = nb;
            const int l = nl;
            nl = -1;
            if (hit) nl = next_leaf(nb);
            box_grow(lb, thr);
            const bool on = l <= last && (PARTIAL || l > p0) && meets(lb);
            const unsigned long long left = __ballot(on);
            if (!left) continue;
            const int l0 = __builtin_amdgcn_readfirstlane(l - lane);
            if (l0 + kChunk - ebase > 1 << (32 - kPairQ)) {
                // entries hold positions relative to ebase in 16 bits
                finish_list();
                if (nent) flush();
                ebase = l0;
            }
            if (on) {
                const int e = cnt + (int)lanes_below(left);
                s_box[e].box = lb;
                s_leaf[e] = l;
                if (PARTIAL) {
                    const int id = ids ? (int)ids[4 * (int64_t)l] : l;
                    s_id[e] = id | (to_check[id] ? (int)0x80000000 : 0);
                }
            }
            cnt += (int)__popcll(left);
            wave_sync();
            for (; cnt >= 2 * kPairSub; cnt -= 2 * kPairSub) step2(cnt - kPairSub + sub);
            if (cnt >= kPairSub) {
                step(cnt - kPairSub + sub, true);
                cnt -= kPairSub;
            }
            wave_sync();
            if (nent > kPairEnt - kList - kPairSub) flush();
        }
    }
    finish_list();
    // the waves' last entries: one reservation for the block
    if (lane == 0) s_base[w] = total;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long sum = 0;
        for (int k = 0; k < kPairWaves; ++k) {
            const unsigned long long t = s_base[k];
            s_base[k] = sum;
            sum += t;
        }
        const unsigned long long base = sum ? atomicAdd(&ctr->cand, sum) : 0ull;
        for (int k = 0; k < kPairWaves; ++k) s_base[k] += base;
    }
    __syncthreads();
    if (nent) emit(readfirstlane_u64(s_base[w]));
}

// ---- sub-primitive filter -----------------------------------------------------------------
// Candidate pairs -> the pairs of sub-primitives (9 edge-edge, 6 vertex-face) whose boxes
// overlap, with PP pairs per thread and one reservation per PP * kThreads pairs (the item
// counter is one contended device address: every reservation is a returning atomic on it).
//   SUB_STATIC: boxes grown by the threshold (proximity_static.cu:11-118) -> packed items;
//   SUB_MINCOL: swept boxes, written as (x, y, type) rows (find_minimal_candidates, :321-338).
// Items stay in pair order: pair u * kThreads + t of a tile comes after every pair
// u' * kThreads + t' < u * kThreads + t.  A tile's items are assembled in LDS (a 2-byte entry
// per item: pair in tile and type) and written as one contiguous run.  The moving pairs of
// the continuous narrow phase go through k_items.
enum { SUB_STATIC = 0, SUB_MINCOL = 1 };
// Exclusive block-wide scan of cnt (< 16) over the NT threads in thread order, without a
// reservation: the thread's offset; the block's sum in `total`.  Every thread calls it.
template <int NT = kThreads>
__device__ __forceinline__ unsigned block_scan_excl(unsigned cnt, unsigned &total) {
    __shared__ unsigned s_part[NT / 64 + 1];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    unsigned long long b0 = __ballot(cnt & 1u), b1 = __ballot(cnt & 2u), b2 = __ballot(cnt & 4u), b3 = __ballot(cnt & 8u);
    unsigned below = lanes_below(b0) + 2u * lanes_below(b1) + 4u * lanes_below(b2) + 8u * lanes_below(b3);
    if (lane == 0) s_part[w] = (unsigned)(__popcll(b0) + 2 * __popcll(b1) + 4 * __popcll(b2) + 8 * __popcll(b3));
    __syncthreads();
    unsigned before = 0, tot = 0;
#pragma unroll
    for (int q = 0; q < NT / 64; ++q) {
        const unsigned v = s_part[q];
        if (q < w) before += v;
        tot += v;
    }
    __syncthreads();
    total = tot;
    return before + below;
}

template <typename T, int KIND, int PP>
__global__ __launch_bounds__(kThreads) void k_subprim(const int2 *__restrict__ pairs_all, int64_t capK, int64_t c0, int64_t c1,
                                                      const T *__restrict__ src_all, int64_t n, T thr,
                                                      void *__restrict__ out_all, int64_t capM,
                                                      DevCounters *__restrict__ ctr_all) {
    static_assert(PP >= 1 && PP * kThreads <= 4096, "pair index and type fit 16 bits");
    constexpr int kEnt = 15 * PP * kThreads;      // (pair in tile) << 4 | type
    __shared__ unsigned short s_ent[kEnt];
    __shared__ int2 s_pair[PP * kThreads];
    __shared__ unsigned long long s_base;
    const int b = blockIdx.y, tid = threadIdx.x;
    DevCounters *ctr = ctr_all + b;
    const unsigned long long kc = ctr->cand;
    int64_t K = (int64_t)(kc < (unsigned long long)capK ? kc : (unsigned long long)capK);
    if (K > c1) K = c1;     // this launch covers the pairs [c0, c1)
    const int2 *pairs = pairs_all + (int64_t)b * capK;
    // SUB_STATIC: the t0 soup; otherwise the vertex records [x0 y0 z0 dx dy dz] per corner
    const T *src = src_all + (int64_t)b * n * (KIND == SUB_STATIC ? 9 : 18);
    int64_t *out = static_cast<int64_t *>(out_all) + (int64_t)b * capM * (KIND == SUB_MINCOL ? 3 : 1);
    constexpr int kTile = PP * kThreads;
    const int64_t ntiles = K > c0 ? (K - c0 + kTile - 1) / kTile : 0;
    CCC_FOR_TILES(tile, ntiles) {
        unsigned tot = 0;
#pragma unroll
        for (int u = 0; u < PP; ++u) {
            const int64_t i = c0 + tile * kTile + u * kThreads + tid;
            uint32_t mask = 0;
            int x = 0, y = 0;
            if (i < K) {
                const int2 pr = pairs[i];
                x = pr.x;
                y = pr.y;
                if (KIND == SUB_STATIC) {
                    V3<T> a[3], c[3];
#pragma unroll
                    for (int k = 0; k < 3; ++k) { a[k] = ld3(src + 9 * (int64_t)x + 3 * k); c[k] = ld3(src + 9 * (int64_t)y + 3 * k); }
                    if (!share_vertex(a, c)) mask = static_mask(a, c, thr);
                } else {
                    mask = moving_mask_axes(src, x, y);
                }
            }
            s_pair[u * kThreads + tid] = make_int2(x, y);
            unsigned t;
            unsigned k = tot + block_scan_excl((unsigned)__popc(mask), t);
            tot += t;
            while (mask) {
                const int type = __ffs(mask) - 1;
                mask &= mask - 1;
                s_ent[k++] = (unsigned short)(((u * kThreads + tid) << 4) | type);
            }
        }
        if (tid == 0) s_base = tot ? atomicAdd(&ctr->items, (unsigned long long)tot) : 0ull;
        __syncthreads();
        const unsigned long long base = s_base;
        const unsigned long long room = base < (unsigned long long)capM ? (unsigned long long)capM - base : 0ull;
        const unsigned lim = room < tot ? (unsigned)room : tot;
        for (unsigned k = tid; k < lim; k += kThreads) {
            const unsigned e = s_ent[k];
            const unsigned long long slot = base + k;
            const int2 pr = s_pair[e >> 4];
            if (KIND == SUB_MINCOL) {
                out[3 * slot] = pr.x; out[3 * slot + 1] = pr.y; out[3 * slot + 2] = (int64_t)(e & 15u);
            } else {
                out[slot] = pack_item(pr.x, pr.y, (int)(e & 15u));
            }
        }
        __syncthreads();
    }
}

// ---- items of the continuous narrow phase ---------------------------------------------------
// Moving candidate pairs -> the sub-primitive pairs whose swept boxes overlap
// (collisions_continuous.cu:234-318, :340-396), as 32-bit items (pair index within the chunk)
// << 4 | type for k_ccd.
// Each wave takes a contiguous run of pairs, 64 at a time (lane = pair), and keeps its
// edge-edge items in the kSegEE slots per pair that the run's place in the list gives it and
// its vertex-face items in the kSegVF behind them, so that k_ccd's 64-item tiles hold one kind,
// nothing is reserved while it runs and the list is as long as its pairs can make it; at the
// end the block reserves its tiles' descriptors (first slot, a multiple of 64, plus the number
// of items less one), which is all that k_ccd needs to find them.  A batch's
// entries are assembled in LDS and written as whole lines.  Bound by its record reads (0.95 L1
// accesses per cycle and CU: 18 of 16 bytes per lane and pair; vector issue 65%): 1.10 ms per pass of the 130k cloth
// (1.20 with blocks of 512 pairs and one reservation each), 33k f32 pass 56 -> 42 us.
constexpr int kBatch = 64;       // pairs per wave at a time
constexpr int kSegEE = 9, kSegVF = 6;
constexpr int kItemBlock = 4;    // waves per block

template <typename T>
__global__ __launch_bounds__(64 * kItemBlock) void k_items(const int2 *__restrict__ pairs_all, int64_t capK, int64_t c0, int64_t c1,
                                              const T *__restrict__ tv_all, int64_t n, uint32_t *__restrict__ list_all, int64_t capM,
                                              uint32_t *__restrict__ tile_all, int64_t capT,
                                              DevPartial *__restrict__ part_all, int nparts, DevCounters *__restrict__ ctr_all) {
    // (pair in batch) << 4 | type: edge-edge entries from the front, vertex-face ones from kSegEE kBatch on
    __shared__ unsigned short s_ents[kItemBlock][(kSegEE + kSegVF) * kBatch];
    __shared__ unsigned s_tiles[kItemBlock];
    const int b = blockIdx.y, lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned short *s_ent = s_ents[w];
    const unsigned long long kc = ctr_all[b].cand;
    int64_t K = (int64_t)(kc < (unsigned long long)capK ? kc : (unsigned long long)capK);
    if (K > c1) K = c1;         // this launch covers the pairs [c0, c1)
    const int64_t nbatch = K > c0 ? (K - c0 + kBatch - 1) / kBatch : 0;
    // the XCD's contiguous share of the batches, and this wave's run of it
    const int64_t per = (nbatch + kXcds - 1) / kXcds, step = (int64_t)gridDim.x / kXcds * kItemBlock, run = (per + step - 1) / step;
    const int64_t base = (int64_t)(blockIdx.x % kXcds) * per, k0 = ((int64_t)(blockIdx.x / kXcds) * kItemBlock + w) * run;
    const int64_t first = base + k0, last = base + (k0 + run < per ? k0 + run : per), stop = last < nbatch ? last : nbatch;
    const int2 *pairs = pairs_all + (int64_t)b * capK + c0;
    const T *tv = tv_all + (int64_t)b * n * 18;
    const uint32_t mine = first < stop ? (uint32_t)(stop - first) : 0u;       // this wave's batches
    const uint32_t slot_ee = (uint32_t)first * ((kSegEE + kSegVF) * kBatch), slot_vf = slot_ee + mine * (kSegEE * kBatch);
    uint32_t *list_ee = list_all + (int64_t)b * capM + slot_ee, *list_vf = list_all + (int64_t)b * capM + slot_vf;
    unsigned nee = 0, nvf = 0;      // items in the two segments
    int2 pr = make_int2(0, 0);
    if (first < stop && first * kBatch + lane < K - c0) pr = pairs[first * kBatch + lane];
    for (int64_t bt = first; bt < stop; ++bt) {
        const int64_t i = bt * kBatch + lane;
        uint32_t mask = 0;
        if (i < K - c0) mask = moving_mask_axes(tv, pr.x, pr.y);
        if (bt + 1 < stop && i + kBatch < K - c0) pr = pairs[i + kBatch];      // on its way for the next round
        // the batch's entries, each kind in pair order
        uint32_t mee = mask & 0x1ffu, mvf = mask >> 9;
        const unsigned ce = (unsigned)__popc(mee), cv = (unsigned)__popc(mvf);
        unsigned ke = 0, kv = 0, te = 0, tvf = 0;
#pragma unroll
        for (int bit = 0; bit < 4; ++bit) {
            const unsigned long long m = __ballot((ce >> bit) & 1u);
            ke += lanes_below(m) << bit;
            te += (unsigned)__popcll(m) << bit;
        }
#pragma unroll
        for (int bit = 0; bit < 3; ++bit) {
            const unsigned long long m = __ballot((cv >> bit) & 1u);
            kv += lanes_below(m) << bit;
            tvf += (unsigned)__popcll(m) << bit;
        }
        while (mee) {
            const int type = __ffs(mee) - 1;
            mee &= mee - 1;
            s_ent[ke++] = (unsigned short)((lane << 4) | type);
        }
        kv += kSegEE * kBatch;
        while (mvf) {
            const int type = 9 + __ffs(mvf) - 1;
            mvf &= mvf - 1;
            s_ent[kv++] = (unsigned short)((lane << 4) | type);
        }
        wave_sync();
        const uint32_t code = (uint32_t)(bt * kBatch) << 4;      // < 2^32: the chunk holds at most 2^28 pairs
        for (unsigned k = lane; k < te; k += 64) list_ee[nee + k] = code + s_ent[k];
        for (unsigned k = lane; k < tvf; k += 64) list_vf[nvf + k] = code + s_ent[kSegEE * kBatch + k];
        nee += te;
        nvf += tvf;
        wave_sync();
    }
    const unsigned tee = (nee + 63u) >> 6, tvf = (nvf + 63u) >> 6;
    if (lane == 0) s_tiles[w] = tee + tvf;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned sum = 0;
        for (int k = 0; k < kItemBlock; ++k) {
            const unsigned t = s_tiles[k];
            s_tiles[k] = sum;
            sum += t;
        }
        const unsigned at = sum ? (unsigned)atomicAdd(&ctr_all[b].tiles, (unsigned long long)sum) : 0u;
        for (int k = 0; k < kItemBlock; ++k) s_tiles[k] += at;
    }
    __syncthreads();
    uint32_t *tiles = tile_all + (int64_t)b * capT + s_tiles[w];
    for (unsigned k = lane; k < tee; k += 64) tiles[k] = slot_ee + 64 * k + (nee - 64 * k < 64u ? nee - 64 * k - 1u : 63u);
    for (unsigned k = lane; k < tvf; k += 64) tiles[tee + k] = slot_vf + 64 * k + (nvf - 64 * k < 64u ? nvf - 64 * k - 1u : 63u);
    if (lane == 0 && nee + nvf > 0)
        atomicAdd(&part_all[(int64_t)b * nparts + (blockIdx.x & (nparts - 1))].items, (unsigned long long)(nee + nvf));
}

// ---- fused narrow phase --------------------------------------------------------------------
// Per (x, y, type) item: tetrahedron (collisions_continuous.cu:36-124), coefficients
// (:409-445), solveCubic (:511-613), flatten of roots in [0, 1] (:732-765, including
// duplicates), filterCollisions (:640-684); then
//   COLLECT: rows (x, y, type) + root, truncated at the output capacity (:1028-1063);
//   IMPULSE: the accepted collisions of the block are staged in LDS and, once at least a
//            block's worth has gathered, every thread takes one and scatters its impulse
//            with atomics into dv / dx / cnt (collisions_impulses.cu:1312-1366).
// The tetrahedron is gathered again for the filter so that it is not live across the
// cubic solver (fewer VGPRs, more waves per SIMD).
enum { MODE_COLLECT = 0, MODE_IMPULSE = 1 };
// Threads (items) per k_ccd tile, in both modes: one wave per block, so that its phases need
// no workgroup barrier (k_ccd per step on the 130k cloth: 4 waves per block 206 ms, 2 waves
// 193 then 175, 1 wave 172.5 with barriers; the collect call 20.8 -> 17.1 ms once its tiles
// were one wave too).
constexpr int kCcdThreads = 64;
template <int MODE> constexpr int ccd_threads() { return kCcdThreads; }   // one wavefront per workgroup in both modes
// Staged collisions are scattered kFlush at a time, one lane each for their impulse
// parameters and in two halves of kFlush / 2 for the corner sums; fewer than kFlush stay
// staged between tiles and a tile adds at most 3 * kCcdThreads.
constexpr int kFlush = kCcdThreads;
constexpr int kHalfFlush = kFlush / 2;
constexpr int kImpStage = kFlush + 3 * kCcdThreads;

template <typename T>
__device__ __forceinline__ void scatter_impulse(const MTet<T> &m, int type, T root, int64_t x, int64_t y, const T *masses,
                                                T *dv, T *dx, int *cnt) {
    T q[4];
    int side[4], idx[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        type_corner(type, k, side[k], idx[k]);
        q[k] = masses[3 * (side[k] ? y : x) + idx[k]];
    }
    const ImpulseParams<T> ip = collision_impulse(m, type, root, q);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        V3<T> imp, imd;
        corner_impulse(ip, type, k, m.dv[k], imp, imd);
        const int64_t c = 3 * (side[k] ? y : x) + idx[k];
        atomicAdd(dv + 3 * c + 0, imp.x);
        atomicAdd(dv + 3 * c + 1, imp.y);
        atomicAdd(dv + 3 * c + 2, imp.z);
        atomicAdd(dx + 3 * c + 0, imd.x);
        atomicAdd(dx + 3 * c + 1, imd.y);
        atomicAdd(dx + 3 * c + 2, imd.z);
        atomicAdd(cnt + c, 1);
    }
}

// ---- order-independent impulse sums (deterministic mode) ----------------------------------
// A finite value v with |v| < 2^45 is held as the integer trunc(|v| * 2^80) with v's sign,
// split into three 42-bit limbs; every limb of every contribution is added with a 64-bit
// integer atomic, which is exact and associative, so the sums do not depend on the order of
// the additions (2^21 additions per limb fit in 64 bits).  Values that cannot be held set
// flag bits in a fourth word instead: 1 NaN, 2 +inf, 4 -inf, 8 out of range; the result
// is then what an fp64 sum gives (NaN, or the infinity) and NaN when out of range.
// Per triangle corner: 6 components (dv xyz, dx xyz) x 4 words; the upper half of the first
// component's flag word is the corner's collision count.
constexpr int kDetWords = kDetWordsPerCorner;
constexpr unsigned long long kDetOne = 1ull << 32;      // one collision in that word
constexpr double kTwo42 = 4398046511104.0, kTwo45 = 35184372088832.0, kTwo80 = 1208925819614629174706176.0;

// The three limbs of v (returns 0), or its flag bit when v cannot be held.
__device__ __forceinline__ unsigned det_split(double v, long long &l0, long long &l1, long long &l2) {
    if (!(fabs(v) < kTwo45))       // NaN fails this test too
        return v != v ? 1u : v == (double)INFINITY ? 2u : v == -(double)INFINITY ? 4u : 8u;
    const double sc = fabs(v) * kTwo80;                  // exact: a power-of-two scaling, < 2^125
    const double hi = floor(sc / (kTwo42 * kTwo42));    // < 2^41; exact
    const double r1 = sc - hi * (kTwo42 * kTwo42);      // the bits of sc below 2^84: exact
    const double mid = floor(r1 / kTwo42);              // < 2^42
    const double lo = floor(r1 - mid * kTwo42);         // < 2^42, fraction truncated
    l0 = (long long)lo;
    l1 = (long long)mid;
    l2 = (long long)hi;
    if (v < 0) { l0 = -l0; l1 = -l1; l2 = -l2; }
    return 0u;
}

__device__ __forceinline__ void det_add1(long long *a, double v) {
    long long l0, l1, l2;
    unsigned long long *u = reinterpret_cast<unsigned long long *>(a);
    const unsigned f = det_split(v, l0, l1, l2);
    if (f) {
        atomicOr(u + 3, (unsigned long long)f);
        return;
    }
    if (l0) atomicAdd(u + 0, (unsigned long long)l0);
    if (l1) atomicAdd(u + 1, (unsigned long long)l1);
    if (l2) atomicAdd(u + 2, (unsigned long long)l2);
}

// Limbs -> dv / dx of every corner: carries normalise the two low limbs into [0, 2^42),
// then hi * 2^84 + mid * 2^42 + lo is formed in double in that order and scaled by 2^-80.
template <typename T>
__global__ void k_det_finalize(const long long *__restrict__ acc, int64_t corners, T *__restrict__ dv, T *__restrict__ dx,
                               int *__restrict__ cnt) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= corners) return;
    const long long *a = acc + kDetWords * c;
    cnt[c] = (int)((unsigned long long)a[3] >> 32);
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        long long l0 = a[4 * k], l1 = a[4 * k + 1], l2 = a[4 * k + 2];
        const unsigned long long f = (unsigned long long)a[4 * k + 3];
        double v;
        if (f & 9ull) v = (double)NAN;
        else if ((f & 6ull) == 6ull) v = (double)NAN;
        else if (f & 2ull) v = (double)INFINITY;
        else if (f & 4ull) v = -(double)INFINITY;
        else {
            const long long c0 = l0 >> 42;
            l0 -= c0 * (1ll << 42);
            l1 += c0;
            const long long c1 = l1 >> 42;
            l1 -= c1 * (1ll << 42);
            l2 += c1;
            v = ((double)l2 * (kTwo42 * kTwo42) + (double)l1 * kTwo42 + (double)l0) / kTwo80;
        }
        T *o = k < 3 ? dv + 3 * c + k : dx + 3 * c + (k - 3);
        *o = (T)v;
    }
}

// Per-block sums of corner impulses: open addressing on the corner key 3 * triangle +
// corner, kImpSlots slots (a power of two), linear probing up to kImpProbe slots; a
// contribution that finds no slot goes to the global arrays directly.  A half flush adds
// 4 kHalfFlush = 128 corner shares, on fewer distinct corners (neighbouring collisions share
// corners); a whole flush at once overfilled the table (every share that found no slot
// spent the whole probe window first): k_ccd 16.2 -> 23.4 ms per pass on the 130k cloth.
constexpr int kImpSlots = 64;
constexpr int kImpProbe = 16;
constexpr int log2_exact(int v) { return v <= 1 ? 0 : 1 + log2_exact(v / 2); }
constexpr int kImpBits = log2_exact(kImpSlots);

template <typename T> struct ImpulseOut {
    T *dv, *dx;
    int *cnt;
    double *lines;
};

// Where the floating sums go: straight to dv, dx and cnt, or to one 64-byte line per corner
// (dv xyz, dx xyz, count, in double for both types; the pad stays 0), which k_line_sums or the
// simulation's update turns into them.  Atomics are bound by the lines they touch, not by
// words: 23.7e9 lane adds per second on random corners in the first form, 187e9 with eight
// lanes on each line, 64e9 in the first form on 64 neighbouring corners.  So lines serve
// where a slot's neighbours are not its neighbours in memory: given rows (from_collisions
// 104 -> 54 us) and simulations that fit their tree to a mesh in arbitrary order (k_ccd of ten
// passes on 32k shuffled triangles 6.96 -> 6.55 ms).  On meshes in spatial order k_ccd is
// bound by its instructions and L1 accesses, and the wider buffer costs more to clear and read
// (122k garment scene 4.31 direct, 4.36 by lines, its updates 115 and 143 us; 130k cloth 103.7
// and 103.9 ms).
enum : int { SUMS_DIRECT = 0, SUMS_LINES = 1, SUMS_DET = 2, SUMS_BY_ROWS = 3 };
constexpr int kLineWords = kLineWordsPerCorner;

// SUMS_BY_ROWS: in lines where the call has some (ImpulseOut::lines), else direct.
template <typename T, int SUMS> struct ImpTable {
    int *key;
    int *count;
    T *acc;     // [slot][dv.xyz, dx.xyz]
    __device__ static bool by_lines(const ImpulseOut<T> &to) { return SUMS == SUMS_LINES || (SUMS == SUMS_BY_ROWS && to.lines); }

    static constexpr size_t bytes() { return (size_t)kImpSlots * (2 * sizeof(int) + 6 * sizeof(T)); }
    __device__ static ImpTable over(unsigned char *raw) {
        ImpTable t;
        t.acc = reinterpret_cast<T *>(raw);
        t.key = reinterpret_cast<int *>(raw + (size_t)kImpSlots * 6 * sizeof(T));
        t.count = t.key + kImpSlots;
        return t;
    }
    __device__ void clear(int tid) {
        for (int s = tid; s < kImpSlots; s += kCcdThreads) {
            key[s] = -1;
            count[s] = 0;
#pragma unroll
            for (int c = 0; c < 6; ++c) acc[6 * s + c] = (T)0;
        }
    }
    // slot of `k`, inserting it if absent; -1 when the probe window is full
    __device__ int slot(int k) {
        int h = (int)(((unsigned)k * 2654435761u) >> (32 - kImpBits)) & (kImpSlots - 1);
        for (int p = 0; p < kImpProbe; ++p) {
            const int old = atomicCAS(&key[h], -1, k);
            if (old == -1 || old == k) return h;
            h = (h + 1) & (kImpSlots - 1);
        }
        return -1;
    }
    // adds one corner's impulse and position correction; to the global arrays directly
    // when the probe window is full
    __device__ void add(int64_t c, const V3<T> &imp, const V3<T> &imd, const ImpulseOut<T> &to) {
        const int s = slot((int)c);
        if (s >= 0) {
            atomicAdd(&acc[6 * s + 0], imp.x);
            atomicAdd(&acc[6 * s + 1], imp.y);
            atomicAdd(&acc[6 * s + 2], imp.z);
            atomicAdd(&acc[6 * s + 3], imd.x);
            atomicAdd(&acc[6 * s + 4], imd.y);
            atomicAdd(&acc[6 * s + 5], imd.z);
            atomicAdd(&count[s], 1);
        } else if (by_lines(to)) {
            double *l = to.lines + kLineWords * c;
            atomicAdd(l + 0, (double)imp.x);
            atomicAdd(l + 1, (double)imp.y);
            atomicAdd(l + 2, (double)imp.z);
            atomicAdd(l + 3, (double)imd.x);
            atomicAdd(l + 4, (double)imd.y);
            atomicAdd(l + 5, (double)imd.z);
            atomicAdd(l + 6, 1.0);
        } else {
            atomicAdd(to.dv + 3 * c + 0, imp.x);
            atomicAdd(to.dv + 3 * c + 1, imp.y);
            atomicAdd(to.dv + 3 * c + 2, imp.z);
            atomicAdd(to.dx + 3 * c + 0, imd.x);
            atomicAdd(to.dx + 3 * c + 1, imd.y);
            atomicAdd(to.dx + 3 * c + 2, imd.z);
            atomicAdd(to.cnt + c, 1);
        }
    }
    __device__ void drain(int tid, const ImpulseOut<T> &to) {
        if (by_lines(to)) {
            // eight lanes per slot, one line per slot
            const int word = tid & 7;
#pragma unroll 2
            for (int r = 0; r < kImpSlots * 8 / kCcdThreads; ++r) {
                const int s = r * (kCcdThreads / 8) + tid / 8, k = key[s];
                if (k < 0 || word > 6) continue;
                const double v = word < 6 ? (double)acc[6 * s + word] : (double)count[s];
                atomicAdd(to.lines + kLineWords * (int64_t)k + word, v);
            }
            return;
        }
        for (int s = tid; s < kImpSlots; s += kCcdThreads) {
            const int k = key[s];
            if (k < 0) continue;
            atomicAdd(to.dv + 3 * (int64_t)k + 0, acc[6 * s + 0]);
            atomicAdd(to.dv + 3 * (int64_t)k + 1, acc[6 * s + 1]);
            atomicAdd(to.dv + 3 * (int64_t)k + 2, acc[6 * s + 2]);
            atomicAdd(to.dx + 3 * (int64_t)k + 0, acc[6 * s + 3]);
            atomicAdd(to.dx + 3 * (int64_t)k + 1, acc[6 * s + 4]);
            atomicAdd(to.dx + 3 * (int64_t)k + 2, acc[6 * s + 5]);
            atomicAdd(to.cnt + k, count[s]);
        }
    }
};
static_assert(kImpSlots == 1 << kImpBits, "the slot count is a power of two");

// Lines -> dv, dx and cnt of every corner; with given rows (or none: NULL) if they were summed
// in lines.
template <typename T>
__global__ void k_line_sums(const double *__restrict__ lines, int64_t corners, T *__restrict__ dv, T *__restrict__ dx,
                            int *__restrict__ cnt, GivenRows given) {
    if (given.at[0] && !many_rows(given)) return;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < corners; c += (int64_t)gridDim.x * blockDim.x) {
        const double2 *l = reinterpret_cast<const double2 *>(lines + kLineWords * c);
        const double2 a = l[0], b = l[1], d = l[2], e = l[3];
        dv[3 * c + 0] = (T)a.x;
        dv[3 * c + 1] = (T)a.y;
        dv[3 * c + 2] = (T)b.x;
        dx[3 * c + 0] = (T)b.y;
        dx[3 * c + 1] = (T)d.x;
        dx[3 * c + 2] = (T)d.y;
        cnt[c] = (int)e.x;
    }
}

// The deterministic mode's per-block table: the same slots and probing as ImpTable, holding
// the two low limbs of each component as 64-bit integers (LDS integer atomics: exact, so the
// table's merge is order-independent too).  High limbs and flags, which cloth-scale
// corrections rarely have, go to the global limbs directly; each occupied slot then adds its
// two limbs per component and its count with global atomics.
struct DetTable {
    int *key;
    int *count;
    unsigned long long *acc;    // [slot][component][lo, mid]

    static constexpr size_t bytes() { return (size_t)kImpSlots * (2 * sizeof(int) + 12 * sizeof(unsigned long long)); }
    __device__ static DetTable over(unsigned char *raw) {
        DetTable t;
        t.acc = reinterpret_cast<unsigned long long *>(raw);
        t.key = reinterpret_cast<int *>(raw + (size_t)kImpSlots * 12 * sizeof(unsigned long long));
        t.count = t.key + kImpSlots;
        return t;
    }
    __device__ void clear(int tid) {
        for (int s = tid; s < kImpSlots; s += kCcdThreads) {
            key[s] = -1;
            count[s] = 0;
#pragma unroll
            for (int c = 0; c < 12; ++c) acc[12 * s + c] = 0ull;
        }
    }
    __device__ int slot(int k) {
        int h = (int)(((unsigned)k * 2654435761u) >> (32 - kImpBits)) & (kImpSlots - 1);
        for (int p = 0; p < kImpProbe; ++p) {
            const int old = atomicCAS(&key[h], -1, k);
            if (old == -1 || old == k) return h;
            h = (h + 1) & (kImpSlots - 1);
        }
        return -1;
    }
    __device__ void add(int64_t c, const double v[6], long long *det) {
        const int s = slot((int)c);
        unsigned long long *g = reinterpret_cast<unsigned long long *>(det + kDetWords * c);
        if (s < 0) {
#pragma unroll
            for (int k = 0; k < 6; ++k) det_add1(det + kDetWords * c + 4 * k, v[k]);
            atomicAdd(g + 3, kDetOne);
            return;
        }
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            long long l0, l1, l2;
            const unsigned f = det_split(v[k], l0, l1, l2);
            if (f) {
                atomicOr(g + 4 * k + 3, (unsigned long long)f);
                continue;
            }
            if (l0) atomicAdd(&acc[12 * s + 2 * k], (unsigned long long)l0);
            if (l1) atomicAdd(&acc[12 * s + 2 * k + 1], (unsigned long long)l1);
            if (l2) atomicAdd(g + 4 * k + 2, (unsigned long long)l2);
        }
        atomicAdd(&count[s], 1);
    }
    // sixteen lanes per slot: the two low limbs of the six components, then the count
    __device__ void drain(int tid, long long *det) {
        const int word = tid & 15;
#pragma unroll 2
        for (int r = 0; r < kImpSlots * 16 / kCcdThreads; ++r) {
            const int s = r * (kCcdThreads / 16) + tid / 16, k = key[s];
            if (k < 0 || word > 12) continue;
            const unsigned long long v = word < 12 ? acc[12 * s + word] : kDetOne * (unsigned long long)count[s];
            unsigned long long *g = reinterpret_cast<unsigned long long *>(det + kDetWords * (int64_t)k);
            if (v) atomicAdd(g + (word < 12 ? 4 * (word >> 1) + (word & 1) : 3), v);
        }
    }
};

// The same pointer, offset by a zero the optimiser cannot see through, so that loads
// through it are not merged with earlier loads of the same addresses.  The pointer itself
// keeps its provenance (a kernel argument), so its loads stay global-memory loads rather
// than flat ones.
template <typename P> __device__ __forceinline__ P *opaque_ptr(P *p) {
    int64_t z;
    asm volatile("s_mov_b64 %0, 0" : "=s"(z));
    return p + z;
}

// One tile of kCcdThreads items per step, in four phases.  Every workgroup of this kernel is
// one wavefront, so its list counters are wave-uniform registers (a lane's place in a list
// comes from a ballot) and the LDS exchanges between phases need only wave-level ordering
// (wave_sync), not a workgroup barrier, whose fence would also wait for the wave's
// outstanding global loads and atomics.
//   A  item ((pair index within the chunk) << 4 | type, its candidate pair read one tile
//      ahead) -> tetrahedron -> coefficients -> cubic_prepare, in registers;
//   B  the lane's roots inside [0, 1] (at most three) go to an LDS root list (item, root),
//      placed by a wave-wide scan of the counts;
//   C  filterCollisions per root in whole rounds of kCcdThreads roots (the tetrahedron is
//      gathered again); fewer than a round are carried to the next tile;
//   D  (impulse mode) accepted collisions wait in an LDS stage; kFlush at a time they are
//      scattered through an LDS hash table that reuses the root-list memory: one lane per
//      collision computes its impulse parameters (gathering the tetrahedron once for the
//      weights and once for the rest, so that this step needs no more registers than the
//      CCD phases); lanes l and l ^ 32 exchange them, and each half of the chunk adds its
//      corners' shares to the table and drains it.  The scatter stays in this
//      kernel: run as a kernel of its own over per-workgroup collision lists it took 14 ms
//      per pass on the 130k cloth against ~6 here (both with one sum per word), where other
//      workgroups' fp64 work hides its atomic latency.
//      (collect mode) accepted rows are written kCollectFlush at a time with one
//      reservation (the row counter is one contended device address).
// Each lane's item of the next tile is loaded while this tile is solved.  The cubic's
// branches diverge within the wave whatever the order of the items, so the items are not
// grouped by branch.  Occupancy: the impulse mode four waves per SIMD (128 VGPRs).  At five
// waves the impulse mode spills 41 registers (155 ms per step of the 130k cloth instead of
// 104); at three it was 13% slower.  What bounds it at four (10.4 ms per pass there, 6.2 M
// tiles): vector instructions issue 77% of the time, 750 per tile of which 55% fp64, and each
// CU's L1 takes 0.83 accesses per cycle with the corner gathers, 24.5 per gather instruction;
// fewer of one alone buys a third of its share.  A single-precision test of the roots from the
// registers of the item's lane, ahead of the filter's gather, took the gathers down by a fifth
// but left 56% of the roots undecided and cost 16% more instructions: 110 ms; not kept.
constexpr int kCollectFlush = 128;

// k_ccd's arguments, all of them, so that late_args finds them at the start of the kernel's
// argument memory.
template <typename T> struct CcdArgs {
    const uint32_t *items;      // [B][cap_items]
    const uint32_t *tiles;      // [B][cap_tiles]: first slot | items - 1
    const int2 *pairs;          // [B][cap_pairs], this chunk's from first_pair on
    const T *tv;                // vertex records
    DevCounters *ctr;
    DevPartial *parts;          // [B][nparts]
    int64_t cap_items, cap_tiles, cap_pairs, first_pair, n;
    // impulse mode
    const T *masses;
    T *dv, *dx;
    int *cnt;
    long long *det;
    double *lines;
    // collect mode
    int64_t *coll;
    T *roots;
    int64_t out_cap;
    int nparts;
};
// The arguments read again where they are used: what only the scatter or the output needs
// would otherwise sit in scalar registers, or in lanes of vector registers, through the solver
// (each spilled scalar costs a vector instruction per use, and the kernel is bound by those).
template <typename T> __device__ __forceinline__ const __attribute__((address_space(4))) CcdArgs<T> *late_args() {
    auto *p = (const __attribute__((address_space(4))) CcdArgs<T> *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}

// Waves per SIMD asked of the compiler: the deterministic table's LDS (12.3 KB) allows only
// 3.25 waves, and at four its registers spilled (37.28 against 37.06 ms per pass at three).
template <typename T, int MODE, int SUMS>
__global__ __launch_bounds__(kCcdThreads, MODE == MODE_IMPULSE ? (SUMS == SUMS_DET ? 3 : 4) : 5) void k_ccd(CcdArgs<T> arg) {
    constexpr int NT = kCcdThreads;     // items per tile: the lanes of the one wavefront
    constexpr bool DET = SUMS == SUMS_DET;
    using Table = ImpTable<T, SUMS == SUMS_LINES ? SUMS_LINES : SUMS_DIRECT>;
    static_assert(NT == 64, "one wavefront per workgroup");
    constexpr int kRootCapT = 3 * NT;
    // the root list (phases B-C) shares its LDS with the impulse table of phase D
    constexpr size_t kListBytes = (sizeof(int64_t) + sizeof(T)) * kRootCapT;
    constexpr size_t kTableBytes = DET ? DetTable::bytes() : Table::bytes();
    constexpr size_t kScatterBytes = MODE == MODE_IMPULSE ? kTableBytes : 0;
    __shared__ __align__(16) unsigned char s_raw[kListBytes > kScatterBytes ? kListBytes : kScatterBytes];
    int64_t *s_ritem = reinterpret_cast<int64_t *>(s_raw);
    T *s_rroot = reinterpret_cast<T *>(s_raw + sizeof(int64_t) * kRootCapT);
    // accepted collisions wait here: impulse mode until kFlush of them are scattered,
    // collect mode until kCollectFlush of them are written as output rows
    constexpr int kStageCap = MODE == MODE_IMPULSE ? kImpStage : kCollectFlush + 3 * NT;
    __shared__ int64_t s_item[kStageCap];
    __shared__ T s_root[kStageCap];
    // roots waiting for a whole round of the filter phase: fewer than NT, carried from tile to
    // tile as (item, root) so that the filter runs full waves
    __shared__ int64_t s_citem[NT];
    __shared__ T s_croot[NT];
    __shared__ uint32_t s_corner[16];
    const int b = blockIdx.y, tid = threadIdx.x;
    if (tid < 15) s_corner[tid] = corner_bytes(tid);
    wave_sync();
    const uint32_t *__restrict__ items = arg.items + (int64_t)b * arg.cap_items;
    const uint32_t *__restrict__ tiles = arg.tiles + (int64_t)b * arg.cap_tiles;
    const int2 *__restrict__ pairs = arg.pairs + (int64_t)b * arg.cap_pairs + arg.first_pair;     // this chunk's candidate pairs
    const T *__restrict__ tv = arg.tv + (int64_t)b * arg.n * 18;
    // wave-uniform counts: roots found, collisions scattered, staged collisions, carried roots
    unsigned long long nroots = 0, ncoll = 0;
    int fill = 0, ncarry = 0;

    // Staged collisions are scattered kFlush at a time: their corner impulses are first
    // summed per corner in an LDS hash table, then each occupied slot adds its sums to dv /
    // dx / cnt with one set of global atomics.
    static_assert(kScatterBytes <= sizeof(s_raw), "the impulse table fits the root-list buffer");
    static_assert(kFlush == NT && kHalfFlush == 32, "one lane per collision of a flush; halves of 32 lanes");
    Table tab = Table::over(s_raw);
    DetTable dtab = DetTable::over(s_raw);
    // Scatters staged collisions [0, f) in chunks of kFlush.  One lane per collision computes
    // its impulse parameters; the parameters of lanes l and l ^ 32 are then exchanged, and
    // each half of the chunk is summed in the LDS table and drained: collision j of the half
    // has corners 0 and 2 added by lane j and corners 1 and 3 by lane j + 32 (the corner
    // steps hold few registers, so the parameter step alone bounds this phase's register
    // use).
    auto flush = [&](int f) {
        for (int base = 0; base < f; base += kFlush) {
            const int nf = f - base < kFlush ? f - base : kFlush;
            auto *late = late_args<T>();
            const int64_t corner0 = (int64_t)blockIdx.y * late->n * 3;
            const T *masses = late->masses + corner0;
            ImpulseParams<T> ip{};
            if (tid < nf) {
                int64_t x, y;
                int type;
                unpack_item(s_item[base + tid], x, y, type);
                const T root = s_root[base + tid];
                // the tetrahedron is gathered once per step (from L2) rather than held
                // across both: that keeps this phase within the CCD phases' registers
                const ImpulseWeights<T> w = impulse_weights(gather_mtet_rec(opaque_ptr(tv), x, y, type, s_corner[type]), type, root);
                T q[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    int side, idx;
                    type_corner(type, k, side, idx);
                    q[k] = masses[3 * (side ? y : x) + idx];
                }
                ip = impulse_params(gather_mtet_rec(opaque_ptr(tv), x, y, type, s_corner[type]), type, root, w, q);
            }
            ImpulseParams<T> pp;      // lane l ^ 32's parameters
            pp.nrm.x = __shfl_xor(ip.nrm.x, 32);
            pp.nrm.y = __shfl_xor(ip.nrm.y, 32);
            pp.nrm.z = __shfl_xor(ip.nrm.z, 32);
            pp.im0 = __shfl_xor(ip.im0, 32);
            pp.im1 = __shfl_xor(ip.im1, 32);
            pp.keep = __shfl_xor(ip.keep, 32);
            const int j = tid & (kHalfFlush - 1), hi = tid >> 5;
            for (int h = 0; h * kHalfFlush < nf; ++h) {
                const int nh = nf - h * kHalfFlush < kHalfFlush ? nf - h * kHalfFlush : kHalfFlush;
                late = late_args<T>();
                ImpulseOut<T> to{};
                if (SUMS == SUMS_DIRECT) to = ImpulseOut<T>{late->dv + 3 * corner0, late->dx + 3 * corner0, late->cnt + corner0, nullptr};
                if (SUMS == SUMS_LINES) to.lines = late->lines + kLineWords * corner0;
                long long *det = DET ? late->det + corner0 * kDetWords : nullptr;
                if (DET) dtab.clear(tid);
                else tab.clear(tid);
                wave_sync();
                if (j < nh) {
                    // collision h * 32 + j: this lane's own when hi == h, else lane l ^ 32's
                    const bool own = hi == h;
                    ImpulseParams<T> cp;
                    cp.nrm.x = own ? ip.nrm.x : pp.nrm.x;
                    cp.nrm.y = own ? ip.nrm.y : pp.nrm.y;
                    cp.nrm.z = own ? ip.nrm.z : pp.nrm.z;
                    cp.im0 = own ? ip.im0 : pp.im0;
                    cp.im1 = own ? ip.im1 : pp.im1;
                    cp.keep = own ? ip.keep : pp.keep;
                    int64_t x, y;
                    int type;
                    unpack_item(s_item[base + h * kHalfFlush + j], x, y, type);
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        const int k = 2 * r + hi;
                        int side, idx;
                        type_corner(type, k, side, idx);
                        const int64_t c = 3 * (side ? y : x) + idx;
                        V3<T> v, dvk;
                        ld_vrec(opaque_ptr(tv), c, v, dvk);
                        V3<T> imp, imd;
                        corner_impulse(cp, type, k, dvk, imp, imd);
                        if (DET) {
                            const double v[6] = {(double)imp.x, (double)imp.y, (double)imp.z, (double)imd.x, (double)imd.y, (double)imd.z};
                            dtab.add(c, v, det);
                        } else {
                            tab.add(c, imp, imd, to);
                        }
                    }
                }
                wave_sync();
                if (DET) dtab.drain(tid, det);
                else tab.drain(tid, to);
                wave_sync();
            }
        }
    };

    // Collect mode: the staged collisions [0, f) to output rows (rows past out_cap are
    // counted, not written).
    auto write_rows = [&](int f) {
        unsigned long long ob = 0;
        auto *late = late_args<T>();
        const int64_t out_cap = late->out_cap;
        if (tid == 0 && f) ob = atomicAdd(&late->ctr[blockIdx.y].coll, (unsigned long long)f);
        ob = readfirstlane_u64(ob);
        int64_t *coll = late->coll + (int64_t)blockIdx.y * out_cap * 3;
        T *roots = late->roots + (int64_t)blockIdx.y * out_cap;
        for (int j = tid; j < f; j += NT) {
            const unsigned long long slot = ob + (unsigned long long)j;
            if (slot < (unsigned long long)out_cap) {
                int64_t x, y;
                int type;
                unpack_item(s_item[j], x, y, type);
                coll[3 * slot] = x; coll[3 * slot + 1] = y; coll[3 * slot + 2] = type;
                roots[slot] = s_root[j];
            }
        }
        wave_sync();
    };

    // Filter of one root per lane where `on` (filterCollisions); accepted collisions join the
    // stage in lane order.  Every lane calls it.
    auto filter_round = [&](bool on, int64_t rit, T root) {
        bool acc = false;
        if (on) {
            int64_t x, y;
            int type;
            unpack_item(rit, x, y, type);
            acc = filter_collision(gather_mtet_rec(opaque_ptr(tv), x, y, type, s_corner[type]), type, root);
        }
        const unsigned long long m = __ballot(acc);
        if (acc) {
            const int p = fill + (int)lanes_below(m);
            s_item[p] = rit;
            s_root[p] = root;
        }
        fill += (int)__popcll(m);
    };

    // The tiles of CCC_FOR_TILES, walked by hand so that each lane's item of the next tile is
    // loaded one tile ahead (after this tile's gathers are issued) and its candidate pair
    // after phase B; kNoItem: no item.  An item is (pair index within the chunk) << 4 | type;
    // the packed (x, y, type) form is made when the tile starts.  A tile's items are of one
    // kind (k_items), so its roots and collisions take one branch of the filter and of the
    // impulse in the whole wave, but for the roots carried over a change.
    // tile counts in 32 bits (at most 15 * 2^28 / 64 tiles): the kernel's uniform values fill
    // the scalar registers
    const int ntiles = (int)arg.ctr[b].tiles;
    const int tper = (ntiles + kXcds - 1) / kXcds, tstep = (int)gridDim.x / kXcds;
    const int tbase = (int)(blockIdx.x % kXcds) * tper;
    // Each block takes one contiguous run of tiles: its collisions share corners, and the
    // blocks running beside it are far away in the list, so that their atomics fall on other
    // corners (tiles dealt out one by one: 129.6 instead of 104 ms per step of the 130k cloth,
    // 8.5 instead of 6.8 of the garment scene, in the order that k_pairs writes its pairs).
    // With few tiles the runs are up to kLongRun tiles long, on fewer blocks, so that 8,192
    // blocks share them: a block's start and its last, partial rounds cost as much as several
    // tiles, and in collect mode one more reservation of rows (23k triangles, 93k tiles on
    // 32,768 blocks: 375 us; runs of 8: 201; of 16 and rows written 128 at a time: 182.  Runs
    // of 16 in impulse mode, pass of 33k triangles in fp32: 335 -> 351).
    constexpr int kLongRun = MODE == MODE_COLLECT ? 16 : 8;
    const int tall = (tper + tstep - 1) / tstep, tfew = (ntiles + 8191) / 8192, tmin = tfew < kLongRun ? tfew : kLongRun;
    const int trun = tall > tmin ? tall : tmin;
    const int tfirst = (int)blockIdx.x / kXcds * trun, tlast = tfirst + trun < tper ? tfirst + trun : tper;
    constexpr uint32_t kNoItem = 0xffffffffu;   // type 15 does not exist
    auto item_of = [&](int k) -> uint32_t {
        if (!(k < tlast && tbase + k < ntiles)) return kNoItem;
        const uint32_t d = tiles[tbase + k];
        return tid <= (int)(d & 63u) ? items[(d & ~63u) + (uint32_t)tid] : kNoItem;
    };
    // the next tile's item waits as its pair (registers) and its type (LDS, 15: no item), so
    // that it holds no more registers than the packed item through phases C and D
    __shared__ unsigned char s_ntype[NT];
    __shared__ int64_t s_myitem[NT];
    uint32_t next_item = item_of(tfirst);
    int2 next_pair = make_int2(0, 0);
    if (next_item != kNoItem) next_pair = pairs[next_item >> 4];
    s_ntype[tid] = (unsigned char)(next_item & 15u);
    for (int tk = tfirst; tk < tlast && tbase + tk < ntiles; ++tk) {
        // ---- A: coefficients and branch of the lane's item
        const int ntype = s_ntype[tid];
        const int64_t it = ntype != 15 ? pack_item(next_pair.x, next_pair.y, ntype) : (int64_t)-1;
        int code = CUBIC_NONE;
        CubicState st;
        if (it >= 0) {
            int64_t x, y;
            int type;
            unpack_item(it, x, y, type);
            T cf[4];
            {
                const MTet<T> m = gather_mtet_rec(tv, x, y, type, s_corner[type]);
                cubic_coeffs(m, cf);
            }
            code = cubic_prepare(cf[0], cf[1], cf[2], cf[3], st);
        }
        s_myitem[tid] = it;     // read back for the root list, not held through the solver
        next_item = item_of(tk + 1);
        // ---- B: the lane's roots in [0, 1], in the order found, to the root list
        T r0, r1, r2;
        const int nk = cubic_roots<T>(code, st, r0, r1, r2);
        {
            const unsigned long long b0 = __ballot(nk & 1), b1 = __ballot(nk & 2);
            const int off = (int)(lanes_below(b0) + 2u * lanes_below(b1));
            // the item as parked in LDS before the solver (the empty asm keeps the compiler
            // from holding it in registers instead: two more VGPRs spilled the solver)
            asm volatile("" ::: "memory");
            const int64_t itb = s_myitem[tid];
            if (nk > 0) { s_ritem[off] = itb; s_rroot[off] = r0; }
            if (nk > 1) { s_ritem[off + 1] = itb; s_rroot[off + 1] = r1; }
            if (nk > 2) { s_ritem[off + 2] = itb; s_rroot[off + 2] = r2; }
            const int nr = (int)(__popcll(b0) + 2 * __popcll(b1));
            nroots += (unsigned long long)nr;
            wave_sync();
            // the next tile's candidate pair (its item arrived during phase B)
            if (next_item != kNoItem) next_pair = pairs[next_item >> 4];
            s_ntype[tid] = (unsigned char)(next_item & 15u);
            // ---- C: filter one root per lane in whole rounds over the carried roots
            // followed by this tile's; the rest (fewer than NT) is carried to the next tile
            const int total = ncarry + nr, full = total / NT * NT;
            for (int base = 0; base < full; base += NT) {
                const int j = base + tid;
                int64_t rit;
                T root;
                if (j < ncarry) {
                    rit = s_citem[j];
                    root = s_croot[j];
                } else {
                    rit = s_ritem[j - ncarry];
                    root = s_rroot[j - ncarry];
                }
                filter_round(true, rit, root);
            }
            wave_sync();      // the carried roots have been read
            // with a whole round the carry was consumed and the rest is this tile's tail;
            // without one, this tile's roots join the carry
            const int from = full > 0 ? full - ncarry : 0, to = full > 0 ? 0 : ncarry;
            for (int k = tid; k < total - full - to; k += NT) {
                s_citem[to + k] = s_ritem[from + k];
                s_croot[to + k] = s_rroot[from + k];
            }
            ncarry = total - full;
            wave_sync();      // the root list has been read (its memory holds the table)
        }
        // ---- D: scatter the staged impulses in whole chunks; the rest moves to the front
        if (MODE == MODE_IMPULSE) {
            if (fill >= kFlush) {
                const int done = fill - fill % kFlush;
                flush(done);
                ncoll += (unsigned long long)done;
                // [done, fill) and [0, fill - done) do not overlap: fill - done < kFlush <= done
                if (tid < fill - done) {
                    s_item[tid] = s_item[done + tid];
                    s_root[tid] = s_root[done + tid];
                }
                wave_sync();
                fill -= done;
            }
        } else if (fill >= kCollectFlush) {
            // ---- D (collect): write the staged rows once kCollectFlush have gathered
            write_rows(fill);
            fill = 0;
        }
    }
    // the carried roots' last, partial round
    filter_round(tid < ncarry, s_citem[tid], s_croot[tid]);
    wave_sync();
    if (MODE == MODE_IMPULSE) {
        flush(fill);
        ncoll += (unsigned long long)fill;
    } else {
        write_rows(fill);
    }
    if (tid == 0) {
        auto *late = late_args<T>();
        DevPartial *part = late->parts + (int64_t)b * late->nparts + (blockIdx.x & (late->nparts - 1));
        if (nroots) atomicAdd(&part->roots, nroots);
        if (MODE == MODE_IMPULSE && ncoll) atomicAdd(&part->coll, ncoll);
    }
}

// The narrow phase's device arithmetic on given inputs, for tests: what 0-4 evaluates the
// portable cbrt / acos / sin / cos / cbrtf of ccc_libm.h at x[i]; what 5 runs cubic_prepare +
// cubic_roots<double> on the coefficients c3 c2 c1 c0 = x[4i..4i+3] and writes the number of
// roots kept in [0, 1] and those roots to y[4i..4i+3].
__global__ void k_device_math(int what, const double *__restrict__ x, double *__restrict__ y, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (what == 5) {
        CubicState st;
        const int code = cubic_prepare(x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3], st);
        double r0, r1, r2;
        const int k = cubic_roots<double>(code, st, r0, r1, r2);
        y[4 * i] = (double)k;
        y[4 * i + 1] = k > 0 ? r0 : 0.0;
        y[4 * i + 2] = k > 1 ? r1 : 0.0;
        y[4 * i + 3] = k > 2 ? r2 : 0.0;
        return;
    }
    const double v = x[i];
    y[i] = what == 0 ? pm_cbrt(v) : what == 1 ? pm_acos(v) : what == 2 ? pm_sin(v) : what == 3 ? pm_cos(v)
         : what == 4 ? (double)pm_cbrtf((float)v) : what == 6 ? div_exact<3>(v) : what == 7 ? div_exact<27>(v)
         : what == 8 ? div_exact_finite<3>(v) : what == 9 ? sqrt_no_rescale(v)
         : what == 10 ? (unit_ratio(v, x[n + i]) ? 1.0 : 0.0)
                      : (unit_ratio((float)v, (float)x[n + i]) ? 1.0 : 0.0);
}

// compute_impulses_from_collisions (collisions_impulses.cu:1736-1880) over given rows;
// rows with a negative or out-of-range index are skipped.  Bound by its atomics: added one by
// one they are 28 per row (450 us for 357k collisions of a 23k-triangle cloth, 22e9 atomics
// per second).  So the corner sums of 32 rows at a time go through the same LDS table as
// k_ccd's first, the collision lists being written in runs of neighbouring pairs: 105 us.
// 64 rows in 128 slots take 143 us, 16 rows in 64 slots 120, tables kept over 128 rows 170 to
// 190: more shares find their slots taken and probe on, or more slots are drained for the same
// sums.  One wave per block takes 64 rows, and then every gridDim.x-th 64 so that all waves
// share the padding at a list's end, read up to four steps ahead.  A short list is bound
// by what one wave does in series: with 128 rows in a row 5,000 rows on 10k triangles took
// 42 us (by single atomics 37.5), with 64 32, and lists of up to kShortRows take 32 per wave
// (30).  Meshes whose corner numbers do not fit the table's 32-bit keys take the atomics one
// by one.
constexpr int64_t kShortRows = 32768;
template <typename T, bool TABLE, int SUMS>
__global__ __launch_bounds__(kCcdThreads) void k_from_collisions(const int64_t *__restrict__ coll_all, const T *__restrict__ roots_all,
                                                                 int64_t m, const T *__restrict__ t0_all, const T *__restrict__ t1_all,
                                                                 const T *__restrict__ masses_all, int64_t n, T *__restrict__ dv_all,
                                                                 T *__restrict__ dx_all, int *__restrict__ cnt_all, double *__restrict__ lines_all,
                                                                 int per_wave, GivenRows given) {
    __shared__ __align__(16) unsigned char s_raw[TABLE ? ImpTable<T, SUMS>::bytes() : 16];
    const int b = blockIdx.y, lane = threadIdx.x;
    const int64_t *coll = coll_all + (int64_t)b * m * 3;
    const T *roots = roots_all + (int64_t)b * m;
    const T *t0 = t0_all + (int64_t)b * n * 9, *t1 = t1_all + (int64_t)b * n * 9, *masses = masses_all + (int64_t)b * n * 3;
    ImpulseOut<T> to{dv_all + (int64_t)b * n * 9, dx_all + (int64_t)b * n * 9, cnt_all + (int64_t)b * n * 3,
                     nullptr};
    bool asked = SUMS != SUMS_BY_ROWS;      // where the sums go, looked up at the first row
    ImpTable<T, SUMS> tab = ImpTable<T, SUMS>::over(s_raw);
    // four rows' first columns are on their way together, so that padding is passed over at the
    // memory's rate
    const int64_t step = (int64_t)gridDim.x * per_wave, end = lane < per_wave ? m : 0;
    int64_t x1 = -1, x2 = -1, x3 = -1, y1 = -1, type1 = -1;
    int left = 0;
    for (int64_t i = (int64_t)blockIdx.x * per_wave + lane; i - lane < m; i += step) {
        int64_t x = x1, y = y1, type = type1;
        if (left == 0) {
            x = x1 = x2 = x3 = -1;
            if (i < end) { x = coll[3 * i]; y = coll[3 * i + 1]; type = coll[3 * i + 2]; }
            if (i + step < end) x1 = coll[3 * (i + step)];
            if (i + 2 * step < end) x2 = coll[3 * (i + 2 * step)];
            if (i + 3 * step < end) x3 = coll[3 * (i + 3 * step)];
            left = 4;
        } else {
            x1 = x2;
            x2 = x3;
        }
        if (--left > 0 && x1 >= 0) { y1 = coll[3 * (i + step) + 1]; type1 = coll[3 * (i + step) + 2]; }
        if (!__any(x >= 0)) continue;
        if (!asked) {
            asked = true;
            if (many_rows(given)) to.lines = lines_all + (int64_t)b * n * 3 * kLineWords;
        }
        const bool on = !(x < 0 || y < 0 || type < 0 || type > 14 || x >= n || y >= n);
        if (!__any(on)) continue;
        MTet<T> mt{};
        T root = (T)0;
        if (on) {
            root = roots[i];
            mt = gather_mtet(t0, t1, x, y, (int)type);
        }
        if (!TABLE) {
            if (on) scatter_impulse(mt, (int)type, root, x, y, masses, to.dv, to.dx, to.cnt);
            continue;
        }
        ImpulseParams<T> ip{};
        if (on) {
            T q[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                int side, idx;
                type_corner((int)type, k, side, idx);
                q[k] = masses[3 * (side ? y : x) + idx];
            }
            ip = collision_impulse(mt, (int)type, root, q);
        }
        for (int h = 0; h < 2; ++h) {
            const bool mine = on && (lane >> 5) == h;
            if (!__any(mine)) continue;
            tab.clear(lane);
            wave_sync();
            if (mine) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    int side, idx;
                    type_corner((int)type, k, side, idx);
                    V3<T> imp, imd;
                    corner_impulse(ip, (int)type, k, mt.dv[k], imp, imd);
                    tab.add(3 * (side ? y : x) + idx, imp, imd, to);
                }
            }
            wave_sync();
            tab.drain(lane, to);
            wave_sync();
        }
    }
}

// Items per thread and reservation of the static narrow phases.  A block's rows take one atomic
// on the row counter, about 10 ns each whatever the number of blocks, which bounded k_proximity
// (597k items in 2.3k blocks: 33.4 us; two items per thread 23.8, four 20.0, eight 24.5) and
// k_sat (629k pairs: 34.7 us; two 26.5, four 28.2, eight 34.7) at one item per thread.  Lists of
// up to 512 blocks keep one: they are too few to be held up, and a thread's items are worked on
// one after another.
constexpr int kProximityItems = 4, kSatPairs = 2;
__device__ __forceinline__ int items_per_thread(int64_t count, int most) { return count > (int64_t)512 * kThreads ? most : 1; }

// Static proximity per item (proximity_static.cu:435-508): distance by type, kept when
// 0 <= d <= threshold; rows (x, y, type) truncated at the output capacity.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_proximity(const int64_t *__restrict__ items_all, int64_t capM,
                                                        const T *__restrict__ t0_all, int64_t n, T thr,
                                                        int64_t *__restrict__ out_all, int64_t out_cap,
                                                        DevCounters *__restrict__ ctr_all) {
    const int b = blockIdx.y;
    DevCounters *ctr = ctr_all + b;
    const unsigned long long mc = ctr->items;
    const int64_t M = (int64_t)(mc < (unsigned long long)capM ? mc : (unsigned long long)capM);
    const int64_t *items = items_all + (int64_t)b * capM;
    const T *t0 = t0_all + (int64_t)b * n * 9;
    int64_t *out = out_all + (int64_t)b * out_cap * 3;
    const int per = items_per_thread(M, kProximityItems);
    const int64_t size = (int64_t)per * kThreads, ntiles = (M + size - 1) / size;
    CCC_FOR_TILES(tile, ntiles) {
        unsigned keep = 0;
        for (int e = 0; e < per; ++e) {
            const int64_t i = tile * size + e * kThreads + threadIdx.x;
            if (i >= M) break;
            int64_t x, y;
            int type;
            unpack_item(items[i], x, y, type);
            V3<T> p[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                int side, idx;
                type_corner(type, k, side, idx);
                p[k] = ld3(t0 + 9 * (side ? y : x) + 3 * idx);
            }
            T d;
            if (type < 9) d = dist_ee(p[0], p[1], p[2], p[3]);
            else if (type < 12) d = dist_vf(p[0], p[1], p[2], p[3]);
            else d = dist_vf(p[1], p[2], p[3], p[0]);
            keep |= (d <= thr && d >= 0) ? 1u << e : 0u;
        }
        unsigned long long slot = block_reserve(&ctr->coll, (unsigned)__popc(keep));
        for (; keep; keep &= keep - 1, ++slot) {
            if (slot >= (unsigned long long)out_cap) break;
            int64_t x, y;
            int type;
            unpack_item(items[tile * size + (__ffs(keep) - 1) * kThreads + threadIdx.x], x, y, type);
            out[3 * slot] = x; out[3 * slot + 1] = y; out[3 * slot + 2] = type;
        }
    }
}

// Static triangle-triangle test per candidate pair (collisions_static.cu:123-159):
// 17-axis SAT with threshold and no shared vertex; rows (x, y).
template <typename T>
__global__ __launch_bounds__(kThreads) void k_sat(const int2 *__restrict__ pairs_all, int64_t capK, const T *__restrict__ t0_all,
                                                  int64_t n, T thr, int64_t *__restrict__ out_all, int64_t out_cap,
                                                  DevCounters *__restrict__ ctr_all) {
    const int b = blockIdx.y;
    DevCounters *ctr = ctr_all + b;
    const unsigned long long kc = ctr->cand;
    const int64_t K = (int64_t)(kc < (unsigned long long)capK ? kc : (unsigned long long)capK);
    const int2 *pairs = pairs_all + (int64_t)b * capK;
    const T *t0 = t0_all + (int64_t)b * n * 9;
    int64_t *out = out_all + (int64_t)b * out_cap * 2;
    const int per = items_per_thread(K, kSatPairs);
    const int64_t size = (int64_t)per * kThreads, ntiles = (K + size - 1) / size;
    CCC_FOR_TILES(tile, ntiles) {
        unsigned keep = 0;
        for (int e = 0; e < per; ++e) {
            const int64_t i = tile * size + e * kThreads + threadIdx.x;
            if (i >= K) break;
            const int2 pr = pairs[i];
            V3<T> a[3], c[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) { a[k] = ld3(t0 + 9 * (int64_t)pr.x + 3 * k); c[k] = ld3(t0 + 9 * (int64_t)pr.y + 3 * k); }
            keep |= (sat_overlap(a, c, thr) && !(count_shared(a, c) > 0)) ? 1u << e : 0u;
        }
        unsigned long long slot = block_reserve(&ctr->coll, (unsigned)__popc(keep));
        for (; keep; keep &= keep - 1, ++slot) {
            if (slot >= (unsigned long long)out_cap) break;
            const int2 pr = pairs[tile * size + (__ffs(keep) - 1) * kThreads + threadIdx.x];
            out[2 * slot] = pr.x; out[2 * slot + 1] = pr.y;
        }
    }
}

// ---- host orchestration ---------------------------------------------------------------------

// Triangle-edge queries over the candidate pairs of a threshold-0 traversal, one pair per
// thread: SAT with at most `allow` shared vertices (collisions_static.cu:123-159), then the
// six edges cid 0..2 = (v0v1, v1v2, v2v0) of x against y and 3..5 of y against x.
//   TE_COLLISIONS  (allow 0) rows (x, y, cid, loop) + edge coefficient for every edge that
//                  pierces the other triangle (collisions_static.cu:445-500, :612-779);
//   TE_CANDIDATES  (allow 1) rows (x, y, cid, loop) for every edge that does not end on a
//                  shared corner (collisions_static.cu:520-604, :782-943);
//   TE_CANDIDATES2 (allow 1) one row (x, y) per pair with bit masks (mx, my) of the same
//                  edges (icontour.cu:11-108, :110-282).
// A thread reserves all of its rows with one block-wide reservation.
enum { TE_COLLISIONS = 0, TE_CANDIDATES = 1, TE_CANDIDATES2 = 2 };

template <typename T, int MODE>
__global__ __launch_bounds__(kThreads) void k_tri_edge(const int2 *__restrict__ pairs_all, int64_t capK,
                                                       const T *__restrict__ t0_all, int64_t n,
                                                       int64_t *__restrict__ rows_all, T *__restrict__ coef_all,
                                                       int32_t *__restrict__ masks_all, int64_t out_cap,
                                                       DevCounters *__restrict__ ctr_all) {
    const int b = blockIdx.y;
    DevCounters *ctr = ctr_all + b;
    const unsigned long long kc = ctr->cand;
    const int64_t K = (int64_t)(kc < (unsigned long long)capK ? kc : (unsigned long long)capK);
    const int2 *pairs = pairs_all + (int64_t)b * capK;
    const T *t0 = t0_all + (int64_t)b * n * 9;
    constexpr int W = MODE == TE_CANDIDATES2 ? 2 : 4;
    int64_t *rows = rows_all + (int64_t)b * out_cap * W;
    const int64_t ntiles = (K + kThreads - 1) / kThreads;
    CCC_FOR_TILES(tile, ntiles) {
        const int64_t i = tile * kThreads + threadIdx.x;
        int x = 0, y = 0;
        unsigned emit = 0;          // bit cid: row for edge cid
        unsigned loops = 0;         // bit cid: loop node (loop id 0)
        int mx = 0, my = 0;
        T coefs[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) coefs[c] = (T)-1;
        bool valid = false;
        if (i < K) {
            const int2 pr = pairs[i];
            x = pr.x;
            y = pr.y;
            V3<T> a[3], c3[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) { a[k] = ld3(t0 + 9 * (int64_t)x + 3 * k); c3[k] = ld3(t0 + 9 * (int64_t)y + 3 * k); }
            const int allow = MODE == TE_COLLISIONS ? 0 : 1;
            valid = sat_overlap(a, c3, (T)0) && !(count_shared(a, c3) > allow);
            if (valid) {
#pragma unroll
                for (int cid = 0; cid < 6; ++cid) {
                    const V3<T> *t1 = cid < 3 ? a : c3;
                    const V3<T> *t2 = cid < 3 ? c3 : a;
                    const int e = cid % 3;
                    const V3<T> e0 = t1[e], e1 = t1[(e + 1) % 3];
                    if (MODE == TE_COLLISIONS) {
                        int64_t loop;
                        T cf;
                        if (te_intersect(t2, e0, e1, cid, loop, cf)) {
                            emit |= 1u << cid;
                            if (loop == 0) loops |= 1u << cid;
                            coefs[cid] = cf;
                        }
                    } else {
                        const bool s0 = has_vertex(t2, e0), s1 = has_vertex(t2, e1);
                        if (s0) {
                            if (cid < 3) { emit |= 1u << cid; loops |= 1u << cid; mx |= 1 << cid; my |= 1 << cid; }
                        } else if (!s1) {
                            // the reference compares t2 with the box of its own edge (collisions_static.cu:594-596)
                            const Box<T> b0 = tri_box(t2[0], t2[1], t2[2]);
                            const Box<T> b1 = unite(point_box(t2[e]), point_box(t2[(e + 1) % 3]));
                            if (overlap(b0, b1, (T)0)) { emit |= 1u << cid; mx |= 1 << cid; }
                        }
                    }
                }
            }
        }
        const unsigned cnt = MODE == TE_CANDIDATES2 ? (valid ? 1u : 0u) : (unsigned)__popc(emit);
        unsigned long long slot = block_reserve(&ctr->coll, cnt);
        if (MODE == TE_CANDIDATES2) {
            if (valid && slot < (unsigned long long)out_cap) {
                rows[2 * slot] = x;
                rows[2 * slot + 1] = y;
                int32_t *masks = masks_all + (int64_t)b * out_cap * 2;
                masks[2 * slot] = mx;
                masks[2 * slot + 1] = my;
            }
        } else {
#pragma unroll
            for (int cid = 0; cid < 6; ++cid) {
                if (!(emit & (1u << cid))) continue;
                if (slot < (unsigned long long)out_cap) {
                    rows[4 * slot] = x;
                    rows[4 * slot + 1] = y;
                    rows[4 * slot + 2] = cid;
                    rows[4 * slot + 3] = (loops & (1u << cid)) ? 0 : -1;
                    if (MODE == TE_COLLISIONS) coef_all[(int64_t)b * out_cap + slot] = coefs[cid];
                }
                ++slot;
            }
        }
    }
}

enum class Narrow { SAT, PROXIMITY, CCD_COLLECT, CCD_IMPULSE, MINCOL, TRI_EDGE };

struct Query {
    ccc_context *ctx;
    const void *bboxes;
    const int64_t *tree;
    const void *t0, *t1, *masses;
    const uint8_t *to_check;
    int64_t B, n;
    int32_t dtype;
    double thr;             // threshold already converted from the binding's float
    int64_t cap_candidates; // per batch element (max_candidates * n)
    int64_t out_cap;        // rows per batch element of the output
    Narrow narrow;
    int64_t *out_rows;      // SAT [B,cap,2] / PROXIMITY, CCD, MINCOL [B,cap,3]
    void *out_roots;        // CCD_COLLECT [B,cap]
    void *dv, *dx;          // CCD_IMPULSE
    int32_t *cnt;
    int te_mode;            // TRI_EDGE: TE_COLLISIONS / TE_CANDIDATES / TE_CANDIDATES2
    const int32_t *mesh_end;  // packed meshes (B = 1): per leaf position, end of its mesh
    int32_t *masks;         // TRI_EDGE candidates2 [B,cap,2]
    ccc_counts *counts;
    uint32_t flags;
    hipStream_t s;
    void *arena;            // non-NULL: every workspace buffer is carved from this block
    size_t arena_bytes;
    // Resident passes (the resident simulation): counters, the candidate list and the
    // deterministic impulse limbs live in the caller's memory, and with `nosync` nothing
    // waits on the host -- the list keeps at most cap_candidates pairs (more are counted),
    // the narrow phase walks [0, cap_candidates) in chunks whose kernels stop at the
    // device's counts, and the counters stay on the device.  Such a pass is capturable.
    bool nosync;
    DevCounters *ctr_ext;   // B counters (zeroed by the pass) or NULL
    int2 *pairs_ext;        // B * cap_candidates pairs or NULL
    int64_t chunk_ext;      // pairs per narrow-phase chunk (0: the context's)
    int ccd_blocks_per_cu;  // grid cap of k_ccd in blocks per CU (0: 128)
    const int64_t *leaf_ids; // resident: the tree when its leaves are in another order than the triangles
    double *lines;          // non-NULL: impulse sums in lines (the caller's, zeroed by the pass and not turned into dv, dx, cnt)
    long long *det_acc;     // non-NULL: impulse sums in fixed-point limbs (n * 3 * 6 * 4 per element)
};

// End of a pair chunk: its sub-primitive items are done; the next chunk refills the list.
__global__ void k_fold_items(DevCounters *__restrict__ ctr, int64_t B) {
    for (int64_t b = threadIdx.x; b < B; b += blockDim.x) {
        ctr[b].items_done += ctr[b].items;
        ctr[b].items = 0;
        ctr[b].tiles = 0;
    }
}

// End of the continuous narrow phase: the blocks' partial counts of every chunk to the
// counters.  One wave per batch element.
__global__ __launch_bounds__(64) void k_fold_partials(const DevPartial *__restrict__ part_all, int nparts, bool coll,
                                                      DevCounters *__restrict__ ctr, DevCounters *__restrict__ host) {
    static_assert(kPartials == 64, "one lane per partial");
    DevPartial p{};
    if ((int)threadIdx.x < nparts) p = part_all[(int64_t)blockIdx.x * nparts + threadIdx.x];
    unsigned long long v[3] = {p.items, p.roots, p.coll};
#pragma unroll
    for (int d = 1; d < 64; d <<= 1)
#pragma unroll
        for (int k = 0; k < 3; ++k) v[k] += __shfl_xor(v[k], d, 64);
    if (threadIdx.x == 0) {
        ctr[blockIdx.x].items_done = v[0];
        ctr[blockIdx.x].roots = v[1];
        if (coll) ctr[blockIdx.x].coll = v[2];
        if (host) host[blockIdx.x] = ctr[blockIdx.x];
    }
}

// The counters to pinned host memory, which the calls' waits then find written (k_fold_partials
// does it itself).  A copy into pageable memory goes through the runtime's staging and its own
// waits, twice per call: pass of 450 triangles 84 -> 68 us, of 20k with a tenth checked
// 132 -> 114, static proximity on 8k 309 -> 284.
__global__ void k_report(const DevCounters *__restrict__ ctr, int64_t B, DevCounters *__restrict__ host) {
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b < B) host[b] = ctr[b];
}

// Pairs per narrow-phase chunk over all batch elements of a call (the context may set
// another size) for 4-byte items, half as many for 8-byte ones: the item list holds at most
// 15 items per pair of a chunk, about 4 GiB either way.  On the 130k cloth one chunk of 2^26
// instead of two of 2^25 took k_ccd from 16.32 to 16.17 ms per pass.
constexpr int64_t kPairChunk = (int64_t)1 << 26;
// Largest chunk: at most 15 * 2^28 items per batch element; the continuous narrow phase's
// 32-bit items hold the pair index within the chunk in 28 bits.
constexpr int64_t kMaxPairChunk = (int64_t)1 << 28;
// Bytes per sub-primitive item: the continuous narrow phase keeps (pair index within the
// chunk) << 4 | type in 32 bits (chunks hold at most 2^28 pairs); the static one (x, y, type)
// in 64.
static size_t item_bytes(Narrow nw) { return nw == Narrow::PROXIMITY ? sizeof(int64_t) : sizeof(uint32_t); }
static int64_t pair_chunk_of(const ccc_context *ctx, int64_t chunk_ext, int64_t pairs, int64_t B, size_t item_size) {
    const int64_t dflt = kPairChunk * (int64_t)sizeof(uint32_t) / (int64_t)item_size;
    const int64_t budget = chunk_ext > 0 ? chunk_ext * B : ctx->pair_chunk > 0 ? ctx->pair_chunk : dflt;
    return std::max<int64_t>(std::min<int64_t>(std::min<int64_t>(pairs, budget / B), kMaxPairChunk), 1);
}
constexpr int kSubprimPairs = 2;   // pairs per thread of k_subprim
constexpr int kItemWaves = 24;   // k_items: waves per CU (about two rounds of the resident ones)

// Grid of the tile-looping kernels: one block per tile up to 128 blocks per CU, each block
// then walking several tiles.  Measured on the 130k cloth (k_ccd per step): 4 blocks per CU
// (all resident at once) 232 ms, 16 215 ms, 32 210, 128 207, 512 214 -- many short blocks
// let the dispatcher balance the uneven tiles; past that the per-block start-up dominates.
static unsigned persistent_grid(const ccc_context *ctx, int64_t items, int64_t B, int block = kThreads, int per_cu = 128) {
    int64_t want = (items + block - 1) / block;
    if (want < 1) want = 1;                        // no items: a grid of idle blocks, never 0
    int64_t limit = (int64_t)ctx->num_cus * per_cu / (B > 0 ? B : 1);
    if (limit < kXcds) limit = kXcds;
    if (want > limit) want = limit;
    want = (want + kXcds - 1) / kXcds * kXcds;    // CCC_FOR_TILES needs a multiple of kXcds
    return (unsigned)want;
}

// The path for every tree that is not the index tree (trees of other builders, fitted trees
// given back to the stateless calls): the tree is checked, its rightmost leaves found, and
// k_traverse walks it with a bounded stack.
template <typename T> class GeneralTree {
  public:
    GeneralTree(const Query &q, Workspace &ws, const T *bb, DevCounters *ctr, hipStream_t s, KernelTimer &tm)
        : q_(q), ws_(ws), bb_(bb), ctr_(ctr), s_(s), tm_(tm) {}
    bool used() const { return used_; }
    bool deep() const { return deep_; }
    void use() { used_ = true; }
    void go_deep() { deep_ = true; }
    bool prepared() const { return prepared_; }
    // The buffers, last in, first out.
    void release() {
        for (void *p : {(void *)qbox_, (void *)frontier_, (void *)recs_, (void *)qnodes_, (void *)nodes_, (void *)lo_, (void *)rm_, (void *)claims_})
            ws_.release(p);
        prepared_ = false;
    }
    ccc_status prepare() {
        prepared_ = true;
        const int64_t B = q_.B, n = q_.n, rows = 2 * n - 1, nint = n > 1 ? n - 1 : 1;
        int *claims = claims_ = ws_.get_as<int>(B * n);
        int *rm = rm_ = ws_.get_as<int>(B * nint);
        int *lo = lo_ = ws_.get_as<int>(B * nint);
        TNode *nodes = nodes_ = ws_.get_as<TNode>(B * nint);
        qnodes_ = ws_.get_as<QNode>(B * nint);
        recs_ = ws_.get_as<LeafRec>(B * n);
        frontier_ = ws_.get_as<Frontier>(B);
        // one block per (start point, query block); query blocks rounded to a multiple of kXcds
        nqb_ = (int)((grid_for(n, kTravThreads) + kXcds - 1) / kXcds * kXcds);
        qbox_ = ws_.get_as<float>(B * (int64_t)nqb_ * 6);
        if (ws_.failed()) return CCC_ERR_NO_MEMORY;
        FillRegions fill;
        fill.add(claims, B * n * 4, 0ull);
        ccc_status st = fill_regions(fill, s_);
        if (st != CCC_OK) return st;
        tm_.begin("tree_prep");
        hipLaunchKernelGGL(k_check_tree, dim3(grid_for(rows, 256), B), dim3(256), 0, s_, q_.tree, n, claims, ctr_);
        if (n > 1) {
            hipLaunchKernelGGL(k_ranges, dim3(grid_for(n - 1, 256), B), dim3(256), 0, s_, q_.tree, n, lo, rm, ctr_);
            hipLaunchKernelGGL(k_order_check, dim3(grid_for(n - 1, 256), B), dim3(256), 0, s_, q_.tree, n, lo, rm, ctr_);
        }
        hipLaunchKernelGGL(k_rightmost, dim3(grid_for(n, 256), B), dim3(256), 0, s_, q_.tree, n, claims, rm, ctr_);
        if (n > 1) {
            hipLaunchKernelGGL((k_nodes<T>), dim3(grid_for(n - 1, 256), B), dim3(256), 0, s_, bb_, q_.tree, rm, n, q_.thr, nodes, ctr_);
            hipLaunchKernelGGL(k_qnodes, dim3(grid_for(n - 1, 256), B), dim3(256), 0, s_, nodes, n, qnodes_, ctr_);
        }
        hipLaunchKernelGGL((k_leaf_recs<T>), dim3(grid_for(n, 256), B), dim3(256), 0, s_, bb_, q_.tree, n, recs_, ctr_);
        hipLaunchKernelGGL((k_frontier<T>), dim3(B), dim3(kFrontier), 0, s_, bb_, q_.tree, rm, n, q_.thr, frontier_, ctr_);
        hipLaunchKernelGGL((k_qblock_boxes<T>), dim3(nqb_, B), dim3(kTravThreads), 0, s_, bb_, n, nqb_, qbox_, ctr_);
        tm_.end();
        CCC_LAUNCH_CHECK("tree preparation");
        return CCC_OK;
    }
    ccc_status traverse(int2 *pairs, int64_t capK) {
        const dim3 g(kFrontier * (unsigned)nqb_, (unsigned)q_.B);
        tm_.begin("traverse");
#define CCC_TRAVERSE(P, D)                                                                                                  \
    hipLaunchKernelGGL((k_traverse<T, P, D>), g, dim3(kTravThreads), 0, s_, bb_, q_.tree, qnodes_, recs_, q_.n, (T)q_.thr, \
                       q_.to_check, pairs, capK, ctr_, frontier_, qbox_)
        if (q_.to_check) {
            if (deep_) CCC_TRAVERSE(true, kStackDeep);
            else CCC_TRAVERSE(true, kStackShort);
        } else {
            if (deep_) CCC_TRAVERSE(false, kStackDeep);
            else CCC_TRAVERSE(false, kStackShort);
        }
#undef CCC_TRAVERSE
        tm_.end();
        CCC_LAUNCH_CHECK("k_traverse");
        return CCC_OK;
    }

  private:
    const Query &q_;
    Workspace &ws_;
    const T *bb_;
    DevCounters *ctr_;
    hipStream_t s_;
    KernelTimer &tm_;
    bool used_ = false, deep_ = false, prepared_ = false;
    int *claims_ = nullptr, *rm_ = nullptr, *lo_ = nullptr;
    TNode *nodes_ = nullptr;
    QNode *qnodes_ = nullptr;
    LeafRec *recs_ = nullptr;
    Frontier *frontier_ = nullptr;
    int nqb_ = 0;
    float *qbox_ = nullptr;
};

// The list of the continuous narrow phase for chunks of at most `chunk` pairs per batch
// element, in whole batches of 64 pairs: 15 slots per pair, a descriptor per 64 of them (a
// wave's items of one kind start at a multiple of 64 and fill at most its slots), and the
// blocks of k_items.
struct ListPlan {
    int64_t chunk, slots, tiles;
    unsigned grid;
    // the slots and the tiles' descriptors, each rounded as a workspace buffer is
    size_t bytes(int64_t B) const {
        auto r = [](size_t b) { return (b + 255) & ~(size_t)255; };
        return r(sizeof(uint32_t) * B * slots) + r(sizeof(uint32_t) * B * tiles);
    }
};
static ListPlan list_plan(const ccc_context *ctx, int64_t chunk, int64_t B) {
    const int64_t batches = (chunk + kBatch - 1) / kBatch, slots = batches * (kSegEE + kSegVF) * kBatch;
    static_assert(kSegEE * kBatch % 64 == 0 && kSegVF * kBatch % 64 == 0, "segments start at multiples of a tile");
    const int64_t waves = std::max<int64_t>(std::min<int64_t>(batches, (int64_t)ctx->num_cus * kItemWaves / B), 1);
    constexpr int kGroup = kXcds * kItemBlock;
    return ListPlan{chunk, slots, slots / 64, (unsigned)((waves + kGroup - 1) / kGroup * kXcds)};
}
// Partial counts per batch element, a power of two: kPartials lines each, and at most sixteen
// times as many over the whole batch (the blocks that add to them are spread over its
// elements; 8 lines on each of six 5,000-triangle meshes instead of 64: 273 -> 282 us).
static int partials_of(int64_t B) {
    int k = kPartials;
    while (k > 1 && k * B > 16 * kPartials) k >>= 1;
    return k;
}

template <typename T>
static ccc_status run_query(const Query &q) {
    hipStream_t s = q.s;
    const int64_t B = q.B, n = q.n, rows = 2 * n - 1;
    Workspace ws(q.ctx, s, q.arena, q.arena_bytes);
    // no event objects in the allocation-free entry point (arena without resident mode)
    KernelTimer tm(q.arena && !q.nosync ? nullptr : q.ctx, s);
    const bool moving = q.narrow == Narrow::CCD_COLLECT || q.narrow == Narrow::CCD_IMPULSE || q.narrow == Narrow::MINCOL;
    const int64_t nc = (n + kChunk - 1) >> kChunkBits;
    DevCounters *ctr = q.ctr_ext ? q.ctr_ext : ws.get_as<DevCounters>(B);
    T *tv = moving ? ws.get_as<T>(B * n * 18) : nullptr;
    const bool ccd_query = q.narrow == Narrow::CCD_COLLECT || q.narrow == Narrow::CCD_IMPULSE;
    // with a scratch block that may be tight the partial counts wait until the traversal's buffers are gone
    int nparts = partials_of(B);
    const bool late_parts = ws.arena() && !q.nosync;
    DevPartial *parts = ccd_query && !late_parts ? ws.get_as<DevPartial>(B * nparts) : nullptr;
    // A context that fits its trees gets them back here: straight to the walk, without a first
    // attempt that only finds out (static query on 8k triangles 189 us with it, 165 without).
    // Packed meshes always have the index tree.
    const bool walk = !q.nosync && !q.mesh_end && q.ctx->morton != CCC_MORTON_COMPAT;
    // what only the index tree's path uses, given back when the tree is another
    unsigned *foreign = q.nosync || walk ? nullptr : ws.get_as<unsigned>(B);
    T *chunks = walk ? nullptr : ws.get_as<T>(B * nc * 6);
    T *groups = walk ? nullptr : ws.get_as<T>(B * nc * (kChunk / kPairQ) * 12);
    T *supers = !walk && nc > kSuperFrom ? ws.get_as<T>(B * ((nc + kChunk - 1) >> kChunkBits) * 6) : nullptr;
    if (ws.failed()) return CCC_ERR_NO_MEMORY;
    ccc_status st;

    // outputs start at -1 (index rows, roots) or 0 (impulses)
    FillRegions fill;
    fill.add(ctr, B * (int64_t)sizeof(DevCounters), 0ull);
    if (foreign) fill.add(foreign, B * 4, 0ull);
    if (parts) fill.add(parts, B * nparts * (int64_t)sizeof(DevPartial), 0ull);
    const uint64_t minus1 = sizeof(T) == 8 ? 0xBFF0000000000000ull : 0xBF800000BF800000ull;
    const int64_t cells = B * q.out_cap, tsz = (int64_t)sizeof(T);
    switch (q.narrow) {
        case Narrow::SAT: fill.add(q.out_rows, cells * 16, ~0ull); break;
        case Narrow::TRI_EDGE:
            fill.add(q.out_rows, cells * (q.te_mode == TE_CANDIDATES2 ? 16 : 32), ~0ull);
            if (q.te_mode == TE_COLLISIONS) fill.add(q.out_roots, cells * tsz, minus1);
            if (q.te_mode == TE_CANDIDATES2) fill.add(q.masks, cells * 8, 0ull);
            break;
        case Narrow::PROXIMITY:
        case Narrow::MINCOL: fill.add(q.out_rows, cells * 24, ~0ull); break;
        case Narrow::CCD_COLLECT:
            fill.add(q.out_rows, cells * 24, ~0ull);
            fill.add(q.out_roots, cells * tsz, minus1);
            break;
        case Narrow::CCD_IMPULSE:
            if (q.det_acc) fill.add(q.det_acc, B * n * 3 * kDetWords * 8, 0ull);
            else if (q.lines) fill.add(q.lines, B * n * 3 * kLineWords * 8, 0ull);
            else {
                fill.add(q.dv, B * n * 9 * tsz, 0ull);
                fill.add(q.dx, B * n * 9 * tsz, 0ull);
                fill.add(q.cnt, B * n * 12, 0ull);
            }
            break;
    }
    if ((st = fill_regions(fill, s)) != CCC_OK) return st;

    const T *bb = (const T *)q.bboxes;
    // a resident pass's tree was built by the pass itself
    const unsigned gr = q.nosync || walk ? 0u : grid_for(rows, 256), gl = walk ? 0u : grid_for(n, 256), gv = moving ? grid_for(3 * n, 256) : 0u;
    if (gr + gl + gv > 0) {
        tm.begin("tree_prep");
        hipLaunchKernelGGL((k_prep<T>), dim3(gr + gl + gv, B), dim3(256), 0, s, bb, q.tree, n, gr, gl, q.to_check, chunks, groups, (const T *)q.t0,
                           (const T *)q.t1, tv, foreign);
        if (supers) hipLaunchKernelGGL((k_super_boxes<T>), dim3(grid_for(nc, 256), B), dim3(256), 0, s, chunks, nc, supers);
        tm.end();
        CCC_LAUNCH_CHECK("tree preparation");
    }

    // traversal, re-run once with the exact size if the capacity was exceeded
    std::vector<DevCounters> h(B);
    HostBlock block(q.ctx, s, !q.nosync && !q.arena && B * sizeof(DevCounters) <= HostBlock::kBytes);
    DevCounters *hp = block.as<DevCounters>();
    // the counters on the host; `reported`: the last kernel has written them to the block
    auto read_counters = [&](bool reported) -> ccc_status {
        if (hp) {
            if (!reported) {
                block.written();
                hipLaunchKernelGGL(k_report, dim3((unsigned)((B + 255) / 256)), dim3(256), 0, s, ctr, B, hp);
                CCC_LAUNCH_CHECK("k_report");
            }
        } else {
            CCC_HIP_TRY(hipMemcpyAsync(h.data(), ctr, sizeof(DevCounters) * B, hipMemcpyDeviceToHost, s));
        }
        CCC_HIP_TRY(hipStreamSynchronize(s));
        block.settled();
        if (hp) std::copy(hp, hp + B, h.begin());
        return CCC_OK;
    };
    int64_t capK = q.cap_candidates > 0 ? q.cap_candidates : 1;
    bool warn_cand = false;
    int2 *pairs = nullptr;
    // Splits per query group: 16,384 waves in all, at least three while the groups alone do not
    // fill the chip twice over (the longest group then ends sooner), at most one per chunk.
    // More waves cost their reservations: 33k-triangle pass (f32) 8k waves 35 us, 16k 38, 32k 55;
    // garment scene 1 split 230 us, 2 144, 4 113; 130k cloth 1 split 410 us, 2 383, 4 409.
    const int64_t nq = (n + kPairQ - 1) / kPairQ, groups_all = nq * B;
    const int splits = (int)std::max<int64_t>(1, std::min<int64_t>(nc, std::max<int64_t>(16384 / groups_all, groups_all < 16384 ? 3 : 1)));
    GeneralTree<T> general(q, ws, bb, ctr, s, tm);
    if (walk) general.use();
    for (int attempt = 0; attempt < 2; ++attempt) {
        if (q.pairs_ext) {
            pairs = q.pairs_ext;
        } else {
            // a re-run: the first attempt's pairs are not kept (in an arena the walk's buffers
            // lie behind them and go first)
            if (general.prepared() && ws.arena()) general.release();
            if (pairs) ws.release(pairs);
            pairs = ws.get_as<int2>(B * capK);
            if (ws.failed()) return CCC_ERR_NO_MEMORY;
        }
        if (general.used() && !general.prepared() && (st = general.prepare()) != CCC_OK) return st;
        if (general.used()) {
            if ((st = general.traverse(pairs, capK)) != CCC_OK) return st;
        } else {
            tm.begin("traverse");
            const dim3 g((unsigned)((nq * splits + kPairWaves - 1) / kPairWaves), (unsigned)B);
            if (q.to_check)
                hipLaunchKernelGGL((k_pairs<T, true>), g, dim3(64 * kPairWaves), 0, s, bb, q.leaf_ids, n, (T)q.thr, chunks, supers, groups, splits, q.to_check,
                                   q.mesh_end, pairs, capK, foreign, ctr);
            else
                hipLaunchKernelGGL((k_pairs<T, false>), g, dim3(64 * kPairWaves), 0, s, bb, q.leaf_ids, n, (T)q.thr, chunks, supers, groups, splits, q.to_check,
                                   q.mesh_end, pairs, capK, foreign, ctr);
            tm.end();
            CCC_LAUNCH_CHECK("k_pairs");
        }
        if (q.nosync) break;          // the caller checks the counters after its step
        if ((st = read_counters(false)) != CCC_OK) return st;
        unsigned flags = 0;
        unsigned long long kmax = 0;
        for (int64_t b = 0; b < B; ++b) {
            flags |= h[b].flags;
            kmax = std::max(kmax, h[b].cand);
        }
        if (flags & DEV_BAD_TREE) { set_error("tree tensor is not a valid BVH over n leaves"); return CCC_ERR_BAD_TREE; }
        if ((flags & DEV_STACK) && general.deep()) { set_error("BVH deeper than the traversal stack"); return CCC_ERR_STACK; }
        if (flags & (DEV_STACK | DEV_FOREIGN)) {
            // again with the deep stack, or by the general path (not a capacity attempt)
            for (int64_t b = 0; b < B; ++b) {
                h[b].cand = 0;
                h[b].flags &= ~(DEV_STACK | DEV_FOREIGN);
            }
            CCC_HIP_TRY(hipMemcpyAsync(ctr, h.data(), sizeof(DevCounters) * B, hipMemcpyHostToDevice, s));
            if (flags & DEV_STACK) general.go_deep();
            else if (q.mesh_end) {
                // (a packed call builds its tree itself, and the walk knows of one mesh)
                set_error("internal error: a packed batch's tree is not the index tree");
                return CCC_ERR_BAD_TREE;
            } else {
                // last in, first out
                if (!q.pairs_ext) { ws.release(pairs); pairs = nullptr; }
                if (supers) ws.release(supers);
                ws.release(groups);
                ws.release(chunks);
                ws.release(foreign);
                foreign = nullptr;
                general.use();
            }
            --attempt;
            continue;
        }
        if (kmax <= (unsigned long long)capK) break;
        warn_cand = true;
        if (q.flags & CCC_FLAG_FIXED_CAPACITY) break;
        if (attempt == 1 || q.pairs_ext) break;   // a caller-owned list does not grow here
        capK = (int64_t)kmax;
        for (int64_t b = 0; b < B; ++b) h[b].cand = 0;
        CCC_HIP_TRY(hipMemcpyAsync(ctr, h.data(), sizeof(DevCounters) * B, hipMemcpyHostToDevice, s));
    }
    if (general.prepared() && ws.arena()) general.release();      // room for the narrow phase
    int64_t kmax = 0;
    if (q.nosync) kmax = capK;        // sizes must not depend on the counts
    else
        for (int64_t b = 0; b < B; ++b) kmax = std::max<int64_t>(kmax, std::min<int64_t>((int64_t)h[b].cand, capK));

    const T thr = (T)q.thr;
    const unsigned gK = persistent_grid(q.ctx, kmax, B);
    if (q.narrow == Narrow::SAT) {
        CCC_TIMED(tm, "sat", hipLaunchKernelGGL((k_sat<T>), dim3(gK, B), dim3(kThreads), 0, s, pairs, capK, (const T *)q.t0, n, thr,
                                                q.out_rows, q.out_cap, ctr));
        CCC_LAUNCH_CHECK("k_sat");
    } else if (q.narrow == Narrow::TRI_EDGE) {
        tm.begin("tri_edge");
        if (q.te_mode == TE_COLLISIONS)
            hipLaunchKernelGGL((k_tri_edge<T, TE_COLLISIONS>), dim3(gK, B), dim3(kThreads), 0, s, pairs, capK, (const T *)q.t0, n,
                               q.out_rows, (T *)q.out_roots, (int32_t *)nullptr, q.out_cap, ctr);
        else if (q.te_mode == TE_CANDIDATES)
            hipLaunchKernelGGL((k_tri_edge<T, TE_CANDIDATES>), dim3(gK, B), dim3(kThreads), 0, s, pairs, capK, (const T *)q.t0, n,
                               q.out_rows, (T *)nullptr, (int32_t *)nullptr, q.out_cap, ctr);
        else
            hipLaunchKernelGGL((k_tri_edge<T, TE_CANDIDATES2>), dim3(gK, B), dim3(kThreads), 0, s, pairs, capK, (const T *)q.t0, n,
                               q.out_rows, (T *)nullptr, q.masks, q.out_cap, ctr);
        tm.end();
        CCC_LAUNCH_CHECK("k_tri_edge");
    } else if (q.narrow == Narrow::MINCOL) {
        const unsigned gS = persistent_grid(q.ctx, (kmax + kSubprimPairs - 1) / kSubprimPairs, B);
        tm.begin("mincol");
        hipLaunchKernelGGL((k_subprim<T, SUB_MINCOL, kSubprimPairs>), dim3(gS, B), dim3(kThreads), 0, s, pairs, capK,
                           (int64_t)0, capK, (const T *)tv, n, thr, q.out_rows, q.out_cap, ctr);
        tm.end();
        CCC_LAUNCH_CHECK("k_subprim");
    } else {
        // sub-primitive items and the narrow phase run over chunks of the pair list; the
        // chunk bounds the pairs of all batch elements together (the item buffer holds B
        // chunks), so the workspace does not grow with the batch
        const bool ccd = q.narrow != Narrow::PROXIMITY;
        int64_t chunk = pair_chunk_of(q.ctx, q.chunk_ext, kmax, B, item_bytes(q.narrow));
        ListPlan plan = list_plan(q.ctx, chunk, B);
        if (ccd && late_parts) {
            while (nparts > 1 && nparts * (int64_t)kBatch > chunk) nparts >>= 1;
            parts = ws.get_as<DevPartial>(B * nparts);
            if (ws.failed()) return CCC_ERR_NO_MEMORY;
            FillRegions zero;
            zero.add(parts, B * nparts * (int64_t)sizeof(DevPartial), 0ull);
            if ((st = fill_regions(zero, s)) != CCC_OK) return st;
        }
        if (ws.arena()) {
            // the item list takes what the arena has left (results do not depend on the chunk)
            if (ccd) {
                while (plan.bytes(B) > ws.arena_left() && chunk > 1) {
                    chunk = std::min(chunk / 2, std::max<int64_t>((int64_t)(ws.arena_left() / ((size_t)B * 15 * sizeof(uint32_t))), 1));
                    plan = list_plan(q.ctx, chunk, B);
                }
                if (plan.bytes(B) > ws.arena_left()) chunk = 0;
            } else {
                chunk = std::min(chunk, (int64_t)(ws.arena_left() / ((size_t)B * 15 * item_bytes(q.narrow))));
            }
            if (chunk < 1) {
                set_error("the scratch buffer has no room left for the sub-primitive items of one candidate pair");
                return CCC_ERR_NO_MEMORY;
            }
        }
        const int64_t capM = ccd ? plan.slots : 15 * chunk;
        uint32_t *tiles = ccd ? ws.get_as<uint32_t>(B * plan.tiles) : nullptr;
        void *items = ws.get_as<unsigned char>(B * capM * (int64_t)item_bytes(q.narrow));
        const unsigned gS = persistent_grid(q.ctx, (chunk + kSubprimPairs - 1) / kSubprimPairs, B);
        const unsigned gM = persistent_grid(q.ctx, capM, B);
        const unsigned gCcdC = persistent_grid(q.ctx, capM, B, ccd_threads<MODE_COLLECT>());
        // one-wave impulse blocks, up to 128 per CU: on the 130k cloth 256 per CU took 171.6 ms
        // per step against 173.7 and 64 took 178.3, but 256 cost the 122k garment scene (fewer
        // items per pass) 23% of its step rate
        const unsigned gCcdI = persistent_grid(q.ctx, capM, B, ccd_threads<MODE_IMPULSE>(),
                                               q.ccd_blocks_per_cu > 0 ? q.ccd_blocks_per_cu : 128);
        if (ws.failed()) return CCC_ERR_NO_MEMORY;
        auto narrow_phase = [&]() -> ccc_status {
            for (int64_t c0 = 0; c0 < kmax; c0 += chunk) {
                const int64_t c1 = c0 + chunk;
                tm.begin("subprim");
                if (q.narrow == Narrow::PROXIMITY)
                    hipLaunchKernelGGL((k_subprim<T, SUB_STATIC, kSubprimPairs>), dim3(gS, B), dim3(kThreads), 0, s, pairs, capK,
                                       c0, c1, (const T *)q.t0, n, thr, items, capM, ctr);
                else
                    hipLaunchKernelGGL((k_items<T>), dim3(plan.grid, B), dim3(64 * kItemBlock), 0, s, pairs, capK, c0, c1, (const T *)tv, n,
                                       (uint32_t *)items, capM, tiles, plan.tiles, parts, nparts, ctr);
                tm.end();
                CCC_LAUNCH_CHECK(ccd ? "k_items" : "k_subprim");
                tm.begin(q.narrow == Narrow::PROXIMITY ? "proximity" : q.narrow == Narrow::CCD_COLLECT ? "ccd_collect" : "ccd_impulse");
                if (q.narrow == Narrow::PROXIMITY)
                    hipLaunchKernelGGL((k_proximity<T>), dim3(gM, B), dim3(kThreads), 0, s, (const int64_t *)items, capM, (const T *)q.t0, n, thr,
                                       q.out_rows, q.out_cap, ctr);
                else {
                    CcdArgs<T> ca{};
                    ca.items = (const uint32_t *)items;
                    ca.tiles = tiles;
                    ca.pairs = pairs;
                    ca.tv = tv;
                    ca.ctr = ctr;
                    ca.parts = parts;
                    ca.nparts = nparts;
                    ca.cap_items = capM;
                    ca.cap_tiles = plan.tiles;
                    ca.cap_pairs = capK;
                    ca.first_pair = c0;
                    ca.n = n;
                    ca.masses = (const T *)q.masses;
                    ca.dv = (T *)q.dv;
                    ca.dx = (T *)q.dx;
                    ca.cnt = q.cnt;
                    ca.det = q.det_acc;
                    ca.lines = q.lines;
                    ca.coll = q.out_rows;
                    ca.roots = (T *)q.out_roots;
                    ca.out_cap = q.out_cap;
#define CCC_CCD(MODE, SUMS, G) hipLaunchKernelGGL((k_ccd<T, MODE, SUMS>), dim3(G, B), dim3(ccd_threads<MODE>()), 0, s, ca)
                    if (q.narrow == Narrow::CCD_COLLECT) CCC_CCD(MODE_COLLECT, SUMS_DIRECT, gCcdC);
                    else if (q.det_acc) CCC_CCD(MODE_IMPULSE, SUMS_DET, gCcdI);
                    else if (q.lines) CCC_CCD(MODE_IMPULSE, SUMS_LINES, gCcdI);
                    else CCC_CCD(MODE_IMPULSE, SUMS_DIRECT, gCcdI);
#undef CCC_CCD
                }
                tm.end();
                CCC_LAUNCH_CHECK("narrow phase");
                if (!ccd || c0 + chunk < kmax) {
                    hipLaunchKernelGGL(k_fold_items, dim3(1), dim3(64), 0, s, ctr, B);
                    CCC_LAUNCH_CHECK("k_fold_items");
                }
            }
            if (ccd) {
                block.written();
                hipLaunchKernelGGL(k_fold_partials, dim3(B), dim3(64), 0, s, parts, nparts, q.narrow == Narrow::CCD_IMPULSE, ctr, hp);
                CCC_LAUNCH_CHECK("k_fold_partials");
            }
            return CCC_OK;
        };
        if ((st = narrow_phase()) != CCC_OK) return st;
        if (q.det_acc) {
            hipLaunchKernelGGL((k_det_finalize<T>), dim3(grid_for(B * n * 3, 256)), dim3(256), 0, s, q.det_acc, B * n * 3,
                               (T *)q.dv, (T *)q.dx, q.cnt);
            CCC_LAUNCH_CHECK("k_det_finalize");
        }
    }
    if (q.nosync) return CCC_OK;
    if ((st = read_counters(hp && ccd_query)) != CCC_OK) return st;
    bool truncated = false;
    for (int64_t b = 0; b < B; ++b) {
        const int64_t K = std::min<int64_t>((int64_t)h[b].cand, capK);
        if (q.counts) {
            q.counts[b].candidates = (int64_t)h[b].cand;
            q.counts[b].subprims = (int64_t)(q.narrow == Narrow::MINCOL ? h[b].items : h[b].items_done);
            q.counts[b].roots = (int64_t)h[b].roots;
            q.counts[b].collisions = q.narrow == Narrow::MINCOL ? (int64_t)h[b].items : (int64_t)h[b].coll;
        }
        (void)K;
        const int64_t produced = q.narrow == Narrow::MINCOL ? (int64_t)h[b].items : (int64_t)h[b].coll;
        if (q.narrow != Narrow::CCD_IMPULSE && produced > q.out_cap) truncated = true;
    }
    ccc_status out = CCC_OK;
    if (warn_cand) out |= CCC_WARN_CANDIDATES;
    if (truncated) out |= CCC_WARN_TRUNCATED;
    return out;
}

// Workspace bytes of a resident CCD_IMPULSE pass (nosync, caller-owned counters and pair
// list): the same buffers, sizes and 256-byte rounding as run_query's requests.
static size_t resident_bytes(const Query &q) {
    const int64_t B = q.B, n = q.n, nc = (n + kChunk - 1) >> kChunkBits;
    const size_t esz = q.dtype == CCC_FLOAT64 ? 8 : 4;
    auto r = [](size_t b) { return ((b ? b : 256) + 255) & ~(size_t)255; };
    size_t tot = 0;
    if (!q.ctr_ext) tot += r(sizeof(DevCounters) * B);
    tot += r(esz * B * nc * 6) + r(esz * B * nc * (kChunk / kPairQ) * 12);
    if (nc > kSuperFrom) tot += r(esz * B * ((nc + kChunk - 1) >> kChunkBits) * 6);
    const int64_t capK = q.cap_candidates > 0 ? q.cap_candidates : 1;
    if (!q.pairs_ext) tot += r(sizeof(int2) * B * capK);
    const int64_t chunk = pair_chunk_of(q.ctx, q.chunk_ext, capK, B, item_bytes(q.narrow));
    const ListPlan plan = list_plan(q.ctx, chunk, B);
    tot += r(esz * B * n * 18) + r(sizeof(DevPartial) * B * partials_of(B)) + plan.bytes(B);
    return tot;
}

static Query resident_query(ccc_context *ctx, const ResidentPass &p, hipStream_t s) {
    Query q{};
    q.ctx = ctx;
    q.bboxes = p.bboxes;
    q.tree = p.tree;
    q.t0 = p.t0;
    q.t1 = p.t1;
    q.masses = p.masses;
    q.B = 1;
    q.n = p.n;
    q.dtype = p.dtype;
    q.thr = 0.0;
    q.cap_candidates = p.cap_pairs;
    q.narrow = Narrow::CCD_IMPULSE;
    q.dv = p.dv;
    q.dx = p.dx;
    q.cnt = p.cnt;
    q.mesh_end = p.mesh_end;
    q.flags = CCC_FLAG_FIXED_CAPACITY;
    q.s = s;
    q.nosync = true;
    q.ctr_ext = p.ctr;
    q.pairs_ext = p.pairs;
    q.chunk_ext = p.chunk;
    q.ccd_blocks_per_cu = p.ccd_blocks_per_cu;
    q.leaf_ids = p.leaf_ids;
    q.det_acc = p.det_acc;
    q.lines = p.lines;
    return q;
}

size_t resident_pass_arena_bytes(ccc_context *ctx, const ResidentPass &p) { return resident_bytes(resident_query(ctx, p, nullptr)); }

ccc_status line_sums(const double *lines, int64_t corners, int32_t dtype, void *dv, void *dx, int32_t *cnt, hipStream_t s) {
    if (dtype == CCC_FLOAT64)
        hipLaunchKernelGGL((k_line_sums<double>), dim3(grid_for(corners, 256)), dim3(256), 0, s, lines, corners, (double *)dv, (double *)dx, cnt, GivenRows{});
    else
        hipLaunchKernelGGL((k_line_sums<float>), dim3(grid_for(corners, 256)), dim3(256), 0, s, lines, corners, (float *)dv, (float *)dx, cnt, GivenRows{});
    CCC_LAUNCH_CHECK("k_line_sums");
    return CCC_OK;
}

ccc_status resident_pass(ccc_context *ctx, const ResidentPass &p, void *arena, size_t arena_bytes, hipStream_t s) {
    Query q = resident_query(ctx, p, s);
    q.arena = arena;
    q.arena_bytes = arena_bytes;
    if (p.dtype == CCC_FLOAT64) return run_query<double>(q);
    if (p.dtype == CCC_FLOAT32) return run_query<float>(q);
    return bad_arg("dtype must be CCC_FLOAT32 or CCC_FLOAT64");
}

static ccc_status run(const Query &q) {
    clear_error();
    if (!q.ctx) return bad_arg("context is NULL");
    if (q.B < 0 || q.n < 1) return bad_arg("need batch >= 0 and n >= 1 triangles");
    if (q.n >= ((int64_t)1 << 28)) return bad_arg("at most 2^28 - 1 triangles per mesh");
    if (q.B == 0) return CCC_OK;
    if (!q.bboxes || !q.tree || !q.t0) return bad_arg("NULL tensor pointer");
    if ((q.narrow == Narrow::CCD_COLLECT || q.narrow == Narrow::CCD_IMPULSE || q.narrow == Narrow::MINCOL) && !q.t1)
        return bad_arg("triangles_next is NULL");
    if (q.narrow == Narrow::CCD_IMPULSE && (!q.masses || !q.dv || !q.dx || !q.cnt)) return bad_arg("NULL impulse tensor");
    if (q.narrow != Narrow::CCD_IMPULSE && (!q.out_rows || q.out_cap < 0)) return bad_arg("NULL output tensor");
    if (q.narrow == Narrow::CCD_COLLECT && !q.out_roots) return bad_arg("NULL roots tensor");
    if (q.narrow == Narrow::TRI_EDGE && q.te_mode == TE_COLLISIONS && !q.out_roots) return bad_arg("NULL coefficient tensor");
    if (q.narrow == Narrow::TRI_EDGE && q.te_mode == TE_CANDIDATES2 && !q.masks) return bad_arg("NULL mask tensor");
    CCC_HIP_TRY(hipSetDevice(q.ctx->device));
    if (q.dtype == CCC_FLOAT64) return run_query<double>(q);
    if (q.dtype == CCC_FLOAT32) return run_query<float>(q);
    return bad_arg("dtype must be CCC_FLOAT32 or CCC_FLOAT64");
}

// Whether `m` given rows on each of B meshes of n triangles may be summed in lines.  Lines take a
// launch and 420 bytes of traffic per triangle more and up to six atomic requests per table
// slot less: on 130k triangles with 16 rows each 113 us against 148 direct, with 4 84 and 102,
// with one 82 and 87, with half of one 80 and 74; collections of a folded cloth (23k triangles,
// 15 rows each) 48 us less.  How many rows there are the device finds out (many_rows): an empty
// list of 8 rows per triangle takes 32 us on 130k triangles (41 when capacity alone chose
// lines, 28 without the choice) and 93 on 1M (164, 84).
static bool lines_pay(int64_t m, int64_t B, int64_t n) { return m * B >= 65536 && m >= n && n < ((int64_t)1 << 28); }

template <typename T>
static ccc_status from_collisions(ccc_context *ctx, const int64_t *coll, const void *roots, int64_t m, const void *t0,
                                  const void *t1, const void *masses, int64_t B, int64_t n, void *dv, void *dx, int32_t *cnt,
                                  hipStream_t s) {
    Workspace ws(ctx, s);
    double *lines = lines_pay(m, B, n) ? ws.try_get_as<double>(B * n * 3 * kLineWords) : nullptr;
    const GivenRows given = lines ? given_rows(coll, m, n, B) : GivenRows{};
    FillRegions direct;
    direct.add(dv, B * n * 9 * (int64_t)sizeof(T), 0ull);
    direct.add(dx, B * n * 9 * (int64_t)sizeof(T), 0ull);
    direct.add(cnt, B * n * 12, 0ull);
    ccc_status st;
    if (lines) {
        FillRegions many;
        many.add(lines, B * n * 3 * kLineWords * 8, 0ull);
        st = fill_by_rows(many, direct, given, s);
    } else {
        st = fill_regions(direct, s);
    }
    if (st != CCC_OK) return st;
    KernelTimer tm(ctx, s);
    if (m > 0) {
        tm.begin("from_collisions");
        const int per_wave = m * B <= kShortRows ? kCcdThreads / 2 : kCcdThreads;
        const unsigned g = (unsigned)std::min<int64_t>((m + per_wave - 1) / per_wave, 16384);
#define CCC_ROWS(TABLE, SUMS)                                                                                             \
    hipLaunchKernelGGL((k_from_collisions<T, TABLE, SUMS>), dim3(g, B), dim3(kCcdThreads), 0, s, coll, (const T *)roots, \
                       m, (const T *)t0, (const T *)t1, (const T *)masses, n, (T *)dv, (T *)dx, cnt, lines, per_wave, given)
        if (lines) CCC_ROWS(true, SUMS_BY_ROWS);
        else if (n < ((int64_t)1 << 28)) CCC_ROWS(true, SUMS_DIRECT);
        else CCC_ROWS(false, SUMS_DIRECT);
#undef CCC_ROWS
        tm.end();
        CCC_LAUNCH_CHECK("k_from_collisions");
        if (lines) {
            hipLaunchKernelGGL((k_line_sums<T>), dim3(std::min(grid_for(B * n * 3, 256), 1024u)), dim3(256), 0, s, lines, B * n * 3, (T *)dv, (T *)dx, cnt, given);
            CCC_LAUNCH_CHECK("k_line_sums");
        }
    }
    CCC_HIP_TRY(hipStreamSynchronize(s));
    return CCC_OK;
}

// mesh_end[i] = offsets[m + 1] for the mesh m that owns triangle i (offsets ascending).
__global__ void k_mesh_end(const int64_t *__restrict__ offsets, int64_t meshes, int64_t total, int32_t *__restrict__ mesh_end) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    int64_t lo = 0, hi = meshes - 1;      // first m with offsets[m + 1] > i
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (offsets[mid + 1] > i) hi = mid;
        else lo = mid + 1;
    }
    mesh_end[i] = (int32_t)offsets[lo + 1];
}

// Independent meshes of different sizes stored back to back, handled as one soup: one BVH
// over the concatenation (compat Morton codes are all zero, so leaf position = triangle
// index and every subtree covers a contiguous index range) and one traversal whose queries
// never enter index ranges of later meshes.  Every stage after the traversal works on the
// resulting pairs unchanged.  The pair set of each mesh is exactly its own single-mesh set.
static ccc_status packed_impulses(ccc_context *ctx, const void *t0, const void *t1, const void *masses, const int64_t *offsets,
                                  int64_t meshes, int32_t dtype, int32_t max_candidates, void *dv, void *dx, int32_t *cnt,
                                  ccc_counts *counts, uint32_t flags, hipStream_t s) {
    clear_error();
    if (!ctx) return bad_arg("context is NULL");
    if (meshes < 0 || (meshes > 0 && !offsets)) return bad_arg("offsets is NULL");
    if (meshes == 0) return CCC_OK;
    if (offsets[0] != 0) return bad_arg("offsets[0] must be 0");
    for (int64_t m = 0; m < meshes; ++m)
        if (offsets[m + 1] <= offsets[m]) return bad_arg("every mesh needs at least one triangle (offsets strictly increasing)");
    const int64_t n = offsets[meshes];
    if (n >= ((int64_t)1 << 28)) return bad_arg("at most 2^28 - 1 triangles in a packed batch");
    if (!t0 || !t1 || !masses || !dv || !dx || !cnt) return bad_arg("NULL tensor pointer");
    if (max_candidates < 1) return bad_arg("max_candidates must be >= 1");
    if (dtype != CCC_FLOAT32 && dtype != CCC_FLOAT64) return bad_arg("dtype must be CCC_FLOAT32 or CCC_FLOAT64");
    CCC_HIP_TRY(hipSetDevice(ctx->device));
    const size_t esz = dtype == CCC_FLOAT64 ? 8 : 4;
    Workspace ws(ctx, s);
    void *bboxes = ws.get((size_t)(2 * n - 1) * 6 * esz);
    int64_t *tree = ws.get_as<int64_t>((2 * n - 1) * 4);
    int32_t *mesh_end = ws.get_as<int32_t>(n);
    int64_t *d_off = ws.get_as<int64_t>(meshes + 1);
    if (ws.failed()) return CCC_ERR_NO_MEMORY;
    CCC_HIP_TRY(hipMemcpyAsync(d_off, offsets, sizeof(int64_t) * (meshes + 1), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_mesh_end, dim3(grid_for(n, 256)), dim3(256), 0, s, d_off, meshes, n, mesh_end);
    CCC_LAUNCH_CHECK("k_mesh_end");
    // the packed traversal needs leaf position = triangle index (the reference's codes)
    ccc_status st = build_bvh_device(ctx, t0, t1, 1, n, dtype, CCC_MORTON_COMPAT, bboxes, tree, s);
    if ((st & CCC_ERR_MASK) != CCC_OK) return st;
    Query q{};
    q.ctx = ctx;
    q.bboxes = bboxes;
    q.tree = tree;
    q.t0 = t0;
    q.t1 = t1;
    q.masses = masses;
    q.B = 1;
    q.n = n;
    q.dtype = dtype;
    q.flags = flags;
    q.s = s;
    q.cap_candidates = (int64_t)max_candidates * n;
    q.narrow = Narrow::CCD_IMPULSE;
    q.dv = dv;
    q.dx = dx;
    q.cnt = cnt;
    q.counts = counts;
    q.mesh_end = mesh_end;
    if (dtype == CCC_FLOAT64) return run_query<double>(q);
    return run_query<float>(q);
}

// Scratch of the allocation-free entry point (ccc_compute_impulses_noalloc): every buffer
// of a call is carved from this array.  Each GPU that loads this code object holds its own
// copy until the process ends; host code reaches it only through the address
// hipGetSymbolAddress returns for the current device (the array's name on the host is a
// stand-in, not a device address).
static __device__ __align__(256) unsigned char scratch[CCC_NOALLOC_SCRATCH_BYTES];

ccc_status scratch_address(int device, void **out) {
    static std::mutex mu;
    static std::map<int, void *> cached;
    std::lock_guard<std::mutex> lock(mu);
    auto it = cached.find(device);
    if (it != cached.end()) {
        *out = it->second;
        return CCC_OK;
    }
    int prev = 0;
    CCC_HIP_TRY(hipGetDevice(&prev));
    CCC_HIP_TRY(hipSetDevice(device));
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    (void)hipSetDevice(prev);
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    cached[device] = p;
    *out = p;
    return CCC_OK;
}

}  // namespace ccc

using ccc::Narrow;
using ccc::Query;

static Query base_query(ccc_context *ctx, const void *bboxes, const int64_t *tree, const void *t0, int64_t B, int64_t n,
                        int32_t dtype, uint32_t flags, void *stream) {
    Query q{};
    q.ctx = ctx;
    q.bboxes = bboxes;
    q.tree = tree;
    q.t0 = t0;
    q.B = B;
    q.n = n;
    q.dtype = dtype;
    q.flags = flags;
    q.s = (hipStream_t)stream;
    return q;
}

static ccc_status tri_edge_query(ccc_context *ctx, const void *bboxes, const int64_t *tree, const void *triangles,
                                 int64_t batch, int64_t n, int32_t dtype, int32_t max_collisions, int mode, int64_t *out,
                                 void *coefs, int32_t *masks, ccc_counts *counts, uint32_t flags, void *stream) {
    Query q = base_query(ctx, bboxes, tree, triangles, batch, n, dtype, flags, stream);
    q.thr = 0.0;
    q.cap_candidates = (int64_t)max_collisions * n;
    q.out_cap = (int64_t)max_collisions * n;
    q.narrow = Narrow::TRI_EDGE;
    q.te_mode = mode;
    q.out_rows = out;
    q.out_roots = coefs;
    q.masks = masks;
    q.counts = counts;
    if (max_collisions < 1) return ccc::bad_arg("max_collisions must be >= 1");
    return ccc::run(q);
}

extern "C" {

ccc_status ccc_find_collisions(ccc_context *ctx, const void *bboxes, const int64_t *tree, const void *triangles, int64_t batch,
                               int64_t n, int32_t dtype, float threshold, int32_t max_collisions, int64_t *out,
                               ccc_counts *counts, uint32_t flags, void *stream) {
    Query q = base_query(ctx, bboxes, tree, triangles, batch, n, dtype, flags, stream);
    q.thr = (double)threshold;
    q.cap_candidates = (int64_t)max_collisions * n;
    q.out_cap = (int64_t)max_collisions * n;
    q.narrow = Narrow::SAT;
    q.out_rows = out;
    q.counts = counts;
    if (max_collisions < 1) return ccc::bad_arg("max_collisions must be >= 1");
    return ccc::run(q);
}

ccc_status ccc_find_triangle_edge_collisions(ccc_context *ctx, const void *bboxes, const int64_t *tree, const void *triangles,
                                             int64_t batch, int64_t n, int32_t dtype, int32_t max_collisions, int64_t *out,
                                             void *coefs, ccc_counts *counts, uint32_t flags, void *stream) {
    return tri_edge_query(ctx, bboxes, tree, triangles, batch, n, dtype, max_collisions, ccc::TE_COLLISIONS, out, coefs, nullptr,
                          counts, flags, stream);
}

ccc_status ccc_find_triangle_edge_candidates(ccc_context *ctx, const void *bboxes, const int64_t *tree, const void *triangles,
                                             int64_t batch, int64_t n, int32_t dtype, int32_t max_collisions, int64_t *out,
                                             ccc_counts *counts, uint32_t flags, void *stream) {
    return tri_edge_query(ctx, bboxes, tree, triangles, batch, n, dtype, max_collisions, ccc::TE_CANDIDATES, out, nullptr, nullptr,
                          counts, flags, stream);
}

ccc_status ccc_find_triangle_edge_candidates2(ccc_context *ctx, const void *bboxes, const int64_t *tree, const void *triangles,
                                              int64_t batch, int64_t n, int32_t dtype, int32_t max_collisions, int64_t *pairs,
                                              int32_t *masks, ccc_counts *counts, uint32_t flags, void *stream) {
    return tri_edge_query(ctx, bboxes, tree, triangles, batch, n, dtype, max_collisions, ccc::TE_CANDIDATES2, pairs, nullptr, masks,
                          counts, flags, stream);
}

ccc_status ccc_compute_impulses_packed(ccc_context *ctx, const void *triangles, const void *triangles_next, const void *masses,
                                       const int64_t *offsets, int64_t num_meshes, int32_t dtype, int32_t max_candidates,
                                       void *dv, void *dx, int32_t *cnt, ccc_counts *counts, uint32_t flags, void *stream) {
    return ccc::packed_impulses(ctx, triangles, triangles_next, masses, offsets, num_meshes, dtype, max_candidates, dv, dx, cnt,
                                counts, flags, (hipStream_t)stream);
}

ccc_status ccc_find_proximity(ccc_context *ctx, const void *bboxes, const int64_t *tree, const void *triangles, int64_t batch,
                              int64_t n, int32_t dtype, float threshold, int32_t max_candidates, int64_t *out,
                              ccc_counts *counts, uint32_t flags, void *stream) {
    Query q = base_query(ctx, bboxes, tree, triangles, batch, n, dtype, flags, stream);
    q.thr = (double)threshold;
    q.cap_candidates = (int64_t)max_candidates * n;
    q.out_cap = (int64_t)max_candidates * n;
    q.narrow = Narrow::PROXIMITY;
    q.out_rows = out;
    q.counts = counts;
    if (max_candidates < 1) return ccc::bad_arg("max_candidates_per_triangle must be >= 1");
    return ccc::run(q);
}

static ccc_status continuous(ccc_context *ctx, const void *bboxes, const int64_t *tree, const void *t0, const void *t1,
                             const uint8_t *to_check, int64_t batch, int64_t n, int32_t dtype, int32_t max_candidates,
                             int32_t max_collisions, int64_t *collisions, void *roots, ccc_counts *counts, uint32_t flags,
                             void *stream) {
    Query q = base_query(ctx, bboxes, tree, t0, batch, n, dtype, flags, stream);
    q.t1 = t1;
    q.to_check = to_check;
    q.thr = 0.0;
    q.cap_candidates = (int64_t)max_candidates * n;
    q.out_cap = (int64_t)max_collisions * n;
    q.narrow = Narrow::CCD_COLLECT;
    q.out_rows = collisions;
    q.out_roots = roots;
    q.counts = counts;
    if (max_candidates < 1 || max_collisions < 1) return ccc::bad_arg("capacities must be >= 1");
    return ccc::run(q);
}

ccc_status ccc_find_collisions_continuous(ccc_context *ctx, const void *bboxes, const int64_t *tree, const void *triangles,
                                          const void *triangles_next, int64_t batch, int64_t n, int32_t dtype,
                                          int32_t max_candidates, int32_t max_collisions, int64_t *collisions, void *roots,
                                          ccc_counts *counts, uint32_t flags, void *stream) {
    return continuous(ctx, bboxes, tree, triangles, triangles_next, nullptr, batch, n, dtype, max_candidates, max_collisions,
                      collisions, roots, counts, flags, stream);
}

ccc_status ccc_find_collisions_continuous_partial(ccc_context *ctx, const void *bboxes, const int64_t *tree,
                                                  const void *triangles, const void *triangles_next, const uint8_t *to_check,
                                                  int64_t batch, int64_t n, int32_t dtype, int32_t max_candidates,
                                                  int32_t max_collisions, int64_t *collisions, void *roots,
                                                  ccc_counts *counts, uint32_t flags, void *stream) {
    if (!to_check) { ccc::set_error("triangles_to_check is NULL"); return CCC_ERR_BAD_ARG; }
    return continuous(ctx, bboxes, tree, triangles, triangles_next, to_check, batch, n, dtype, max_candidates, max_collisions,
                      collisions, roots, counts, flags, stream);
}

ccc_status ccc_find_mincol_cand(ccc_context *ctx, const void *bboxes, const int64_t *tree, const void *triangles,
                                const void *triangles_next, int64_t batch, int64_t n, int32_t dtype, int32_t max_collisions,
                                int64_t *out, ccc_counts *counts, uint32_t flags, void *stream) {
    Query q = base_query(ctx, bboxes, tree, triangles, batch, n, dtype, flags, stream);
    q.t1 = triangles_next;
    q.thr = 0.0;
    q.cap_candidates = (int64_t)max_collisions * n;
    q.out_cap = (int64_t)max_collisions * n * 15;
    q.narrow = Narrow::MINCOL;
    q.out_rows = out;
    q.counts = counts;
    if (max_collisions < 1) return ccc::bad_arg("max_collisions must be >= 1");
    return ccc::run(q);
}

static ccc_status impulses(ccc_context *ctx, const void *bboxes, const int64_t *tree, const void *t0, const void *t1,
                           const void *masses, const uint8_t *to_check, int64_t batch, int64_t n, int32_t dtype,
                           int32_t max_candidates, void *dv, void *dx, int32_t *cnt, ccc_counts *counts, uint32_t flags,
                           void *stream) {
    Query q = base_query(ctx, bboxes, tree, t0, batch, n, dtype, flags, stream);
    q.t1 = t1;
    q.masses = masses;
    q.to_check = to_check;
    q.thr = 0.0;
    q.cap_candidates = (int64_t)max_candidates * n;
    q.out_cap = 0;
    q.narrow = Narrow::CCD_IMPULSE;
    q.dv = dv;
    q.dx = dx;
    q.cnt = cnt;
    q.counts = counts;
    if (max_candidates < 1) return ccc::bad_arg("max_candidates_per_triangle must be >= 1");
    return ccc::run(q);
}

ccc_status ccc_compute_impulses(ccc_context *ctx, const void *bboxes, const int64_t *tree, const void *triangles,
                                const void *triangles_next, const void *masses, int64_t batch, int64_t n, int32_t dtype,
                                int32_t max_candidates, int32_t max_collisions, void *dv, void *dx, int32_t *cnt,
                                ccc_counts *counts, uint32_t flags, void *stream) {
    (void)max_collisions;
    return impulses(ctx, bboxes, tree, triangles, triangles_next, masses, nullptr, batch, n, dtype, max_candidates, dv, dx, cnt,
                    counts, flags, stream);
}

ccc_status ccc_compute_impulses_noalloc(ccc_context *ctx, const void *bboxes, const int64_t *tree, const void *triangles,
                                        const void *triangles_next, const void *masses, int64_t batch, int64_t n, int32_t dtype,
                                        int32_t max_candidates, int32_t max_collisions, void *dv, void *dx, int32_t *cnt,
                                        ccc_counts *counts, uint32_t flags, void *stream) {
    (void)max_collisions;
    ccc::clear_error();
    if (!ctx) return ccc::bad_arg("context is NULL");
    if (!ctx->scratch) { ccc::set_error("the context has no scratch address"); return CCC_ERR_HIP; }
    Query q = base_query(ctx, bboxes, tree, triangles, batch, n, dtype, flags, stream);
    q.t1 = triangles_next;
    q.masses = masses;
    q.thr = 0.0;
    q.cap_candidates = (int64_t)max_candidates * n;
    q.out_cap = 0;
    q.narrow = Narrow::CCD_IMPULSE;
    q.dv = dv;
    q.dx = dx;
    q.cnt = cnt;
    q.counts = counts;
    q.arena = ctx->scratch;
    q.arena_bytes = CCC_NOALLOC_SCRATCH_BYTES;
    if (max_candidates < 1) return ccc::bad_arg("max_candidates_per_triangle must be >= 1");
    return ccc::run(q);
}

ccc_status ccc_compute_impulses_partial(ccc_context *ctx, const void *bboxes, const int64_t *tree, const void *triangles,
                                        const void *triangles_next, const void *masses, const uint8_t *to_check, int64_t batch,
                                        int64_t n, int32_t dtype, int32_t max_candidates, int32_t max_collisions, void *dv,
                                        void *dx, int32_t *cnt, ccc_counts *counts, uint32_t flags, void *stream) {
    (void)max_collisions;
    if (!to_check) { ccc::set_error("triangles_to_check is NULL"); return CCC_ERR_BAD_ARG; }
    return impulses(ctx, bboxes, tree, triangles, triangles_next, masses, to_check, batch, n, dtype, max_candidates, dv, dx, cnt,
                    counts, flags, stream);
}

ccc_status ccc_compute_impulses_from_collisions(ccc_context *ctx, const int64_t *collisions, const void *roots, int64_t m,
                                                const void *triangles, const void *triangles_next, const void *masses,
                                                int64_t batch, int64_t n, int32_t dtype, void *dv, void *dx, int32_t *cnt,
                                                uint32_t flags, void *stream) {
    (void)flags;
    ccc::clear_error();
    if (!ctx) return ccc::bad_arg("context is NULL");
    if (batch < 0 || n < 1 || m < 0) return ccc::bad_arg("invalid sizes");
    if (batch == 0) return CCC_OK;
    if (!triangles || !triangles_next || !masses || !dv || !dx || !cnt || (m > 0 && (!collisions || !roots)))
        return ccc::bad_arg("NULL tensor pointer");
    CCC_HIP_TRY(hipSetDevice(ctx->device));
    hipStream_t s = (hipStream_t)stream;
    if (dtype == CCC_FLOAT64)
        return ccc::from_collisions<double>(ctx, collisions, roots, m, triangles, triangles_next, masses, batch, n, dv, dx, cnt, s);
    if (dtype == CCC_FLOAT32)
        return ccc::from_collisions<float>(ctx, collisions, roots, m, triangles, triangles_next, masses, batch, n, dv, dx, cnt, s);
    return ccc::bad_arg("dtype must be CCC_FLOAT32 or CCC_FLOAT64");
}

}  // extern "C"

extern "C" ccc_status ccc_debug_device_math(ccc_context *ctx, int what, const double *x, double *y, int64_t n,
                                            void *stream) {
    ccc::clear_error();
    if (!ctx) return ccc::bad_arg("context is NULL");
    if (what < 0 || what > 11) return ccc::bad_arg("what must be 0-11");
    if (n < 0 || (n > 0 && (!x || !y))) return ccc::bad_arg("x and y must be device arrays of n doubles (what 5: 4 n each; what 10, 11: x 2 n)");
    if (n == 0) return CCC_OK;
    CCC_HIP_TRY(hipSetDevice(ctx->device));
    hipLaunchKernelGGL(ccc::k_device_math, dim3(ccc::grid_for(n, 256)), dim3(256), 0, (hipStream_t)stream, what, x, y, n);
    CCC_LAUNCH_CHECK("k_device_math");
    return CCC_OK;
}

extern "C" ccc_status ccc_debug_query_groups(ccc_context *ctx, const void *bboxes, const uint8_t *to_check, int64_t n, int32_t dtype, void *chunks,
                                             void *groups, void *stream) {
    ccc::clear_error();
    if (!ctx) return ccc::bad_arg("context is NULL");
    if (n < 1 || n >= ((int64_t)1 << 28) || !bboxes || !chunks || !groups) return ccc::bad_arg("need n in [1, 2^28) and device arrays");
    CCC_HIP_TRY(hipSetDevice(ctx->device));
    const unsigned g = ccc::grid_for(n, 256);
    if (dtype == CCC_FLOAT64)
        hipLaunchKernelGGL((ccc::k_prep<double>), dim3(g), dim3(256), 0, (hipStream_t)stream, (const double *)bboxes, (const int64_t *)nullptr, n, 0u, g, to_check,
                           (double *)chunks, (double *)groups, (const double *)nullptr, (const double *)nullptr, (double *)nullptr, (unsigned *)nullptr);
    else if (dtype == CCC_FLOAT32)
        hipLaunchKernelGGL((ccc::k_prep<float>), dim3(g), dim3(256), 0, (hipStream_t)stream, (const float *)bboxes, (const int64_t *)nullptr, n, 0u, g, to_check,
                           (float *)chunks, (float *)groups, (const float *)nullptr, (const float *)nullptr, (float *)nullptr, (unsigned *)nullptr);
    else return ccc::bad_arg("dtype must be CCC_FLOAT32 or CCC_FLOAT64");
    CCC_LAUNCH_CHECK("k_prep");
    return CCC_OK;
}
