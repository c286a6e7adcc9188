// Host-side plumbing shared by the C-ABI translation units: context, workspace
// allocation, error reporting, launch helpers and wave-level primitives.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/cccollisions_amd.h"

struct ccc_context {
    int device;
    ccc_alloc_fn alloc;
    ccc_free_fn free_fn;
    void *user;
    int num_cus;
    // pairs per narrow-phase chunk over the whole batch (0: the default)
    int64_t pair_chunk = 0;
    // this device's copy of the allocation-free entry point's scratch array
    void *scratch = nullptr;
    // Morton mode of the trees bvh / bvh_motion build (CCC_MORTON_*)
    int morton = CCC_MORTON_COMPAT;
    // opt-in kernel timing (HIP events on the call's stream), accumulated per kernel name
    bool profiling = false;
    std::mutex prof_mu;
    std::map<std::string, std::pair<double, int64_t>> prof;
    // pinned blocks that calls read their counters from (HostBlock), free ones; the context
    // keeps as many as it ever had calls at once and frees them with itself
    std::mutex host_mu;
    std::vector<void *> host_free;
};

namespace ccc {

void set_error(const std::string &msg);
void clear_error();

// A pinned host block of kBytes for the time of one call, from the context's free ones.  NULL
// when `on` is false or none can be had.  Kernels of `s` may write to it: settled() says that
// the stream was waited for since; without it the destructor waits.
class HostBlock {
  public:
    static constexpr size_t kBytes = 16384;
    HostBlock(ccc_context *ctx, hipStream_t s, bool on);
    ~HostBlock();
    template <typename P> P *as() const { return static_cast<P *>(p_); }
    void written() { settled_ = false; }
    void settled() { settled_ = true; }

  private:
    ccc_context *ctx_;
    hipStream_t s_;
    void *p_ = nullptr;
    bool settled_ = true;
};

// Per-call device workspace.  Buffers come from the context's allocator (or
// hipMallocAsync on the call's stream) and are released when the Workspace goes out of
// scope; the call has synchronised its stream before that happens.
// Arena mode (arena != NULL): buffers are carved from [arena, arena + arena_bytes) in
// order, 256-byte aligned, and nothing is allocated or freed; a request that does not fit
// fails like an allocation failure.
class Workspace {
  public:
    Workspace(ccc_context *ctx, hipStream_t s, void *arena = nullptr, size_t arena_bytes = 0)
        : ctx_(ctx), s_(s), arena_(static_cast<char *>(arena)), arena_bytes_(arena_bytes) {}
    ~Workspace();
    void *get(size_t bytes);
    template <typename P> P *get_as(size_t count) { return static_cast<P *>(get(count * sizeof(P))); }
    // NULL when there is no room; the Workspace has not failed then.
    template <typename P> P *try_get_as(size_t count) {
        const bool failed = failed_;
        P *p = get_as<P>(count);
        if (!p) {
            failed_ = failed;
            if (!arena_) (void)hipGetLastError();
            clear_error();
        }
        return p;
    }
    // Returns a buffer obtained from get() before the Workspace ends (stream-ordered).  In
    // arena mode only the most recent buffer can be returned (its bytes become free again).
    void release(void *p);
    bool failed() const { return failed_; }
    bool arena() const { return arena_ != nullptr; }
    // Arena mode: bytes not yet handed out (after 256-byte alignment of the next request).
    size_t arena_left() const { return arena_bytes_ > used_ ? arena_bytes_ - used_ : 0; }

  private:
    ccc_context *ctx_;
    hipStream_t s_;
    std::vector<void *> ptrs_;
    bool failed_ = false;
    char *arena_ = nullptr;
    size_t arena_bytes_ = 0, used_ = 0;
    std::vector<size_t> marks_;   // arena mode: offset of each buffer handed out
};

// Records HIP events around kernel launches when the context profiles; collect() runs
// after the call's stream synchronisation and adds the elapsed times to the context.
class KernelTimer {
  public:
    KernelTimer(ccc_context *ctx, hipStream_t s) : ctx_(ctx), s_(s), on_(ctx && ctx->profiling) {}
    ~KernelTimer() { collect(); }
    void begin(const char *name) {
        if (!on_) return;
        Rec r{name, nullptr, nullptr};
        if (hipEventCreate(&r.a) != hipSuccess || hipEventCreate(&r.b) != hipSuccess) { on_ = false; return; }
        (void)hipEventRecord(r.a, s_);
        recs_.push_back(r);
    }
    void end() {
        if (!on_ || recs_.empty()) return;
        (void)hipEventRecord(recs_.back().b, s_);
    }
    void collect() {
        if (recs_.empty()) return;
        (void)hipStreamSynchronize(s_);
        std::lock_guard<std::mutex> lock(ctx_->prof_mu);
        for (auto &r : recs_) {
            float ms = 0.f;
            if (hipEventElapsedTime(&ms, r.a, r.b) == hipSuccess) {
                auto &e = ctx_->prof[r.name];
                e.first += ms;
                e.second += 1;
            }
            (void)hipEventDestroy(r.a);
            (void)hipEventDestroy(r.b);
        }
        recs_.clear();
    }

  private:
    struct Rec { const char *name; hipEvent_t a, b; };
    ccc_context *ctx_;
    hipStream_t s_;
    bool on_;
    std::vector<Rec> recs_;
};

#define CCC_TIMED(timer, name, launch) \
    do {                               \
        (timer).begin(name);           \
        launch;                        \
        (timer).end();                 \
    } while (0)

inline ccc_status hip_fail(hipError_t e, const char *what) {
    set_error(std::string(what) + ": " + hipGetErrorString(e));
    return CCC_ERR_HIP;
}

#define CCC_HIP_TRY(expr)                                                                       \
    do {                                                                                        \
        hipError_t _e = (expr);                                                                 \
        if (_e != hipSuccess) return ::ccc::hip_fail(_e, #expr);                                \
    } while (0)

#define CCC_LAUNCH_CHECK(what)                                                                  \
    do {                                                                                        \
        hipError_t _e = hipGetLastError();                                                      \
        if (_e != hipSuccess) return ::ccc::hip_fail(_e, what);                                 \
    } while (0)

inline ccc_status bad_arg(const std::string &msg) {
    set_error(msg);
    return CCC_ERR_BAD_ARG;
}

inline unsigned grid_for(int64_t items, int block) {
    int64_t g = (items + block - 1) / block;
    if (g < 1) g = 1;
    return (unsigned)g;
}

// Device error bits reported by kernels.
// DEV_UNORDERED is informational: the tree's subtrees do not cover contiguous, ordered
// leaf ranges (or are deeper than 64), so the rightmost leaves come from the climb.
// DEV_FOREIGN: the tree is not the index tree that bvh / bvh_motion build by default.
enum : unsigned { DEV_BAD_TREE = 1u, DEV_STACK = 2u, DEV_UNORDERED = 4u, DEV_FOREIGN = 8u };

// The compat tree is the radix tree over leaf indices (every Morton code is 0).  Node i covers
// the aligned block of 2^k leaves that starts at i (i even, k = trailing zeros of i) or ends
// at i (i odd, k = trailing zeros of i + 1), cut off at n; node 0 covers everything.  That is
// Karras' Algorithm 1 (k_karras) with delta(i, j) = 32 + clz(i ^ j) solved in closed form: the
// direction and range follow from i's neighbours, and the split is at the highest differing
// bit of the range's ends.
__device__ __forceinline__ int index_node_level(int64_t i) { return __ffsll((long long)((i & 1) ? i + 1 : i)) - 1; }

__device__ __forceinline__ void index_node_row(int64_t i, int64_t n, int64_t &left, int64_t &right) {
    int64_t lo = 0, hi = n - 1;
    if (i > 0) {
        const int64_t len = (int64_t)1 << index_node_level(i);
        lo = (i & 1) ? i + 1 - len : i;
        hi = (i & 1) ? i : (i + len <= n ? i + len - 1 : n - 1);
    }
    const int bit = 63 - __clzll((long long)(lo ^ hi));
    const int64_t split = ((hi >> bit) << bit) - 1;
    left = lo == split ? n - 1 + split : split;
    right = hi == split + 1 ? n - 1 + split + 1 : split + 1;
}

// Per-batch-element counters kept on the device during a call.
struct alignas(64) DevCounters {
    unsigned long long cand;    // K (total, may exceed the candidate capacity)
    unsigned long long items;   // M of the current pair chunk
    unsigned long long roots;   // V
    unsigned long long coll;    // R (total, may exceed the output capacity)
    unsigned long long items_done;  // M of the pair chunks already finished
    unsigned long long tiles;   // item tiles of the current pair chunk (continuous narrow phase)
    unsigned int flags;         // DEV_* bits
    unsigned int pad[3];
};
static_assert(sizeof(DevCounters) == 64, "DevCounters is one 64-byte line");

// Counts that nobody reads before the call ends: every block of the narrow phase adds its own
// to one of up to kPartials lines of its batch element, and k_fold_partials sums them.  An atomic on one device address
// takes 6-13 ns however many waves issue them: on the shared counters the 32,768 blocks of
// k_ccd spent 0.4-0.8 ms of a pass on two of them each (all of its time on the 33k f32 pass).
struct alignas(128) DevPartial {
    unsigned long long items, roots, coll;
};
constexpr int kPartials = 64;

// Device address of the allocation-free entry point's scratch array on `device` (looked up
// once per device with that device current, then cached).
ccc_status scratch_address(int device, void **out);

// One compute_impulses pass of one mesh (or one packed set of meshes) over caller-owned,
// resident buffers, for the resident simulation.  Nothing waits on the host and nothing is
// allocated: workspace comes from `arena` in a fixed order (so the buffers have the same
// addresses on every call with the same sizes and the pass can be captured in a HIP graph),
// the candidate list keeps at most cap_pairs pairs (more are counted in ctr->cand and must
// be detected by the caller after synchronising), the narrow phase covers [0, cap_pairs)
// in chunks of `chunk` pairs whose kernels stop at the counts on the device, and the
// counters stay in `ctr` (zeroed by the pass).  det_acc != NULL: the impulse sums are
// order-independent (fixed-point limbs, kDetWords int64 per corner) and then written to dv
// / dx, so that a pass gives the same bits however its atomics interleave.
struct ResidentPass {
    const void *bboxes;
    const int64_t *tree;
    const void *t0, *t1, *masses;
    int64_t n;
    int32_t dtype;
    const int32_t *mesh_end;     // packed meshes: per triangle, the end of its mesh; else NULL
    int2 *pairs;
    int64_t cap_pairs;
    int64_t chunk;
    int ccd_blocks_per_cu;       // grid cap of k_ccd (0: 128)
    const int64_t *leaf_ids;     // the tree when its leaves are in another order than the triangles (fitted), else NULL
    long long *det_acc;
    double *lines;               // non-NULL: the sums as lines, dv / dx / cnt not written (line_sums)
    void *dv, *dx;
    int32_t *cnt;
    DevCounters *ctr;
};
ccc_status resident_pass(ccc_context *ctx, const ResidentPass &p, void *arena, size_t arena_bytes, hipStream_t s);
size_t resident_pass_arena_bytes(ccc_context *ctx, const ResidentPass &p);
constexpr int kDetWordsPerCorner = 24;
constexpr int kLineWordsPerCorner = 8;     // dv xyz, dx xyz, count, 0
// dv, dx and cnt of every corner from its line.
ccc_status line_sums(const double *lines, int64_t corners, int32_t dtype, void *dv, void *dx, int32_t *cnt, hipStream_t s);

// Buffers a call fills before it starts (a kernel instead of hipMemsetAsync, so that the
// calls stay capturable): `words` 32-bit words of the repeated 64-bit `value`.
struct FillRegion {
    void *p;
    int64_t words;
    uint64_t value;
};
struct FillRegions {
    FillRegion r[8];
    unsigned blocks[8] = {};     // of each region's, in one launch
    int count = 0;
    void add(void *p, int64_t bytes, uint64_t value) { r[count++] = FillRegion{p, bytes / 4, value}; }
};
ccc_status fill_regions(const FillRegions &r, hipStream_t s);

// Lists of given rows, -1 from each list's end on.  Whether they hold a row per triangle is only
// known on the device: the kernels that depend on it look at the same four places.  (Rows in
// another order than that may be taken for fewer or more than they are; both ways are right.)
struct GivenRows {
    const int64_t *at[4];       // all NULL: nothing depends on the rows
};
// B lists of m rows on meshes of n <= m triangles: at quarters of the first n, each in a quarter
// of the lists.
inline GivenRows given_rows(const int64_t *rows, int64_t m, int64_t n, int64_t B) {
    GivenRows g;
    for (int q = 0; q < 4; ++q) g.at[q] = rows + 3 * (q * B / 4 * m + ((q + 1) * n + 3) / 4 - 1);
    return g;
}
__device__ __forceinline__ bool many_rows(const GivenRows &g) {
    return (*g.at[0] >= 0) & (*g.at[1] >= 0) & (*g.at[2] >= 0) & (*g.at[3] >= 0);
}
// Fills `many` or `few`, as many_rows says.
ccc_status fill_by_rows(const FillRegions &many, const FillRegions &few, const GivenRows &g, hipStream_t s);

// BVH over B soups of n triangles each (t1 = NULL: static boxes) into the wire format, with
// Morton mode `morton` (CCC_MORTON_*); arguments already validated, the device already
// current.
ccc_status build_bvh_device(ccc_context *ctx, const void *t0, const void *t1, int64_t B, int64_t n, int32_t dtype, int morton,
                            void *bboxes, int64_t *tree, hipStream_t s, void *arena = nullptr, size_t arena_bytes = 0);
// Workspace bytes of build_bvh_device (all of its buffers, 256-byte rounded).
size_t build_bvh_arena_bytes(int64_t B, int64_t n, int32_t dtype, int morton);

}  // namespace ccc

// Leaf positions are grouped in chunks of 64, one per lane of a wave.
namespace ccc {
constexpr int kChunkBits = 6;
constexpr int kChunk = 1 << kChunkBits;
}

// ---- wave primitives (wave64) ---------------------------------------------------------
namespace ccc {
// Number of lanes below the calling lane whose bit is set in `mask`.
__device__ __forceinline__ unsigned lanes_below(unsigned long long mask) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}
__device__ __forceinline__ unsigned long long readfirstlane_u64(unsigned long long v) {
    unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}
// Slot of the calling lane in a list whose length is the LDS counter *counter: every active
// lane appends one entry, the wave's entries go in lane order after one atomic.
__device__ __forceinline__ int wave_append1(int *counter) {
    const unsigned long long act = __ballot(1);
    const unsigned below = lanes_below(act);
    int base = 0;
    if (below == 0) base = atomicAdd(counter, (int)__popcll(act));
    base = __builtin_amdgcn_readfirstlane(base);
    return base + (int)below;
}
// Reserve `cnt` consecutive slots (cnt < 16) per active lane of the wave from `counter`
// with a single atomic; returns this lane's first slot.
__device__ __forceinline__ unsigned long long wave_reserve(unsigned long long *counter, unsigned cnt) {
    unsigned long long b0 = __ballot(cnt & 1u), b1 = __ballot(cnt & 2u), b2 = __ballot(cnt & 4u), b3 = __ballot(cnt & 8u);
    unsigned below = lanes_below(b0) + 2u * lanes_below(b1) + 4u * lanes_below(b2) + 8u * lanes_below(b3);
    unsigned long long total = (unsigned long long)__popcll(b0) + 2ull * __popcll(b1) + 4ull * __popcll(b2) + 8ull * __popcll(b3);
    unsigned long long base = 0;
    if (lanes_below(__ballot(1)) == 0 && total) base = atomicAdd(counter, total);
    base = readfirstlane_u64(base);
    return base + below;
}

// Orders the wave's LDS accesses before this point against those after it.  The lanes of a
// wavefront run in lockstep and the LDS serves one wave's accesses in issue order, so no
// instruction is needed: the fences and the barrier only keep the compiler from moving
// memory accesses across the point.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace ccc
