// Context, workspace and error plumbing of the C ABI.
#include <limits.h>

#include <algorithm>

#include "ccc_internal.h"

#include <cstring>
#include <new>

namespace ccc {

static thread_local std::string g_last_error;

void set_error(const std::string &msg) { g_last_error = msg; }
void clear_error() { g_last_error.clear(); }

HostBlock::HostBlock(ccc_context *ctx, hipStream_t s, bool on) : ctx_(ctx), s_(s) {
    if (!on) return;
    {
        std::lock_guard<std::mutex> lock(ctx->host_mu);
        if (!ctx->host_free.empty()) {
            p_ = ctx->host_free.back();
            ctx->host_free.pop_back();
            return;
        }
    }
    if (hipHostMalloc(&p_, kBytes) != hipSuccess) {
        (void)hipGetLastError();
        p_ = nullptr;
    }
}

HostBlock::~HostBlock() {
    if (!p_) return;
    if (!settled_) (void)hipStreamSynchronize(s_);
    std::lock_guard<std::mutex> lock(ctx_->host_mu);
    ctx_->host_free.push_back(p_);
}

Workspace::~Workspace() {
    if (arena_) return;
    for (void *p : ptrs_) {
        if (ctx_ && ctx_->free_fn) ctx_->free_fn(ctx_->user, p, (void *)s_);
        else (void)hipFreeAsync(p, s_);
    }
}

void Workspace::release(void *p) {
    if (arena_) {
        if (!marks_.empty() && arena_ + marks_.back() == static_cast<char *>(p)) {
            used_ = marks_.back();
            marks_.pop_back();
        }
        return;
    }
    for (size_t i = 0; i < ptrs_.size(); ++i) {
        if (ptrs_[i] != p) continue;
        if (ctx_ && ctx_->free_fn) ctx_->free_fn(ctx_->user, p, (void *)s_);
        else (void)hipFreeAsync(p, s_);
        ptrs_.erase(ptrs_.begin() + (std::ptrdiff_t)i);
        return;
    }
}

void *Workspace::get(size_t bytes) {
    if (bytes == 0) bytes = 256;
    bytes = (bytes + 255) & ~(size_t)255;
    if (arena_) {
        if (bytes > arena_left()) {
            failed_ = true;
            set_error("the call needs more than the " + std::to_string(arena_bytes_) +
                      "-byte scratch buffer: " + std::to_string(used_) + " bytes in use, " + std::to_string(bytes) +
                      " more requested");
            return nullptr;
        }
        marks_.push_back(used_);
        void *p = arena_ + used_;
        used_ += bytes;
        return p;
    }
    void *p = nullptr;
    if (ctx_ && ctx_->alloc) {
        p = ctx_->alloc(ctx_->user, bytes, (void *)s_);
    } else {
        if (hipMallocAsync(&p, bytes, s_) != hipSuccess) p = nullptr;
    }
    if (!p) {
        failed_ = true;
        set_error("workspace allocation of " + std::to_string(bytes) + " bytes failed");
        return nullptr;
    }
    ptrs_.push_back(p);
    return p;
}

// One launch for all the buffers a call starts from (seven fills of 2-5 us each otherwise).  A
// thread stores four words, 16 bytes where the region's address allows it, and a block 4 KiB:
// 6.4 to 6.9 TB/s on 1 to 6 GiB, where a loop over 8,192 blocks reached 4.3 to 5.0 and 8-byte
// stores over 65,536 blocks 5.7; up to 50 MB they are alike.
constexpr int64_t kFillWords = 4 * 256;     // per block
__device__ __forceinline__ void fill_block(const FillRegions &r, unsigned block) {
    unsigned first = 0;
    int k = 0;
    while (k + 1 < r.count && block >= first + r.blocks[k]) first += r.blocks[k++];
    const FillRegion f = r.r[k];
    const uint32_t lo = (uint32_t)f.value, hi = (uint32_t)(f.value >> 32);
    const int64_t i = (int64_t)(block - first) * kFillWords + 4 * threadIdx.x;
    uint32_t *p = reinterpret_cast<uint32_t *>(f.p);
    if (i + 4 <= f.words && ((uintptr_t)f.p & 15) == 0) {
        *reinterpret_cast<uint4 *>(p + i) = make_uint4(lo, hi, lo, hi);
        return;
    }
    for (int64_t j = i; j < i + 4 && j < f.words; ++j) p[j] = (j & 1) ? hi : lo;
}
__global__ __launch_bounds__(256) void k_fill_regions(FillRegions r, unsigned base) { fill_block(r, base + blockIdx.x); }
// Every gridDim.x-th block's worth, as a block starts with a wait for its four rows: 156 MB on
// 4,096 blocks in 30 us (8 blocks' worth in a row each: 33; 38,000 blocks of one: about 60).  What
// lies past the chosen regions finds no words left in the last of them.
constexpr int64_t kRowsFillBlocks = 4096;
__global__ __launch_bounds__(256) void k_fill_by_rows(FillRegions many, FillRegions few, GivenRows g, unsigned total) {
    const bool all = many_rows(g);
    for (unsigned j = blockIdx.x; j < total; j += gridDim.x) {
        if (all) fill_block(many, j);
        else fill_block(few, j);
    }
}

// A launch holds fewer than 2^32 work items (hip_runtime_api.h), which is 64 GiB here: larger
// fills take one launch per 32 GiB.
constexpr int64_t kFillLaunchBlocks = (int64_t)1 << 23;

// Blocks of each region, and of all of them.
static int64_t count_fill_blocks(FillRegions &r) {
    int64_t total = 0;
    for (int k = 0; k < r.count; ++k) {
        const int64_t blocks = r.r[k].words > 0 ? (r.r[k].words + kFillWords - 1) / kFillWords : 0;
        r.blocks[k] = (unsigned)blocks;
        total += blocks;
    }
    return total;
}
// launch(first block, blocks) for every launch of a fill of `total` blocks.
template <typename F> static void each_fill_launch(int64_t total, F launch) {
    for (int64_t base = 0; base < total; base += kFillLaunchBlocks)
        launch((unsigned)base, (unsigned)std::min(total - base, kFillLaunchBlocks));
}

ccc_status fill_regions(const FillRegions &regions, hipStream_t s) {
    FillRegions r = regions;
    const int64_t total = count_fill_blocks(r);
    if (total > INT_MAX) return bad_arg("an output of more than 8 TiB");
    each_fill_launch(total, [&](unsigned base, unsigned blocks) {
        hipLaunchKernelGGL(k_fill_regions, dim3(blocks), dim3(256), 0, s, r, base);
    });
    CCC_LAUNCH_CHECK("fill_regions");
    return CCC_OK;
}

ccc_status fill_by_rows(const FillRegions &many, const FillRegions &few, const GivenRows &g, hipStream_t s) {
    FillRegions a = many, b = few;
    const int64_t total = std::max(count_fill_blocks(a), count_fill_blocks(b));
    if (total > INT_MAX) return bad_arg("an output of more than 8 TiB");
    const int64_t blocks = std::min<int64_t>(total, std::max<int64_t>(kRowsFillBlocks, total / 64));
    if (total > 0) hipLaunchKernelGGL(k_fill_by_rows, dim3((unsigned)blocks), dim3(256), 0, s, a, b, g, (unsigned)total);
    CCC_LAUNCH_CHECK("fill_by_rows");
    return CCC_OK;
}

}  // namespace ccc

extern "C" {

ccc_status ccc_context_create(ccc_context **out, int device, ccc_alloc_fn alloc, ccc_free_fn free_fn, void *user) {
    ccc::clear_error();
    if (!out) return ccc::bad_arg("ccc_context_create: out is NULL");
    *out = nullptr;
    int ndev = 0;
    CCC_HIP_TRY(hipGetDeviceCount(&ndev));
    if (device < 0 || device >= ndev) return ccc::bad_arg("ccc_context_create: invalid device " + std::to_string(device));
    int cus = 0;
    CCC_HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
    ccc_context *c = new (std::nothrow) ccc_context;
    if (!c) return CCC_ERR_NO_MEMORY;
    c->device = device;
    c->alloc = alloc;
    c->free_fn = free_fn;
    c->user = user;
    c->num_cus = cus > 0 ? cus : 256;
    ccc_status st = ccc::scratch_address(device, &c->scratch);
    if (st != CCC_OK) {
        delete c;
        return st;
    }
    *out = c;
    return CCC_OK;
}

void ccc_context_destroy(ccc_context *ctx) {
    if (ctx)
        for (void *p : ctx->host_free) (void)hipHostFree(p);
    delete ctx;
}

const char *ccc_status_string(ccc_status status) {
    switch (status & CCC_ERR_MASK) {
        case CCC_OK: return (status & CCC_WARN_TRUNCATED) ? "ok (output truncated)" : (status & CCC_WARN_CANDIDATES) ? "ok (candidate capacity exceeded)" : "ok";
        case CCC_ERR_BAD_ARG: return "invalid argument";
        case CCC_ERR_HIP: return "HIP runtime error";
        case CCC_ERR_NO_MEMORY: return "out of device memory";
        case CCC_ERR_BAD_TREE: return "malformed BVH tree";
        case CCC_ERR_STACK: return "BVH deeper than the traversal stack";
        default: return "unknown status";
    }
}

const char *ccc_last_error(void) { return ccc::g_last_error.c_str(); }

int ccc_abi_version(void) { return CCC_ABI_VERSION; }

ccc_status ccc_context_set_pair_chunk(ccc_context *ctx, int64_t pairs) {
    if (!ctx) return ccc::bad_arg("context is NULL");
    if (pairs < 0) return ccc::bad_arg("pair chunk must be >= 0");
    ctx->pair_chunk = pairs;
    return CCC_OK;
}

ccc_status ccc_context_set_morton(ccc_context *ctx, int mode) {
    if (!ctx) return ccc::bad_arg("context is NULL");
    if (mode != CCC_MORTON_COMPAT && mode != CCC_MORTON_30 && mode != CCC_MORTON_63)
        return ccc::bad_arg("Morton mode must be CCC_MORTON_COMPAT, CCC_MORTON_30 or CCC_MORTON_63");
    ctx->morton = mode;
    return CCC_OK;
}

ccc_status ccc_context_set_profiling(ccc_context *ctx, int on) {
    if (!ctx) return ccc::bad_arg("context is NULL");
    std::lock_guard<std::mutex> lock(ctx->prof_mu);
    ctx->profiling = on != 0;
    ctx->prof.clear();
    return CCC_OK;
}

ccc_status ccc_context_kernel_time(ccc_context *ctx, const char *kernel, double *total_ms, int64_t *launches) {
    if (!ctx || !kernel || !total_ms || !launches) return ccc::bad_arg("NULL argument");
    std::lock_guard<std::mutex> lock(ctx->prof_mu);
    auto it = ctx->prof.find(kernel);
    *total_ms = it == ctx->prof.end() ? 0.0 : it->second.first;
    *launches = it == ctx->prof.end() ? 0 : it->second.second;
    return CCC_OK;
}

int ccc_context_kernel_names(ccc_context *ctx, char *buf, size_t len) {
    if (!ctx) return -1;
    std::string all;
    {
        std::lock_guard<std::mutex> lock(ctx->prof_mu);
        for (auto &kv : ctx->prof) { if (!all.empty()) all += ","; all += kv.first; }
    }
    if (buf && len > 0) {
        size_t n = all.size() < len - 1 ? all.size() : len - 1;
        memcpy(buf, all.data(), n);
        buf[n] = 0;
    }
    return (int)all.size();
}

int ccc_debug_fill_launches(const int64_t *bytes, int count, int64_t *blocks, int capacity) {
    ccc::FillRegions r;
    if (!bytes || !blocks || count < 0 || count > (int)(sizeof(r.r) / sizeof(r.r[0]))) return -1;
    for (int k = 0; k < count; ++k) r.add(nullptr, bytes[k], 0ull);
    const int64_t total = ccc::count_fill_blocks(r);
    if (total > INT_MAX) return -1;
    int launches = 0;
    ccc::each_fill_launch(total, [&](unsigned base, unsigned n) {
        if (launches < capacity) {
            blocks[2 * launches] = base;
            blocks[2 * launches + 1] = n;
        }
        ++launches;
    });
    return launches;
}

}  // extern "C"
