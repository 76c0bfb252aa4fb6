// Context: device, stream, HBM budget, scratch pool, operand cache, timing.
// Replaces the role of Aquarius's Arena (src/util/distributed.hpp:28-74): the
// place every tensor of one job lives.  One context = one HIP stream; nothing
// here is global, so contexts on one device are independent.
#include "internal.hpp"

#include <atomic>

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>

namespace aqamd {

static thread_local std::string g_last_error;

void set_last_error(const std::string& msg) { g_last_error = msg; }

size_t ctx_in_use(const aq_ctx* ctx) { return ctx->tensor_bytes + ctx->pool_bytes + ctx->cache_bytes; }

// Blocks that a server's jobs have freed, kept for its next jobs.  The device
// pool releases its free memory to the driver once that exceeds what is in use
// (36 to 46 ms per release here, twice in a burst of eight small jobs), and
// every job's end frees nearly all it had.  Safe across the slots' streams: a
// block goes to other slots only when its job has ended and its stream is
// synchronised (before that to the same stream, in order), so no slot ever waits
// for another's events.  Such waits do not go together with graphs: an event of
// a stream that another thread captures by now cannot be waited for, and a host
// wait for it ends that capture.  Bounded by the server's budget (BlockLedger):
// what does not fit beside the running jobs' reservations goes to the device
// pool, oldest first.
struct BlockCache {
    int device = 0;
    std::mutex mu;
    BlockLedger led;

    void* take(size_t n) {
        std::lock_guard<std::mutex> lk(mu);
        KeptBlock b;
        return led.take(n, b) ? b.p : nullptr;
    }
    void lend(void* p, size_t bytes, size_t asked) noexcept {
        std::lock_guard<std::mutex> lk(mu);
        try {
            led.lend(p, bytes, asked);
        } catch (...) {   // no host memory: not tracked, and freed as any other block
        }
    }
    BlockLedger::Lent back(void* p) {
        std::lock_guard<std::mutex> lk(mu);
        return led.back(p);
    }
    // An idle block; false: no room (the caller frees it).  pooled: the device
    // pool got older blocks instead.
    bool keep(const KeptBlock& b, hipStream_t stream, bool& pooled) noexcept {
        std::lock_guard<std::mutex> lk(mu);
        if (!led.fits(b.bytes)) return false;
        try {
            led.keep(b);
        } catch (...) {   // no host memory for the bookkeeping
            return false;
        }
        release_over(stream, pooled);
        return true;
    }
    void set_limit(size_t bytes) {
        std::lock_guard<std::mutex> lk(mu);
        led.limit = bytes;
    }
    // what may be lent beyond the requests' sizes
    size_t spare() {
        std::lock_guard<std::mutex> lk(mu);
        return led.limit > led.slack() ? led.limit - led.slack() : 0;
    }
    size_t slack() {
        std::lock_guard<std::mutex> lk(mu);
        return led.slack();
    }
    size_t kept() {
        std::lock_guard<std::mutex> lk(mu);
        return led.kept();
    }
    // Kept blocks beyond the limit (all: every kept block) to the device pool.
    void release(hipStream_t stream, bool all, bool& pooled) {
        std::lock_guard<std::mutex> lk(mu);
        release_over(stream, pooled);
        while (all && !led.empty()) release_oldest(stream, pooled);
    }
    ~BlockCache() {
        bool pooled = false;
        release(nullptr, true, pooled);
        (void)hipStreamSynchronize(nullptr);
    }

  private:
    void release_oldest(hipStream_t stream, bool& pooled) noexcept {   // mu held
        (void)hipFreeAsync(led.pop_oldest().p, stream);
        pooled = true;
    }
    void release_over(hipStream_t stream, bool& pooled) noexcept {
        while (led.over()) release_oldest(stream, pooled);
    }
};

// Every server's cache: a context that runs short of memory, or is trimmed,
// takes back what servers on its device keep.  Locked before a cache's own mutex.
static std::mutex g_caches_mu;
static std::vector<BlockCache*> g_caches;

size_t kept_bytes(int device) {
    std::lock_guard<std::mutex> lk(g_caches_mu);
    size_t n = 0;
    for (auto* c : g_caches)
        if (c->device == device) n += c->kept();
    return n;
}

static void release_kept_blocks(aq_ctx* ctx) {
    std::lock_guard<std::mutex> lk(g_caches_mu);
    for (auto* c : g_caches)
        if (c->device == ctx->device) c->release(ctx->stream, true, ctx->pooled);
}

BlockCache* block_cache_create(int device) {
    std::unique_ptr<BlockCache> c(new BlockCache());
    c->device = device;
    std::lock_guard<std::mutex> lk(g_caches_mu);
    g_caches.push_back(c.get());
    return c.release();
}
void block_cache_destroy(BlockCache* c) {
    {
        std::lock_guard<std::mutex> lk(g_caches_mu);
        g_caches.erase(std::remove(g_caches.begin(), g_caches.end(), c), g_caches.end());
    }
    delete c;
}
void block_cache_limit(BlockCache* c, size_t bytes) { c->set_limit(bytes); }
size_t block_cache_slack(BlockCache* c) { return c->slack(); }

// A job starts: kept blocks that its reservation displaces go, and so do all
// servers' where the device runs short for what the runtime allocates by itself
// (the scratch of a queue's first spilling kernel: up to 0.2 GB a queue, and
// the queue aborts without it).
void block_cache_settle(aq_ctx* ctx) {
    constexpr size_t kDeviceReserve = size_t(4) << 30;
    ctx->drained = false;
    ctx->blocks->release(ctx->stream, false, ctx->pooled);
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) == hipSuccess && free_b < kDeviceReserve) {
        release_kept_blocks(ctx);
        (void)hipStreamSynchronize(ctx->stream);
        trim_device_pool(ctx->device);   // also what other contexts left there
    }
    (void)hipGetLastError();
    block_cache_trim(ctx);
}

// What the device pool got from this slot, back to the driver.
void block_cache_trim(aq_ctx* ctx) {
    if (!ctx->pooled) return;
    ctx->pooled = false;
    (void)hipStreamSynchronize(ctx->stream);   // the frees are complete
    trim_device_pool(ctx->device);
}

// Stream-ordered device memory: allocations and frees are ordered on the
// context's stream, so one context releasing memory never synchronises the
// device under other contexts (concurrent serving).
static void pool_free(aq_ctx* ctx, void* p) {
    (void)hipFreeAsync(p, ctx->stream);
    ctx->pooled = true;
}

void* dmalloc(aq_ctx* ctx, size_t bytes) {
    if (ctx->blocks) {
        KeptBlock b;
        if (ctx->own.take(bytes, ctx->blocks->spare(), b)) {
            ctx->blocks->lend(b.p, b.bytes, bytes);
            ctx->blocks->release(ctx->stream, false, ctx->pooled);
            return b.p;
        }
        if (void* p = ctx->blocks->take(bytes)) return p;
        // within the reservation also with what the job has freed
        while (!ctx->own.blocks.empty() && ctx_in_use(ctx) + bytes + ctx->own.bytes > ctx->budget)
            pool_free(ctx, ctx->own.pop_oldest().p);
    }
    void* p = nullptr;
    if (hipMallocAsync(&p, bytes, ctx->stream) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    if (ctx->blocks) ctx->blocks->lend(p, bytes, bytes);
    return p;
}

void dfree(aq_ctx* ctx, void* p) {
    if (!p) return;
    ctx->mem_gen += 1;
    if (!ctx->blocks) {
        (void)hipFreeAsync(p, ctx->stream);
        return;
    }
    const BlockLedger::Lent l = ctx->blocks->back(p);
    if (l.bytes && ctx->drained) {
        if (ctx->blocks->keep({p, l.bytes}, ctx->stream, ctx->pooled)) return;
    } else if (l.bytes && ctx_in_use(ctx) - l.asked + ctx->own.bytes + l.bytes <= ctx->budget) {
        try {
            ctx->own.keep({p, l.bytes});
            return;
        } catch (const std::bad_alloc&) {
        }
    }
    pool_free(ctx, p);
}

// A job has ended and its stream is synchronised: what it frees from here on, and
// has freed, is idle.
void block_cache_drained(aq_ctx* ctx) {
    ctx->drained = true;
    while (!ctx->own.blocks.empty()) {
        const KeptBlock b = ctx->own.pop_oldest();
        if (!ctx->blocks->keep(b, ctx->stream, ctx->pooled)) pool_free(ctx, b.p);
    }
}

// Return the memory the device's default pool holds but no allocation uses
// (blocks whose stream-ordered frees have completed, on any stream) to the
// driver.  The pool keeps freed blocks between synchronisations (release
// threshold at its maximum), which is what makes repeated allocation cheap
// within a job; across jobs of different sizes those cached blocks can be
// the wrong shapes for the next request, and memory that sits there is missing
// to everything else on the device, the runtime's own allocations among it.
// They are trimmed when a served job ends, when a server starts and before an
// allocation is retried.
void trim_device_pool(int device) {
    hipMemPool_t pool;
    if (hipDeviceGetDefaultMemPool(&pool, device) == hipSuccess) (void)hipMemPoolTrimTo(pool, 0);
    (void)hipGetLastError();
}

static void note_peak(aq_ctx* ctx) { ctx->peak_bytes = std::max(ctx->peak_bytes, ctx_in_use(ctx)); }

static void pool_release_all(aq_ctx* ctx) {
    for (auto& kv : ctx->pool_free) {
        for (void* p : kv.second) {
            dfree(ctx, p);
            ctx->pool_bytes -= kv.first;
        }
    }
    ctx->pool_free.clear();
}

void evict_cache(aq_ctx* ctx, size_t need) {
    // least recently used first; copies pinned by the running operation stay
    auto it = ctx->cache_lru.end();
    while (it != ctx->cache_lru.begin() && ctx_in_use(ctx) + need > ctx->budget) {
        --it;
        auto ce = ctx->cache.find(*it);
        if (ce == ctx->cache.end() || ce->second.pins > 0) continue;
        dfree(ctx, ce->second.ptr);
        ctx->cache_bytes -= ce->second.bytes;
        ctx->cache.erase(ce);
        it = ctx->cache_lru.erase(it);
    }
}

void invalidate_cache(aq_ctx* ctx) {
    for (auto& kv : ctx->cache) kv.second.valid = false;
}

// AQ_ALLOC_TRACE=1: one line on stderr per allocation that needed the retry path
static bool alloc_trace() {
    static const bool on = [] {
        const char* e = getenv("AQ_ALLOC_TRACE");
        return e && e[0] == '1';
    }();
    return on;
}

static void* raw_alloc(aq_ctx* ctx, size_t bytes) {
    // under graph capture an allocation would become part of the graph;
    // the capturing caller abandons the capture and runs eagerly instead
    AQ_CHECK(!ctx->capture, AQ_ERR_UNSUPPORTED, "device allocation during graph capture");
    if (ctx_in_use(ctx) + bytes > ctx->budget) {
        pool_release_all(ctx);
        evict_cache(ctx, bytes);
        while (ctx_in_use(ctx) + bytes > ctx->budget && !ctx->reclaimable.empty()) ctx->reclaimable.front()->reclaim();
    }
    AQ_CHECK(ctx_in_use(ctx) + bytes <= ctx->budget, AQ_ERR_OOM,
             "HBM budget exceeded: need " + std::to_string(bytes) + " B, in use " +
                 std::to_string(ctx_in_use(ctx)) + " of " + std::to_string(ctx->budget));
    void* p = dmalloc(ctx, bytes);
    if (!p) {
        // The device pool holds freed blocks of other sizes (and other contexts'
        // memory), and servers keep finished jobs' blocks: hand the unused
        // memory back to the driver and retry before giving up any cached
        // operand copy.
        const auto t0 = std::chrono::steady_clock::now();
        pool_release_all(ctx);
        while (!ctx->own.blocks.empty()) pool_free(ctx, ctx->own.pop_oldest().p);
        release_kept_blocks(ctx);
        AQ_HIP(hipStreamSynchronize(ctx->stream));
        trim_device_pool(ctx->device);
        p = dmalloc(ctx, bytes);
        if (!p) {
            evict_cache(ctx, ctx->budget);   // drop every cached copy
            while (!ctx->reclaimable.empty()) ctx->reclaimable.front()->reclaim();
            while (!ctx->own.blocks.empty()) pool_free(ctx, ctx->own.pop_oldest().p);
            release_kept_blocks(ctx);
            AQ_HIP(hipStreamSynchronize(ctx->stream));
            trim_device_pool(ctx->device);
            p = dmalloc(ctx, bytes);
        }
        if (alloc_trace())
            fprintf(stderr, "aq_alloc retry: %zu B, %s, %.1f ms\n", bytes, p ? "served" : "failed",
                    std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count());
        if (!p) throw Error(AQ_ERR_OOM, "device allocation of " + std::to_string(bytes) + " B failed");
    }
    return p;
}

static size_t round_up(size_t b) {
    const size_t g = b >= (1u << 20) ? (size_t(1) << 20) : 256;
    return (b + g - 1) / g * g;
}

void* dev_alloc(aq_ctx* ctx, size_t bytes) {
    bytes = round_up(bytes);
    auto it = ctx->pool_free.find(bytes);
    if (it != ctx->pool_free.end() && !it->second.empty()) {
        void* p = it->second.back();
        it->second.pop_back();
        return p;
    }
    void* p = raw_alloc(ctx, bytes);
    ctx->pool_bytes += bytes;
    note_peak(ctx);
    return p;
}

void dev_free(aq_ctx* ctx, void* p, size_t bytes) {
    // stream-ordered reuse: later work on the same stream may reuse p
    ctx->pool_free[round_up(bytes)].push_back(p);
}

size_t alloc_bytes(size_t bytes) { return std::max<size_t>(round_up(bytes), 256); }

double* tensor_alloc(aq_ctx* ctx, size_t bytes) {
    bytes = alloc_bytes(bytes);
    void* p = raw_alloc(ctx, bytes);
    ctx->tensor_bytes += bytes;
    note_peak(ctx);
    return static_cast<double*>(p);
}

void tensor_free(aq_ctx* ctx, double* p, size_t bytes) {
    bytes = alloc_bytes(bytes);
    dfree(ctx, p);
    ctx->tensor_bytes -= bytes;
}

void note_cache_alloc(aq_ctx* ctx) { note_peak(ctx); }

// cached operand copies and pooled scratch back to the device pool
void drop_caches(aq_ctx* ctx) {
    pool_release_all(ctx);
    for (auto& kv : ctx->cache) dfree(ctx, kv.second.ptr);
    ctx->cache.clear();
    ctx->cache_lru.clear();
    ctx->cache_bytes = 0;
}

// ---------------------------------------------------------------- timing

TimedLaunch::TimedLaunch(aq_ctx* c, const char* name, double flops, double bytes) : ctx(c), on(c->timing) {
    if (!on) return;
    rec.name = name;
    rec.flops = flops;
    rec.bytes = bytes;
    auto take = [&]() {
        if (!ctx->event_pool.empty()) {
            hipEvent_t e = ctx->event_pool.back();
            ctx->event_pool.pop_back();
            return e;
        }
        hipEvent_t e;
        AQ_HIP(hipEventCreate(&e));
        return e;
    };
    rec.start = take();
    rec.stop = take();
    AQ_HIP(hipEventRecord(rec.start, ctx->stream));
}

TimedLaunch::~TimedLaunch() {
    if (!on) return;
    if (hipEventRecord(rec.stop, ctx->stream) == hipSuccess) ctx->pending.push_back(rec);
}

void resolve_timing(aq_ctx* ctx) {
    for (auto& p : ctx->pending) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, p.start, p.stop) == hipSuccess) {
            auto& c = ctx->timing_classes[p.name];
            c.launches += 1;
            c.total_ms += ms;
            c.flops += p.flops;
            c.bytes += p.bytes;
        }
        ctx->event_pool.push_back(p.start);
        ctx->event_pool.push_back(p.stop);
    }
    ctx->pending.clear();
}

}  // namespace aqamd

uint64_t new_tensor_id() {
    static std::atomic<uint64_t> next{1};
    return next.fetch_add(1, std::memory_order_relaxed);
}

using namespace aqamd;

extern "C" {

const char* aq_last_error(void) { return g_last_error.c_str(); }

int aq_version(void) { return 100; }

int aq_ctx_create(int device, size_t hbm_budget, aq_ctx** out) {
    return guarded([&] {
        AQ_CHECK(out, AQ_ERR_INVALID, "null output pointer");
        int ndev = 0;
        AQ_HIP(hipGetDeviceCount(&ndev));
        AQ_CHECK(device >= 0 && device < ndev, AQ_ERR_INVALID, "no such HIP device");
        AQ_HIP(hipSetDevice(device));
        noalloc_scratch_init(device);
        {
            // keep memory released by hipFreeAsync in the device pool instead of
            // returning it to the driver at every synchronisation
            hipMemPool_t pool;
            if (hipDeviceGetDefaultMemPool(&pool, device) == hipSuccess) {
                uint64_t thr = UINT64_MAX;
                (void)hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &thr);
            }
            (void)hipGetLastError();
        }
        auto* ctx = new aq_ctx();
        ctx->device = device;
        try {
            AQ_HIP(hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking));
            size_t free_b = 0, total_b = 0;
            AQ_HIP(hipMemGetInfo(&free_b, &total_b));
            free_b += kept_bytes(device);   // given up on request
            ctx->budget = hbm_budget ? hbm_budget : static_cast<size_t>(0.9 * double(free_b));
            ctx->d_partials = static_cast<double*>(dmalloc(ctx, sizeof(double) * kRedSlots * kRedPartials));
            AQ_CHECK(ctx->d_partials, AQ_ERR_OOM, "device allocation of reduction slots failed");
            AQ_HIP(hipHostMalloc(&ctx->h_result, sizeof(double) * kRedSlots, hipHostMallocDefault));
            AQ_HIP(hipHostGetDevicePointer(reinterpret_cast<void**>(&ctx->d_result), ctx->h_result, 0));
        } catch (...) {
            if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
            delete ctx;
            throw;
        }
        *out = ctx;
    });
}

int aq_ctx_destroy(aq_ctx* ctx) {
    return guarded([&] {
        if (!ctx) return;
        (void)hipSetDevice(ctx->device);
        (void)hipStreamSynchronize(ctx->stream);
        resolve_timing(ctx);
        pool_release_all(ctx);
        for (auto& kv : ctx->cache) dfree(ctx, kv.second.ptr);
        for (auto e : ctx->event_pool) (void)hipEventDestroy(e);
        if (ctx->group_ready) (void)hipEventDestroy(ctx->group_ready);
        dfree(ctx, ctx->d_partials);
        (void)hipStreamSynchronize(ctx->stream);
        (void)hipHostFree(ctx->h_result);
        (void)hipStreamDestroy(ctx->stream);
        delete ctx;
    });
}

int aq_ctx_sync(aq_ctx* ctx) {
    return guarded([&] {
        AQ_CHECK(ctx, AQ_ERR_INVALID, "null context");
        AQ_HIP(hipStreamSynchronize(ctx->stream));
        resolve_timing(ctx);
    });
}

int aq_ctx_set_precision(aq_ctx* ctx, int precision, double min_reduced_flops) {
    return guarded([&] {
        AQ_CHECK(ctx, AQ_ERR_INVALID, "null context");
        AQ_CHECK(precision == AQ_PREC_FP64 || precision == AQ_PREC_FP32 || precision == AQ_PREC_BF16X3,
                 AQ_ERR_INVALID, "unknown precision");
        ctx->precision = precision;
        ctx->min_reduced_flops = min_reduced_flops;
    });
}

int aq_ctx_set_autotune(aq_ctx* ctx, int enable) {
    return guarded([&] {
        AQ_CHECK(ctx, AQ_ERR_INVALID, "null context");
        ctx->autotune = enable != 0;
    });
}

int aq_autotune_table(aq_tune_entry* out, int cap, int* n) {
    return guarded([&] {
        AQ_CHECK(n && cap >= 0, AQ_ERR_INVALID, "null count");
        *n = autotune_entries(out, cap);
    });
}

int aq_ctx_set_gemm_variant(aq_ctx* ctx, int precision, int variant) {
    return guarded([&] {
        AQ_CHECK(ctx, AQ_ERR_INVALID, "null context");
        AQ_CHECK(precision >= 0 && precision <= 2, AQ_ERR_INVALID, "unknown precision");
        AQ_CHECK(variant >= -1 && variant <= (precision == AQ_PREC_BF16X3 ? 4 : 2), AQ_ERR_INVALID,
                 "unknown GEMM variant");
        // AQ_PREC_* and the internal format ids coincide: FP64 = 0, FP32 = 1, BF16x3 = 2
        ctx->gemm_variant[precision] = variant;
    });
}

int aq_ctx_get_precision(const aq_ctx* ctx, int* precision) {
    return guarded([&] {
        AQ_CHECK(ctx && precision, AQ_ERR_INVALID, "null argument");
        *precision = ctx->precision;
    });
}

int aq_ctx_memory(const aq_ctx* ctx, size_t* in_use, size_t* budget) {
    return guarded([&] {
        AQ_CHECK(ctx, AQ_ERR_INVALID, "null context");
        if (in_use) *in_use = ctx_in_use(ctx);
        if (budget) *budget = ctx->budget;
    });
}

int aq_ctx_peak_memory(aq_ctx* ctx, size_t* peak, int reset) {
    return guarded([&] {
        AQ_CHECK(ctx && peak, AQ_ERR_INVALID, "null argument");
        *peak = ctx->peak_bytes;
        if (reset) ctx->peak_bytes = ctx_in_use(ctx);
    });
}

int aq_ctx_trim(aq_ctx* ctx) {
    return guarded([&] {
        AQ_CHECK(ctx, AQ_ERR_INVALID, "null context");
        AQ_HIP(hipStreamSynchronize(ctx->stream));
        drop_caches(ctx);
        release_kept_blocks(ctx);
        AQ_HIP(hipStreamSynchronize(ctx->stream));
        trim_device_pool(ctx->device);
    });
}

int aq_ctx_enable_timing(aq_ctx* ctx, int enable) {
    return guarded([&] {
        AQ_CHECK(ctx, AQ_ERR_INVALID, "null context");
        ctx->timing = enable != 0;
    });
}

int aq_ctx_timing(aq_ctx* ctx, aq_timing_record* rec, int cap, int* n) {
    return guarded([&] {
        AQ_CHECK(ctx && n, AQ_ERR_INVALID, "null argument");
        AQ_HIP(hipStreamSynchronize(ctx->stream));
        resolve_timing(ctx);
        int i = 0;
        for (auto& kv : ctx->timing_classes) {
            if (rec && i < cap) {
                std::memset(rec[i].name, 0, sizeof(rec[i].name));
                std::strncpy(rec[i].name, kv.first.c_str(), sizeof(rec[i].name) - 1);
                rec[i].launches = kv.second.launches;
                rec[i].total_ms = kv.second.total_ms;
                rec[i].flops = kv.second.flops;
                rec[i].bytes = kv.second.bytes;
            }
            ++i;
        }
        *n = i;
    });
}

int aq_ctx_timing_reset(aq_ctx* ctx) {
    return guarded([&] {
        AQ_CHECK(ctx, AQ_ERR_INVALID, "null context");
        AQ_HIP(hipStreamSynchronize(ctx->stream));
        resolve_timing(ctx);
        ctx->timing_classes.clear();
    });
}

}  // extern "C"
