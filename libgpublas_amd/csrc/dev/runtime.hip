// runtime.hip -- device bring-up, per-thread streams, the caching device
// pool, host<->device copies, deterministic input generation and kernel
// timing for the gfx950 device layer.
//
// Replaces the reference's device runtime shim (runtime.h:78-125,
// runtime.c:195-260): backend-neutral alloc / memcpy there, one HIP device,
// one stream per host thread and a size-class cache of device blocks here.
#include "devcommon.hpp"
#include "gpublas_dev.h"

#include <atomic>
#include <mutex>
#include <unordered_map>
#include <vector>
#include <string.h>
#include <stdio.h>
#include <stdlib.h>

namespace {

std::once_flag g_init_once;
int g_init_status = -1;
hipDeviceProp_t g_prop;

// ---- caching pool --------------------------------------------------------
// Device blocks are rounded to a size class (powers of two up to 2 MiB,
// multiples of 2 MiB above) and kept on per-class free lists after release,
// so steady-state BLAS calls on untracked operands do not hit hipMalloc /
// hipFree (hipFree synchronises the whole device).
std::mutex g_pool_mu;
std::unordered_map<size_t, std::vector<void *>> *g_free;
std::unordered_map<void *, size_t> *g_live;
size_t g_pool_bytes = 0;
// blocks released behind a stream event: reusable once the event completes
struct Deferred {
    void *p;
    size_t c;
    hipEvent_t ev;
};
std::vector<Deferred> *g_deferred;

size_t size_class(size_t b)
{
    if (b <= 256) return 256;
    const size_t two_mib = 2u << 20;
    if (b <= two_mib) {
        size_t c = 256;
        while (c < b) c <<= 1;
        return c;
    }
    return (b + two_mib - 1) / two_mib * two_mib;
}

// Blocks whose graph is gone.  The runtime calls block_of_graph_done() from inside
// its own destroy functions, so it takes no lock under which the pool calls the
// runtime; the next allocation or trim moves them to the free lists.
std::mutex g_returned_mu;
std::vector<void *> *g_returned;
std::atomic<bool> g_any_returned{false};

void block_of_graph_done(void *p)
{
    std::lock_guard<std::mutex> g(g_returned_mu);
    g_returned->push_back(p);
    g_any_returned.store(true, std::memory_order_release);
}

void take_returned_locked()  // the pool's lock is held
{
    if (!g_any_returned.load(std::memory_order_acquire)) return;
    std::vector<void *> v;
    {
        std::lock_guard<std::mutex> g(g_returned_mu);
        v.swap(*g_returned);
        g_any_returned.store(false, std::memory_order_relaxed);
    }
    for (void *p : v) {
        auto it = g_live->find(p);
        if (it == g_live->end()) continue;
        (*g_free)[it->second].push_back(p);
        g_live->erase(it);
    }
}

// The calling thread's stream capture mode set to relaxed while in scope: an
// allocation belongs to no stream and must not end a capture that is under way.
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// The stream of the calling thread's current (or last) call, and whether it records a
// graph: 1, 0, or -1 while no part of the call has asked (52 ns).
thread_local hipStream_t t_call_stream = nullptr;
thread_local signed char t_call_recorded = 0;

// Move deferred blocks whose event has completed to the free lists
// (all of them when `wait`).
void pool_reap_locked(bool wait)
{
    auto &d = *g_deferred;
    size_t keep = 0;
    for (size_t i = 0; i < d.size(); ++i) {
        if (wait) (void)hipEventSynchronize(d[i].ev);
        if (hipEventQuery(d[i].ev) == hipSuccess) {
            (void)hipEventDestroy(d[i].ev);
            (*g_free)[d[i].c].push_back(d[i].p);
        } else {
            d[keep++] = d[i];
        }
    }
    d.resize(keep);
    (void)hipGetLastError();  // a not-ready query is not an error
}

void pool_trim_locked()
{
    pool_reap_locked(true);
    take_returned_locked();
    for (auto &kv : *g_free) {
        for (void *p : kv.second) {
            (void)hipFree(p);
            g_pool_bytes -= kv.first;
        }
        kv.second.clear();
    }
}

// ---- timing ----------------------------------------------------------------
struct Pending {
    hipEvent_t a, b;
    int name;
};
std::mutex g_prof_mu;
std::vector<Pending> *g_pending;
std::vector<hipEvent_t> *g_event_cache;
const int kMaxNames = 128;
const char *g_names[kMaxNames];
int g_nnames = 0;
struct Stat {
    long count;
    double total, mn, mx;
};
Stat g_stats[kMaxNames];
thread_local hipEvent_t t_begin_ev = nullptr;
thread_local int t_begin_name = -1;

hipEvent_t ev_get()
{
    hipEvent_t e = nullptr;
    if (!g_event_cache->empty()) {
        e = g_event_cache->back();
        g_event_cache->pop_back();
        return e;
    }
    (void)hipEventCreate(&e);
    return e;
}

int name_id(const char *n)
{
    for (int i = 0; i < g_nnames; ++i)
        if (g_names[i] == n || strcmp(g_names[i], n) == 0) return i;
    if (g_nnames == kMaxNames) return kMaxNames - 1;
    g_names[g_nnames] = n;
    g_stats[g_nnames] = Stat{0, 0, 1e300, 0};
    return g_nnames++;
}

void prof_resolve_locked()
{
    for (auto &p : *g_pending) {
        (void)hipEventSynchronize(p.b);
        float ms = 0;
        (void)hipEventElapsedTime(&ms, p.a, p.b);
        Stat &s = g_stats[p.name];
        s.count++;
        s.total += ms;
        if (ms < s.mn) s.mn = ms;
        if (ms > s.mx) s.mx = ms;
        g_event_cache->push_back(p.a);
        g_event_cache->push_back(p.b);
    }
    g_pending->clear();
}

// ---- deterministic inputs ------------------------------------------------
__device__ __forceinline__ uint64_t splitmix_at(uint64_t seed, uint64_t i)
{
    uint64_t z = seed + (i + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__global__ void fill_uniform_kernel(uint64_t seed, int64_t n, double *out)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        uint64_t z = splitmix_at(seed, (uint64_t)i);
        double u = (double)(z >> 11) * 0x1.0p-53;
        out[i] = 2.0 * u - 1.0;
    }
}

__global__ void fill_uniform_f32_kernel(uint64_t seed, int64_t n, float *out)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        uint64_t z = splitmix_at(seed, (uint64_t)i);
        double u = (double)(z >> 11) * 0x1.0p-53;
        out[i] = (float)(2.0 * u - 1.0);
    }
}

void do_init()
{
    if (__atomic_load_n(&g_init_status, __ATOMIC_ACQUIRE) == -5) return;  // a fork child
    g_free = new std::unordered_map<size_t, std::vector<void *>>();
    g_live = new std::unordered_map<void *, size_t>();
    g_deferred = new std::vector<Deferred>();
    g_returned = new std::vector<void *>();
    g_pending = new std::vector<Pending>();
    g_event_cache = new std::vector<hipEvent_t>();
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n < 1) {
        g_init_status = -1;
        return;
    }
    if (hipSetDevice(0) != hipSuccess || hipGetDeviceProperties(&g_prop, 0) != hipSuccess) {
        g_init_status = -2;
        return;
    }
    if (strncmp(g_prop.gcnArchName, "gfx950", 6) != 0) {
        g_init_status = -3;  // code objects are built for gfx950 only
        return;
    }
    // the allocation-free DGEMV's fixed scratch array: its address on device 0
    // (current since hipSetDevice above); if it cannot be taken here, that
    // entry point's first call tries again and reports the error
    (void)noalloc_scratch_setup(0);
    g_init_status = 0;
}

}  // namespace

int g_prof_on = 0;

// ---- per-thread context ------------------------------------------------------
namespace {
std::mutex g_ctx_mu;
std::vector<DevCtx *> *g_ctx_all;   // every context ever made (stream registry)
std::vector<DevCtx *> *g_ctx_free;  // contexts of exited threads

DevCtx *ctx_create()
{
    DevCtx *c = new DevCtx();
    (void)hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    (void)hipMalloc(&c->tickets, kTicketSlots * sizeof(unsigned));
    (void)hipMemsetAsync(c->tickets, 0, kTicketSlots * sizeof(unsigned), c->stream);
    (void)hipHostMalloc(&c->pinned, 256, hipHostMallocDefault);
    memset(c->pinned, 0, 256);
    (void)hipStreamSynchronize(c->stream);
    return c;
}

struct CtxHolder {
    DevCtx *c = nullptr;
    ~CtxHolder()
    {
        // Thread exit: park the context for the next thread.  No HIP call
        // here (the runtime may already be tearing down this thread's
        // state); work still queued on the stream stays ordered before
        // whatever the next owner enqueues, and tracked objects that name
        // the stream wait on its sequence numbers as before.
        if (c && g_init_status == 0) {
            std::lock_guard<std::mutex> g(g_ctx_mu);
            g_ctx_free->push_back(c);
        }
    }
};
thread_local CtxHolder t_ctx;
DevCtx g_null_ctx{};
}  // namespace

DevCtx *dev_ctx()
{
    if (t_ctx.c) return t_ctx.c;
    if (gpublas_dev_init() != 0) return &g_null_ctx;
    std::lock_guard<std::mutex> g(g_ctx_mu);
    if (!g_ctx_all) {
        g_ctx_all = new std::vector<DevCtx *>();
        g_ctx_free = new std::vector<DevCtx *>();
    }
    if (!g_ctx_free->empty()) {
        t_ctx.c = g_ctx_free->back();
        g_ctx_free->pop_back();
    } else {
        t_ctx.c = ctx_create();
        g_ctx_all->push_back(t_ctx.c);
    }
    return t_ctx.c;
}

DevCtx *ctx_of(hipStream_t stream)
{
    DevCtx *mine = dev_ctx();
    if (!stream || mine->stream == stream) return mine;
    std::lock_guard<std::mutex> g(g_ctx_mu);
    for (DevCtx *c : *g_ctx_all)
        if (c->stream == stream) return c;
    return nullptr;
}

static hipStream_t stream_of(void *s) { return s ? (hipStream_t)s : dev_ctx()->stream; }

hipStream_t pick_stream(void *stream)
{
    t_call_recorded = -1;
    return t_call_stream = stream_of(stream);
}
bool call_is_recorded()
{
    if (t_call_recorded < 0) {
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        if (dev_ready() && hipStreamIsCapturing(t_call_stream, &st) != hipSuccess)
            (void)hipGetLastError();
        t_call_recorded = st == hipStreamCaptureStatusActive;
    }
    return t_call_recorded != 0;
}
void *dev_block(size_t bytes)
{
    (void)call_is_recorded();
    return gpublas_dev_alloc(bytes);
}

Scratch dev_scratch(size_t bytes, hipStream_t s)
{
    Scratch r;
    DevCtx *c = dev_ctx();
    r.s = s ? s : c->stream;
    if (r.s != c->stream || call_is_recorded()) {
        r.p = dev_block(bytes);
        r.pooled = r.p != nullptr;
        return r;
    }
    if (c->ws_bytes < bytes) {
        if (c->ws) {
            // the workspace is only ever used on c->stream: once that stream
            // has drained, no kernel can still be using it
            (void)hipStreamSynchronize(c->stream);
            gpublas_dev_release(c->ws);
        }
        size_t want = bytes < (1u << 20) ? (1u << 20) : bytes;
        c->ws = gpublas_dev_alloc(want);
        c->ws_bytes = c->ws ? want : 0;
    }
    r.p = c->ws;
    return r;
}

void prof_begin(hipStream_t s, const char *name)
{
    std::lock_guard<std::mutex> g(g_prof_mu);
    t_begin_ev = ev_get();
    t_begin_name = name_id(name);
    (void)hipEventRecord(t_begin_ev, s);
}

void prof_end(hipStream_t s)
{
    std::lock_guard<std::mutex> g(g_prof_mu);
    if (!t_begin_ev) return;
    hipEvent_t b = ev_get();
    (void)hipEventRecord(b, s);
    g_pending->push_back(Pending{t_begin_ev, b, t_begin_name});
    t_begin_ev = nullptr;
}

bool dev_ready() { return __atomic_load_n(&g_init_status, __ATOMIC_ACQUIRE) == 0; }

extern "C" {

int gpublas_dev_init(void)
{
    std::call_once(g_init_once, do_init);
    return g_init_status;
}

int gpublas_dev_count(void)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

const char *gpublas_dev_arch(void)
{
    if (gpublas_dev_init() != 0) return "none";
    return g_prop.gcnArchName;
}

size_t gpublas_dev_total_mem(void)
{
    if (gpublas_dev_init() != 0) return 0;
    return g_prop.totalGlobalMem;
}

void *gpublas_dev_stream(void) { return (void *)dev_ctx()->stream; }

int gpublas_dev_sync(void *stream)
{
    hipStream_t s = stream_of(stream);
    DevCtx *c = ctx_of(s);
    const uint64_t sub = c ? __atomic_load_n(&c->submitted, __ATOMIC_ACQUIRE) : 0;
    int err = (int)hipStreamSynchronize(s);
    if (c && !err) {
        uint64_t cur = __atomic_load_n(&c->completed, __ATOMIC_RELAXED);
        while (cur < sub && !__atomic_compare_exchange_n(&c->completed, &cur, sub, false,
                                                         __ATOMIC_RELEASE, __ATOMIC_RELAXED)) {
        }
    }
    return err;
}

uint64_t gpublas_dev_stream_mark(void *stream)
{
    DevCtx *c = ctx_of(stream_of(stream));
    return c ? __atomic_add_fetch(&c->submitted, 1, __ATOMIC_ACQ_REL) : 0;
}

int gpublas_dev_stream_done(void *stream, uint64_t seq)
{
    hipStream_t s = stream_of(stream);
    DevCtx *c = ctx_of(s);
    if (c && __atomic_load_n(&c->completed, __ATOMIC_ACQUIRE) >= seq) return 1;
    if (hipStreamQuery(s) != hipSuccess) return 0;
    if (c) {
        // the stream is idle: everything marked before this query is complete
        uint64_t cur = __atomic_load_n(&c->completed, __ATOMIC_RELAXED);
        while (cur < seq && !__atomic_compare_exchange_n(&c->completed, &cur, seq, false,
                                                         __ATOMIC_RELEASE, __ATOMIC_RELAXED)) {
        }
    }
    return 1;
}

void gpublas_dev_forked_child(void)
{
    __atomic_store_n(&g_init_status, -5, __ATOMIC_RELEASE);  // -5: after fork
    res_forget_after_fork();
}

int gpublas_dev_stream_known_done(void *stream, uint64_t seq)
{
    DevCtx *c = ctx_of(stream_of(stream));
    return c && __atomic_load_n(&c->completed, __ATOMIC_ACQUIRE) >= seq;
}

void gpublas_dev_stream_observed(void *stream, uint64_t seq)
{
    DevCtx *c = ctx_of(stream_of(stream));
    if (!c) return;
    uint64_t cur = __atomic_load_n(&c->completed, __ATOMIC_RELAXED);
    while (cur < seq && !__atomic_compare_exchange_n(&c->completed, &cur, seq, false,
                                                     __ATOMIC_RELEASE, __ATOMIC_RELAXED)) {
    }
}

int gpublas_dev_stream_wait(void *stream, uint64_t seq)
{
    DevCtx *c = ctx_of(stream_of(stream));
    if (!c) return (int)hipStreamSynchronize(stream_of(stream));
    if (__atomic_load_n(&c->completed, __ATOMIC_ACQUIRE) >= seq) return 0;
    return gpublas_dev_sync(c->stream);
}

uint64_t gpublas_dev_scalar_next(void)
{
    DevCtx *c = dev_ctx();
    return ++c->scalar_seq;
}

int gpublas_dev_scalar_wait(void *stream, uint64_t seq)
{
    // The reduction kernels publish [value, seq] into this thread's pinned
    // slot; poll the flag (a system-scope store after a system fence) rather
    // than paying a full stream synchronisation.  Every 4096 polls the stream
    // is queried so an error or a lost publication ends the wait.
    DevCtx *c = dev_ctx();
    volatile uint64_t *flag = (volatile uint64_t *)((char *)c->pinned + 8);
    for (unsigned spin = 1;; ++spin) {
        if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) == seq) return 0;
        if ((spin & 4095) == 0) {
            hipError_t q = hipStreamQuery(stream_of(stream));
            if (q == hipSuccess) {
                // stream drained: the flag must be there now
                if (__atomic_load_n(flag, __ATOMIC_ACQUIRE) == seq) return 0;
                return (int)hipErrorUnknown;
            }
            if (q != hipErrorNotReady) return (int)q;
        }
    }
}

void *gpublas_dev_alloc(size_t bytes)
{
    if (gpublas_dev_init() != 0) return nullptr;
    size_t c = size_class(bytes ? bytes : 1);
    std::lock_guard<std::mutex> g(g_pool_mu);
    // (querying an event of a stream that records would end its capture)
    if (!g_deferred->empty() && t_call_recorded <= 0) pool_reap_locked(false);
    take_returned_locked();
    auto it = g_free->find(c);
    void *p = nullptr;
    if (it != g_free->end() && !it->second.empty()) {
        p = it->second.back();
        it->second.pop_back();
    } else {
        RelaxedCapture relaxed;
        if (hipMalloc(&p, c) != hipSuccess) {
            (void)hipGetLastError();
            (void)hipDeviceSynchronize();
            pool_trim_locked();
            if (hipMalloc(&p, c) != hipSuccess) {
                (void)hipGetLastError();
                return nullptr;
            }
        }
        g_pool_bytes += c;
    }
    (*g_live)[p] = c;
    return p;
}

void gpublas_dev_release(void *d_ptr)
{
    if (!d_ptr) return;
    std::lock_guard<std::mutex> g(g_pool_mu);
    auto it = g_live->find(d_ptr);
    if (it == g_live->end()) return;
    (*g_free)[it->second].push_back(d_ptr);
    g_live->erase(it);
}

// Release a block whose last users are queued on stream s: it returns to
// the free lists once the work queued so far on s has completed, so the
// caller need not wait for it.  While s records a graph the users run at every
// replay: the block then belongs to the graph and the executables made of it (a
// user object), and returns when the last of them is destroyed.
extern "C++" void dev_release_after(void *d_ptr, hipStream_t s)
{
    if (!d_ptr) return;
    if (call_is_recorded()) {
        hipStreamCaptureStatus st;
        hipGraph_t graph = nullptr;
        hipUserObject_t obj = nullptr;
        if (hipStreamGetCaptureInfo_v2(s, &st, nullptr, &graph, nullptr, nullptr) != hipSuccess ||
            !graph || hipUserObjectCreate(&obj, d_ptr, block_of_graph_done, 1,
                                          hipUserObjectNoDestructorSync) != hipSuccess ||
            hipGraphRetainUserObject(graph, obj, 1, hipGraphUserObjectMove) != hipSuccess)
            (void)hipGetLastError();  // not tied to the graph: kept until the process ends
        return;
    }
    std::lock_guard<std::mutex> g(g_pool_mu);
    auto it = g_live->find(d_ptr);
    if (it == g_live->end()) return;
    hipEvent_t ev = nullptr;
    bool ok = hipEventCreateWithFlags(&ev, hipEventDisableTiming) == hipSuccess;
    ok = ok && hipEventRecord(ev, s) == hipSuccess;
    if (ok) {
        g_deferred->push_back(Deferred{d_ptr, it->second, ev});
    } else {
        // cannot order the release behind the stream: wait for it instead
        (void)hipGetLastError();
        if (ev) (void)hipEventDestroy(ev);
        (void)hipStreamSynchronize(s);
        (*g_free)[it->second].push_back(d_ptr);
    }
    g_live->erase(it);
}

int gpublas_dev_trim(void)
{
    std::lock_guard<std::mutex> g(g_pool_mu);
    (void)hipDeviceSynchronize();
    pool_trim_locked();
    return 0;
}

size_t gpublas_dev_pool_bytes(void)
{
    std::lock_guard<std::mutex> g(g_pool_mu);
    return g_pool_bytes;
}

int gpublas_dev_h2d(void *d_dst, const void *h_src, size_t bytes, void *stream)
{
    if (!bytes) return 0;
    return (int)hipMemcpyAsync(d_dst, h_src, bytes, hipMemcpyHostToDevice, stream_of(stream));
}

int gpublas_dev_d2h(void *h_dst, const void *d_src, size_t bytes, void *stream)
{
    if (!bytes) return 0;
    return (int)hipMemcpyAsync(h_dst, d_src, bytes, hipMemcpyDeviceToHost, stream_of(stream));
}

int gpublas_dev_d2d(void *d_dst, const void *d_src, size_t bytes, void *stream)
{
    if (!bytes) return 0;
    return (int)hipMemcpyAsync(d_dst, d_src, bytes, hipMemcpyDeviceToDevice, stream_of(stream));
}

int gpublas_dev_h2d_2d(void *d_dst, size_t ldd, const void *h_src, size_t lds, size_t m, size_t n,
                       size_t es, void *stream)
{
    if (!m || !n) return 0;
    return (int)hipMemcpy2DAsync(d_dst, ldd * es, h_src, lds * es, m * es, n,
                                 hipMemcpyHostToDevice, stream_of(stream));
}

int gpublas_dev_d2h_2d(void *h_dst, size_t ldd, const void *d_src, size_t lds, size_t m, size_t n,
                       size_t es, void *stream)
{
    if (!m || !n) return 0;
    return (int)hipMemcpy2DAsync(h_dst, ldd * es, d_src, lds * es, m * es, n,
                                 hipMemcpyDeviceToHost, stream_of(stream));
}

void *gpublas_dev_host_alloc(size_t bytes)
{
    if (gpublas_dev_init() != 0) return nullptr;
    void *p = nullptr;
    if (hipHostMalloc(&p, bytes, hipHostMallocDefault) != hipSuccess) return nullptr;
    return p;
}

void gpublas_dev_host_free(void *p)
{
    if (p) (void)hipHostFree(p);
}

int gpublas_dev_fill_uniform(void *stream, uint64_t seed, int64_t n, double *d_out)
{
    if (n <= 0) return 0;
    hipStream_t s = pick_stream(stream);
    int blocks = (int)((n + 255) / 256);
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(fill_uniform_kernel, dim3(blocks), dim3(256), 0, s, seed, n, d_out);
    return (int)hipGetLastError();
}

int gpublas_dev_fill_uniform_f32(void *stream, uint64_t seed, int64_t n, float *d_out)
{
    if (n <= 0) return 0;
    hipStream_t s = pick_stream(stream);
    int blocks = (int)((n + 255) / 256);
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(fill_uniform_f32_kernel, dim3(blocks), dim3(256), 0, s, seed, n, d_out);
    return (int)hipGetLastError();
}

void *gpublas_dev_result_slot(void) { return dev_ctx()->pinned; }

void gpublas_dev_prof_enable(int on)
{
    // no device work here: the library's constructor calls this before every
    // object's kernels are registered with the HIP runtime
    g_prof_on = on;
}

void gpublas_dev_prof_reset(void)
{
    std::lock_guard<std::mutex> g(g_prof_mu);
    if (g_pending) prof_resolve_locked();
    for (int i = 0; i < g_nnames; ++i) g_stats[i] = Stat{0, 0, 1e300, 0};
}

int gpublas_dev_prof_query(const char *kernel, double *total_ms, double *min_ms, double *max_ms)
{
    std::lock_guard<std::mutex> g(g_prof_mu);
    if (!g_pending) return 0;
    prof_resolve_locked();
    for (int i = 0; i < g_nnames; ++i)
        if (strcmp(g_names[i], kernel) == 0) {
            if (total_ms) *total_ms = g_stats[i].total;
            if (min_ms) *min_ms = g_stats[i].count ? g_stats[i].mn : 0;
            if (max_ms) *max_ms = g_stats[i].mx;
            return (int)g_stats[i].count;
        }
    if (total_ms) *total_ms = 0;
    return 0;
}

int gpublas_dev_prof_dump(char *buf, size_t len)
{
    std::lock_guard<std::mutex> g(g_prof_mu);
    if (!g_pending) return 0;
    prof_resolve_locked();
    size_t off = 0;
    for (int i = 0; i < g_nnames && off < len; ++i) {
        int w = snprintf(buf + off, len - off, "%s %ld %.6f\n", g_names[i], g_stats[i].count,
                         g_stats[i].total);
        if (w < 0) break;
        off += (size_t)w;
    }
    return (int)off;
}

}  // extern "C"
