// C ABI of libpwmhip.so (declared in include/pwm_hip.h): handle lifetime,
// matrix loading, planning, and the SpMV / power-method entry points.
#include <math.h>
#include <string.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <memory>
#include <mutex>
#include <thread>
#include <numeric>
#include <vector>

#include "api_internal.hpp"
#include "engine.hpp"

using namespace pwm_impl;
using pwmk::CrsDev;
using pwmk::PowerArgs;

namespace pwm_impl {

static thread_local std::string g_err;
void set_global_error(const std::string& msg) { g_err = msg; }

hipError_t DevBuf::alloc(size_t n) {
    release();
    if (n == 0) return hipSuccess;
    hipError_t e = hipMalloc(&p, n);
    if (e != hipSuccess) {
        p = nullptr;
        return e;
    }
    bytes = n;
    return hipSuccess;
}
hipError_t alloc_padded(DevBuf& b, int64_t n, size_t elem) {
    hipError_t e = b.alloc((size_t)(n + kPadEntries) * elem);
    if (e == hipSuccess) e = hipMemset((char*)b.p + (size_t)n * elem, 0, (size_t)kPadEntries * elem);
    if (e == hipSuccess) e = hipStreamSynchronize(nullptr);  // before any handle stream reads it
    return e;
}
void DevBuf::release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
}

// ---- host thread pool behind parallel_for
namespace {
constexpr int kMaxWorkers = 16;  // the GPU host grants 16 cores per GPU

void run_chunks(std::atomic<int64_t>& next, int64_t n, int64_t chunk, const LoopFn& fn, int worker) {
    for (;;) {
        const int64_t b = next.fetch_add(chunk);
        if (b >= n) break;
        fn(b, std::min(n, b + chunk), worker);
    }
}

// one job at a time: workers 1..nworkers join the caller (worker 0)
struct HostPool {
    std::mutex run_mu;  // held by the caller whose job the pool runs
    std::mutex mu;
    std::condition_variable cv_work, cv_done;
    const LoopFn* fn = nullptr;
    int64_t n = 0, chunk = 0;
    std::atomic<int64_t> next{0};
    int nworkers = 0, active = 0, pending = 0;
    uint64_t epoch = 0;
    pid_t pid = 0;  // the process whose threads these are (a forked child has none of them)
};
HostPool* g_pool = nullptr;  // created once, never destroyed (its threads are detached)
std::once_flag g_pool_once;

void pool_worker(HostPool* p, int id) {
    uint64_t seen = 0;
    for (;;) {
        const LoopFn* fn;
        int64_t n, chunk;
        {
            std::unique_lock<std::mutex> lk(p->mu);
            p->cv_work.wait(lk, [&] { return p->epoch != seen; });
            seen = p->epoch;
            if (id > p->active) continue;  // not needed for this job
            fn = p->fn;
            n = p->n;
            chunk = p->chunk;
        }
        run_chunks(p->next, n, chunk, *fn, id);
        std::lock_guard<std::mutex> lk(p->mu);
        if (--p->pending == 0) p->cv_done.notify_all();
    }
}

void spawn_run(int64_t n, int64_t chunk, const LoopFn& fn, int nt, const LeadFn* lead) {
    std::atomic<int64_t> next(0);
    std::vector<std::thread> ts;
    for (int t = 1; t < nt; ++t) ts.emplace_back([&, t]() { run_chunks(next, n, chunk, fn, t); });
    if (lead) (*lead)(next);
    run_chunks(next, n, chunk, fn, 0);
    for (auto& th : ts) th.join();
}
}  // namespace

void parallel_run(int64_t n, int64_t chunk, const LoopFn& fn, const LeadFn* lead) {
    const unsigned hw = std::thread::hardware_concurrency();
    const int64_t pieces = (n + chunk - 1) / chunk;
    const int nt = (int)std::min<int64_t>(std::min<int64_t>(hw ? hw : 4, kMaxWorkers), pieces);
    if (nt <= 1) {
        std::atomic<int64_t> next(0);
        if (lead) (*lead)(next);
        run_chunks(next, n, lead ? chunk : n, fn, 0);
        return;
    }
    std::call_once(g_pool_once, [&] {
        HostPool* p = new HostPool();
        p->pid = getpid();
        const int want = (int)std::min<unsigned>(hw ? hw : 4, kMaxWorkers) - 1;
        for (int i = 1; i <= want; ++i) {
            try {
                std::thread(pool_worker, p, i).detach();
                p->nworkers = i;
            } catch (...) {
                break;
            }
        }
        g_pool = p;
    });
    HostPool* p = g_pool;
    std::unique_lock<std::mutex> run(p->run_mu, std::try_to_lock);
    if (!run.owns_lock() || p->nworkers == 0 || p->pid != getpid()) {
        spawn_run(n, chunk, fn, nt, lead);
        return;
    }
    {
        std::lock_guard<std::mutex> lk(p->mu);
        p->fn = &fn;
        p->n = n;
        p->chunk = chunk;
        p->next = 0;
        p->active = std::min(p->nworkers, nt - 1);
        p->pending = p->active;
        ++p->epoch;
    }
    p->cv_work.notify_all();
    if (lead) (*lead)(p->next);
    run_chunks(p->next, n, chunk, fn, 0);
    std::unique_lock<std::mutex> lk(p->mu);
    p->cv_done.wait(lk, [&] { return p->pending == 0; });
}

// Pinned staging for transfers: two process-wide buffers of kStageBytes, held
// until the process ends; one transfer at a time uses them.
namespace {
constexpr size_t kStageBytes = (size_t)64 << 20;
std::mutex g_stage_mu;
void* g_stage[2] = {nullptr, nullptr};
hipEvent_t g_stage_ev[2] = {nullptr, nullptr};
constexpr size_t kRingChunks = 16;  // most chunks per buffer
hipEvent_t g_ring_ev[2 * kRingChunks] = {};
bool g_stage_failed = false;

// Vectors of at most kInlineBytes go through a piece of their own, one per call
// under way: they wait for nobody's transfer.  At most kShortSlots pieces, each
// allocated when first needed and kept for the process.
constexpr size_t kInlineBytes = (size_t)1 << 20;
constexpr int kShortSlots = 16;
std::mutex g_short_mu;
char* g_short_free[kShortSlots];
int g_short_n = 0, g_short_made = 0;  // free ones, all

struct ShortSlot {
    char* p = nullptr;  // nullptr: none to be had
    ShortSlot() {
        std::lock_guard<std::mutex> lk(g_short_mu);
        if (g_short_n > 0) {
            p = g_short_free[--g_short_n];
        } else if (g_short_made < kShortSlots) {
            void* q = nullptr;
            if (hipHostMalloc(&q, kInlineBytes, hipHostMallocCoherent | hipHostMallocPortable) == hipSuccess) {
                p = (char*)q;
                ++g_short_made;
            } else {
                (void)hipGetLastError();
            }
        }
    }
    ~ShortSlot() {
        if (!p) return;
        std::lock_guard<std::mutex> lk(g_short_mu);
        g_short_free[g_short_n++] = p;
    }
    ShortSlot(const ShortSlot&) = delete;
    ShortSlot& operator=(const ShortSlot&) = delete;
};
}  // namespace

// Chunk of one staged transfer: about an eighth of it (whole MB, at least
// 2 MB, at most a buffer), so that the host copy into one buffer overlaps the
// DMA of the other from the second chunk on; host threads copy pieces of at
// least 256 KB.
static size_t stage_chunk(size_t bytes) {
    constexpr size_t MB = (size_t)1 << 20;
    const size_t c = (bytes / 8 + MB - 1) & ~(MB - 1);
    return std::min(kStageBytes, std::max(c, 2 * MB));
}
static int64_t stage_piece(size_t chunk) { return std::max<int64_t>((int64_t)(chunk / 16), (int64_t)256 << 10); }

// Allocates the staging pair once (the caller holds g_stage_mu); false when
// pinned memory cannot be had.
static bool stage_ready() {
    if (!g_stage[0] && !g_stage_failed) {
        for (int i = 0; i < 2 && !g_stage_failed; ++i)
            if (hipHostMalloc(&g_stage[i], kStageBytes, hipHostMallocCoherent | hipHostMallocPortable) != hipSuccess ||
                hipEventCreateWithFlags(&g_stage_ev[i], hipEventDisableTiming) != hipSuccess)
                g_stage_failed = true;
        for (hipEvent_t& v : g_ring_ev)
            if (!g_stage_failed && hipEventCreateWithFlags(&v, hipEventDisableTiming | hipEventReleaseToSystem) != hipSuccess)
                g_stage_failed = true;
        if (g_stage_failed) {
            for (int i = 0; i < 2; ++i) {
                if (g_stage[i]) (void)hipHostFree(g_stage[i]);
                if (g_stage_ev[i]) (void)hipEventDestroy(g_stage_ev[i]);
                g_stage[i] = nullptr;
                g_stage_ev[i] = nullptr;
            }
            for (hipEvent_t& v : g_ring_ev) {
                if (v) (void)hipEventDestroy(v);
                v = nullptr;
            }
            (void)hipGetLastError();
        }
    }
    return !g_stage_failed;
}

// FP64 value k as stored: FP32, or BF16 as the upper half of the FP32 value
// (exact for values exact in BF16, which the callers check).
static inline void narrow_value(const double* v, int vt, int64_t k, char* out) {
    const float f = (float)v[k];
    if (vt == PWM_VALUES_F32) {
        memcpy(out, &f, 4);
    } else {
        uint32_t u;
        memcpy(&u, &f, 4);
        const uint16_t h = (uint16_t)(u >> 16);
        memcpy(out, &h, 2);
    }
}

// What the threads do to a piece, bytes [a0, a1) of the transfer (whole values:
// pieces are multiples of 64 KB): host arrays into the staging buffers, as they
// are or in the stored type, and vectors out of them.
static auto bytes_in(const void* src) {
    return [src](char* to, size_t a0, size_t a1) { memcpy(to, (const char*)src + a0, a1 - a0); };
}
static auto values_in(const double* src, int vt) {
    return [src, vt](char* to, size_t a0, size_t a1) {
        if (vt == PWM_VALUES_F32)
            for (size_t k = a0 / 4; k < a1 / 4; ++k) ((float*)to)[k - a0 / 4] = (float)src[k];
        else
            for (size_t k = a0 / 2; k < a1 / 2; ++k) narrow_value(src, vt, (int64_t)k, to + 2 * k - a0);
    };
}
static auto bytes_out(double* dst) {
    return [dst](const char* from, size_t a0, size_t a1) { memcpy((char*)dst + a0, from, a1 - a0); };
}
static auto floats_out(double* dst) {
    return [dst](const char* from, size_t a0, size_t a1) {
        const float* f = (const float*)from;
        for (size_t i = 0; i < (a1 - a0) / 4; ++i) dst[a0 / 4 + i] = f[i];
    };
}

// ---- transfers in one parallel loop
// A transfer goes in windows of one staging buffer (64 MB), in turn through the
// two: while the threads fill or empty one, the copies of the other run.  A
// window holds chunks; host threads take pieces of the whole window in order,
// and the calling thread queues a chunk's copy as soon as its pieces are in
// (uploads) or hands a chunk to the threads as soon as it has arrived
// (downloads): the threads are woken once per window, not once per chunk.  Up to
// one buffer, chunks of 1 to 4 MB copied by kernels that read or write the
// pinned memory: eight of 1 MB take 183 us up and 185 down, where the copy
// engine takes 225 and 260 (about 10 us more per copy), and 154 for the 8 MB at
// once.  Beyond, where the host's copies set the pace, chunks of 16 MB by the
// copy engine in pieces of 1 MB (2 x 200 MB: 8.16 ms, with chunks of 4 MB 8.27).
// mv(x, y) on host arrays of a Poisson grid, FP64: 300 x 300 165 -> 75 us, 1000 x
// 999 575 -> 450, 5000 x 5000 as before; FP32, which used to convert in separate
// loops, 1000 x 999 590 -> 280 and 4000 x 3000 9300 -> 2170.
namespace {
// Transfers of at most kInlineBytes are copied by the calling thread: waking the
// others costs more (mv of 0.7 MB vectors takes 75 us, through the threads 97; of
// 1.4 MB 143 through the threads, without them 155).
struct Window {
    size_t bytes, chunk, piece, nch;
    int64_t pieces;
    std::unique_ptr<std::atomic<int>[]> left;  // pieces of a chunk not yet copied
    Window(size_t n, size_t transfer) : bytes(n) {
        constexpr size_t KB = 1024, MB = KB * KB;
        chunk = transfer > kStageBytes ? 16 * MB : MB;
        piece = transfer > kStageBytes ? MB : 128 * KB;
        while (chunk < 4 * MB && chunk * 16 < transfer) chunk *= 2;
        nch = (n + chunk - 1) / chunk;
        pieces = (int64_t)((n + piece - 1) / piece);
        left.reset(new std::atomic<int>[nch]);
        for (size_t k = 0; k < nch; ++k) left[k] = (int)((size(k) + piece - 1) / piece);
    }
    size_t size(size_t k) const { return std::min(chunk, bytes - k * chunk); }
    size_t chunk_of(int64_t p) const { return (size_t)p * piece / chunk; }
};
}  // namespace

// Host -> device: fill(stage, a0, a1) writes bytes [a0, a1) of the transfer to
// `stage`.  The caller holds g_stage_mu and stage_ready() is true.  Without
// `wait` the last copies are still under way: the caller synchronizes s before
// it gives the buffers up.
template <typename Fill>
static hipError_t window_upload(void* dst, size_t bytes, hipStream_t s, Fill fill, bool wait = true) {
    hipError_t e = hipSuccess;
    int b = 0, used = 0;
    for (size_t off = 0; off < bytes && e == hipSuccess; off += kStageBytes, b ^= 1, ++used) {
        const size_t n = std::min(kStageBytes, bytes - off);
        char* stage = (char*)g_stage[b];
        char* to = (char*)dst + off;
        if (used >= 2 && (e = hipEventSynchronize(g_stage_ev[b])) != hipSuccess) break;
        if (n <= kInlineBytes) {
            fill(stage, off, off + n);
            e = pwmk::launch_copy_bytes(to, stage, n, false, s);
        } else {
            Window W(n, bytes);
            const LoopFn work = [&](int64_t p0, int64_t p1, int) {
                for (int64_t p = p0; p < p1; ++p) {
                    const size_t a0 = (size_t)p * W.piece, a1 = std::min(n, a0 + W.piece);
                    fill(stage + a0, off + a0, off + a1);
                    W.left[W.chunk_of(p)].fetch_sub(1, std::memory_order_release);
                }
            };
            const LeadFn lead = [&](std::atomic<int64_t>& next) {
                for (size_t k = 0; k < W.nch; ++k) {
                    while (W.left[k].load(std::memory_order_acquire) != 0) {
                        const int64_t p = next.load() < W.pieces ? next.fetch_add(1) : W.pieces;
                        if (p < W.pieces)
                            work(p, p + 1, 0);
                        else
                            std::this_thread::yield();
                    }
                    if (e == hipSuccess)
                        e = pwmk::launch_copy_bytes(to + k * W.chunk, stage + k * W.chunk, W.size(k), false, s);
                }
            };
            parallel_run(W.pieces, 1, work, &lead);
        }
        if (e == hipSuccess && bytes > 2 * kStageBytes) e = hipEventRecord(g_stage_ev[b], s);
    }
    if (!wait && e == hipSuccess) return e;
    const hipError_t e2 = hipStreamSynchronize(s);  // the buffers are the next transfer's
    return e != hipSuccess ? e : e2;
}

// Device -> host: empty(stage, a0, a1) takes bytes [a0, a1) from `stage`.  Waits
// for the work queued on s.  The caller holds g_stage_mu and stage_ready() is
// true.  b: the buffer to begin with.  The host threads are woken when the work
// before the copies has ended, or (soon) at once, where that is short: waking takes
// some 40 us (mv of 2 MB vectors 150 us, with the threads woken behind the SpMV 189;
// of 8 MB 449 and 453, of 32 MB 1425 and 1440).
template <typename Empty>
static hipError_t window_download(const void* src, size_t bytes, hipStream_t s, Empty empty, int b = 0, bool soon = true) {
    if (bytes <= kInlineBytes) {  // (an event costs 5 us more than the stream)
        hipError_t e = pwmk::launch_copy_bytes(g_stage[b], src, bytes, true, s);
        const hipError_t e2 = hipStreamSynchronize(s);
        if (e == hipSuccess) e = e2;
        if (e == hipSuccess) empty((const char*)g_stage[b], 0, bytes);
        return e;
    }
    auto issue = [&](size_t off, int to) {
        const Window W(std::min(kStageBytes, bytes - off), bytes);
        hipError_t e = hipSuccess;
        for (size_t k = 0; k < W.nch && e == hipSuccess; ++k) {
            e = pwmk::launch_copy_bytes((char*)g_stage[to] + k * W.chunk, (const char*)src + off + k * W.chunk, W.size(k),
                                        true, s);
            if (e == hipSuccess) e = hipEventRecord(g_ring_ev[to * kRingChunks + k], s);
        }
        return e;
    };
    hipError_t e = soon ? hipSuccess : hipEventRecord(g_stage_ev[b], s);
    if (e == hipSuccess) e = issue(0, b);
    if (e == hipSuccess && !soon) e = hipEventSynchronize(g_stage_ev[b]);
    for (size_t off = 0; off < bytes && e == hipSuccess; off += kStageBytes, b ^= 1) {
        if (off + kStageBytes < bytes && (e = issue(off + kStageBytes, b ^ 1)) != hipSuccess) break;
        const size_t n = std::min(kStageBytes, bytes - off);
        const char* stage = (const char*)g_stage[b];
        const Window W(n, bytes);
        std::atomic<size_t> ready{0};  // chunks that have arrived
        std::atomic<bool> bad{false};
        const LoopFn work = [&](int64_t p0, int64_t p1, int) {
            for (int64_t p = p0; p < p1; ++p) {
                while (ready.load(std::memory_order_acquire) <= W.chunk_of(p)) std::this_thread::yield();
                const size_t a0 = (size_t)p * W.piece, a1 = std::min(n, a0 + W.piece);
                if (!bad) empty(stage + a0, off + a0, off + a1);
            }
        };
        const LeadFn lead = [&](std::atomic<int64_t>&) {
            for (size_t k = 0; k < W.nch; ++k) {
                if (e == hipSuccess) e = hipEventSynchronize(g_ring_ev[b * kRingChunks + k]);
                if (e != hipSuccess) bad = true;
                ready.store(k + 1, std::memory_order_release);
            }
        };
        parallel_run(W.pieces, 1, work, &lead);
    }
    const hipError_t e2 = hipStreamSynchronize(s);
    return e != hipSuccess ? e : e2;
}

// Host -> device chunk by chunk (a caller that works between the chunks):
// fill(stage, a0, a1) writes bytes [a0, a1) of the transfer into `stage`
// (called by host threads on pieces of a chunk); host threads fill one buffer
// while the other is in flight.  The caller holds g_stage_mu and stage_ready()
// is true.
template <typename Fill>
static hipError_t staged_upload(void* dst, size_t bytes, hipStream_t s, Fill fill,
                                const std::function<void()>* between) {
    hipError_t e = hipSuccess;
    bool busy[2] = {false, false};
    int b = 0;
    const size_t chunk = stage_chunk(bytes);
    const int64_t piece = stage_piece(chunk);
    for (size_t off = 0; off < bytes && e == hipSuccess; off += chunk, b ^= 1) {
        const size_t n = std::min(chunk, bytes - off);
        if (busy[b] && (e = hipEventSynchronize(g_stage_ev[b])) != hipSuccess) break;
        char* stage = (char*)g_stage[b];
        parallel_for((int64_t)n, piece, [&](int64_t a0, int64_t a1, int) { fill(stage + a0, off + a0, off + a1); });
        e = hipMemcpyAsync((char*)dst + off, stage, n, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipEventRecord(g_stage_ev[b], s);
        busy[b] = true;
        if (between && *between) (*between)();
    }
    // the buffers are the next upload's: wait until the copies have read them
    const hipError_t e2 = hipStreamSynchronize(s);
    return e != hipSuccess ? e : e2;
}

hipError_t upload_staged(void* dst, const void* src, size_t bytes, hipStream_t s,
                         const std::function<void()>* between) {
    if (bytes == 0) return hipSuccess;
    std::lock_guard<std::mutex> lk(g_stage_mu);
    if (!stage_ready()) {  // no pinned memory: a plain copy from pageable memory
        hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e;
    }
    if (between && *between) return staged_upload(dst, bytes, s, bytes_in(src), between);
    return window_upload(dst, bytes, s, bytes_in(src));
}

hipError_t upload_indices_staged(void* dst, const int32_t* src, int64_t n, int64_t bound, bool* out_of_range,
                                 hipStream_t s, const std::function<void()>* between) {
    std::atomic<bool> bad{false};
    *out_of_range = false;
    if (n <= 0) return hipSuccess;
    const uint64_t ub = (uint64_t)bound;
    auto scan = [&bad, ub](const int32_t* p, int64_t m) {
        bool b = false;
        for (int64_t k = 0; k < m; ++k) b |= (uint64_t)(uint32_t)p[k] >= ub;  // negative values wrap above bound
        if (b) bad = true;
    };
    hipError_t e;
    {
        std::lock_guard<std::mutex> lk(g_stage_mu);
        if (!stage_ready()) {  // no pinned memory: check, then a plain copy from pageable memory
            parallel_for(n, 1 << 20, [&](int64_t a0, int64_t a1, int) { scan(src + a0, a1 - a0); });
            if (bad) {
                *out_of_range = true;
                return hipSuccess;
            }
            e = hipMemcpyAsync(dst, src, (size_t)n * 4, hipMemcpyHostToDevice, s);
            return e == hipSuccess ? hipStreamSynchronize(s) : e;
        }
        // pieces start and end on whole indices (multiples of 64 KB)
        const char* from = (const char*)src;
        e = staged_upload(
            dst, (size_t)n * 4, s,
            [from, &scan](char* to, size_t a0, size_t a1) {
                memcpy(to, from + a0, a1 - a0);
                scan((const int32_t*)to, (int64_t)((a1 - a0) / 4));
            },
            between);
    }
    *out_of_range = bad;
    return e;
}

hipError_t upload_values_staged(void* dst, const double* src, int64_t n, int vt, hipStream_t s,
                                const std::function<void()>* between) {
    if (vt == PWM_VALUES_F64) return upload_staged(dst, src, (size_t)n * 8, s, between);
    if (n <= 0) return hipSuccess;
    const size_t es = vt == PWM_VALUES_F32 ? 4 : 2;
    std::lock_guard<std::mutex> lk(g_stage_mu);
    if (!stage_ready()) {  // no pinned memory: narrow into host memory, then a plain copy
        std::vector<char> tmp((size_t)n * es);
        char* o = tmp.data();
        parallel_for(n, 1 << 20, [&](int64_t a0, int64_t a1, int) {
            for (int64_t k = a0; k < a1; ++k) narrow_value(src, vt, k, o + k * es);
        });
        hipError_t e = hipMemcpyAsync(dst, o, tmp.size(), hipMemcpyHostToDevice, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e;
    }
    if (between && *between) return staged_upload(dst, (size_t)n * es, s, values_in(src, vt), between);
    return window_upload(dst, (size_t)n * es, s, values_in(src, vt));
}

hipError_t download_doubles(double* dst, const void* src, int64_t n, bool f64, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const size_t bytes = (size_t)n * (f64 ? 8 : 4);
    if (bytes <= kInlineBytes) {
        ShortSlot slot;
        if (slot.p) {
            hipError_t e = pwmk::launch_copy_bytes(slot.p, src, bytes, true, s);
            const hipError_t e2 = hipStreamSynchronize(s);
            if (e == hipSuccess) e = e2;
            if (e == hipSuccess) f64 ? bytes_out(dst)(slot.p, 0, bytes) : floats_out(dst)(slot.p, 0, bytes);
            return e;
        }
    }
    hipError_t e = hipStreamSynchronize(s);  // before the lock
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lk(g_stage_mu);
    if (!stage_ready()) {  // no pinned memory: a plain copy to pageable memory
        std::vector<float> f(f64 ? 0 : n);
        e = hipMemcpyAsync(f64 ? (void*)dst : f.data(), src, bytes, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        for (size_t i = 0; i < f.size() && e == hipSuccess; ++i) dst[i] = f[i];
        return e;
    }
    return f64 ? window_download(src, bytes, s, bytes_out(dst)) : window_download(src, bytes, s, floats_out(dst));
}

int fail(pwm_matrix* h, int code, const std::string& msg) {
    if (h)
        h->err = msg;
    else
        g_err = msg;
    return code;
}
int hip_fail(pwm_matrix* h, hipError_t e, const char* what) {
    std::string m = std::string(what) + ": " + hipGetErrorString(e);
    return fail(h, e == hipErrorOutOfMemory ? PWM_ERR_NOMEM : PWM_ERR_HIP, m);
}
size_t value_size(int vtype) { return vtype == PWM_VALUES_F64 ? 8 : (vtype == PWM_VALUES_F32 ? 4 : 2); }

bool exact_in_bf16(const double* v, int64_t n) {
    std::atomic<bool> ok{true};
    parallel_for(n, 1 << 20, [&](int64_t b, int64_t e, int) {
        for (int64_t k = b; k < e && ok.load(std::memory_order_relaxed); ++k) {
            const float f = (float)v[k];
            uint32_t bits;
            memcpy(&bits, &f, 4);
            if ((double)f != v[k] || (bits & 0xffffu)) ok = false;
        }
    });
    return ok;
}
size_t vector_size(int vtype) { return vtype == PWM_VALUES_F64 ? 8 : 4; }

static CrsDev crs_of(const pwm_matrix* h) {
    CrsDev A;
    A.nrows = h->nor;
    A.ncols = h->noc;
    A.nnz = h->nnz;
    A.rs = h->rs.as<int32_t>();
    A.ci = h->ci.as<int32_t>();
    A.val = h->val.p;
    A.vtype = h->vtype;
    A.nt = h->crs_nt_used;
    return A;
}

// The CRS arrays the one-workgroup power method reads: the handle's own, or
// those a blocked format keeps of a small matrix.
static CrsDev small_crs_of(const pwm_matrix* h) {
    CrsDev A = crs_of(h);
    if (h->sm_rs.p) {
        A.rs = h->sm_rs.as<int32_t>();
        A.ci = h->sm_ci.as<int32_t>();
        A.val = h->sm_val.p;
    }
    return A;
}

// Whether the power method of the handle about to be planned runs in one
// workgroup (k_power.hip): the matrix fits it, and the caller chose no kernel,
// layout or partition count, which a power step would otherwise have to run.
static bool wants_power_small(const pwm_matrix* h) {
    bool chosen = false;
    switch (h->format) {
        case PWM_FORMAT_CRS: chosen = h->crs_kernel || h->group_opt || h->vec_blocks_opt || h->long_row || h->crs_nt >= 0; break;
        case PWM_FORMAT_CRS_MERGE: chosen = h->threads > 0 || h->ipt != 8; break;
        case PWM_FORMAT_CSB:
            chosen = h->csb_bits_override || h->csb_groups || h->csb_layout || h->csb_window_bits || h->csb_unroll ||
                     h->csb_nt >= 0;
            break;
        case PWM_FORMAT_BLOCKCOH: chosen = h->threads > 0 || h->coh_occ8 >= 0; break;
    }
    CrsDev A = crs_of(h);
    return !chosen && pwmk::power_small_fits(A, h->stats.row_max);
}

static int pow2_ceil(int64_t v) {
    int g = 1;
    while (g < v && g < 64) g <<= 1;
    return g;
}

// CRS tiles kernel: the engine's row-aligned tile plan, kept as merge-path
// splits (split_a/split_b = each tile's first row / nonzero) for the fix-up.
static int plan_crs_tiles(pwm_matrix* h) {
    const int ipt = pwmk::tiles_items_per_thread();
    const int32_t nt = pwmk::engine_tiles_for(h->nor, h->nnz, ipt);
    hipError_t e;
    if ((e = h->tiles.alloc((size_t)nt * sizeof(pwmk::ETile))) != hipSuccess ||
        (e = h->split_a.alloc((nt + 1) * 8)) != hipSuccess || (e = h->split_b.alloc((nt + 1) * 8)) != hipSuccess ||
        (e = h->carry_row.alloc(nt * 4)) != hipSuccess || (e = h->carry_val.alloc(nt * 8)) != hipSuccess)
        return hip_fail(h, e, "tiles plan allocation");
    e = pwmk::engine_plan_tiles(h->rs.as<int32_t>(), h->nor, h->nnz, ipt, h->tiles.as<pwmk::ETile>(), h->stream);
    std::vector<pwmk::ETile> t(nt);
    if (e == hipSuccess)
        e = hipMemcpyAsync(t.data(), h->tiles.p, (size_t)nt * sizeof(pwmk::ETile), hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return hip_fail(h, e, "tiles plan");
    std::vector<int64_t> sa(nt + 1), sb(nt + 1);
    h->tiles_carry = false;
    for (int32_t i = 0; i < nt; ++i) {
        sa[i] = t[i].a0;
        sb[i] = t[i].b0;
        if (!t[i].stream) h->tiles_carry = true;
    }
    sa[nt] = h->nor;
    sb[nt] = h->nnz;
    if ((e = hipMemcpy(h->split_a.p, sa.data(), (nt + 1) * 8, hipMemcpyHostToDevice)) != hipSuccess ||
        (e = hipMemcpy(h->split_b.p, sb.data(), (nt + 1) * 8, hipMemcpyHostToDevice)) != hipSuccess)
        return hip_fail(h, e, "tiles plan upload");
    h->mp = pwmk::MergePlan{};
    h->mp.P = nt;
    h->mp.ipt = ipt;
    h->mp.items_per_tile = 0;
    h->mp.split_a = h->split_a.as<int64_t>();
    h->mp.split_b = h->split_b.as<int64_t>();
    h->mp.carry_row = h->carry_row.as<int32_t>();
    h->mp.carry_val = h->carry_val.p;
    return PWM_OK;
}

static hipError_t crs_kernel_launch(pwm_matrix* h, int which, const void* x, void* y, const PowerArgs* pw) {
    const CrsDev A = crs_of(h);
    hipError_t e;
    if (which == 0) {  // CRS_MERGE
        e = pwmk::launch_merge_spmv(A, h->mp, x, y, pw, h->stream);
        if (e == hipSuccess) e = pwmk::launch_merge_fixup(A, h->mp, y, pw, h->stream);
        return e;
    }
    if (which == 3) {
        e = pwmk::launch_rows(A, h->rp, x, y, pw, h->stream);
        if (e == hipSuccess && pw) e = pwmk::launch_power_reduce(*pw, pwmk::rows_power_blocks(h->rp.nt), h->stream);
        return e;
    }
    if (which == 2) {
        // a plain SpMV whose tiles are all row-aligned stream tiles has no
        // carries to add; power steps always finish in the fix-up (norms)
        e = pwmk::launch_tiles_spmv(A, h->tiles.as<pwmk::ETile>(), h->mp, x, y, pw, h->stream);
        if (e == hipSuccess && (pw || h->tiles_carry)) e = pwmk::launch_merge_fixup(A, h->mp, y, pw, h->stream);
        return e;
    }
    e = pwmk::launch_crs_vector(A, h->group, h->vec_blocks, h->lr, x, y, pw, h->stream);
    if (e == hipSuccess && (pw || h->lr.n_rows > 0)) e = pwmk::launch_crs_finalize(A, h->vec_blocks, h->lr, y, pw, h->stream);
    return e;
}

// Mean of 5 SpMVs after 2 warm-up ones.  From 4 M entries on (25 us a run and
// more: one run pages everything in, two give its time to a few percent) 2 after
// 1, unless these 2 took less than 0.1 ms.  Loading power-law rows in CSB, which
// times 13 layouts: 6.4 M entries 16.6 -> 13.7 ms, 48 M 87 -> 56; in CRS 6.4 ->
// 5.3 and 38 -> 30.
hipError_t time_launches(pwm_matrix* h, const std::function<hipError_t()>& launch, float* ms) {
    hipEvent_t a = nullptr, b = nullptr;
    hipError_t e = hipEventCreate(&a);
    if (e == hipSuccess) e = hipEventCreate(&b);
    auto run = [&](int warm, int timed) {
        float t = 0.0f;
        for (int i = 0; i < warm && e == hipSuccess; ++i) e = launch();
        if (e == hipSuccess) e = hipEventRecord(a, h->stream);
        for (int i = 0; i < timed && e == hipSuccess; ++i) e = launch();
        if (e == hipSuccess) e = hipEventRecord(b, h->stream);
        if (e == hipSuccess) e = hipEventSynchronize(b);
        if (e == hipSuccess) e = hipEventElapsedTime(&t, a, b);
        return t / timed;
    };
    const bool large = h->nnz >= ((int64_t)4 << 20);
    *ms = large ? run(1, 2) : run(2, 5);
    if (large && e == hipSuccess && 2 * *ms < 0.1f) *ms = run(0, 5);
    if (a) (void)hipEventDestroy(a);
    if (b) (void)hipEventDestroy(b);
    return e;
}

// Time of an SpMV by CRS kernel `which` on the device vectors x, y.
static hipError_t time_crs_kernel(pwm_matrix* h, int which, const void* x, void* y, float* ms) {
    return time_launches(h, [&] { return crs_kernel_launch(h, which, x, y, nullptr); }, ms);
}

constexpr int64_t kXcdL2 = (int64_t)4 << 20;  // an XCD's L2

// Stencils and banded matrices have some 10 to 20, with 2 random entries per row
// about 55, uniformly random columns all 256.
hipError_t column_lines(pwm_matrix* h, double* per_group) {
    *per_group = 0.0;
    const int64_t xb = (int64_t)vector_size(h->vtype);
    if (h->noc * xb <= kXcdL2 || h->nnz < 256) return hipSuccess;
    const int64_t groups = std::min<int64_t>(h->nnz / 256, 2048);
    DevBuf lines;
    unsigned n = 0;
    hipError_t e = lines.alloc(4);
    if (e == hipSuccess) e = hipMemsetAsync(lines.p, 0, 4, h->stream);
    if (e == hipSuccess)
        e = pwmk::launch_scatter(h->ci.as<int32_t>(), h->nnz, groups, xb == 8 ? 4 : 5, lines.as<unsigned>(), h->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(&n, lines.p, 4, hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    *per_group = (double)n / (double)groups;
    return e;
}

// Entry loads of the wave tiles: non-temporal, so that the entries leave the L2
// to x, where x is beyond one L2 and some of its lines are far apart.  9-point
// stencil with 2 random entries per row, us, plain and non-temporal: FP64 1001^2
// 45.9 44.1, 1448^2 103 99.5, 2000^2 205 201, FP32 1448^2 76.0 70.0; 500^2 (2 MB
// of x) 10.2 12.8.  Poisson: FP64 1024^2 13.7 17.0, 3000^2 123 140, 5000^2 335
// 381; FP32 5000^2 231 238.
constexpr double kSpreadLines = 32.0;
static int rows_nt(const pwm_matrix* h, double lines) { return h->crs_nt >= 0 ? h->crs_nt : lines > kSpreadLines; }

// Time of an SpMV by the swept slabs beside the CRS arrays, entry loads plain or
// non-temporal, the faster kept.
static hipError_t time_swept(pwm_matrix* h, const void* x, void* y, float* best) {
    hipError_t e = hipSuccess;
    int best_nt = 0;
    *best = -1.0f;
    for (int nt = 0; nt < 2 && e == hipSuccess; ++nt) {
        h->csb.nt = nt;
        float ms = 0.0f;
        e = time_launches(h, [&] { return csb_launch(h, x, y, nullptr); }, &ms);
        if (*best < 0.0f || ms < *best) {
            *best = ms;
            best_nt = nt;
        }
    }
    h->csb.nt = best_nt;
    return e;
}

// Swept slabs for scattered columns (k_csb_sweep, turns), more than 128 lines
// per 256 entries: a sweep in row order then fetches about one 128-byte line per
// entry from beyond the L2.  Built beside the CRS arrays and timed into *ms, on a
// vector of ones x; *ms < 0 when not built.  csb_layout = 4 builds them for any
// columns and returns 0 ms (always the
// faster), 1 to 3 never.  Power-law rows of 16 entries, warm: FP64 1.2 M rows
// 228 -> 76 us, 2.1 M 487 -> 161; FP32 3 M 586 -> 159; below 4 MB of x the row
// order is at most a third slower (FP64 600 000 rows, 4.8 MB: 85 -> 60 us) and
// the build is not worth its time (8 ms at 1.2 M rows).
// CRS_MERGE, which times nothing otherwise, takes them from 8 MB of x on: its load
// becomes half as long again (6.2 M entries: 6.5 -> 9.8 ms), which 33 SpMVs bring
// back at 9.6 MB of x (250 -> 108 us each) and 130 at 6.2 MB (65 -> 40).  A CRS
// load times its kernels in any case (11.0 ms, with the slabs 10.0).
//
// The slabs are a second copy of the matrix, which nobody asked for: they are kept
// only while three quarters of the device memory stay free, so that all handles'
// slabs together take about an eighth of it at most.
static bool leaves_room(const pwm_matrix* h) {
    size_t free = 0, total = 0;
    if (hipMemGetInfo(&free, &total) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return free >= total / 4 * 3 + (size_t)h->nnz * (4 + value_size(h->vtype));
}
static bool wants_swept(const pwm_matrix* h, double lines) {
    if (h->csb_layout == 4) return h->nnz > 0;
    const int64_t xbytes = h->noc * (int64_t)vector_size(h->vtype);
    return h->csb_layout == 0 && lines > 128.0 && (h->format == PWM_FORMAT_CRS || xbytes > 2 * kXcdL2) && leaves_room(h);
}
static int plan_swept(pwm_matrix* h, double lines, const void* x, void* y, float* ms) {
    *ms = -1.0f;
    h->csb.clear();
    const bool asked = h->csb_layout == 4;
    if (!wants_swept(h, lines)) return PWM_OK;
    const int rc = build_swept_beside_crs(h);
    if (rc != PWM_OK || !h->csb.sweep) return rc;
    hipError_t e;
    if ((e = time_swept(h, x, y, ms)) != hipSuccess) return hip_fail(h, e, "swept slabs");
    if (asked) *ms = 0.0f;
    return PWM_OK;
}

// The faster of plain and non-temporal entry loads (the caller's choice, else
// both are timed) for the CRS tiles, and its time.
static hipError_t time_entry_loads(pwm_matrix* h, const void* x, void* y, float* best) {
    int best_nt = 0;
    *best = -1.0f;
    for (int nt : {0, 1}) {
        if (h->crs_nt >= 0 && nt != h->crs_nt) continue;
        h->crs_nt_used = nt;
        float ms = 0.0f;
        const hipError_t e = time_crs_kernel(h, 2, x, y, &ms);
        if (e != hipSuccess) return e;
        if (*best < 0.0f || ms < *best) {
            *best = ms;
            best_nt = nt;
        }
    }
    h->crs_nt_used = best_nt;
    return hipSuccess;
}

// CRS vector kernel with G lanes per row: grid size and the long-row chunk
// plan (rows longer than max(1024, 128 G) are cut into chunks).
static int plan_crs_vector(pwm_matrix* h, int G) {
    h->group = G;
    const int64_t rpw = 64 / G;
    const int64_t units = (h->nor + rpw - 1) / rpw;
    int64_t blocks = h->vec_blocks_opt > 0 ? h->vec_blocks_opt : std::min<int64_t>((units + 3) / 4, 2048);
    h->vec_blocks = (int)std::max<int64_t>(blocks, 1);

    int64_t thr = h->long_row > 0 ? h->long_row : std::max<int64_t>(1024, 128 * G);
    h->lr = pwmk::LongRows{};
    h->lr.threshold = (int32_t)std::min<int64_t>(thr, INT32_MAX);
    std::vector<pwmk::LongChunk> chunks;
    std::vector<int32_t> ids, begin;
    // the row offsets: the host copy when the load kept one, else read back
    // from the device (every row longer than the threshold must be planned,
    // since the vector kernel skips them)
    std::vector<int32_t> rs_dev;
    const int32_t* rsh = h->h_rs.empty() ? nullptr : h->h_rs.data();
    if (!rsh && h->nor > 0) {
        rs_dev.resize(h->nor + 1);
        hipError_t e = hipMemcpy(rs_dev.data(), h->rs.p, (h->nor + 1) * 4, hipMemcpyDeviceToHost);
        if (e != hipSuccess) return hip_fail(h, e, "long-row plan: row offsets");
        rsh = rs_dev.data();
    }
    if (rsh) {
        for (int64_t r = 0; r < h->nor; ++r) {
            const int64_t s = rsh[r], e = rsh[r + 1];
            if (e - s <= thr) continue;
            begin.push_back((int32_t)chunks.size());
            for (int64_t k = s; k < e; k += h->chunk) {
                pwmk::LongChunk c;
                c.row = (int32_t)r;
                c.slot = (int32_t)ids.size();
                c.k0 = (int32_t)k;
                c.k1 = (int32_t)std::min<int64_t>(e, k + h->chunk);
                chunks.push_back(c);
            }
            ids.push_back((int32_t)r);
        }
    }
    begin.push_back((int32_t)chunks.size());
    h->lr.n_rows = (int32_t)ids.size();
    h->lr.n_chunks = (int32_t)chunks.size();
    if (!ids.empty()) {
        hipError_t e;
        if ((e = h->lr_chunks.alloc(chunks.size() * sizeof(pwmk::LongChunk))) != hipSuccess ||
            (e = h->lr_rows.alloc(ids.size() * 4)) != hipSuccess ||
            (e = h->lr_begin.alloc(begin.size() * 4)) != hipSuccess ||
            (e = h->lr_partial.alloc(chunks.size() * 8)) != hipSuccess)
            return hip_fail(h, e, "long-row plan allocation");
        if ((e = hipMemcpy(h->lr_chunks.p, chunks.data(), chunks.size() * sizeof(pwmk::LongChunk),
                           hipMemcpyHostToDevice)) != hipSuccess ||
            (e = hipMemcpy(h->lr_rows.p, ids.data(), ids.size() * 4, hipMemcpyHostToDevice)) != hipSuccess ||
            (e = hipMemcpy(h->lr_begin.p, begin.data(), begin.size() * 4, hipMemcpyHostToDevice)) != hipSuccess)
            return hip_fail(h, e, "long-row plan upload");
        h->lr.chunks = h->lr_chunks.as<pwmk::LongChunk>();
        h->lr.row_ids = h->lr_rows.as<int32_t>();
        h->lr.chunk_begin = h->lr_begin.as<int32_t>();
        h->lr.chunk_partial = h->lr_partial.p;
    }
    return PWM_OK;
}

// Wave tiles (k_rows.hip), where every row is short and no tile has too many
// rows; PWM_OK with rp.nt = 0 where not.
static int plan_crs_rows(pwm_matrix* h) {
    h->rp = pwmk::RowsPlan{};
    h->rows_cut.release();
    const int64_t step = pwmk::rows_step(h->stats.row_max);
    if (step <= 0 || h->nnz == 0) return PWM_OK;
    pwmk::RowsPlan rp;
    rp.nt = (h->nnz + step - 1) / step;
    // the cuts and, behind them, the plan kernel's flag
    hipError_t e = h->rows_cut.alloc((rp.nt + 2) * sizeof(int2));
    if (e != hipSuccess) return hip_fail(h, e, "wave tile plan");
    int2* cut = h->rows_cut.as<int2>();
    int* flag = (int*)(cut + rp.nt + 1);
    int too_many = 0;
    e = hipMemsetAsync(flag, 0, 4, h->stream);
    if (e == hipSuccess) e = pwmk::launch_rows_plan(crs_of(h), step, rp.nt, cut, flag, h->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(&too_many, flag, 4, hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return hip_fail(h, e, "wave tile plan");
    if (too_many) {
        h->rows_cut.release();
        return PWM_OK;
    }
    rp.cut = cut;
    h->rp = rp;
    return PWM_OK;
}

// Where the wave tiles need no timing: up to `mean` entries per row, and on small
// matrices (0.5 M entries), whose kernels differ by less than a microsecond of a
// call.  A lane sums a row alone, and of longer rows a tile has few.  Rows of L
// columns near the diagonal, FP64 SpMV in us, wave tiles, CRS tiles, vector and merge
// kernel: 150 000 rows L = 12 5.2 5.5 6.1 11.4, 20 8.0 9.6 10.3 15.6, 28 10.7 11.9
// 11.4 18.6, 48 26.9 20.5 17.1 23.6, 64 39.8 25.8 19.3 28.4; 1 M rows L = 12 23.8 25.2
// 29.8 35.9, 16 40.7 37.5 34.2 43.7, 28 68 72 88 80, 48 153 123 160 129.  Random
// columns hide it: 150 000 rows L = 64 49 48 50 54.
constexpr int64_t kRowsMeanCrs = 12, kRowsMeanMerge = 28;
static bool rows_untimed(const pwm_matrix* h, int64_t mean) {
    return h->nnz <= mean * h->nor || h->nnz < (int64_t)1 << 19;
}

// Time of an SpMV by the wave tiles.  Less 1.5 us where their power steps defer the
// norms, half of what that saves a step: the other kernels' do not.
static hipError_t time_rows(pwm_matrix* h, const void* x, void* y, float* ms) {
    const hipError_t e = time_crs_kernel(h, 3, x, y, ms);
    if (pwmk::rows_power_blocks(h->rp.nt) <= pwmk::kDeferSlots) *ms -= 0.0015f;
    return e;
}

static void drop_rows(pwm_matrix* h) {
    h->rp = pwmk::RowsPlan{};
    h->rows_cut.release();
}

// CRS planning and the autotuner.  Where no row has more than 64 entries the wave
// tiles (k_rows.hip) run, on a mean of at most 12 by rule (FP64, us, against the
// fastest of the others: Poisson 300 x 301 2.7 against 3.4, 5000 x 5000 332 against
// 441, 9-point stencil with 2 random entries per row, 1448 x 1448, 100 against
// 100), but where x has far lines and more than 24 MB (that stencil on 2896 x
// 2896: FP64 441 against 434, FP32, 33.5 MB of x, 369 against 364; on 2200 x 2200
// in FP32, 19 MB, 197 against 196).  Otherwise, or when the caller named a kernel
// or set up the vector kernel: candidates are that one with the
// rows-per-wave heuristic G0 = pow2(avg row length / 2) in [2, 32] and with
// G0/2 and 2 G0 when the longest row fills them (only G0 when the caller
// fixed group_size), the tiles kernel (unless crs_kernel excludes
// either) and the wave tiles.  With more than one candidate,
// each is timed on x = 1 and the fastest is kept.
int plan_crs(pwm_matrix* h) {
    const double avg = h->nor > 0 ? (double)h->nnz / (double)h->nor : 0.0;
    const int G0 = h->group_opt > 0 ? h->group_opt : std::min(32, std::max(2, pow2_ceil((int64_t)ceil(avg / 2.0))));
    // more lanes per row than the longest row has entries leave lanes idle
    // in every row: such candidates (other than G0) are not timed
    std::vector<int> gs;
    if (h->crs_kernel != 2) {
        if (h->group_opt > 0) {
            gs.push_back(G0);
        } else {
            for (int g : {G0 / 2, G0, 2 * G0})
                if (g >= 1 && g <= 64 && (g == G0 || g <= std::max<int64_t>(1, h->stats.row_max))) gs.push_back(g);
        }
    }
    int rc;
    drop_rows(h);
    h->csb.clear();
    const bool automatic = h->crs_kernel == 0 && h->group_opt == 0 && h->vec_blocks_opt == 0 && h->long_row == 0;
    hipError_t e;
    double lines = 0.0;
    if (automatic && (e = column_lines(h, &lines)) != hipSuccess) return hip_fail(h, e, "column lines");
    const int64_t xbytes = h->noc * (int64_t)vector_size(h->vtype);
    if (automatic && !(lines > kSpreadLines && xbytes > 6 * kXcdL2) && (rc = plan_crs_rows(h)) != PWM_OK) return rc;
    const bool rows = h->rp.nt > 0, rows_only = rows && rows_untimed(h, kRowsMeanCrs);
    bool tiles = !rows_only && h->crs_kernel != 1;
    const bool sweep = automatic && h->crs_nt < 0 && wants_swept(h, lines);
    if (rows_only) {
        gs.clear();
        h->lr = pwmk::LongRows{};
        h->crs_nt_used = rows_nt(h, lines);
        h->crs_used = 3;
        if (!sweep) return PWM_OK;
    } else {
        h->crs_nt_used = h->crs_nt > 0 ? 1 : 0;
    }
    if (!rows && (int)gs.size() + (tiles ? 1 : 0) == 1 && (!tiles || h->crs_nt >= 0)) {
        if (tiles && (rc = plan_crs_tiles(h)) != PWM_OK) return rc;
        h->crs_used = tiles ? 2 : 1;
        return plan_crs_vector(h, tiles ? G0 : gs[0]);
    }
    const size_t vs = vector_size(h->vtype);
    DevBuf x, y;
    if ((e = x.alloc(std::max<int64_t>(h->noc, 1) * vs)) != hipSuccess ||
        (e = y.alloc(std::max<int64_t>(h->nor, 1) * vs)) != hipSuccess)
        return hip_fail(h, e, "CRS autotune vectors");
    e = pwmk::launch_fill(x.p, h->noc, h->vtype == PWM_VALUES_F64 ? 1 : 0, 1.0, h->stream);
    if (e != hipSuccess) return hip_fail(h, e, "CRS autotune vectors");
    float best = -1.0f, swept = -1.0f;
    int best_kernel = 1, best_g = G0, best_nt = 0;
    if (sweep && (rc = plan_swept(h, lines, x.p, y.p, &swept)) != PWM_OK) return rc;
    if (rows) {
        best_kernel = 3;
        best_nt = h->crs_nt_used = rows_nt(h, lines);
        if ((e = time_rows(h, x.p, y.p, &best)) != hipSuccess) return hip_fail(h, e, "CRS autotune");
        // those below gather in row order too
        if (swept >= 0.0f && swept < 0.7f * best) {
            tiles = false;
            gs.clear();
        }
    }
    if (tiles) {
        float ms = 0.0f;
        if ((rc = plan_crs_tiles(h)) != PWM_OK) return rc;
        if ((e = time_entry_loads(h, x.p, y.p, &ms)) != hipSuccess) return hip_fail(h, e, "CRS autotune");
        if (!rows || ms < best) {
            best = ms;
            best_kernel = 2;
            best_nt = h->crs_nt_used;
        }
    }
    // the vector kernel gathers in row order like the tiles and was never a
    // third faster than they: it is not timed against a sweep that is
    if (swept >= 0.0f && swept < 0.7f * best) gs.clear();
    for (int g : gs) {
        if ((rc = plan_crs_vector(h, g)) != PWM_OK) return rc;
        float ms = 0.0f;
        if ((e = time_crs_kernel(h, 1, x.p, y.p, &ms)) != hipSuccess) return hip_fail(h, e, "CRS autotune");
        if ((!rows && !tiles && best < 0.0f) || ms < best) {
            best = ms;
            best_kernel = 1;
            best_g = g;
        }
    }
    h->crs_used = best_kernel;
    if (best_kernel != 1) h->crs_nt_used = best_nt;
    if (swept >= 0.0f && swept >= best) h->csb.clear();
    if (best_kernel != 3) drop_rows(h);
    if (best_kernel == 3 || h->csb.sweep) {
        h->lr = pwmk::LongRows{};
        h->vec_blocks = 0;
        return PWM_OK;
    }
    return plan_crs_vector(h, best_kernel == 1 ? best_g : G0);
}

// Merge path: P tiles of at most 256*ipt merge items (the threads count
// given to the constructor is used when its tiles fit that capacity).
int plan_merge(pwm_matrix* h) {
    const int64_t total = h->nor + h->nnz;
    const int64_t cap = 256 * (int64_t)h->ipt;
    int64_t P = (total + cap - 1) / cap;
    if (P < 1) P = 1;
    if (h->threads > 0) {
        const int64_t want = h->threads;
        const int64_t items = (total + want - 1) / want;
        if (items <= cap) P = want;
    }
    h->mp = pwmk::MergePlan{};
    h->mp.P = P;
    h->mp.items_per_tile = (total + P - 1) / P;
    h->mp.ipt = h->ipt;
    hipError_t e;
    if ((e = h->split_a.alloc((P + 1) * 8)) != hipSuccess || (e = h->split_b.alloc((P + 1) * 8)) != hipSuccess ||
        (e = h->carry_row.alloc(P * 4)) != hipSuccess || (e = h->carry_val.alloc(P * 8)) != hipSuccess)
        return hip_fail(h, e, "merge plan allocation");
    h->mp.split_a = h->split_a.as<int64_t>();
    h->mp.split_b = h->split_b.as<int64_t>();
    h->mp.carry_row = h->carry_row.as<int32_t>();
    h->mp.carry_val = h->carry_val.p;
    e = pwmk::launch_merge_splits(crs_of(h), h->mp, h->stream);
    if (e != hipSuccess) return hip_fail(h, e, "merge split search");
    // Unless the caller chose the partition or the tile size, the SpMV takes
    // the CRS format's wave tiles when the rows are short (Poisson 80 x 80: 8.0
    // -> 3.0 us, 1024 x 1024: 23.2 -> 13.8, 5000 x 5000: 405 -> 338, FP64; the
    // merge of each thread's items is what they save; timed against the merge
    // kernel above a mean of 28 entries) and its swept slabs when
    // the columns are scattered and the slabs time faster.
    h->csb.clear();
    drop_rows(h);
    h->crs_used = 0;
    const bool chosen = (h->threads > 0 && P == h->threads) || h->ipt != 8;
    int rc = chosen ? PWM_OK : plan_crs_rows(h);
    if (rc != PWM_OK) return rc;
    const bool rows = h->rp.nt > 0, contest = rows && !rows_untimed(h, kRowsMeanMerge);
    double lines = 0.0;
    if (!chosen && (rows || h->csb_layout == 0) && (e = column_lines(h, &lines)) != hipSuccess)
        return hip_fail(h, e, "column lines");
    if (rows) {
        h->crs_used = 3;
        h->crs_nt_used = rows_nt(h, lines);
    }
    if (chosen || (!contest && !wants_swept(h, lines))) {
        e = rows ? hipSuccess : hipStreamSynchronize(h->stream);
        return e == hipSuccess ? PWM_OK : hip_fail(h, e, "merge split search");
    }
    const size_t vs = vector_size(h->vtype);
    DevBuf x, y;
    if ((e = x.alloc(h->noc * vs)) == hipErrorOutOfMemory ||
        (e == hipSuccess && (e = y.alloc(std::max<int64_t>(h->nor, 1) * vs)) == hipErrorOutOfMemory)) {
        (void)hipGetLastError();  // nothing to time on: the kernel chosen so far stays
        e = hipStreamSynchronize(h->stream);
        return e == hipSuccess ? PWM_OK : hip_fail(h, e, "merge split search");
    }
    if (e != hipSuccess ||
        (e = pwmk::launch_fill(x.p, h->noc, h->vtype == PWM_VALUES_F64 ? 1 : 0, 1.0, h->stream)) != hipSuccess)
        return hip_fail(h, e, "merge plan vectors");
    float swept = -1.0f, best = -1.0f;
    if (contest) {
        float merge = 0.0f;
        if ((e = time_rows(h, x.p, y.p, &best)) != hipSuccess ||
            (e = time_crs_kernel(h, 0, x.p, y.p, &merge)) != hipSuccess)
            return hip_fail(h, e, "merge plan");
        if (merge < best) {
            best = merge;
            h->crs_used = 0;
            drop_rows(h);
        }
    }
    if ((rc = plan_swept(h, lines, x.p, y.p, &swept)) != PWM_OK) return rc;
    if (swept < 0.0f) return PWM_OK;
    if (!contest && (e = time_crs_kernel(h, h->crs_used, x.p, y.p, &best)) != hipSuccess) return hip_fail(h, e, "merge plan");
    if (swept >= best) h->csb.clear();
    return PWM_OK;
}

// A CRS or CRS_MERGE handle whose SpMV sweeps its slabs.
static bool swept_crs(const pwm_matrix* h) {
    return (h->format == PWM_FORMAT_CRS || h->format == PWM_FORMAT_CRS_MERGE) && h->csb.sweep;
}

int spmv_launch(pwm_matrix* h, const void* x, void* y, const PowerArgs* pw) {
    hipError_t e = hipSuccess;
    switch (swept_crs(h) ? PWM_FORMAT_CSB : h->format) {
        case PWM_FORMAT_CRS:
        case PWM_FORMAT_CRS_MERGE: e = crs_kernel_launch(h, h->crs_used, x, y, pw); break;
        case PWM_FORMAT_CSB: e = csb_launch(h, x, y, pw); break;
        case PWM_FORMAT_BLOCKCOH: e = coh_launch(h, x, y, pw); break;
        default: return fail(h, PWM_ERR_INVALID, "unknown format");
    }
    if (e != hipSuccess) return hip_fail(h, e, "SpMV launch");
    return PWM_OK;
}

static int64_t partial_slots(const pwm_matrix* h) {
    switch (swept_crs(h) ? PWM_FORMAT_CSB : h->format) {
        case PWM_FORMAT_CRS:
            if (h->crs_used == 3) return pwmk::rows_power_blocks(h->rp.nt);
            return std::max<int64_t>(h->vec_blocks, h->tiles.p ? h->mp.P + pwmk::merge_fix_blocks(h->mp.P) : 0);
        case PWM_FORMAT_CRS_MERGE:
            return h->crs_used == 3 ? pwmk::rows_power_blocks(h->rp.nt) : h->mp.P + pwmk::merge_fix_blocks(h->mp.P);
        case PWM_FORMAT_CSB: return csb_partials(h);
        case PWM_FORMAT_BLOCKCOH: return coh_partials(h);
    }
    return 0;
}

// Whether a fixed number of power steps defers the norms: few slots, and kernels
// that can add them up (wave tiles, slab streams that write y, swept slabs,
// BlockCOH).
static bool defers_norms(const pwm_matrix* h) {
    bool can = h->crs_used == 3;
    if (swept_crs(h) || h->format == PWM_FORMAT_CSB)
        can = h->csb.sweep || (h->csb.stream && h->csb.groups == 1);
    else if (h->format == PWM_FORMAT_BLOCKCOH)
        can = h->coh.n_tasks > 0;
    const int64_t slots = partial_slots(h);
    return can && !h->power_small && slots > 0 && slots <= pwmk::kDeferSlots;
}

// deferred norms: two steps' slots
static int64_t partials_needed(const pwm_matrix* h) { return partial_slots(h) * (defers_norms(h) ? 2 : 1); }

}  // namespace pwm_impl

// ---------------------------------------------------------------- lifetime

static int noalloc_scratch(pwm_matrix* h, char** out);

extern "C" int pwm_create(int format, int threads, int value_type, pwm_matrix** out) {
    if (!out) return fail(nullptr, PWM_ERR_INVALID, "pwm_create: out is NULL");
    *out = nullptr;
    if (format != PWM_FORMAT_CRS && format != PWM_FORMAT_CRS_MERGE && format != PWM_FORMAT_CSB &&
        format != PWM_FORMAT_BLOCKCOH)
        return fail(nullptr, PWM_ERR_INVALID, "pwm_create: unknown format id " + std::to_string(format));
    if (value_type < PWM_VALUES_F64 || value_type > PWM_VALUES_BF16)
        return fail(nullptr, PWM_ERR_INVALID, "pwm_create: unknown value type");
    int ndev = 0;
    hipError_t e = hipGetDeviceCount(&ndev);
    if (e != hipSuccess || ndev < 1)
        return fail(nullptr, PWM_ERR_HIP, "pwm_create: no HIP device available");
    pwm_matrix* h = new pwm_matrix();
    h->format = format;
    h->threads = threads;
    h->vtype = value_type;
    e = hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        delete h;
        return hip_fail(nullptr, e, "pwm_create: stream");
    }
    // set-up of the no-allocation power method: the per-GPU workspace array
    // is made resident on this device and its address looked up, once per
    // device, so that pwm_power_method_device_noalloc itself allocates nothing
    char* ws = nullptr;
    if (int rc = noalloc_scratch(nullptr, &ws)) {
        (void)hipStreamDestroy(h->stream);
        delete h;
        return rc;
    }
    *out = h;
    return PWM_OK;
}

extern "C" int pwm_destroy(pwm_matrix* h) {
    if (!h) return PWM_OK;
    if (h->stream) {
        (void)hipStreamSynchronize(h->stream);
        (void)hipStreamDestroy(h->stream);
    }
    delete h;
    return PWM_OK;
}

extern "C" const char* pwm_last_error(const pwm_matrix* h) { return h ? h->err.c_str() : g_err.c_str(); }

extern "C" int pwm_set_option(pwm_matrix* h, const char* key, int64_t value) {
    if (!h || !key) return fail(h, PWM_ERR_INVALID, "pwm_set_option: NULL argument");
    const std::string k(key);
    if (k == "group_size") {
        if (value != 0 && (value < 1 || value > 64 || (value & (value - 1))))
            return fail(h, PWM_ERR_INVALID, "group_size must be 0 or a power of two in 1..64");
        h->group_opt = (int)value;
    } else if (k == "vec_blocks") {
        h->vec_blocks_opt = (int)std::max<int64_t>(0, value);
    } else if (k == "long_row") {
        h->long_row = std::max<int64_t>(0, value);
    } else if (k == "long_chunk") {
        if (value < 256) return fail(h, PWM_ERR_INVALID, "long_chunk must be >= 256");
        h->chunk = (int)value;
    } else if (k == "items_per_thread") {
        if (value != 4 && value != 8 && value != 12 && value != 16)
            return fail(h, PWM_ERR_INVALID, "items_per_thread must be 4, 8, 12 or 16");
        h->ipt = (int)value;
    } else if (k == "block_bits") {
        if (value < 0 || value > 16) return fail(h, PWM_ERR_INVALID, "block_bits must be 0..16");
        h->csb_bits_override = (int32_t)value;
    } else if (k == "csb_groups") {
        if (value < 0 || value > 64) return fail(h, PWM_ERR_INVALID, "csb_groups must be 0..64");
        h->csb_groups = (int32_t)value;
    } else if (k == "csb_layout") {
        if (value < 0 || value > 4)
            return fail(h, PWM_ERR_INVALID,
                        "csb_layout must be 0 (automatic), 1 (slab pieces), 2 (slab streams), 3 (wide slab streams) "
                        "or 4 (swept slabs)");
        h->csb_layout = (int32_t)value;
    } else if (k == "csb_window_bits") {
        if (value != 0 && (value < 10 || value > 24))
            return fail(h, PWM_ERR_INVALID, "csb_window_bits must be 0 (1 MB of x) or in [10, 24]");
        h->csb_window_bits = (int32_t)value;
    } else if (k == "csb_sync_every") {
        if (value != 1 && value != 2 && value != 4 && value != 8)
            return fail(h, PWM_ERR_INVALID, "csb_sync_every must be 1, 2, 4 or 8");
        h->csb_sync_every = (int32_t)value;
    } else if (k == "csb_sweep_unroll") {
        if (value != 1 && value != 2 && value != 4) return fail(h, PWM_ERR_INVALID, "csb_sweep_unroll must be 1, 2 or 4");
        h->csb_sweep_unroll = (int32_t)value;
    } else if (k == "csb_sweep_order") {
        if (value < 0 || value > 1) return fail(h, PWM_ERR_INVALID, "csb_sweep_order must be 0 (rows) or 1 (columns)");
        h->csb_sweep_order = (int32_t)value;
    } else if (k == "csb_sweep_waves") {
        if (value < 1 || value > 8) return fail(h, PWM_ERR_INVALID, "csb_sweep_waves must be 1..8");
        h->csb_sweep_waves = (int32_t)value;
    } else if (k == "coh_occ8") {
        if (value < -1 || value > 1) return fail(h, PWM_ERR_INVALID, "coh_occ8 must be -1 (automatic), 0 or 1");
        h->coh_occ8 = (int32_t)value;
    } else if (k == "csb_unroll") {
        if (value != 0 && value != 2 && value != 4) return fail(h, PWM_ERR_INVALID, "csb_unroll must be 0, 2 or 4");
        h->csb_unroll = (int32_t)value;
    } else if (k == "crs_nt") {
        if (value < -1 || value > 1) return fail(h, PWM_ERR_INVALID, "crs_nt must be -1 (timed), 0 or 1");
        h->crs_nt = (int)value;
    } else if (k == "csb_nt") {
        if (value < -1 || value > 1) return fail(h, PWM_ERR_INVALID, "csb_nt must be -1 (timed), 0 or 1");
        h->csb_nt = (int32_t)value;
    } else if (k == "csb_build") {
        if (value < 0 || value > 1) return fail(h, PWM_ERR_INVALID, "csb_build must be 0 (device) or 1 (host)");
        h->csb_build = (int32_t)value;
    } else if (k == "coh_build") {
        if (value < 0 || value > 1) return fail(h, PWM_ERR_INVALID, "coh_build must be 0 (device) or 1 (host)");
        h->coh_build = (int32_t)value;
    } else if (k == "crs_kernel") {
        if (value < 0 || value > 2) return fail(h, PWM_ERR_INVALID, "crs_kernel must be 0 (time both), 1 (vector) or 2 (tiles)");
        h->crs_kernel = (int)value;
    } else {
        return fail(h, PWM_ERR_UNSUPPORTED, "unknown option " + k);
    }
    if (h->loaded && (k == "group_size" || k == "vec_blocks" || k == "long_row" || k == "long_chunk" || k == "crs_kernel" ||
                      k == "crs_nt") &&
        h->format == PWM_FORMAT_CRS) {
        h->power_small = wants_power_small(h);
        return plan_crs(h);
    }
    if (h->loaded && k == "items_per_thread" && h->format == PWM_FORMAT_CRS_MERGE) {
        h->power_small = wants_power_small(h);
        return plan_merge(h);
    }
    return PWM_OK;
}

// ---------------------------------------------------------------- loading

static int upload_values(pwm_matrix* h, const double* vals, int64_t nnz) {
    hipError_t e = alloc_padded(h->val, nnz, value_size(h->vtype));
    if (e != hipSuccess) return hip_fail(h, e, "value allocation");
    if (nnz == 0) return PWM_OK;
    if (h->vtype == PWM_VALUES_BF16 && !exact_in_bf16(vals, nnz)) {
        for (int64_t i = 0; i < nnz; ++i) {  // name the first value that is not
            const float f = (float)vals[i];
            uint32_t b;
            memcpy(&b, &f, 4);
            if ((double)f != vals[i] || (b & 0xffffu))
                return fail(h, PWM_ERR_INVALID, "BF16 storage needs values exact in BF16 (entry " +
                                                    std::to_string(i) + ")");
        }
    }
    e = upload_values_staged(h->val.p, vals, nnz, h->vtype, h->stream);
    if (e != hipSuccess) return hip_fail(h, e, "value upload");
    return PWM_OK;
}

static void reset_matrix(pwm_matrix* h) {
    h->loaded = false;
    h->rs.release();
    h->ci.release();
    h->val.release();
    h->h_rs.clear();
    h->lr = pwmk::LongRows{};
    h->mp = pwmk::MergePlan{};
    h->tiles.release();
    h->rp = pwmk::RowsPlan{};
    h->rows_cut.release();
    h->crs_used = 1;
    h->csb.clear();
    h->coh.clear();
    h->power_small = false;
    h->sm_rs.release();
    h->sm_ci.release();
    h->sm_val.release();
}

static int finish_load(pwm_matrix* h, const int32_t* hrs, const int32_t* hci, const double* hval) {
    int rc = compute_matrix_stats(h);
    if (rc != PWM_OK) return rc;
    h->power_small = wants_power_small(h);
    switch (h->format) {
        case PWM_FORMAT_CRS: rc = plan_crs(h); break;
        case PWM_FORMAT_CRS_MERGE: rc = plan_merge(h); break;
        case PWM_FORMAT_CSB: rc = build_csb(h, hrs, hci, hval); break;
        case PWM_FORMAT_BLOCKCOH: rc = build_blockcoh(h, hrs, hci, hval); break;
    }
    if (rc == PWM_OK) h->loaded = true;
    return rc;
}

// Validated host CRS -> device.
static int load_crs_host(pwm_matrix* h, int64_t nor, int64_t noc, const int32_t* rs, const int32_t* ci,
                         const double* vals) {
    const int64_t nnz = rs[nor];
    h->nor = nor;
    h->noc = noc;
    h->nnz = nnz;
    hipError_t e;
    if ((e = h->rs.alloc((nor + 1) * 4)) != hipSuccess || (e = alloc_padded(h->ci, nnz, 4)) != hipSuccess)
        return hip_fail(h, e, "CRS allocation");
    if ((e = upload_staged(h->rs.p, rs, (nor + 1) * 4, h->stream)) != hipSuccess ||
        (e = upload_staged(h->ci.p, ci, nnz * 4, h->stream)) != hipSuccess)
        return hip_fail(h, e, "CRS upload");
    int rc = upload_values(h, vals, nnz);
    if (rc != PWM_OK) return rc;
    h->h_rs.assign(rs, rs + nor + 1);
    return finish_load(h, rs, ci, vals);
}

extern "C" int pwm_load_crs(pwm_matrix* h, int64_t nor, int64_t noc, const int32_t* rs, const int32_t* ci,
                            const double* vals, int partitions) {
    (void)partitions;
    if (!h) return fail(nullptr, PWM_ERR_INVALID, "pwm_load_crs: NULL handle");
    if (nor <= 0 || noc <= 0 || nor > INT32_MAX - 1 || noc > INT32_MAX || !rs)
        return fail(h, PWM_ERR_INVALID, "pwm_load_crs: need 0 < nor, noc < 2^31 and row_start");
    if (rs[0] != 0) return fail(h, PWM_ERR_INVALID, "pwm_load_crs: row_start[0] must be 0");
    for (int64_t r = 0; r < nor; ++r)
        if (rs[r + 1] < rs[r]) return fail(h, PWM_ERR_INVALID, "pwm_load_crs: row_start must be non-decreasing");
    const int64_t nnz = rs[nor];
    if (nnz > PWM_MAX_NNZ) return fail(h, PWM_ERR_INVALID, "pwm_load_crs: more than PWM_MAX_NNZ nonzeros");
    if (nnz > 0 && (!ci || !vals)) return fail(h, PWM_ERR_INVALID, "pwm_load_crs: NULL col_ind/values");
    std::atomic<bool> bad{false};
    parallel_for(nnz, 1 << 20, [&](int64_t k0, int64_t k1, int) {
        bool b = false;
        for (int64_t k = k0; k < k1; ++k) b |= (ci[k] < 0) | (ci[k] >= noc);
        if (b) bad = true;
    });
    if (bad) return fail(h, PWM_ERR_INVALID, "pwm_load_crs: column index out of range");
    reset_matrix(h);
    return load_crs_host(h, nor, noc, rs, ci, vals);
}

// COO -> CRS (Util/TripletToCRS.hpp:135-172): rows ascending, columns
// ascending inside a row, duplicates kept in input order.  The indices are
// validated on the host (in parallel); the sort runs on the device
// (coo_to_crs_device).  A host-built BlockCOH then takes the sorted arrays
// back; the other builds need only row_start on the host.
extern "C" int pwm_load_triplets(pwm_matrix* h, int64_t nor, int64_t noc, int64_t nnz, const int32_t* rows,
                                 const int32_t* cols, const double* vals, int partitions) {
    (void)partitions;
    if (!h) return fail(nullptr, PWM_ERR_INVALID, "pwm_load_triplets: NULL handle");
    if (nor <= 0 || noc <= 0 || nnz < 0 || nor > INT32_MAX - 1 || noc > INT32_MAX || nnz > PWM_MAX_NNZ)
        return fail(h, PWM_ERR_INVALID, "pwm_load_triplets: need 0 < nor, noc < 2^31 and 0 <= nnz <= PWM_MAX_NNZ");
    if (nnz > 0 && (!rows || !cols || !vals)) return fail(h, PWM_ERR_INVALID, "pwm_load_triplets: NULL arrays");
    // first out-of-range entry and first value not exact in BF16 (when BF16 storage)
    std::atomic<int64_t> bad_idx{INT64_MAX}, bad_val{INT64_MAX};
    const bool bf16 = h->vtype == PWM_VALUES_BF16;
    parallel_for(nnz, 1 << 16, [&](int64_t i0, int64_t i1, int) {
        for (int64_t i = i0; i < i1; ++i) {
            if (rows[i] < 0 || rows[i] >= nor || cols[i] < 0 || cols[i] >= noc) {
                int64_t cur = bad_idx.load();
                while (i < cur && !bad_idx.compare_exchange_weak(cur, i)) {
                }
                break;
            }
        }
        if (!bf16) return;
        for (int64_t i = i0; i < i1; ++i) {
            const float f = (float)vals[i];
            uint32_t b;
            memcpy(&b, &f, 4);
            if ((double)f != vals[i] || (b & 0xffffu)) {
                int64_t cur = bad_val.load();
                while (i < cur && !bad_val.compare_exchange_weak(cur, i)) {
                }
                break;
            }
        }
    });
    if (bad_idx.load() != INT64_MAX)
        return fail(h, PWM_ERR_INVALID, "pwm_load_triplets: index out of range at entry " + std::to_string(bad_idx.load()));
    if (bad_val.load() != INT64_MAX)
        return fail(h, PWM_ERR_INVALID,
                    "BF16 storage needs values exact in BF16 (entry " + std::to_string(bad_val.load()) + ")");
    reset_matrix(h);
    h->nor = nor;
    h->noc = noc;
    h->nnz = nnz;
    const bool f64 = h->vtype == PWM_VALUES_F64;
    DevBuf dtmp;
    int rc = coo_to_crs_device(h, nor, noc, nnz, rows, cols, vals, h->rs, h->ci, f64 ? h->val : dtmp);
    if (rc != PWM_OK) return rc;
    hipError_t e;
    if (!f64) {
        if ((e = alloc_padded(h->val, nnz, value_size(h->vtype))) != hipSuccess)
            return hip_fail(h, e, "value allocation");
        if (nnz > 0) {
            e = pwmk::launch_convert_values(dtmp.as<double>(), h->val.p, nnz, h->vtype, h->stream);
            if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
            if (e != hipSuccess) return hip_fail(h, e, "value conversion");
        }
    }
    std::vector<int32_t> hrs(nor + 1);
    if ((e = hipMemcpy(hrs.data(), h->rs.p, (nor + 1) * 4, hipMemcpyDeviceToHost)) != hipSuccess)
        return hip_fail(h, e, "row_start download");
    h->h_rs = hrs;
    if (h->format == PWM_FORMAT_CSB || (h->format == PWM_FORMAT_BLOCKCOH && h->coh_build != 1))
        return finish_load(h, h->h_rs.data(), nullptr, nullptr);
    if (h->format == PWM_FORMAT_BLOCKCOH) {
        std::vector<int32_t> hci(std::max<int64_t>(nnz, 1));
        std::vector<double> hdv(std::max<int64_t>(nnz, 1));
        const DevBuf& dsrc = f64 ? h->val : dtmp;
        if (nnz && (e = hipMemcpy(hci.data(), h->ci.p, nnz * 4, hipMemcpyDeviceToHost)) != hipSuccess)
            return hip_fail(h, e, "CRS download");
        if (nnz && (e = hipMemcpy(hdv.data(), dsrc.p, nnz * 8, hipMemcpyDeviceToHost)) != hipSuccess)
            return hip_fail(h, e, "CRS download");
        return finish_load(h, hrs.data(), hci.data(), hdv.data());
    }
    return finish_load(h, nullptr, nullptr, nullptr);
}

// SparseMatrix::generatePoissonMatrix: CRS filled on the device
// (Util/Poisson.hpp:32-83).  The blocked formats build from the same matrix.
extern "C" int pwm_generate_poisson(pwm_matrix* h, int64_t m, int64_t n, int partitions) {
    (void)partitions;
    if (!h) return fail(nullptr, PWM_ERR_INVALID, "pwm_generate_poisson: NULL handle");
    if (m <= 0 || n <= 0 || m * n > INT32_MAX - 1 || 5 * m * n > PWM_MAX_NNZ)
        return fail(h, PWM_ERR_INVALID, "pwm_generate_poisson: need m, n > 0 and 5*m*n <= PWM_MAX_NNZ");
    reset_matrix(h);
    const int64_t N = m * n, Z = n * (m + 2 * (m - 1)) + 2 * (n - 1) * m;
    h->nor = h->noc = N;
    h->nnz = Z;
    hipError_t e;
    if ((e = h->rs.alloc((N + 1) * 4)) != hipSuccess || (e = alloc_padded(h->ci, Z, 4)) != hipSuccess ||
        (e = alloc_padded(h->val, Z, value_size(h->vtype))) != hipSuccess)
        return hip_fail(h, e, "Poisson allocation");
    e = pwmk::launch_fill_poisson(m, n, h->rs.as<int32_t>(), h->ci.as<int32_t>(), h->val.p, h->vtype, h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return hip_fail(h, e, "Poisson fill");
    if (h->format == PWM_FORMAT_CSB || (h->format == PWM_FORMAT_BLOCKCOH && h->coh_build != 1)) {
        // the device builds need only row_start on the host (block-row sums,
        // band cuts); CSB's host-built fallback downloads the rest itself
        h->h_rs.resize(N + 1);
        if ((e = hipMemcpy(h->h_rs.data(), h->rs.p, (N + 1) * 4, hipMemcpyDeviceToHost)) != hipSuccess)
            return hip_fail(h, e, "Poisson download");
        return finish_load(h, h->h_rs.data(), nullptr, nullptr);
    }
    if (h->format == PWM_FORMAT_BLOCKCOH) {
        // the host builder works from host CRS arrays
        std::vector<int32_t> rs(N + 1), ci(Z);
        std::vector<double> dv(Z);
        DevBuf tmp;
        if ((e = tmp.alloc(Z * 8)) != hipSuccess) return hip_fail(h, e, "staging allocation");
        e = pwmk::launch_fill_poisson(m, n, h->rs.as<int32_t>(), h->ci.as<int32_t>(), tmp.p, pwmk::VT_F64, h->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
        if (e == hipSuccess) e = hipMemcpy(rs.data(), h->rs.p, (N + 1) * 4, hipMemcpyDeviceToHost);
        if (e == hipSuccess) e = hipMemcpy(ci.data(), h->ci.p, Z * 4, hipMemcpyDeviceToHost);
        if (e == hipSuccess) e = hipMemcpy(dv.data(), tmp.p, Z * 8, hipMemcpyDeviceToHost);
        if (e != hipSuccess) return hip_fail(h, e, "Poisson download");
        h->h_rs = rs;
        return finish_load(h, rs.data(), ci.data(), dv.data());
    }
    return finish_load(h, nullptr, nullptr, nullptr);
}

extern "C" int pwm_info(const pwm_matrix* h, pwm_info_t* out) {
    if (!h || !out) return fail(const_cast<pwm_matrix*>(h), PWM_ERR_INVALID, "pwm_info: NULL argument");
    memset(out, 0, sizeof(*out));
    out->nor = h->nor;
    out->noc = h->noc;
    out->nnz = h->nnz;
    out->format = h->format;
    out->value_type = h->vtype;
    // CRS: the lanes per row of the vector kernel, 0 when a tiles kernel runs
    out->group_size = h->format == PWM_FORMAT_CSB ? h->csb.groups
                      : (h->format == PWM_FORMAT_CRS && (h->crs_used >= 2 || swept_crs(h))) ? 0
                                                                           : h->group;
    out->long_rows = h->lr.n_rows;
    out->threads = swept_crs(h) && h->format == PWM_FORMAT_CRS ? (int32_t)h->csb.n_tasks
                   : (h->format == PWM_FORMAT_CRS_MERGE || (h->format == PWM_FORMAT_CRS && h->crs_used == 2))
                       ? (int32_t)h->mp.P
                   : h->format == PWM_FORMAT_CRS && h->crs_used == 3 ? (int32_t)h->rp.nt
                   : h->format == PWM_FORMAT_BLOCKCOH ? (int32_t)h->coh.bands.size()
                   : h->format == PWM_FORMAT_CSB      ? (int32_t)h->csb.n_tasks
                                                      : h->vec_blocks;
    out->block_bits = h->format == PWM_FORMAT_CSB ? h->csb.bits : 0;
    out->balanced = h->format == PWM_FORMAT_CSB ? h->csb.balanced : 0;
    out->unroll = h->format == PWM_FORMAT_CSB && h->csb.stream ? h->csb.unroll : 0;
    out->layout = h->format != PWM_FORMAT_CSB ? 0 : h->csb.sweep ? 4 : !h->csb.stream ? 1 : h->csb.wide ? 3 : 2;
    switch (h->format) {
        case PWM_FORMAT_CRS:
            out->kernels = 1 + (h->crs_used == 2 ? (h->tiles_carry ? 1 : 0) : (h->lr.n_rows > 0 ? 1 : 0));
            break;
        case PWM_FORMAT_CRS_MERGE: out->kernels = h->crs_used == 3 ? 1 : 2; break;
        case PWM_FORMAT_CSB: out->kernels = h->csb.sweep ? 1 : 1 + (h->csb.groups > 1 ? 1 : 0); break;
        case PWM_FORMAT_BLOCKCOH: out->kernels = 1 + (h->coh.n_pieces > 0 ? 1 : 0); break;
    }
    if (swept_crs(h)) out->kernels = 1;
    if (h->format == PWM_FORMAT_CSB && h->csb.n_tasks <= 0) out->kernels = 0;
    out->high_occupancy = h->format == PWM_FORMAT_BLOCKCOH ? !h->coh.one_wave : 0;
    out->non_temporal = h->format == PWM_FORMAT_CSB || swept_crs(h)         ? h->csb.nt
                        : (h->format == PWM_FORMAT_CRS && h->crs_used == 2) || h->crs_used == 3 ? h->crs_nt_used
                                                                           : 0;
    const pwm_impl::DevBuf* bufs[] = {&h->rs, &h->ci, &h->val, &h->lr_chunks, &h->lr_rows, &h->lr_begin,
                                      &h->lr_partial, &h->split_a, &h->split_b, &h->carry_row, &h->carry_val, &h->tiles,
                                      &h->rows_cut, &h->csb.ind, &h->csb.data, &h->csb.blk_ptr, &h->csb.work, &h->csb.ypart,
                                      &h->csb.soff, &h->csb.srows, &h->csb.sweep_start,
                                      &h->coh.ent, &h->coh.data, &h->coh.row_jump_block,
                                      &h->coh.col_jump_block, &h->coh.block_nnz, &h->coh.block_coords,
                                      &h->coh.band_table, &h->coh.tasks, &h->coh.ysum, &h->sm_rs, &h->sm_ci, &h->sm_val, &h->pw_ctrl, &h->pw_rec, &h->pw_partials,
                                      &h->hx, &h->hy};
    int64_t b = 0;
    for (auto* d : bufs) b += (int64_t)d->bytes;
    out->device_bytes = b;
    return PWM_OK;
}

// ---------------------------------------------------------------- SpMV

// A vector handed to a _device entry point must be coarse-grained device
// memory (hipMalloc) that holds `bytes` from p.  Host memory, pinned
// (hipHostMalloc) or not, managed memory and fine-grained device allocations
// are refused: the kernels add into y with hardware FP64 atomics (the library
// is built with unsafe FP atomics), which are not performed on fine-grained
// or host memory.
static int check_device_vec(pwm_matrix* h, const void* p, size_t bytes, const char* who, const char* name) {
    hipPointerAttribute_t a;
    hipError_t e = hipPointerGetAttributes(&a, p);
    if (e != hipSuccess) {
        (void)hipGetLastError();  // a refused pointer must not show up as a later launch error
        return fail(h, PWM_ERR_INVALID, std::string(who) + ": " + name + " is not device memory");
    }
    if (a.type != hipMemoryTypeDevice || a.isManaged)
        return fail(h, PWM_ERR_INVALID, std::string(who) + ": " + name + " is host or managed memory, not hipMalloc device memory");
    if (a.allocationFlags & hipDeviceMallocFinegrained)
        return fail(h, PWM_ERR_INVALID, std::string(who) + ": " + name + " is fine-grained device memory");
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    e = hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)p);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return fail(h, PWM_ERR_INVALID, std::string(who) + ": " + name + " has no device allocation");
    }
    if ((const char*)p + bytes > (const char*)base + size)
        return fail(h, PWM_ERR_INVALID, std::string(who) + ": " + name + " is shorter than the vector");
    return PWM_OK;
}

static int check_device_xy(pwm_matrix* h, const void* x, size_t x_elems, const void* y, size_t y_elems,
                           const char* who) {
    const size_t vs = vector_size(h->vtype);
    int rc = check_device_vec(h, x, x_elems * vs, who, "x");
    if (rc == PWM_OK) rc = check_device_vec(h, y, y_elems * vs, who, "y");
    return rc;
}

extern "C" int pwm_mv_device(pwm_matrix* h, const void* x, void* y) {
    if (!h) return fail(nullptr, PWM_ERR_INVALID, "pwm_mv_device: NULL handle");
    if (!h->loaded) return fail(h, PWM_ERR_STATE, "pwm_mv_device: no matrix loaded");
    if (!x || !y) return fail(h, PWM_ERR_INVALID, "pwm_mv_device: NULL vector");
    const size_t vs = vector_size(h->vtype);
    const char* xb = (const char*)x;
    const char* yb = (const char*)y;
    if (xb < yb + h->nor * vs && yb < xb + h->noc * vs)
        return fail(h, PWM_ERR_INVALID, "pwm_mv_device: x and y overlap");
    if (int rc0 = check_device_xy(h, x, h->noc, y, h->nor, "pwm_mv_device")) return rc0;
    int rc = spmv_launch(h, x, y, nullptr);
    if (rc != PWM_OK) return rc;
    hipError_t e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return hip_fail(h, e, "pwm_mv_device");
    return PWM_OK;
}

static int stage_vectors(pwm_matrix* h) {
    const size_t vs = vector_size(h->vtype);
    const size_t need = (size_t)std::max(h->nor, h->noc) * vs;
    hipError_t e;
    if (h->hx.bytes < need && (e = h->hx.alloc(need)) != hipSuccess) return hip_fail(h, e, "staging allocation");
    if (h->hy.bytes < need && (e = h->hy.alloc(need)) != hipSuccess) return hip_fail(h, e, "staging allocation");
    return PWM_OK;
}

// Host double vector -> device vector of the handle's type.
static int upload_vec(pwm_matrix* h, const double* src, void* dst, int64_t n) {
    const int vt = h->vtype == PWM_VALUES_F64 ? PWM_VALUES_F64 : PWM_VALUES_F32;
    const hipError_t e = upload_values_staged(dst, src, n, vt, h->stream);
    return e == hipSuccess ? PWM_OK : hip_fail(h, e, "vector upload");
}
static int download_vec(pwm_matrix* h, const void* src, double* dst, int64_t n) {
    const hipError_t e = download_doubles(dst, src, n, h->vtype == PWM_VALUES_F64, h->stream);
    return e == hipSuccess ? PWM_OK : hip_fail(h, e, "vector download");
}

// y = A x on short host vectors: x and y go through one piece of pinned memory,
// in the stream's order, and the host waits once, for y.
static int mv_short(pwm_matrix* h, const double* x, double* y, char* stage) {
    const bool f64 = h->vtype == PWM_VALUES_F64;
    const size_t vs = vector_size(h->vtype), nx = (size_t)h->noc * vs, ny = (size_t)h->nor * vs;
    f64 ? bytes_in(x)(stage, 0, nx) : values_in(x, PWM_VALUES_F32)(stage, 0, nx);
    hipError_t e = pwmk::launch_copy_bytes(h->hx.p, stage, nx, false, h->stream);
    int rc = e == hipSuccess ? spmv_launch(h, h->hx.p, h->hy.p, nullptr) : hip_fail(h, e, "vector upload");
    if (rc == PWM_OK && (e = pwmk::launch_copy_bytes(stage, h->hy.p, ny, true, h->stream)) != hipSuccess)
        rc = hip_fail(h, e, "vector download");
    e = hipStreamSynchronize(h->stream);
    if (rc == PWM_OK && e != hipSuccess) rc = hip_fail(h, e, "SpMV on host vectors");
    if (rc == PWM_OK) f64 ? bytes_out(y)(stage, 0, ny) : floats_out(y)(stage, 0, ny);
    return rc;
}

// y = A x on host vectors of at most one staging buffer each: x goes through one,
// y through the other, y's copies are queued behind the SpMV and the host waits
// once, for y.  Without that an FP64 call on a 1000 x 999 grid takes 482 instead of
// 453 us, an FP32 one 320 instead of 280.  g_stage_mu is held meanwhile, so only for
// SpMVs that are short beside their transfers.
constexpr int64_t kShortSpmv = (int64_t)1 << 26;  // entries, some 0.2 to 0.5 ms
constexpr int64_t kSoonSpmv = (int64_t)1 << 25;   // at most 0.1 ms or so
static int mv_staged(pwm_matrix* h, const double* x, double* y, bool* done) {
    const bool f64 = h->vtype == PWM_VALUES_F64;
    const size_t vs = vector_size(h->vtype);
    if (h->nnz > kShortSpmv || (size_t)std::max(h->nor, h->noc) * vs > kStageBytes) return PWM_OK;
    std::lock_guard<std::mutex> lk(g_stage_mu);
    if (!stage_ready()) return PWM_OK;  // no pinned memory: the general path
    *done = true;
    const bool soon = h->nnz <= kSoonSpmv;
    hipError_t e = f64 ? window_upload(h->hx.p, (size_t)h->noc * vs, h->stream, bytes_in(x), false)
                       : window_upload(h->hx.p, (size_t)h->noc * vs, h->stream, values_in(x, PWM_VALUES_F32), false);
    const int rc = e == hipSuccess ? spmv_launch(h, h->hx.p, h->hy.p, nullptr) : hip_fail(h, e, "vector upload");
    if (rc != PWM_OK) {
        (void)hipStreamSynchronize(h->stream);
        return rc;
    }
    e = f64 ? window_download(h->hy.p, (size_t)h->nor * vs, h->stream, bytes_out(y), 1, soon)
            : window_download(h->hy.p, (size_t)h->nor * vs, h->stream, floats_out(y), 1, soon);
    return e == hipSuccess ? PWM_OK : hip_fail(h, e, "vector download");
}

extern "C" int pwm_mv(pwm_matrix* h, const double* x, double* y) {
    if (!h) return fail(nullptr, PWM_ERR_INVALID, "pwm_mv: NULL handle");
    if (!h->loaded) return fail(h, PWM_ERR_STATE, "pwm_mv: no matrix loaded");
    if (!x || !y) return fail(h, PWM_ERR_INVALID, "pwm_mv: NULL vector");
    if (x < y + h->nor && y < x + h->noc) return fail(h, PWM_ERR_INVALID, "pwm_mv: x and y overlap");
    int rc = stage_vectors(h);
    if (rc != PWM_OK) return rc;
    if ((size_t)std::max(h->nor, h->noc) * vector_size(h->vtype) <= kInlineBytes) {
        ShortSlot slot;
        if (slot.p) return mv_short(h, x, y, slot.p);
    }
    bool done = false;
    rc = mv_staged(h, x, y, &done);
    if (done) return rc;
    if (rc == PWM_OK) rc = upload_vec(h, x, h->hx.p, h->noc);
    if (rc == PWM_OK) rc = spmv_launch(h, h->hx.p, h->hy.p, nullptr);
    if (rc == PWM_OK) rc = download_vec(h, h->hy.p, y, h->nor);
    return rc;
}

// ---------------------------------------------------------------- power method

static int power_workspace(pwm_matrix* h, int64_t max_it) {
    hipError_t e;
    if (!h->pw_ctrl.p && (e = h->pw_ctrl.alloc(64)) != hipSuccess) return hip_fail(h, e, "power workspace");
    const int64_t np = std::max<int64_t>(partials_needed(h), 1);
    if ((int64_t)h->pw_partials.bytes < np * 24 && (e = h->pw_partials.alloc(np * 24)) != hipSuccess)
        return hip_fail(h, e, "power workspace");
    if (h->pw_rec_cap < max_it) {
        if ((e = h->pw_rec.alloc(std::max<int64_t>(max_it, 1) * 32)) != hipSuccess)
            return hip_fail(h, e, "power workspace");
        h->pw_rec_cap = max_it;
    }
    return PWM_OK;
}

// Device workspace of one power method: step control (2 ints), one record
// of 4 doubles per step, 3 FP64 partial sums per partial slot.
struct PowerWs {
    int* ctrl;
    double* rec;
    double* partials;
};

// Runs the device power loop on buf0 (start vector) / buf1 with workspace ws
// (NULL: the handle's own, allocated on first use); returns steps done.
static int run_power(pwm_matrix* h, void* buf0, void* buf1, int64_t max_it, double tol, int64_t* steps,
                     double* lambda, double* ynorm, const PowerWs* ws = nullptr) {
    if (h->nor != h->noc) return fail(h, PWM_ERR_NOT_SQUARE, "power method needs a square matrix");
    if (max_it < 0) return fail(h, PWM_ERR_INVALID, "negative iteration count");
    if (max_it == 0) {
        if (steps) *steps = 0;
        return PWM_OK;
    }
    int rc;
    PowerWs own;
    if (!ws) {
        if ((rc = power_workspace(h, max_it)) != PWM_OK) return rc;
        own = PowerWs{h->pw_ctrl.as<int>(), h->pw_rec.as<double>(), h->pw_partials.as<double>()};
        ws = &own;
    }
    PowerArgs pw;
    pw.buf0 = buf0;
    pw.buf1 = buf1;
    pw.ctrl = ws->ctrl;
    pw.rec = ws->rec;
    pw.partials = ws->partials;
    pw.max_it = max_it;
    pw.tol = tol;
    pw.k = 0;
    const int64_t slots = partial_slots(h);
    pw.defer = tol < 0 && defers_norms(h);
    pw.prev = nullptr;
    pw.prev_n = 0;
    // what the loop leaves in ctrl: the step count, the done flag, and the
    // last step's lambda and |y|^2
    struct {
        int steps, done;
        double pad, lambda, yy;
    } out = {};
    static_assert(sizeof(out) == 32, "step control and result are read back as one record");
    hipError_t e = hipSuccess;
    auto read_back = [&] {
        e = hipMemcpyAsync(&out, ws->ctrl, sizeof(out), hipMemcpyDeviceToHost, h->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
        return e == hipSuccess;
    };
    // Steps issued between looks at the stop test (none: all at once).  A
    // small matrix runs its steps in one workgroup (k_power.hip), at most 4096
    // (a few ms) per launch, and leaves the vectors finished.
    const CrsDev small = small_crs_of(h);
    const int64_t chunk = h->power_small ? 4096 : tol < 0 ? max_it : 32;
    while (pw.k < max_it) {
        const int64_t end = std::min(max_it, pw.k + chunk);
        if (h->power_small) {
            e = pwmk::launch_power_small(small, h->stats.row_max, pw, pw.k, chunk, h->stream);
            if (e != hipSuccess) return hip_fail(h, e, "power loop");
            pw.k = end;
        }
        for (; pw.k < end; ++pw.k) {
            if ((rc = spmv_launch(h, nullptr, nullptr, &pw)) != PWM_OK) return rc;
            if (pw.defer) {
                pw.prev = pw.partials;
                pw.prev_n = slots;
                pw.partials = ws->partials + (pw.k & 1 ? 0 : 3 * slots);
            }
        }
        if (tol >= 0 && end < max_it) {
            if (!read_back()) return hip_fail(h, e, "power loop");
            if (out.done) break;
        }
    }
    if (pw.defer) {  // the last step's norms
        pw.k = max_it - 1;
        e = pwmk::launch_power_final(pw, pw.prev, slots, 1, h->stream);
        if (e != hipSuccess) return hip_fail(h, e, "power norms");
        pw.k = max_it;
    }
    if (!h->power_small) {
        e = pwmk::launch_power_finish(pw, h->nor, h->vtype == PWM_VALUES_F64, h->stream);
        if (e != hipSuccess) return hip_fail(h, e, "power finish");
    }
    if (!read_back()) return hip_fail(h, e, "power finish");
    if (steps) *steps = out.steps;
    if (lambda) *lambda = out.lambda;
    if (ynorm) *ynorm = sqrt(out.yy);
    return PWM_OK;
}

extern "C" int pwm_power_iteration(pwm_matrix* h, double* x, double* y, int64_t it) {
    if (!h) return fail(nullptr, PWM_ERR_INVALID, "pwm_power_iteration: NULL handle");
    if (!h->loaded) return fail(h, PWM_ERR_STATE, "pwm_power_iteration: no matrix loaded");
    if (!x || !y) return fail(h, PWM_ERR_INVALID, "pwm_power_iteration: NULL vector");
    if (h->nor != h->noc) return fail(h, PWM_ERR_NOT_SQUARE, "power method needs a square matrix");
    if (x < y + h->nor && y < x + h->nor) return fail(h, PWM_ERR_INVALID, "pwm_power_iteration: x and y overlap");
    if (it <= 0) return it < 0 ? fail(h, PWM_ERR_INVALID, "negative iteration count") : PWM_OK;
    int rc = stage_vectors(h);
    if (rc == PWM_OK) rc = upload_vec(h, x, h->hx.p, h->nor);
    int64_t steps = 0;
    if (rc == PWM_OK) rc = run_power(h, h->hx.p, h->hy.p, it, -1.0, &steps, nullptr, nullptr);
    if (rc == PWM_OK) rc = download_vec(h, h->hx.p, x, h->nor);
    if (rc == PWM_OK) rc = download_vec(h, h->hy.p, y, h->nor);
    return rc;
}

extern "C" int pwm_power_method_device(pwm_matrix* h, void* x, void* y, int64_t max_it, double tol, double* lambda,
                                       double* ynorm, int64_t* iterations) {
    if (!h) return fail(nullptr, PWM_ERR_INVALID, "pwm_power_method_device: NULL handle");
    if (!h->loaded) return fail(h, PWM_ERR_STATE, "pwm_power_method_device: no matrix loaded");
    if (!x || !y) return fail(h, PWM_ERR_INVALID, "pwm_power_method_device: NULL vector");
    const size_t vs = vector_size(h->vtype);
    if ((const char*)x < (const char*)y + h->nor * vs && (const char*)y < (const char*)x + h->nor * vs)
        return fail(h, PWM_ERR_INVALID, "pwm_power_method_device: x and y overlap");
    if (int rc0 = check_device_xy(h, x, h->nor, y, h->nor, "pwm_power_method_device")) return rc0;
    int64_t steps = 0;
    int rc = run_power(h, x, y, max_it, tol, &steps, lambda, ynorm);
    if (iterations) *iterations = steps;
    return rc;
}

// ---------------------------------------------------------------- row partitions

// TripletToMultipleCRS (Util/TripletToCRS.hpp:309-385) over the device CRS:
// partition p holds the rows [first_rows[p], first_rows[p] + thread_rows[p])
// with am_rows = nor / partitions rows each (integer division, :320) and the
// remainder in the last partition (:325-326).
static void row_partitions(int64_t nor, int partitions, std::vector<int64_t>& first, std::vector<int64_t>& rows) {
    first.assign(partitions, 0);
    rows.assign(partitions, 0);
    const int64_t am_rows = nor / partitions;
    int64_t last = 0;
    for (int p = 0; p < partitions; ++p) {
        first[p] = last;
        last = p == partitions - 1 ? nor : first[p] + am_rows;
        rows[p] = last - first[p];
    }
}

static int partition_args(pwm_matrix* h, int partitions, const char* who) {
    if (!h) return fail(nullptr, PWM_ERR_INVALID, std::string(who) + ": NULL handle");
    if (!h->loaded || !h->rs.p) return fail(h, PWM_ERR_STATE, std::string(who) + ": needs a loaded CRS or CRS_MERGE handle");
    if (partitions < 1) return fail(h, PWM_ERR_INVALID, std::string(who) + ": partitions must be at least 1");
    return PWM_OK;
}

extern "C" int pwm_crs_partitions(pwm_matrix* h, int partitions, int32_t* first_rows, int32_t* thread_rows,
                                  int64_t* part_nnz) {
    if (int rc = partition_args(h, partitions, "pwm_crs_partitions")) return rc;
    std::vector<int64_t> first, rows;
    row_partitions(h->nor, partitions, first, rows);
    for (int p = 0; p < partitions; ++p) {
        if (first_rows) first_rows[p] = (int32_t)first[p];
        if (thread_rows) thread_rows[p] = (int32_t)rows[p];
        if (part_nnz) {
            int32_t b[2] = {0, 0};
            hipError_t e = hipMemcpy(&b[0], h->rs.as<int32_t>() + first[p], 4, hipMemcpyDeviceToHost);
            if (e == hipSuccess) e = hipMemcpy(&b[1], h->rs.as<int32_t>() + first[p] + rows[p], 4, hipMemcpyDeviceToHost);
            if (e != hipSuccess) return hip_fail(h, e, "pwm_crs_partitions");
            part_nnz[p] = (int64_t)b[1] - b[0];
        }
    }
    return PWM_OK;
}

extern "C" int pwm_crs_partition_export(pwm_matrix* h, int partitions, int part, int32_t* row_start, int32_t* col_ind,
                                        double* values) {
    if (int rc = partition_args(h, partitions, "pwm_crs_partition_export")) return rc;
    if (part < 0 || part >= partitions || !row_start)
        return fail(h, PWM_ERR_INVALID, "pwm_crs_partition_export: bad partition or NULL row_start");
    std::vector<int64_t> first, rows;
    row_partitions(h->nor, partitions, first, rows);
    const int64_t f = first[part], n = rows[part];
    hipError_t e = hipMemcpy(row_start, h->rs.as<int32_t>() + f, (n + 1) * 4, hipMemcpyDeviceToHost);
    if (e != hipSuccess) return hip_fail(h, e, "pwm_crs_partition_export");
    const int32_t base = row_start[0];
    for (int64_t j = 0; j <= n; ++j) row_start[j] -= base;
    const int64_t nz = row_start[n];
    if (nz > 0 && (!col_ind || !values)) return fail(h, PWM_ERR_INVALID, "pwm_crs_partition_export: NULL arrays");
    if (nz > 0) {
        e = hipMemcpy(col_ind, h->ci.as<int32_t>() + base, nz * 4, hipMemcpyDeviceToHost);
        DevBuf tmp;
        if (e == hipSuccess) e = tmp.alloc(nz * 8);
        if (e == hipSuccess)
            e = pwmk::launch_copy_values_f64((const char*)h->val.p + (size_t)base * value_size(h->vtype), h->vtype,
                                             tmp.as<double>(), nz, h->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
        if (e == hipSuccess) e = hipMemcpy(values, tmp.p, nz * 8, hipMemcpyDeviceToHost);
        if (e != hipSuccess) return hip_fail(h, e, "pwm_crs_partition_export");
    }
    return PWM_OK;
}

// ---------------------------------------------------------------- no-allocation power method

// Workspace of pwm_power_method_device_noalloc: one fixed device array per
// GPU (each device holds its own copy until the process ends).  Layout:
// step control at 0, kNoAllocMaxIt step records (32 B) from 256, then the
// FP64 partial sums (24 B per slot) up to the end.
constexpr int64_t kNoAllocBytes = (int64_t)8 << 20;
constexpr int64_t kNoAllocMaxIt = 65536;
constexpr int64_t kNoAllocRecOff = 256;
constexpr int64_t kNoAllocPartOff = kNoAllocRecOff + 32 * kNoAllocMaxIt;
constexpr int64_t kNoAllocMaxSlots = (kNoAllocBytes - kNoAllocPartOff) / 24;
static_assert(PWM_NOALLOC_MAX_IT == kNoAllocMaxIt, "header and library disagree on the iteration limit");
static_assert(PWM_NOALLOC_MAX_SLOTS == kNoAllocMaxSlots, "header and library disagree on the slot limit");
static __device__ __align__(256) char scratch[kNoAllocBytes];

// Device address of `scratch` on the current device, looked up once per
// device with that device current (pwm_create does it for every device it
// runs on; the lookup loads the array onto the device).  The host-side name
// `scratch` is only a stand-in: host code passes this address to kernels,
// never the name.
static int noalloc_scratch(pwm_matrix* h, char** out) {
    static std::mutex mu;
    static std::vector<char*> addr;  // per device ordinal
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(h, e, "pwm_power_method_device_noalloc: hipGetDevice");
    std::lock_guard<std::mutex> lock(mu);
    if ((int)addr.size() <= dev) addr.resize(dev + 1, nullptr);
    if (!addr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            (void)hipGetLastError();
            return hip_fail(h, e != hipSuccess ? e : hipErrorInvalidSymbol,
                            "pwm_power_method_device_noalloc: workspace address");
        }
        addr[dev] = (char*)p;
    }
    *out = addr[dev];
    return PWM_OK;
}

extern "C" int pwm_power_method_device_noalloc(pwm_matrix* h, void* x, void* y, int64_t max_it, double tol,
                                               double* lambda, double* ynorm, int64_t* iterations) {
    if (!h) return fail(nullptr, PWM_ERR_INVALID, "pwm_power_method_device_noalloc: NULL handle");
    if (!h->loaded) return fail(h, PWM_ERR_STATE, "pwm_power_method_device_noalloc: no matrix loaded");
    if (!x || !y) return fail(h, PWM_ERR_INVALID, "pwm_power_method_device_noalloc: NULL vector");
    const size_t vs = vector_size(h->vtype);
    if ((const char*)x < (const char*)y + h->nor * vs && (const char*)y < (const char*)x + h->nor * vs)
        return fail(h, PWM_ERR_INVALID, "pwm_power_method_device_noalloc: x and y overlap");
    if (max_it > kNoAllocMaxIt)
        return fail(h, PWM_ERR_INVALID, "pwm_power_method_device_noalloc: max_it above " +
                                            std::to_string(kNoAllocMaxIt) + ", the workspace's step records");
    const int64_t slots = std::max<int64_t>(partials_needed(h), 1);
    if (slots > kNoAllocMaxSlots)
        return fail(h, PWM_ERR_INVALID, "pwm_power_method_device_noalloc: the matrix's plan needs " +
                                            std::to_string(slots) + " partial-sum slots, above the workspace's " +
                                            std::to_string(kNoAllocMaxSlots));
    if (int rc0 = check_device_xy(h, x, h->nor, y, h->nor, "pwm_power_method_device_noalloc")) return rc0;
    char* base = nullptr;
    if (int rc0 = noalloc_scratch(h, &base)) return rc0;
    // the first step ignores the step control that another call left; records
    // and partial sums are written before they are read
    const PowerWs ws{(int*)base, (double*)(base + kNoAllocRecOff), (double*)(base + kNoAllocPartOff)};
    int64_t steps = 0;
    int rc = run_power(h, x, y, max_it, tol, &steps, lambda, ynorm, &ws);
    if (iterations) *iterations = steps;
    return rc;
}

// ---------------------------------------------------------------- exports

extern "C" int pwm_merge_splits(pwm_matrix* h, int64_t* P, int64_t* a, int64_t* b) {
    if (!h || !P) return fail(h, PWM_ERR_INVALID, "pwm_merge_splits: NULL argument");
    if (h->format != PWM_FORMAT_CRS_MERGE || !h->loaded)
        return fail(h, PWM_ERR_STATE, "pwm_merge_splits: not a loaded CRS_MERGE handle");
    *P = h->mp.P;
    if (!a || !b) return PWM_OK;
    hipError_t e = hipMemcpy(a, h->split_a.p, (h->mp.P + 1) * 8, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(b, h->split_b.p, (h->mp.P + 1) * 8, hipMemcpyDeviceToHost);
    if (e != hipSuccess) return hip_fail(h, e, "pwm_merge_splits");
    return PWM_OK;
}

extern "C" int pwm_crs_export(pwm_matrix* h, int32_t* row_start, int32_t* col_ind, double* values) {
    if (!h || !row_start || !col_ind || !values) return fail(h, PWM_ERR_INVALID, "pwm_crs_export: NULL argument");
    if (!h->loaded || !h->rs.p) return fail(h, PWM_ERR_STATE, "pwm_crs_export: no CRS arrays on the device");
    hipError_t e = hipMemcpy(row_start, h->rs.p, (h->nor + 1) * 4, hipMemcpyDeviceToHost);
    if (e == hipSuccess && h->nnz) e = hipMemcpy(col_ind, h->ci.p, h->nnz * 4, hipMemcpyDeviceToHost);
    if (e == hipSuccess && h->nnz) {
        DevBuf tmp;
        e = tmp.alloc(h->nnz * 8);
        if (e == hipSuccess) e = pwmk::launch_copy_values_f64(h->val.p, h->vtype, tmp.as<double>(), h->nnz, h->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
        if (e == hipSuccess) e = hipMemcpy(values, tmp.p, h->nnz * 8, hipMemcpyDeviceToHost);
    }
    if (e != hipSuccess) return hip_fail(h, e, "pwm_crs_export");
    return PWM_OK;
}

// ---------------------------------------------------------------- device helpers

extern "C" int pwm_device_alloc(size_t bytes, void** ptr) {
    if (!ptr) return fail(nullptr, PWM_ERR_INVALID, "pwm_device_alloc: NULL out");
    hipError_t e = hipMalloc(ptr, bytes ? bytes : 1);
    if (e != hipSuccess) return hip_fail(nullptr, e, "pwm_device_alloc");
    return PWM_OK;
}
extern "C" int pwm_device_free(void* ptr) {
    if (ptr) {
        hipError_t e = hipFree(ptr);
        if (e != hipSuccess) return hip_fail(nullptr, e, "pwm_device_free");
    }
    return PWM_OK;
}
extern "C" int pwm_memcpy_h2d(void* dst, const void* src, size_t bytes) {
    hipError_t e = hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice);
    return e == hipSuccess ? PWM_OK : hip_fail(nullptr, e, "pwm_memcpy_h2d");
}
extern "C" int pwm_memcpy_d2h(void* dst, const void* src, size_t bytes) {
    hipError_t e = hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
    return e == hipSuccess ? PWM_OK : hip_fail(nullptr, e, "pwm_memcpy_d2h");
}
extern "C" int pwm_device_synchronize(void) {
    hipError_t e = hipDeviceSynchronize();
    return e == hipSuccess ? PWM_OK : hip_fail(nullptr, e, "pwm_device_synchronize");
}
extern "C" int pwm_device_fill(void* ptr, int64_t n, int is_f64, double value) {
    hipError_t e = pwmk::launch_fill(ptr, n, is_f64, value, nullptr);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    return e == hipSuccess ? PWM_OK : hip_fail(nullptr, e, "pwm_device_fill");
}

extern "C" int pwm_device_copy(void* dst, const void* src, int64_t bytes) {
    if (!dst || !src || bytes < 0 || bytes % 16) return fail(nullptr, PWM_ERR_INVALID, "pwm_device_copy: bad argument");
    hipError_t e = pwmk::launch_stream_copy(dst, src, bytes, nullptr);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    return e == hipSuccess ? PWM_OK : hip_fail(nullptr, e, "pwm_device_copy");
}

// ---------------------------------------------------------------- timing

extern "C" int pwm_gather_rate(const void* x_dev, int64_t x_len, int64_t window, int per_xcd, int64_t n,
                               double* ms) {
    const int kind = (per_xcd >> 8) & 0xff;
    if (kind != 0 && (kind < 1 || (kind > 4 && kind < 17) || kind > 20 || window * 8 > INT32_MAX))
        return fail(nullptr, PWM_ERR_INVALID, "pwm_gather_rate: unknown gather load kind (or window over 2 GB)");
    if (!ms || window < 0 || window > UINT32_MAX ||
        (window > 0 && (!x_dev || ((per_xcd & 1) ? 8 * window : window) > x_len)))
        return fail(nullptr, PWM_ERR_INVALID, "pwm_gather_rate: window must fit x (8 windows when per_xcd)");
    const int64_t m = pwmk::gather_probe_entries(n);
    if (m <= 0) return fail(nullptr, PWM_ERR_INVALID, "pwm_gather_rate: n must be at least 8192");
    DevBuf idx, val, out;
    hipError_t e;
    if ((e = idx.alloc(m * 4)) != hipSuccess || (e = val.alloc(m * 8)) != hipSuccess ||
        (e = out.alloc(m / 8192 * 256 * 8)) != hipSuccess)
        return hip_fail(nullptr, e, "pwm_gather_rate buffers");
    e = pwmk::launch_gather_fill(idx.as<uint32_t>(), val.as<double>(), m, (uint32_t)std::max<int64_t>(window, 1), nullptr);
    hipEvent_t a = nullptr, b = nullptr;
    if (e == hipSuccess) e = hipEventCreate(&a);
    if (e == hipSuccess) e = hipEventCreate(&b);
    const double* x = (const double*)x_dev;
    for (int r = 0; r < 2 && e == hipSuccess; ++r)
        e = pwmk::launch_gather_probe(idx.as<uint32_t>(), val.as<double>(), x, out.as<double>(), m, window, per_xcd, nullptr);
    if (e == hipSuccess) e = hipEventRecord(a, nullptr);
    for (int r = 0; r < 10 && e == hipSuccess; ++r)
        e = pwmk::launch_gather_probe(idx.as<uint32_t>(), val.as<double>(), x, out.as<double>(), m, window, per_xcd, nullptr);
    if (e == hipSuccess) e = hipEventRecord(b, nullptr);
    if (e == hipSuccess) e = hipEventSynchronize(b);
    float t = 0.0f;
    if (e == hipSuccess) e = hipEventElapsedTime(&t, a, b);
    if (a) (void)hipEventDestroy(a);
    if (b) (void)hipEventDestroy(b);
    if (e != hipSuccess) return hip_fail(nullptr, e, "pwm_gather_rate");
    *ms = t / 10.0;
    return PWM_OK;
}

// One SpMV of h on h->stream with `mid` recorded after its dominant kernel
// (the tiles / vector / merge / CSB slab kernel; the whole SpMV for BlockCOH).
static int launch_marked(pwm_matrix* h, const void* x, void* y, hipEvent_t mid) {
    const CrsDev A = crs_of(h);
    hipError_t e = hipSuccess;
    switch (swept_crs(h) ? PWM_FORMAT_CSB : h->format) {
        case PWM_FORMAT_CRS:
            if (h->crs_used == 3) {
                e = pwmk::launch_rows(A, h->rp, x, y, nullptr, h->stream);
                (void)hipEventRecord(mid, h->stream);
                break;
            }
            if (h->crs_used == 2) {
                e = pwmk::launch_tiles_spmv(A, h->tiles.as<pwmk::ETile>(), h->mp, x, y, nullptr, h->stream);
                (void)hipEventRecord(mid, h->stream);
                if (e == hipSuccess && h->tiles_carry) e = pwmk::launch_merge_fixup(A, h->mp, y, nullptr, h->stream);
                break;
            }
            e = pwmk::launch_crs_vector(A, h->group, h->vec_blocks, h->lr, x, y, nullptr, h->stream);
            (void)hipEventRecord(mid, h->stream);
            if (e == hipSuccess && h->lr.n_rows > 0)
                e = pwmk::launch_crs_finalize(A, h->vec_blocks, h->lr, y, nullptr, h->stream);
            break;
        case PWM_FORMAT_CRS_MERGE:
            if (h->crs_used == 3) {
                e = pwmk::launch_rows(A, h->rp, x, y, nullptr, h->stream);
                (void)hipEventRecord(mid, h->stream);
                break;
            }
            e = pwmk::launch_merge_spmv(A, h->mp, x, y, nullptr, h->stream);
            (void)hipEventRecord(mid, h->stream);
            if (e == hipSuccess) e = pwmk::launch_merge_fixup(A, h->mp, y, nullptr, h->stream);
            break;
        case PWM_FORMAT_CSB:
            e = csb_launch(h, x, y, nullptr, 1);
            (void)hipEventRecord(mid, h->stream);
            if (e == hipSuccess) e = csb_launch(h, x, y, nullptr, 2);
            break;
        default: {
            const int rc = spmv_launch(h, x, y, nullptr);
            (void)hipEventRecord(mid, h->stream);
            return rc;
        }
    }
    if (e != hipSuccess) return hip_fail(h, e, "timed SpMV");
    return PWM_OK;
}

extern "C" int pwm_time_mv(pwm_matrix* h, const void* x, void* y, int reps, int64_t flush_bytes, double* ms_per_mv,
                           double* kernel_ms) {
    if (!h || !x || !y || reps <= 0) return fail(h, PWM_ERR_INVALID, "pwm_time_mv: bad argument");
    if (!h->loaded) return fail(h, PWM_ERR_STATE, "pwm_time_mv: no matrix loaded");
    if (int rc0 = check_device_xy(h, x, h->noc, y, h->nor, "pwm_time_mv")) return rc0;
    hipError_t e;
    if (flush_bytes > 0 && (int64_t)h->flush.bytes < flush_bytes && (e = h->flush.alloc(flush_bytes)) != hipSuccess)
        return hip_fail(h, e, "flush buffer");
    int rc = PWM_OK;
    if (!kernel_ms && flush_bytes <= 0) {
        // back-to-back SpMVs (the pwm_mv_device launch sequence) between one
        // pair of events: no markers between the steps
        hipEvent_t e0 = nullptr, e1 = nullptr;
        if ((e = hipEventCreate(&e0)) != hipSuccess || (e = hipEventCreate(&e1)) != hipSuccess) {
            if (e0) (void)hipEventDestroy(e0);
            return hip_fail(h, e, "event create");
        }
        (void)hipEventRecord(e0, h->stream);
        for (int r = 0; r < reps && rc == PWM_OK; ++r) rc = spmv_launch(h, x, y, nullptr);
        (void)hipEventRecord(e1, h->stream);
        e = hipStreamSynchronize(h->stream);
        if (rc == PWM_OK && e != hipSuccess) rc = hip_fail(h, e, "timed SpMV");
        float t = 0;
        if (rc == PWM_OK) (void)hipEventElapsedTime(&t, e0, e1);
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        if (rc == PWM_OK && ms_per_mv) *ms_per_mv = t / reps;
        return rc;
    }
    std::vector<hipEvent_t> ev(3 * reps);
    for (auto& v : ev)
        if ((e = hipEventCreate(&v)) != hipSuccess) return hip_fail(h, e, "event create");
    for (int r = 0; r < reps && rc == PWM_OK; ++r) {
        if (flush_bytes > 0) (void)pwmk::launch_flush(h->flush.p, flush_bytes, h->stream);
        (void)hipEventRecord(ev[3 * r], h->stream);
        rc = launch_marked(h, x, y, ev[3 * r + 1]);
        (void)hipEventRecord(ev[3 * r + 2], h->stream);
    }
    e = hipStreamSynchronize(h->stream);
    if (rc == PWM_OK && e != hipSuccess) rc = hip_fail(h, e, "timed SpMV");
    double tot = 0, ker = 0;
    for (int r = 0; r < reps && rc == PWM_OK; ++r) {
        float a = 0, b = 0;
        (void)hipEventElapsedTime(&a, ev[3 * r], ev[3 * r + 2]);
        (void)hipEventElapsedTime(&b, ev[3 * r], ev[3 * r + 1]);
        tot += a;
        ker += b;
    }
    for (auto& v : ev) (void)hipEventDestroy(v);
    if (rc != PWM_OK) return rc;
    if (ms_per_mv) *ms_per_mv = tot / reps;
    if (kernel_ms) *kernel_ms = ker / reps;
    return PWM_OK;
}

// SpMVs of `count` handles in turn, reps rounds, all on the first handle's
// stream: with count independent matrices whose arrays together exceed the
// 256 MB Infinity Cache, every SpMV reads its matrix from HBM, back to back.
extern "C" int pwm_time_mv_rotating(pwm_matrix* const* hs, const void* const* xs, void* const* ys, int count,
                                    int reps, double* ms_per_mv, double* kernel_ms) {
    if (!hs || !xs || !ys || count <= 0 || reps <= 0)
        return fail(nullptr, PWM_ERR_INVALID, "pwm_time_mv_rotating: bad argument");
    for (int k = 0; k < count; ++k) {
        pwm_matrix* h = hs[k];
        if (!h) return fail(nullptr, PWM_ERR_INVALID, "pwm_time_mv_rotating: NULL handle");
        if (!h->loaded) return fail(h, PWM_ERR_STATE, "pwm_time_mv_rotating: no matrix loaded");
        if (!xs[k] || !ys[k]) return fail(h, PWM_ERR_INVALID, "pwm_time_mv_rotating: NULL vector");
        if (int rc0 = check_device_xy(h, xs[k], h->noc, ys[k], h->nor, "pwm_time_mv_rotating")) return rc0;
    }
    pwm_matrix* h0 = hs[0];
    const hipStream_t s = h0->stream;
    // work still queued on a handle's own stream finishes before its SpMVs
    // run on the first handle's stream
    for (int k = 1; k < count; ++k) {
        const hipError_t es = hipStreamSynchronize(hs[k]->stream);
        if (es != hipSuccess) return hip_fail(hs[k], es, "pwm_time_mv_rotating");
    }
    std::vector<hipStream_t> saved(count);
    for (int k = 0; k < count; ++k) {
        saved[k] = hs[k]->stream;
        hs[k]->stream = s;
    }
    const int n = count * reps;
    std::vector<hipEvent_t> ev(kernel_ms ? 3 * n : 2, nullptr);
    int rc = PWM_OK;
    hipError_t e = hipSuccess;
    for (auto& v : ev)
        if (e == hipSuccess) e = hipEventCreate(&v);
    if (e != hipSuccess) rc = hip_fail(h0, e, "event create");
    if (rc == PWM_OK && !kernel_ms) {
        (void)hipEventRecord(ev[0], s);
        for (int i = 0; i < n && rc == PWM_OK; ++i) rc = spmv_launch(hs[i % count], xs[i % count], ys[i % count], nullptr);
        (void)hipEventRecord(ev[1], s);
    } else if (rc == PWM_OK) {
        for (int i = 0; i < n && rc == PWM_OK; ++i) {
            (void)hipEventRecord(ev[3 * i], s);
            rc = launch_marked(hs[i % count], xs[i % count], ys[i % count], ev[3 * i + 1]);
            (void)hipEventRecord(ev[3 * i + 2], s);
        }
    }
    e = hipStreamSynchronize(s);
    if (rc == PWM_OK && e != hipSuccess) rc = hip_fail(h0, e, "timed SpMV");
    for (int k = count - 1; k >= 0; --k) hs[k]->stream = saved[k];  // reverse order: a handle may repeat
    if (rc == PWM_OK) {
        double tot = 0, ker = 0;
        if (!kernel_ms) {
            float t = 0;
            (void)hipEventElapsedTime(&t, ev[0], ev[1]);
            tot = t;
        } else {
            for (int i = 0; i < n; ++i) {
                float a = 0, b = 0;
                (void)hipEventElapsedTime(&a, ev[3 * i], ev[3 * i + 2]);
                (void)hipEventElapsedTime(&b, ev[3 * i], ev[3 * i + 1]);
                tot += a;
                ker += b;
            }
            *kernel_ms = ker / n;
        }
        if (ms_per_mv) *ms_per_mv = tot / n;
    }
    for (auto& v : ev)
        if (v) (void)hipEventDestroy(v);
    return rc;
}
