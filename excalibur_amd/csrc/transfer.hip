// Host <-> device transfers of the library: pinned staging, helper threads for the host side of a copy, and a bounded pool of
// pinned host blocks that results are read into.
//
// What bounds a transfer is the link (56 GB/s each way, measured) as long as nothing else is on the way: handing the HIP
// runtime pageable memory moves 17 GB/s to the host and 27-36 GB/s to the device, one core copies 30 GB/s, and a fresh
// pageable buffer costs 14 GB/s in page faults. So large copies go through pinned chunks of 4 MiB, the host side of a chunk is
// copied by several threads (70 GB/s with six) while the previous chunk is on the link, and small ones are one kernel that
// reads or writes the pinned memory itself (no copy engine, no hand-over between queues: 15 instead of 19 us for 75 KB with
// the kernel behind it; 6 instead of 11 us for a result the host polls for instead of waiting on the stream).
//
// Uploads of every size from pageable memory to a destination on 16 bytes are kernels that read the pinned memory: the copy engine leaves the link idle for some 15 us between two
// copies, a kernel for 3, so an upload can begin with a small piece and needs no hand-over to the kernels behind it (16 groups: 54
// GB/s in launches of 4 MiB, 48 in 1 MiB; the engine 50 and 38; 64 groups 53 and 41). Until everything is there: 4.9 MB 147 -> 130
// us, 19 MB 480 -> 416, 79 MB 1755 -> 1562. Two kinds stay with the engine, in whole chunks: sources in the pinned pool of results, and above
// 256 KiB destinations off 16 bytes, which a kernel would write byte by byte (4.9 MB 138 us, 148 in pieces that grow; 20 MB 465 and 480; 83 MB 1814 and 1800).
#include <string.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <map>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "common.h"

namespace {

constexpr size_t kChunk = (size_t)4 << 20;       // staging chunk, the longest piece on the link
constexpr size_t kPiece = (size_t)128 << 10;     // what one thread copies at a time
constexpr size_t kStep = (size_t)512 << 10;      // what the first launch of an upload takes
constexpr unsigned kUploadGroups = 16;
constexpr size_t kUploadKernel = (size_t)256 << 10;   // small uploads; results up to here leave without staging
constexpr size_t kSmallRing = (size_t)512 << 10;      // small uploads turn in this much of each chunk, so that the GPU's translations of it stay
                                                      // cached (75 KB from pages not seen lately take the kernel 31 us)
constexpr size_t kDownloadKernel = (size_t)64 << 10;  // up to here one group writes the host's memory and a flag
constexpr int kSmallThreads = 1024;

// ---- helper threads: copy pieces of one transfer at a time beside the thread that asked for it ----
// The asking thread claims pieces too and waits for claimed pieces only, so a copy ends whether or not a helper ever runs
// (helpers do not exist in a forked child). A helper that finds nothing to copy looks out for kLookOut, which bridges the wait for a
// transfer's next chunk, and sleeps then, so that nobody spins while a result's kernels run (spinning for the whole transfer took 1.7 s
// of processor time for a result that came over 0.43 s, now 0.02; 5 MB transfers in a row keep 3.2 cores busy, not 4.3, at the same 33 and
// 30 GB/s; 200 us move no more). The object is never destroyed: its threads sleep until the process ends.
class copy_crew {
public:
    static copy_crew& get() {
        static copy_crew* crew = new copy_crew();
        return *crew;
    }
    // A session has the helpers to itself over the chunks of one transfer. Another thread's transfer copies alone meanwhile: with
    // the helpers dealt out to both under a lock, two 80 MB transfers at once moved 23 GB/s each instead of 31.
    class session {
    public:
        explicit session(bool wanted) : crew_(get()), lock_(crew_.busy_, std::defer_lock) {
            if (wanted && crew_.helpers_ > 0 && lock_.try_lock()) {
                std::lock_guard<std::mutex> g(crew_.m_);
                crew_.start();
            }
        }
        void copy(void* dst, const void* src, size_t bytes) {
            if (!lock_.owns_lock() || bytes < 2 * kPiece) memcpy(dst, src, bytes);
            else crew_.copy(static_cast<char*>(dst), static_cast<const char*>(src), bytes);
        }

    private:
        copy_crew& crew_;
        std::unique_lock<std::mutex> lock_;
    };

private:
    struct piece {
        char* dst;
        const char* src;
        size_t bytes;
    };
    static constexpr auto kLookOut = std::chrono::microseconds(50);
    static constexpr unsigned kRing = 64;  // more than the pieces of one copy() call, which waits for all of them

    copy_crew() {
        const unsigned cores = std::thread::hardware_concurrency();
        helpers_ = cores >= 4 ? (int)(cores / 2 < 5 ? cores / 2 : 5) : 0;  // six threads in all reach the memory's rate
    }
    void start() {
        try {
            for (; started_ < helpers_; ++started_) std::thread([this] { help(); }).detach();
        } catch (...) {  // the process may have no more threads: those there are will do
            helpers_ = started_;
        }
    }
    bool take_one() {
        unsigned long long n = next_.load(std::memory_order_acquire);
        while (n < published_.load(std::memory_order_acquire)) {
            if (next_.compare_exchange_weak(n, n + 1, std::memory_order_acq_rel)) {
                const piece p = ring_[n % kRing];
                memcpy(p.dst, p.src, p.bytes);
                done_.fetch_add(1, std::memory_order_acq_rel);
                return true;
            }
        }
        return false;
    }
    void help() {
        for (;;) {
            {
                std::unique_lock<std::mutex> g(m_);
                ++sleeping_;
                cv_.wait(g, [this] { return next_.load() < published_.load(); });
                --sleeping_;
            }
            auto last = std::chrono::steady_clock::now();
            for (;;) {
                bool worked = false;
                while (take_one()) worked = true;
                const auto now = std::chrono::steady_clock::now();
                if (worked) last = now;
                else if (now - last > kLookOut) break;
                for (int i = 0; i < 8; ++i) __builtin_ia32_pause();
            }
        }
    }
    void copy(char* dst, const char* src, size_t bytes) {
        while (bytes) {
            const size_t now = bytes < kPiece * (kRing / 2) ? bytes : kPiece * (kRing / 2);
            unsigned long long at = published_.load(std::memory_order_relaxed);
            for (size_t o = 0; o < now; o += kPiece) ring_[at++ % kRing] = {dst + o, src + o, now - o < kPiece ? now - o : kPiece};
            published_.store(at);  // (before sleeping_ is read: a helper counts itself there before it looks for work the last time)
            if (sleeping_.load() > 0) {
                { std::lock_guard<std::mutex> g(m_); }
                cv_.notify_all();
            }
            while (take_one()) {}
            while (done_.load(std::memory_order_acquire) < at) __builtin_ia32_pause();
            dst += now;
            src += now;
            bytes -= now;
        }
    }

    std::mutex busy_, m_;
    std::condition_variable cv_;
    std::atomic<int> sleeping_{0};
    std::atomic<unsigned long long> published_{0}, next_{0}, done_{0};
    piece ring_[kRing];
    int helpers_ = 0, started_ = 0;
};

// ---- pinned memory: chunks for staging and blocks for results, cached for the process ----
std::mutex g_pinned_mu;
std::vector<void*> g_chunks;                      // idle staging chunks
constexpr size_t kIdleChunks = 16;
struct block_info { size_t bytes; };
std::map<char*, block_info> g_blocks;             // every result block, by address
std::multimap<size_t, char*> g_idle_blocks;       // those nobody holds, by size
size_t g_block_bytes = 0;                         // bytes of all result blocks
constexpr size_t kBlockLimit = (size_t)1 << 30;   // at most this much; callers beyond it get pageable memory
constexpr size_t kIdleBlockLimit = (size_t)512 << 20;
size_t g_idle_block_bytes = 0;

void* take_chunk() {
    {
        std::lock_guard<std::mutex> g(g_pinned_mu);
        if (!g_chunks.empty()) {
            void* p = g_chunks.back();
            g_chunks.pop_back();
            return p;
        }
    }
    void* p = nullptr;
    if (hipHostMalloc(&p, kChunk, 0) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return p;
}

void give_chunk(void* p) {
    if (!p) return;
    {
        std::lock_guard<std::mutex> g(g_pinned_mu);
        if (g_chunks.size() < kIdleChunks) {
            g_chunks.push_back(p);
            return;
        }
    }
    (void)hipHostFree(p);
}

bool is_result_block(const void* p, size_t bytes) {
    std::lock_guard<std::mutex> g(g_pinned_mu);
    auto it = g_blocks.upper_bound(static_cast<char*>(const_cast<void*>(p)));
    if (it == g_blocks.begin()) return false;
    --it;
    return static_cast<const char*>(p) + bytes <= it->first + it->second.bytes;
}

// One group or a few copy `bytes` between device memory and pinned host memory. Bound by the link's latency and rate.
__global__ void __launch_bounds__(256) upload_kernel(const char* __restrict__ src, char* __restrict__ dst, unsigned bytes, int wide) {
    const unsigned stride = gridDim.x * blockDim.x;
    unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (wide) {
        const unsigned n = bytes / 16;
        const uint4* const from = reinterpret_cast<const uint4*>(src);
        uint4* const to = reinterpret_cast<uint4*>(dst);
        unsigned k = i;
        for (; k + 3 * stride < n; k += 4 * stride) {
            const uint4 a = from[k], b = from[k + stride], c = from[k + 2 * stride], d = from[k + 3 * stride];
            to[k] = a;
            to[k + stride] = b;
            to[k + 2 * stride] = c;
            to[k + 3 * stride] = d;
        }
        for (; k < n; k += stride) to[k] = from[k];
        for (unsigned b = n * 16 + i; b < bytes; b += stride) dst[b] = src[b];
    } else {
        for (; i < bytes; i += stride) dst[i] = src[i];
    }
}

__global__ void __launch_bounds__(kSmallThreads) download_kernel(const char* __restrict__ src, char* __restrict__ dst, unsigned bytes, int wide,
                                                                 unsigned* flag, unsigned value) {
    if (wide) {
        const unsigned n = bytes / 16;
        for (unsigned k = threadIdx.x; k < n; k += kSmallThreads) reinterpret_cast<uint4*>(dst)[k] = reinterpret_cast<const uint4*>(src)[k];
        for (unsigned k = n * 16 + threadIdx.x; k < bytes; k += kSmallThreads) dst[k] = src[k];
    } else {
        for (unsigned k = threadIdx.x; k < bytes; k += kSmallThreads) dst[k] = src[k];
    }
    __threadfence_system();  // every thread's bytes are in host memory before the flag
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(flag, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

int is_wide(const void* a, const void* b) { return ((uintptr_t)a | (uintptr_t)b) % 16 == 0; }

void release(exhip_staging* s) {
    for (int i = 0; i < exhip_staging::kChunks; ++i) {
        give_chunk(s->chunk[i]);
        if (s->event[i]) (void)hipEventDestroy((hipEvent_t)s->event[i]);
    }
    delete s;
}

// One copy's staging: the pool's last returned one (a thread that copies alone meets the same chunks again and again) or a new
// one, NULL where the host has no memory for it. More than the pool keeps are only there while as many copies run; `reader` is
// the stream whose queued work may still read the chunks when the loan ends.
class staging_loan {
public:
    explicit staging_loan(exhip_staging_pool& pool, hipStream_t reader = nullptr) : pool_(pool), reader_(reader) {
        std::lock_guard<std::mutex> g(pool_.mu);
        staging = pool_.n_idle > 0 ? pool_.idle[--pool_.n_idle] : new (std::nothrow) exhip_staging();
    }
    ~staging_loan() {
        if (!staging) return;
        {
            std::lock_guard<std::mutex> g(pool_.mu);
            if (pool_.n_idle < exhip_staging_pool::kIdle) {
                pool_.idle[pool_.n_idle++] = staging;
                return;
            }
        }
        if (reader_) (void)hipStreamSynchronize(reader_);
        release(staging);
    }
    staging_loan(const staging_loan&) = delete;
    staging_loan& operator=(const staging_loan&) = delete;
    exhip_staging* staging;

private:
    exhip_staging_pool& pool_;
    const hipStream_t reader_;
};

// Moves on to the next upload chunk (allocating it the first time round) and waits until its last readers are done.
int next_chunk(exhip_ctx* ctx, exhip_staging& s) {
    if (s.at >= 0 && s.used) {
        EXHIP_CHECK(hipEventRecord((hipEvent_t)s.event[s.at], ctx->stream));
        s.pending[s.at] = true;
    }
    s.at = (s.at + 1) % exhip_staging::kChunks;
    s.used = 0;
    if (!s.chunk[s.at]) {
        s.chunk[s.at] = take_chunk();
        if (!s.chunk[s.at]) return EXHIP_ERR_UNSUPPORTED;
        hipEvent_t e;
        EXHIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        s.event[s.at] = e;
    }
    if (s.pending[s.at]) {
        EXHIP_CHECK(hipEventSynchronize((hipEvent_t)s.event[s.at]));
        s.pending[s.at] = false;
    }
    return 0;
}

}  // namespace

// Copies src to the device on the context's stream and returns as soon as src has been read: what is queued on the stream
// afterwards finds the bytes, other streams have to wait for this one.
extern "C" int exhip_upload(exhip_ctx* ctx, void* dst, const void* src, size_t bytes) {
    EXHIP_REQUIRE(ctx && ((dst && src) || !bytes), "exhip_upload: NULL argument");
    const char* from = static_cast<const char*>(src);
    char* to = static_cast<char*>(dst);
    if (!bytes) return 0;
    if (is_result_block(src, bytes)) {  // pinned already: straight to the copy engine, which has to be done with it before the caller is
        EXHIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
        EXHIP_CHECK(hipStreamSynchronize(ctx->stream));
        return 0;
    }
    staging_loan loan(ctx->up, ctx->stream);
    EXHIP_REQUIRE(loan.staging, "exhip_upload: no host memory");
    exhip_staging& s = *loan.staging;
    const bool small = bytes <= kUploadKernel, kernels = small || is_wide(to, to);
    copy_crew::session crew(bytes >= 2 * kStep);
    for (size_t done = 0; bytes;) {
        // kernels: as much again as is on its way, so that the link starts early and later launches are long
        const size_t step = !kernels ? kChunk : done < kStep ? kStep : done < kChunk ? done : kChunk, now = bytes < step ? bytes : step;
        if (s.at < 0 || s.used + now > (small ? kSmallRing : kChunk)) {
            const int rc = next_chunk(ctx, s);
            if (rc == EXHIP_ERR_UNSUPPORTED) {  // no pinned memory left: the runtime's own way
                EXHIP_CHECK(hipMemcpyAsync(to, from, bytes, hipMemcpyHostToDevice, ctx->stream));
                EXHIP_CHECK(hipStreamSynchronize(ctx->stream));
                s.at = -1;
                s.used = 0;
                return 0;
            }
            if (rc != 0) return rc;
        }
        char* stage = static_cast<char*>(s.chunk[s.at]) + s.used;
        crew.copy(stage, from, now);
        if (kernels) {
            const unsigned groups = (unsigned)((now + 4095) / 4096), most = small ? 64 : kUploadGroups;
            upload_kernel<<<groups < most ? groups : most, 256, 0, ctx->stream>>>(stage, to, (unsigned)now, is_wide(stage, to));
            EXHIP_LAUNCH_CHECK();
        } else {  // a destination off 16 bytes would be written byte by byte
            EXHIP_CHECK(hipMemcpyAsync(to, stage, now, hipMemcpyHostToDevice, ctx->stream));
        }
        s.used += (now + 255) / 256 * 256;
        from += now;
        to += now;
        done += now;
        bytes -= now;
    }
    return 0;
}

extern "C" int exhip_memcpy_h2d(exhip_ctx* ctx, void* dst, const void* src, size_t bytes) {
    EXHIP_REQUIRE(ctx && ((dst && src) || !bytes), "exhip_memcpy_h2d: NULL argument");
    if (!bytes) return 0;
    const int rc = exhip_upload(ctx, dst, src, bytes);
    if (rc != 0) return rc;
    EXHIP_CHECK(hipStreamSynchronize(ctx->stream));  // readers on other streams find the bytes too
    return 0;
}

extern "C" int exhip_mark(exhip_ctx* ctx, void** mark) {
    EXHIP_REQUIRE(ctx && mark, "exhip_mark: NULL argument");
    if (!*mark) {
        hipEvent_t e;
        EXHIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        *mark = (void*)e;
    }
    EXHIP_CHECK(hipEventRecord((hipEvent_t)*mark, ctx->stream));
    return 0;
}

extern "C" int exhip_mark_destroy(void* mark) {
    if (mark) EXHIP_CHECK(hipEventDestroy((hipEvent_t)mark));
    return 0;
}

// Everything but small results: through pinned chunks, or straight into a pinned block.
static int download_through(exhip_staging& s, hipStream_t stream, void* dst, const void* src, size_t bytes) {
    auto chunk = [&](int i) {
        if (!s.chunk[i]) s.chunk[i] = take_chunk();
        return static_cast<char*>(s.chunk[i]);
    };
    if (is_result_block(dst, bytes) || bytes <= kUploadKernel || !chunk(0) || !chunk(1)) {
        EXHIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream));
        EXHIP_CHECK(hipStreamSynchronize(stream));
        return 0;
    }
    int chunks = 2;
    while (chunks < exhip_staging::kChunks && (size_t)chunks * kChunk < bytes && chunk(chunks)) ++chunks;
    for (int i = 0; i < chunks; ++i)
        if (!s.event[i]) {
            hipEvent_t e;
            EXHIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
            s.event[i] = e;
        }
    copy_crew::session crew(bytes >= 4 * kStep);
    const size_t total = (bytes + kChunk - 1) / kChunk;
    auto request = [&](size_t i) -> int {
        const size_t o = i * kChunk, n = bytes - o < kChunk ? bytes - o : kChunk;
        EXHIP_CHECK(hipMemcpyAsync(s.chunk[i % chunks], static_cast<const char*>(src) + o, n, hipMemcpyDeviceToHost, stream));
        EXHIP_CHECK(hipEventRecord((hipEvent_t)s.event[i % chunks], stream));
        return 0;
    };
    for (size_t i = 0; i < total && i < (size_t)chunks; ++i)
        if (const int rc = request(i)) return rc;
    for (size_t i = 0; i < total; ++i) {
        const size_t o = i * kChunk, n = bytes - o < kChunk ? bytes - o : kChunk;
        EXHIP_CHECK(hipEventSynchronize((hipEvent_t)s.event[i % chunks]));
        crew.copy(static_cast<char*>(dst) + o, s.chunk[i % chunks], n);
        if (i + chunks < total)
            if (const int rc = request(i + chunks)) return rc;
    }
    return 0;
}

static int download(exhip_ctx* ctx, hipStream_t stream, void* dst, const void* src, size_t bytes) {
    staging_loan loan(ctx->down);
    EXHIP_REQUIRE(loan.staging, "download: no host memory");
    const int rc = download_through(*loan.staging, stream, dst, src, bytes);
    if (rc != 0) (void)hipStreamSynchronize(stream);  // requests may still be writing to its chunks
    return rc;
}

// Streams for copies beside a context's own, cached for the process: one per copy in flight, kept until it ends.
namespace {
std::mutex g_side_mu;
std::map<int, std::vector<hipStream_t>> g_side;  // idle streams by device
}  // namespace

extern "C" int exhip_memcpy_d2h_from(exhip_ctx* ctx, void* mark, void* dst, const void* src, size_t bytes) {
    EXHIP_REQUIRE(ctx && mark && ((dst && src) || !bytes), "exhip_memcpy_d2h_from: NULL argument");
    if (!bytes) return 0;
    hipStream_t side = nullptr;
    {
        std::lock_guard<std::mutex> g(g_side_mu);
        auto& idle = g_side[ctx->device];
        if (!idle.empty()) {
            side = idle.back();
            idle.pop_back();
        }
    }
    if (!side) {
        EXHIP_CHECK(hipSetDevice(ctx->device));
        EXHIP_CHECK(hipStreamCreateWithFlags(&side, hipStreamNonBlocking));
    }
    int rc = (int)hipStreamWaitEvent(side, (hipEvent_t)mark, 0);
    if (rc == 0) rc = download(ctx, side, dst, src, bytes);
    else exhip_set_error("exhip_memcpy_d2h_from: hipStreamWaitEvent failed: %s", hipGetErrorString((hipError_t)rc));
    std::lock_guard<std::mutex> g(g_side_mu);
    g_side[ctx->device].push_back(side);  // download() has waited for it
    return rc;
}

extern "C" int exhip_memcpy_d2h(exhip_ctx* ctx, void* dst, const void* src, size_t bytes) {
    EXHIP_REQUIRE(ctx && ((dst && src) || !bytes), "exhip_memcpy_d2h: NULL argument");
    if (!bytes) return 0;
    if (bytes > kDownloadKernel) return download(ctx, ctx->stream, dst, src, bytes);
    staging_loan loan(ctx->down);
    EXHIP_REQUIRE(loan.staging, "exhip_memcpy_d2h: no host memory");
    exhip_staging& s = *loan.staging;
    if (!s.chunk[0]) s.chunk[0] = take_chunk();
    if (!s.chunk[0]) return download_through(s, ctx->stream, dst, src, bytes);
    // the flag's line and the bytes behind it
    auto* flag = static_cast<unsigned*>(s.chunk[0]);
    char* stage = static_cast<char*>(s.chunk[0]) + 256;
    const unsigned value = ++s.number;
    __atomic_store_n(flag, value - 1, __ATOMIC_RELAXED);
    download_kernel<<<1, kSmallThreads, 0, ctx->stream>>>(static_cast<const char*>(src), stage, (unsigned)bytes, is_wide(src, stage), flag, value);
    EXHIP_LAUNCH_CHECK();
    const auto start = std::chrono::steady_clock::now();
    for (int i = 0; __atomic_load_n(flag, __ATOMIC_ACQUIRE) != value; ++i) {
        __builtin_ia32_pause();
        if (i % 256 == 255 && std::chrono::steady_clock::now() - start > std::chrono::milliseconds(2)) {
            EXHIP_CHECK(hipStreamSynchronize(ctx->stream));  // a long queue in front (or an error): wait without spinning
            break;
        }
    }
    memcpy(dst, stage, bytes);
    return 0;
}

// A pinned host block for results of a megabyte and more: the copy engine writes it directly. Blocks are cached for reuse
// (at most 512 MiB idle, 1 GiB in all, process-wide); NULL where the limit is reached or no pinned memory is to be had, and the
// caller then takes memory of its own. A new block's first access by the host costs 0.3 ms per MiB in page faults, so it is
// touched here, by several threads, and not under the caller's first read.
extern "C" void* exhip_host_alloc(size_t bytes) {
    if (bytes == 0 || bytes > kBlockLimit) return nullptr;
    size_t rounded = (size_t)1 << 20;
    while (rounded < bytes) rounded <<= 1;
    if (rounded > ((size_t)8 << 20)) {  // in eighths of the power of two above 8 MiB
        const size_t step = rounded >> 4;
        rounded = (bytes + step - 1) / step * step;
    }
    std::vector<char*> dropped;
    {
        std::lock_guard<std::mutex> g(g_pinned_mu);
        auto it = g_idle_blocks.find(rounded);
        if (it != g_idle_blocks.end()) {
            char* p = it->second;
            g_idle_blocks.erase(it);
            g_idle_block_bytes -= rounded;
            return p;
        }
        while (g_block_bytes + rounded > kBlockLimit && !g_idle_blocks.empty()) {  // idle blocks of other sizes make room
            auto old = std::prev(g_idle_blocks.end());
            dropped.push_back(old->second);
            g_block_bytes -= old->first;
            g_idle_block_bytes -= old->first;
            g_blocks.erase(old->second);
            g_idle_blocks.erase(old);
        }
        if (g_block_bytes + rounded > kBlockLimit) rounded = 0;
        else g_block_bytes += rounded;
    }
    for (char* p : dropped) (void)hipHostFree(p);
    if (!rounded) return nullptr;
    void* p = nullptr;
    if (hipHostMalloc(&p, rounded, 0) != hipSuccess) {
        (void)hipGetLastError();
        std::lock_guard<std::mutex> g(g_pinned_mu);
        g_block_bytes -= rounded;
        return nullptr;
    }
    {
        const unsigned cores = std::thread::hardware_concurrency();
        const int threads = cores >= 4 ? (cores / 2 < 8 ? (int)(cores / 2) : 8) : 1;
        std::thread crew[8];
        auto touch = [p, rounded, threads](int t) {
            for (size_t o = rounded / threads * t; o < (t + 1 == threads ? rounded : rounded / threads * (t + 1)); o += 4096)
                static_cast<volatile char*>(p)[o] = 0;
        };
        int started = 1;
        try {
            for (; started < threads; ++started) crew[started] = std::thread(touch, started);
        } catch (...) {  // the process may have no more threads
        }
        touch(0);
        for (int t = started; t < threads; ++t) touch(t);
        for (int t = 1; t < started; ++t) crew[t].join();
    }
    std::lock_guard<std::mutex> g(g_pinned_mu);
    g_blocks[static_cast<char*>(p)] = {rounded};
    return p;
}

extern "C" void exhip_host_free(void* p) {
    if (!p) return;
    {
        std::lock_guard<std::mutex> g(g_pinned_mu);
        auto it = g_blocks.find(static_cast<char*>(p));
        if (it == g_blocks.end()) return;
        const size_t bytes = it->second.bytes;
        if (g_idle_block_bytes + bytes <= kIdleBlockLimit) {
            g_idle_blocks.emplace(bytes, it->first);
            g_idle_block_bytes += bytes;
            return;
        }
        g_block_bytes -= bytes;
        g_blocks.erase(it);
    }
    (void)hipHostFree(p);
}

void exhip_release_staging(exhip_ctx* ctx) {
    for (exhip_staging_pool* pool : {&ctx->up, &ctx->down})
        while (pool->n_idle > 0) release(pool->idle[--pool->n_idle]);
}
