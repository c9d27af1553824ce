// The library's runtime on host_device.hip, from several threads: transfer_check <name of the check>.
#include <cstdio>
#include <cstring>
#include <thread>
#include <vector>

#include <time.h>

#include "../../excalibur_amd/csrc/common.h"
#include "host_device.h"

namespace {
constexpr int kThreads = 7;  // more than a context keeps staging for
#define OK(call)                                                             \
    do {                                                                     \
        const int rc_ = (call);                                              \
        if (rc_ != 0) {                                                      \
            std::printf("%s: %d %s\n", #call, rc_, exhip_last_error());      \
            std::exit(1);                                                    \
        }                                                                    \
    } while (0)

template <typename F>
int on_threads(F f) {
    std::atomic<int> bad{0};
    std::vector<std::thread> threads;
    for (int t = 0; t < kThreads; ++t) threads.emplace_back([&, t] { bad += f(t); });
    for (auto& t : threads) t.join();
    return bad;
}

// The scratch of the convolution's split reduction, first needed by all threads at once.
int scratch(exhip_ctx* ctx) {
    g_malloc_us = 3000;
    const int before = g_mallocs;
    const int bad = on_threads([&](int) {
        int* acc = nullptr;
        unsigned* count = nullptr;
        OK(exhip_split_scratch(ctx, 1 << 20, 16, &acc, &count));
        return acc == nullptr || acc != ctx->split_acc || count == nullptr || count != ctx->split_count || count[kSplitGroups - 1] != 0;
    });
    return bad + (g_mallocs - before != 2);
}

// Every thread sends bytes of its own to a block of its own and reads them back, all on one context: the sizes take each way
// through the staging memory.
int shared(exhip_ctx* ctx) {
    g_copy_us = 50;
    return on_threads([&](int t) {
        int bad = 0;
        void* mark = nullptr;
        for (int i = 0; i < 12; ++i) {
            const size_t sizes[] = {300, 75 << 10, (size_t)900 << 10, (size_t)9 << 20};
            const size_t bytes = sizes[(i + t) % 4] + t;
            std::vector<char> want(bytes), got(bytes);
            for (size_t k = 0; k < bytes; ++k) want[k] = (char)(k * 7 + t * 50 + i);
            const std::vector<char> sent = want;
            void* dev = nullptr;
            OK(exhip_malloc(ctx, bytes, &dev));
            if (i % 3 == 0) OK(exhip_memcpy_h2d(ctx, dev, want.data(), bytes));
            else OK(exhip_upload(ctx, dev, want.data(), bytes));
            std::memset(want.data(), 0x55, bytes);  // the source may change at once
            if (i % 3 == 1) {
                OK(exhip_mark(ctx, &mark));
                OK(exhip_memcpy_d2h_from(ctx, mark, got.data(), dev, bytes));
            } else {
                OK(exhip_memcpy_d2h(ctx, got.data(), dev, bytes));
            }
            if (got != sent) {
                std::printf("thread %d copy %d of %zu bytes differs\n", t, i, bytes);
                ++bad;
            }
            OK(exhip_free(ctx, dev));
        }
        OK(exhip_mark_destroy(mark));
        return bad;
    });
}

// Results that the link brings slowly: the helper threads take the processor while there is something to copy, not while they wait.
int idle(exhip_ctx* ctx) {
    const size_t bytes = (size_t)40 << 20;
    std::vector<char> got(bytes);
    void* dev = nullptr;
    OK(exhip_malloc(ctx, bytes, &dev));
    std::memset(dev, 3, bytes);
    OK(exhip_memcpy_d2h(ctx, got.data(), dev, bytes));  // threads and pages are there
    auto seconds = [](clockid_t id) {
        timespec t;
        clock_gettime(id, &t);
        return t.tv_sec + t.tv_nsec * 1e-9;
    };
    g_copy_us = 40000;
    const double wall = seconds(CLOCK_MONOTONIC), cpu = seconds(CLOCK_PROCESS_CPUTIME_ID);
    OK(exhip_memcpy_d2h(ctx, got.data(), dev, bytes));
    const double wall_s = seconds(CLOCK_MONOTONIC) - wall, cpu_s = seconds(CLOCK_PROCESS_CPUTIME_ID) - cpu;
    std::printf("%.3f s of processor time in %.3f s\n", cpu_s, wall_s);
    OK(exhip_free(ctx, dev));
    return got[bytes - 1] != 3 || cpu_s > wall_s / 2;
}

// A process that cannot have another thread copies without helpers.
int limit(exhip_ctx* ctx) {
    g_no_threads = true;
    const size_t bytes = (size_t)9 << 20;
    std::vector<char> sent(bytes, 5), got(bytes);
    void *dev = nullptr, *block = exhip_host_alloc(bytes);
    OK(exhip_malloc(ctx, bytes, &dev));
    OK(exhip_memcpy_h2d(ctx, dev, sent.data(), bytes));
    OK(exhip_memcpy_d2h(ctx, got.data(), dev, bytes));
    OK(exhip_free(ctx, dev));
    const bool zero = block && static_cast<char*>(block)[bytes - 1] == 0;
    exhip_host_free(block);
    return got != sent || !zero;
}
}  // namespace

int main(int, char** argv) {
    exhip_ctx* ctx = nullptr;
    OK(exhip_init(0, &ctx));
    const int bad = !std::strcmp(argv[1], "scratch") ? scratch(ctx) : !std::strcmp(argv[1], "shared") ? shared(ctx) : !std::strcmp(argv[1], "idle") ? idle(ctx) : !std::strcmp(argv[1], "limit") ? limit(ctx) : 1;
    OK(exhip_destroy(ctx));
    std::printf("%s: %s\n", argv[1], bad ? "wrong" : "ok");
    return bad != 0;
}
