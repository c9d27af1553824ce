// The library's runtime on host_device.hip, from several threads: transfer_check <name of the check>.
#include <cstdio>
#include <cstring>
#include <thread>
#include <vector>

#include "../../excalibur_amd/csrc/common.h"
#include "host_device.h"

namespace {
constexpr int kThreads = 4;
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
}  // namespace

int main(int, char** argv) {
    exhip_ctx* ctx = nullptr;
    OK(exhip_init(0, &ctx));
    const int bad = !std::strcmp(argv[1], "scratch") ? scratch(ctx) : 1;
    OK(exhip_destroy(ctx));
    std::printf("%s: %s\n", argv[1], bad ? "wrong" : "ok");
    return bad != 0;
}
