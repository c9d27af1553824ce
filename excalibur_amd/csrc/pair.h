// Two layers in one launch (conv_pw.hip, conv_f32.hip): while a layer of the pair is run, a launch of a form that can share one is left waiting instead.
#pragma once
#include "common.h"

template <typename P>
struct exhip_waiting {
    int kind = -1, dt = 0;
    unsigned groups = 0;
    const void* kernel = nullptr;
    P p;
};

// place: the thread's place for the next launch. both(w): launches the two as one, EXHIP_ERR_UNSUPPORTED where they cannot share one after all.
template <typename P, typename BOTH>
int exhip_run_pair(exhip_ctx* ctx, exhip_waiting<P>** place, int (*layer)(exhip_ctx*, const void*), const void* first, const void* second, BOTH both) {
    exhip_waiting<P> w[2];
    int rc = 0;
    for (int i = 0; i < 2 && !rc; ++i) {
        *place = &w[i];
        rc = layer(ctx, i ? second : first);
        *place = nullptr;
    }
    // (a layer that ran by itself is done; it reads nothing of the other's)
    if (!rc && w[0].kind >= 0 && w[1].kind >= 0 && (long long)w[0].groups + w[1].groups < (1ll << 31)) {
        const int one = both(w);
        if (one != EXHIP_ERR_UNSUPPORTED) return one;
    }
    for (exhip_waiting<P>& one : w) {
        if (one.kind < 0) continue;
        void* args[] = {&one.p};
        EXHIP_CHECK(hipLaunchKernel(one.kernel, dim3(one.groups), dim3(256), args, 0, ctx->stream));
        EXHIP_LAUNCH_CHECK();
    }
    return rc;
}
