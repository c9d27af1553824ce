// The kernel that stages the input of 3x3 fp16 and int8 layers in LDS, on the CPU: every load and store of every form, over all channel counts from 32 to 512 that it
// takes, lies inside its operand.
#include <strict.h>
#include <sys/mman.h>

#include "../../excalibur_amd/csrc/conv_staged.hip"

void exhip_set_error(const char*, ...) {}
exhip_options g_exhip_options;

namespace {
char lds_all[kLdsLimit];

// `bytes` bytes whose last one is the last before an unreadable page
char* ending_at_a_page(size_t bytes) {
    const size_t pages = (bytes + 4095) / 4096 * 4096;
    char* p = static_cast<char*>(mmap(nullptr, pages + 4096, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
    mprotect(p + pages, 4096, PROT_NONE);
    return p + pages - bytes;
}

bool layer(int dt, int n, int h, int w, int c, int k, int mts, int stride, int form) {
    const int es = dt == EXHIP_I8 ? 1 : 2, xs_b = c * es, chunk_b = xs_b % 64 ? 32 : 64, steps = 9 * xs_b / 32, kblocks = (k + 31) / 32;
    const int oh = (h - 1) / stride + 1, ow = (w - 1) / stride + 1, ks = kblocks * 32;
    PwParams p = {};
    p.pixels = n * oh * ow; p.x_bytes = n * h * w * xs_b; p.w_bytes = (kblocks + mts - 1) / mts * steps * mts * 1024;
    p.xs_b = xs_b; p.n_ksteps = steps; p.mts = mts; p.K = k; p.kstride = ks; p.act = 0;
    p.in_h = h; p.in_w = w; p.out_h = oh; p.out_w = ow; p.stride = stride; p.pad_t = p.pad_l = 1; p.kh = p.kw = 3; p.chunk_b = chunk_b; p.fs_out = 1;
    p.x = ending_at_a_page(p.x_bytes); p.wp = ending_at_a_page(p.w_bytes + (xs_b % 64 && dt == EXHIP_I8 ? 9 * mts * 1024 : 0));  // (the packing's zeros behind the weights)
    p.bias = (float*)ending_at_a_page(k * 4); p.scale = (float*)ending_at_a_page(k * 4);
    char* const y = ending_at_a_page((size_t)p.pixels * ks * es);
    if (dt == EXHIP_I8) p.y_q = (int8_t*)y;
    else p.y = (uint16_t*)y;
    exhip_host_divisor(oh * ow, &p.image_magic, &p.image_shift);
    exhip_host_divisor(ow, &p.width_magic, &p.width_shift);
    g_exhip_options.staged = form;
    static exhip_ctx context;
    const int rc = exhip_conv3x3_staged(&context, dt, &p, n, kblocks, 0);
    if (rc || host_outside) return printf("%s %d x %d x %d, %d -> %d channels, stride %d, option %d: error %d, %lld accesses outside\n", dt == EXHIP_I8 ? "int8" : "fp16", n, h, w, c, k, stride, form, rc, host_outside), false;
    return true;
}

}  // namespace

int main() {
    for (int form = 2; form <= 4; ++form)
        for (int c = 32; c <= 512; c += 32) {
            const int mts = c % 3 ? 2 : 4, n = c % 5 == 1 ? 2 : 1, w = c % 64 ? 5 : 4;
            if (!layer(EXHIP_I8, n, 3, w, c, c % 7 ? 40 : 96, mts, 1, form)) return 1;
            if (!layer(EXHIP_F16, n, 3, w, c, c % 7 ? 40 : 96, mts, 1, form) || !layer(EXHIP_F16, n, 5, w + 3, c, c % 7 ? 40 : 96, mts, 2, form)) return 1;
        }
    return 0;
}
