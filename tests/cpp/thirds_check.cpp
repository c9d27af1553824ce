// The float32 kernel of bfloat16 thirds on the CPU: every layer of maps up to 40 x 40 has a form whose staged pixels LDS holds, and as few groups as a CU each where
// its pixels are that few; and every load of every form, over all channel counts from 16 to 512, lies inside its operand.
#include <strict.h>
#include <sys/mman.h>

#include "../../excalibur_amd/csrc/conv_f32_thirds.hip"

void exhip_set_error(const char*, ...) {}
exhip_options g_exhip_options;

namespace {
char lds_all[kLdsLimit];

bool small_maps() {
    long long plans = 0;
    for (int h = 1; h <= 40; ++h)
        for (int w = 1; w <= 40; ++w)
            for (long long images : {1, 2, 17, 18, 31, 32, 33, 64, 500})
                for (int csteps : {1, 3, 4, 5, 8, 9, 32}) {
                    F32Params p = {};
                    p.out_h = h; p.out_w = w; p.csteps = csteps;
                    for (int tile = 0; tile <= kForms; ++tile) {
                        const Plan plan = plan_of(p, images, 2, tile);
                        ++plans;
                        const Sizes s(kForm[plan.form]);
                        if (s.lds(plan.strips.staged, csteps > kForm[plan.form].cs ? 2 : 1) > kLdsLimit)
                            return printf("%lld images of %d x %d, %d steps, option %d: %d pixels staged in form %d\n", images, h, w, csteps, tile, plan.strips.staged, plan.form), false;
                    }
                }
    printf("%lld plans\n", plans);
    return true;
}

// Strips of columns that a map does not have make runs: not more of them than there are CUs where the pixels alone need no more and strips that divide the map lie in LDS.
bool one_round() {
    int layers = 0;
    for (int h = 8; h <= 64; ++h)
        for (int w = h - 3; w <= h + 3; ++w)
            for (int images = 1; images <= 4; ++images)
                for (int kblocks : {1, 2, 4, 8, 16})
                    for (int tile = 1; tile <= kForms; ++tile) {
                        F32Params p = {};
                        p.out_h = h; p.out_w = w; p.csteps = 8;
                        const Plan plan = plan_of(p, images, kblocks, tile);
                        const Shape& f = kForm[plan.form];
                        const Sizes s(f);
                        const long long groups = (kblocks + f.mt - 1) / f.mt, runs = ((long long)h * w * images + s.run - 1) / s.run;
                        bool fits = false;
                        for (int width = 4; width <= w; ++width) {
                            const int rows = (s.run + width - 2) / width, staged = (rows + (rows + h - 1) / h * 2 + 3) * (width + 2);
                            fits |= w % width == 0 && s.lds(staged, p.csteps > f.cs ? 2 : 1) <= kLdsLimit;
                        }
                        if (!fits || runs * groups > 256) continue;
                        ++layers;
                        if (plan.strips.tiles * groups > 256)
                            return printf("%d images of %d x %d, %d blocks, form %d: %lld groups for %lld\n", images, h, w, kblocks, plan.form, plan.strips.tiles * groups, runs * groups), false;
                    }
    printf("%d layers of one round\n", layers);
    return layers > 1000;
}

// `count` values whose last one is the last before an unreadable page
float* ending_at_a_page(size_t count) {
    const size_t bytes = count * 4, pages = (bytes + 4095) / 4096 * 4096;
    char* p = static_cast<char*>(mmap(nullptr, pages + 4096, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
    mprotect(p + pages, 4096, PROT_NONE);
    return reinterpret_cast<float*>(p + pages - bytes);
}

bool layer(int n, int h, int w, int c, int k, int tile, bool twice) {
    host_of_class = twice;
    exhip_conv_desc d = {};
    d.n = n; d.h = h; d.w = w; d.c = c; d.k = k; d.kh = d.kw = 3; d.sh = d.sw = 1; d.pt = d.pl = 1;
    F32Params p = {};
    float *const x = ending_at_a_page((size_t)n * h * w * c), *const wp = ending_at_a_page(exhip_conv_f32_thirds_bytes(&d) / 4);
    float *const y = ending_at_a_page((size_t)n * h * w * ((k + 31) / 32 * 32)), *const bias = ending_at_a_page(k);
    p.x = reinterpret_cast<char*>(x); p.wp = reinterpret_cast<char*>(wp); p.bias = bias; p.y = y;
    p.pixels = n * h * w; p.x_bytes = n * h * w * c * 4; p.w_bytes = (unsigned)exhip_conv_f32_thirds_bytes(&d);
    p.in_h = p.out_h = h; p.in_w = p.out_w = w; p.stride = 1; p.pad_t = p.pad_l = 1; p.kh = p.kw = 3;
    p.xs_b = c * 4; p.row_b = w * c * 4; p.csteps = c / 16; p.K = k; p.kstride = p.k_end = (k + 31) / 32 * 32; p.vector_rows = 1;
    exhip_host_divisor(h * w, &p.image_magic, &p.image_shift);
    exhip_host_divisor(w, &p.width_magic, &p.width_shift);
    g_exhip_options.f32_tile = tile;
    static exhip_ctx context;
    const int rc = exhip_conv_f32_thirds_run(&context, {&p, n, (k + 31) / 32});
    if (rc || host_outside) return printf("%d x %d x %d, %d -> %d channels, option %d: error %d, %lld accesses outside\n", n, h, w, c, k, tile, rc, host_outside), false;
    for (size_t i = 0; i < (size_t)n * h * w; ++i)
        for (int ch = 0; ch < p.kstride; ++ch)
            if (y[i * p.kstride + ch] != 0) return printf("%d channels, option %d: pixel %zu\n", c, tile, i), false;  // (biases and products are zeros here)
    return true;
}

}  // namespace

int main() {
    if (!small_maps() || !one_round()) return 1;
    for (int tile = 1; tile <= kForms; ++tile)
        for (int c = 16; c <= 512; c += 16)
            if (!layer(c % 5 == 1 ? 2 : 1, 3, c % 3 ? 5 : 4, c, c % 7 ? 40 : 64, tile, false) || (c % 48 == 32 && (!layer(2, 3, 4, c, 40, tile, true) || !layer(33, 1, 1, c, 40, tile, false)))) return 1;  // (twice: sums that thirds do not hold)
    return 0;
}
