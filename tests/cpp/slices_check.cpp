// The entry points of bandwidth.hip that take slices of wider tensors, on the CPU: every tensor ends where an unreadable page begins, so that
// an access behind it ends the program, and the results are those of plain loops.
#include <sys/mman.h>

#include "../../excalibur_amd/csrc/bandwidth.hip"

void exhip_set_error(const char*, ...) {}
exhip_options g_exhip_options;

namespace {

// `count` values whose last one is the last before an unreadable page (to 16 bytes: the kernels' vector accesses need aligned tensors).
template <typename T>
T* ending_at_a_page(size_t count) {
    const size_t bytes = (count * sizeof(T) + 15) / 16 * 16, pages = (bytes + 4095) / 4096 * 4096;
    char* p = static_cast<char*>(mmap(nullptr, pages + 4096, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
    mprotect(p + pages, 4096, PROT_NONE);
    return reinterpret_cast<T*>(p + pages - bytes);
}

int failures = 0;
void expect(bool ok, const char* what, int c, int stride, int offset, int h, int w) {
    if (ok) return;
    ++failures;
    printf("%s: c %d of %d from %d, %d x %d\n", what, c, stride, offset, h, w);
}

template <typename Tin, typename Tout, typename F>
void nchw(const char* what, F call, int n, int c, int stride, int offset, int h, int w) {
    Tin* x = ending_at_a_page<Tin>((size_t)n * h * w * stride);
    Tout* y = ending_at_a_page<Tout>((size_t)n * h * w * c);
    for (size_t i = 0; i < (size_t)n * h * w * stride; ++i) x[i] = (Tin)(i % 1021);
    int rc = call(x + offset, n, c, h, w, stride, y);
    bool ok = rc == 0;
    for (int i = 0; i < n; ++i)
        for (int k = 0; k < c; ++k)
            for (int p = 0; p < h * w; ++p) {
                const Tin v = x[((size_t)i * h * w + p) * stride + offset + k];
                const Tout want = sizeof(Tin) == 2 && sizeof(Tout) == 4 ? (Tout)exhip_h2f((uint16_t)v) : (Tout)v;
                ok = ok && y[((size_t)i * c + k) * h * w + p] == want;
            }
    expect(ok, what, c, stride, offset, h, w);
}

}  // namespace

int main() {
    static exhip_ctx context;
    exhip_ctx* const ctx = &context;
    struct { int c, stride, offset; } slices[] = {{64, 64, 0}, {8, 24, 16}, {32, 96, 64}, {16, 80, 0}, {72, 144, 72}, {12, 16, 0}, {5, 40, 32}, {24, 56, 8}};
    struct { int n, h, w; } maps[] = {{1, 8, 8}, {2, 9, 13}, {3, 16, 16}, {1, 3, 5}};
    for (const auto& s : slices)
        for (const auto& m : maps) {
            nchw<float, float>("float32", [&](auto* x, int n, int c, int h, int w, int cs, auto* y) { return exhip_nhwc_f32_to_nchw_f32(ctx, x, n, c, h, w, cs, y); },
                               m.n, s.c, s.stride, s.offset, m.h, m.w);
            nchw<uint16_t, uint16_t>("half", [&](auto* x, int n, int c, int h, int w, int cs, auto* y) { return exhip_nhwc_f16_to_nchw_f16(ctx, x, n, c, h, w, cs, y); },
                                     m.n, s.c, s.stride, s.offset, m.h, m.w);
            nchw<uint16_t, float>("half to float32", [&](auto* x, int n, int c, int h, int w, int cs, auto* y) { return exhip_nhwc_f16_to_nchw_f32(ctx, x, n, c, h, w, cs, y); },
                                  m.n, s.c, s.stride, s.offset, m.h, m.w);
            if (s.c % 4 || s.offset % 4) continue;
            // a slice pooled and resized into a slice: the values around it stay
            const size_t pixels = (size_t)m.n * m.h * m.w;
            float* x = ending_at_a_page<float>(pixels * s.stride);
            for (size_t i = 0; i < pixels * s.stride; ++i) x[i] = (float)(i % 1021);
            float* y = ending_at_a_page<float>(pixels * s.stride);
            auto inside = [&](size_t i) { const int k = (int)(i % s.stride); return k >= s.offset && k < s.offset + s.c; };
            std::fill(y, y + pixels * s.stride, -1.f);
            bool ok = exhip_pool2d_nhwc_f32(ctx, x + s.offset, s.stride, y + s.offset, s.stride, m.n, s.c, m.h, m.w, m.h, m.w, 0, 1, 1, 1, 1, 0, 0, 0, 0, 0) == 0;
            for (size_t i = 0; i < pixels * s.stride; ++i) ok = ok && y[i] == (inside(i) ? x[i] : -1.f);
            expect(ok, "pool", s.c, s.stride, s.offset, m.h, m.w);
            std::fill(y, y + pixels * s.stride, -1.f);
            ok = exhip_interp_nearest_nhwc_f32(ctx, x + s.offset, s.stride, y + s.offset, s.stride, m.n, s.c, m.h, m.w, m.h, m.w) == 0;
            for (size_t i = 0; i < pixels * s.stride; ++i) ok = ok && y[i] == (inside(i) ? x[i] : -1.f);
            expect(ok, "interp", s.c, s.stride, s.offset, m.h, m.w);
            const float* from = x + s.offset;
            const int total = s.c;
            if (total % 4 == 0) {
                float* z = ending_at_a_page<float>(pixels * total);
                ok = exhip_concat_batchnorm_unary_nhwc_f32(ctx, &from, &s.c, &s.stride, 1, pixels, nullptr, nullptr, -1, 0.f, 0.f, total, z, nullptr, 0.f) == 0;
                for (size_t i = 0; i < pixels; ++i)
                    for (int k = 0; k < total; ++k) ok = ok && z[i * total + k] == x[i * s.stride + s.offset + k];
                expect(ok, "concat", s.c, s.stride, s.offset, m.h, m.w);
            }
        }
    printf("%d failures\n", failures);
    return failures != 0;
}
