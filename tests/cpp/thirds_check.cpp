// The float32 kernel of bfloat16 thirds on the CPU: every layer of maps up to 40 x 40 has a form whose staged pixels LDS holds; and every load of every form, over
// all channel counts from 16 to 512, lies inside its operand.
#include <strict.h>

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
                    for (int tile = 0; tile <= kForms + 1; ++tile) {
                        const Plan plan = plan_of(p, images, 2, tile);
                        const Sizes s(kForm[plan.form]);
                        ++plans;
                        if (s.lds(plan.staged, csteps > kForm[plan.form].cs ? 2 : 1) > kLdsLimit)
                            return printf("%lld images of %d x %d, %d steps, option %d: %d pixels staged in form %d\n", images, h, w, csteps, tile, plan.staged, plan.form), false;
                    }
                }
    printf("%lld plans\n", plans);
    return true;
}

}  // namespace

int main() {
    if (!small_maps()) return 1;
    return 0;
}
