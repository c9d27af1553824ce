// The float32 convolution (conv_f32.hip, conv_f32_thirds.hip): its checks and weight packing, which exhip_conv_packed_bytes and
// exhip_conv_pack_weights hand on for EXHIP_F32.
#pragma once
#include "common.h"

int exhip_conv_f32_validate(const exhip_conv_desc* d);
size_t exhip_conv_f32_packed_bytes(const exhip_conv_desc* d);  // 0: outside what the convolution takes
int exhip_conv_f32_pack_weights(const exhip_conv_desc* d, const float* w_oihw, float* packed);

// 3x3 layers whose products are taken in thirds (conv_f32_thirds.hip): which, their packing, and a launch of up to 2 GiB of input.
struct F32Launch {
    const void* params;  // F32Params
    long long images;
    int blocks;          // 32-channel blocks to write
};
bool exhip_conv_f32_thirds(const exhip_conv_desc* d);
size_t exhip_conv_f32_thirds_bytes(const exhip_conv_desc* d);
void exhip_conv_f32_thirds_pack(const exhip_conv_desc* d, const float* w_oihw, void* packed);
int exhip_conv_f32_thirds_pack_device(exhip_ctx* ctx, const exhip_conv_desc* d, const float* w_oihw, void* packed);  // both on the device
int exhip_conv_f32_thirds_run(exhip_ctx* ctx, const F32Launch& launch);
