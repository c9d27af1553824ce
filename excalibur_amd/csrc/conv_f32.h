// The float32 convolution (conv_f32.hip): its checks and weight packing, which exhip_conv_packed_bytes and
// exhip_conv_pack_weights hand on for EXHIP_F32.
#pragma once
#include "common.h"

int exhip_conv_f32_validate(const exhip_conv_desc* d);
size_t exhip_conv_f32_packed_bytes(const exhip_conv_desc* d);  // 0: outside what the convolution takes
int exhip_conv_f32_pack_weights(const exhip_conv_desc* d, const float* w_oihw, float* packed);
