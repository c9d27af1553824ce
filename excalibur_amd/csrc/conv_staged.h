// The 3x3 fp16 / int8 convolution with its input staged in LDS (conv_staged.hip): conv_pw.hip fills the launch's parameters (a PwParams of a layer with a
// filter) and hands it over. lean_tiles: groups of conv_i8_lean.hip's fp16 form for the
// layer, 0 where it cannot take it. EXHIP_ERR_UNSUPPORTED, with nothing launched, where another kernel runs the layer.
#pragma once
#include "common.h"
#include "conv_pw.h"

int exhip_conv3x3_staged(exhip_ctx* ctx, int dt, const void* pw_params, long long images, int kblocks, int lean_tiles);
// Int8 layers at stride 1 whose pixels end with half a piece of 64 bytes: zeros behind the packed weights, a 32-byte step's nine taps, that the kernel reads for the other half.
constexpr int exhip_staged_pad(int slab_blocks) { return 9 * slab_blocks * 1024; }
constexpr int kStagedBlocks = 512;  // blocks of 32 pixels x 32 channels that a layer has to have more of
// What can be said of that beforehand, by the layer's kind and size: false where another kernel is faster. y_f: a float32 result is asked for.
bool exhip_staged_wins(int dt, const exhip_pw_geom& g, int stride, int n_ksteps, bool shortcut, bool y_f);
