// Included behind hip_runtime.h and before a kernel source: buffer loads and stores as the hardware lets them through (the range check looks at the
// lane's offset alone), and an access that then lies outside its operand counts as an error. LDS that a launch sizes itself is `lds_all`.
#pragma once
#include <hip/hip_runtime.h>

inline long long host_outside = 0;
inline bool host_lands(host_buffer r, unsigned lane, unsigned scalar, size_t bytes) {
    if ((size_t)lane + bytes > r.bytes) return false;
    if ((size_t)lane + scalar + bytes > r.bytes) {
        ++host_outside;
        return false;
    }
    return true;
}
template <typename V>
V strict_load(host_buffer r, int lane, int scalar) {
    V v = {};
    if (host_lands(r, (unsigned)lane, (unsigned)scalar, sizeof(V))) memcpy((char*)&v, r.at + (unsigned)lane + (unsigned)scalar, sizeof(V));
    return v;
}
template <typename V>
void strict_store(V v, host_buffer r, int lane, int scalar) {
    if (host_lands(r, (unsigned)lane, (unsigned)scalar, sizeof(V))) memcpy(r.at + (unsigned)lane + (unsigned)scalar, (char*)&v, sizeof(V));
}
#undef __builtin_amdgcn_raw_buffer_load_b128
#undef __builtin_amdgcn_raw_buffer_load_b32
#undef __builtin_amdgcn_raw_buffer_store_b128
#undef __builtin_amdgcn_raw_buffer_store_b32
#define __builtin_amdgcn_raw_buffer_load_b128(r, lane, scalar, aux) strict_load<host_words<4>>(r, lane, scalar)
#define __builtin_amdgcn_raw_buffer_load_b32(r, lane, scalar, aux) strict_load<unsigned>(r, lane, scalar)
#define __builtin_amdgcn_raw_buffer_store_b128(v, r, lane, scalar, aux) strict_store(v, r, lane, scalar)
#define __builtin_amdgcn_raw_buffer_store_b32(v, r, lane, scalar, aux) strict_store(v, r, lane, scalar)

// Products are not computed: where a kernel reads and writes does not depend on them.
#define __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, x, y, z) (c)
#define __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, x, y, z) (c)
#define __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, x, y, z) (c)
#define __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, x, y, z) (c)
#define __builtin_amdgcn_readfirstlane(v) (v)
#define __builtin_amdgcn_sched_barrier(v)
#define __builtin_amdgcn_ds_bpermute(at, v) host::of_lane(v, (at) >> 2 & 63)
#define __any(v) (v)
inline bool host_of_class = false;  // what every value's test for its kind says
#define __builtin_amdgcn_classf(v, kinds) host_of_class
inline float __uint_as_float(unsigned u) { return __builtin_bit_cast(float, u); }
inline unsigned __float_as_uint(float f) { return __builtin_bit_cast(unsigned, f); }
constexpr int hipFuncAttributeMaxDynamicSharedMemorySize = 0;
inline hipError_t hipFuncSetAttribute(const void*, int, int) { return hipSuccess; }
#undef __shared__
#define __shared__
