// Loading 8 activations of a row and their products with the input scales, shared by the input-Hadamard kernels that
// hold a 128-block in 16 lanes x 8 values (the grouped experts and the dense linear).
#pragma once
#include "exl3_common.cuh"

namespace exl3 {

typedef uint32_t u32x4_x __attribute__((ext_vector_type(4)));
template <int DT> struct XRaw { u32x4_x w[DT == 2 ? 2 : 1]; };       // 8 activations as loaded
typedef uint32_t u32x4_u __attribute__((ext_vector_type(4), aligned(2)));   // (at any alignment)

template <int DT>
__device__ __forceinline__ void ld_x8(const void* x, size_t i, XRaw<DT>& r) {
    if constexpr (DT == 2) {
        r.w[0] = *(const u32x4_u*)((const float*)x + i);
        r.w[1] = *(const u32x4_u*)((const float*)x + i + 4);
    } else {
        r.w[0] = *(const u32x4_u*)((const uint16_t*)x + i);
    }
}
// fp16(x suh) of value j, the product rounded to fp32 first: a 16-bit x makes it exact in fp32, so rounding it once to
// fp16 gives the same bits
template <int DT>
__device__ __forceinline__ float x_su(const XRaw<DT>& r, int j, half_t s) {
    if constexpr (DT == 2) return (float)to_half(__uint_as_float(r.w[j >> 2][j & 3]) * (float)s);
    const uint32_t w = r.w[0][j >> 1];
    if constexpr (DT == 1) return (float)(half_t)(__uint_as_float(j & 1 ? w & 0xFFFF0000u : w << 16) * (float)s);
    else return (float)(half_t)(__builtin_bit_cast(half2_t, w)[j & 1] * s);
}

}  // namespace exl3
