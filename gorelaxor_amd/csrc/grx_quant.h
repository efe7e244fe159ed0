// grx_quant.h - rounding one block of 32 activations to Q8_0 on eight lanes.
#pragma once
#include "grx_internal.h"

// quantU8 (grx_quant_block) of a block held four values a lane by eight
// consecutive lanes: v are values 4 * l8 .. + 3, q the block's bytes.  The
// maximum is the same in any order.
__device__ __forceinline__ void quant8x4_store(const float (&v)[4], int8_t *q, float *sc, int l8) {
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = fabsf(v[i]);
        amax = a > amax ? a : amax;
    }
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) {
        const float t = __shfl_xor(amax, o, 8);
        amax = t > amax ? t : amax;
    }
    const float id = amax != 0.0f ? __fdiv_rn(127.0f, amax) : 0.0f;
    uint32_t w = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float r = rintf(__fmul_rn(v[i], id));
        r = fminf(fmaxf(r, -128.0f), 127.0f);
        w |= (uint32_t)(uint8_t)(int8_t)(int)r << (8 * i);
    }
    __builtin_memcpy(q + 4 * l8, &w, 4);
    if (l8 == 0) *sc = __fmul_rn(amax, grx_bits_f32(0x3c010204u));
}
