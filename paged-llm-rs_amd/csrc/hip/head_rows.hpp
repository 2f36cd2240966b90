// Rows of heads of 128 values, 16 lanes a row and eight values a lane: the per-head norm and the rotation.  The stand-alone kernel
// (qk_norm_rope_kv_write_128_kernel), the projection that prepares its heads and the near contexts' kernel all go through here, and so write the same bits.
#pragma once

#include "common.hpp"

typedef __bf16 hr_bf16x2 __attribute__((ext_vector_type(2)));
typedef float hr_f32x2 __attribute__((ext_vector_type(2)));
typedef float hr_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t hr_u32x4 __attribute__((ext_vector_type(4)));

#define HR_D 128

__device__ __forceinline__ uint32_t hr_pack2(float lo, float hi) {
    const hr_f32x2 pair = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(pair, hr_bf16x2));
}
template <int CONTROL>
__device__ __forceinline__ float hr_dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CONTROL, 0xf, 0xf, true));
}

// The sum over 16 lanes that stand side by side, by each of them.
__device__ __forceinline__ float hr_sum16(float v) {
    v += hr_dpp<0xB1>(v);          // quad_perm [1,0,3,2]
    v += hr_dpp<0x4E>(v);          // quad_perm [2,3,0,1]
    v += hr_dpp<0x141>(v);         // lane i of 8 takes 7 - i
    v += hr_dpp<0x140>(v);         // lane i of 16 takes 15 - i
    return v;
}

// Eight values of a head's row of 128, of which 16 lanes side by side hold all: normed with the gains g (gain) and turned by c and sn (turn).
__device__ __forceinline__ void hr_norm_turn(float (&x)[8], bool gain, const float (&g)[8], float eps, bool turn, const float (&c)[8], const float (&sn)[8], bool low) {
    if (gain) {
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(x[e], x[e], ss);
        const float rinv = 1.f / sqrtf(hr_sum16(ss) / static_cast<float>(HR_D) + eps);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = x[e] * rinv * g[e];
    }
    if (turn) {
        float px[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) px[e] = hr_dpp<0x128>(x[e]);       // lane i of 16 takes i ^ 8
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = low ? x[e] * c[e] - px[e] * sn[e] : x[e] * c[e] + px[e] * sn[e];
    }
}

// The same of eight values in bfloat16, and rounded.
__device__ __forceinline__ hr_u32x4 hr_prepare(hr_u32x4 raw, bool gain, const float (&g)[8], float eps, bool turn, const float (&c)[8], const float (&sn)[8], bool low) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        x[2 * e] = __uint_as_float(raw[e] << 16);
        x[2 * e + 1] = __uint_as_float(raw[e] & 0xffff0000u);
    }
    hr_norm_turn(x, gain, g, eps, turn, c, sn, low);
    return hr_u32x4{hr_pack2(x[0], x[1]), hr_pack2(x[2], x[3]), hr_pack2(x[4], x[5]), hr_pack2(x[6], x[7])};
}

__device__ __forceinline__ void hr_load8(const float* from, float (&to)[8]) {
    const hr_f32x4 a = *reinterpret_cast<const hr_f32x4*>(from), b = *reinterpret_cast<const hr_f32x4*>(from + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        to[e] = a[e];
        to[4 + e] = b[e];
    }
}

__device__ __forceinline__ void hr_load_gain(const void* gain, int dtype, int chunk, float (&to)[8]) {
    if (dtype == PL_DTYPE_F32) {
        hr_load8(static_cast<const float*>(gain) + chunk * 8, to);
    } else {
        const hr_u32x4 raw = *reinterpret_cast<const hr_u32x4*>(static_cast<const bf16_t*>(gain) + chunk * 8);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            to[2 * e] = __uint_as_float(raw[e] << 16);
            to[2 * e + 1] = __uint_as_float(raw[e] & 0xffff0000u);
        }
    }
}
