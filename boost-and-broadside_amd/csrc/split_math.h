// Float32 values as three bf16 pieces, v = h + m / 128 + l / 128^2: the pieces shared by the kernels that multiply
// float32 operands on the bf16 matrix cores (linear_split.hip says why these pieces and these products).
#pragma once

#include "common.h"

namespace bnb {

constexpr int kLsChunkHalfs = 8 * 3 * 512;  // 32 features x 128 channels x 3 pieces

// erf-GELU, Abramowitz-Stegun 7.1.26 (|error of gelu| <= 5e-7)
__device__ __forceinline__ float gelu_erf_ls(float v)
{
    const float x = fabsf(v) * 0.70710678118654752f;
    const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, x, 1.0f));
    float poly = fmaf(1.061405429f, t, -1.453152027f);
    poly = fmaf(poly, t, 1.421413741f);
    poly = fmaf(poly, t, -0.284496736f);
    poly = fmaf(poly, t, 0.254829592f);
    const float e = __builtin_amdgcn_exp2f((x * x) * -1.4426950408889634f);
    const float erf_abs = fmaf(-(poly * t), e, 1.0f);
    const float hv = 0.5f * v;
    return fmaf(fabsf(hv), erf_abs, hv);
}

constexpr float kLsScale = 128.0f;  // each rest is carried this much larger: it keeps a bf16 exponent down to the smallest values

// eight float32 -> three bf16 operands
__device__ __forceinline__ void split8(const float (&v)[8], bf16x8 &h, bf16x8 &m, bf16x8 &l)
{
    u32x4 hw, mw, lw;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float a = v[2 * q], b = v[2 * q + 1];
        hw[q] = pack_bf16x2(a, b);
        const float ra = (a - __uint_as_float(hw[q] << 16)) * kLsScale, rb = (b - __uint_as_float(hw[q] & 0xffff0000u)) * kLsScale;
        mw[q] = pack_bf16x2(ra, rb);
        lw[q] = pack_bf16x2((ra - __uint_as_float(mw[q] << 16)) * kLsScale, (rb - __uint_as_float(mw[q] & 0xffff0000u)) * kLsScale);
    }
    h = __builtin_bit_cast(bf16x8, hw), m = __builtin_bit_cast(bf16x8, mw), l = __builtin_bit_cast(bf16x8, lw);
}

__device__ __forceinline__ bool not_finite(float v) { return __builtin_amdgcn_classf(v, 0x207); }  // NaNs and infinities

// Weight k of feature m of block `block` as a whole float32, from a stream of `slabs` slabs of 128 channels a block
__device__ __forceinline__ float whole_weight(const uint16_t *w, int slabs, int block, int m, int k)
{
    const uint16_t *wp = w + ((int64_t)block * slabs + (k >> 7)) * kLsChunkHalfs + ((k & 127) >> 4) * 1536 +
                         (((k >> 2) & 1) * 32 + m) * 8 + ((k >> 3) & 1) * 4 + (k & 3);
    const float wm = bf16_bits_to_f32(wp[512]);  // infinite for an infinite weight, whose last piece then says nothing
    const float wv = fmaf(fmaf(bf16_bits_to_f32(wp[1024]), 1.0f / kLsScale, wm), 1.0f / kLsScale, bf16_bits_to_f32(wp[0]));
    return not_finite(wm) ? wm : wv;
}

// The sums of a block by size: products of two leading pieces, of a leading and a second piece (1 / kLsScale of their value),
// and the rest (1 / kLsScale^2).
struct Sums {
    f32x16 big, mid, small;
    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int v = 0; v < 16; ++v) big[v] = mid[v] = small[v] = 0.0f;
    }
    __device__ __forceinline__ float total(int v) const
    {
        return fmaf(fmaf(small[v], 1.0f / kLsScale, mid[v]), 1.0f / kLsScale, big[v]);
    }
};

}  // namespace bnb
