// x as fp16 rows with power-of-two exponents (x16), the activations of the int4 dense gate/up: written by k_x16, or by the
// router's launches when a layer call feeds those tiles.
#pragma once
#include "moe_common.h"
#include "moe_internal.h"

namespace moe {

// Power-of-two exponent e with which the int4 dense tiles store a row (x16: a token's x; h16: a slot's 32-row chunk
// of h) of largest magnitude amax as fp16 v 2^-e: 0 while 2^-8 <= amax < 2^15 (fp16's subnormal rounding, 2^-25,
// then stays below 2^-17 of the row's largest), else floor(log2 amax) - 14, which puts the largest at [2^14, 2^15)
// (large rows: no overflow; small rows: no flush to zero), clamped to [-127, 127]. An all-zero row gives
// H16_ZERO_EXP, which never wins a slot's maximum (its values are 0 under any scaling); NaN gives 0.
constexpr int H16_ZERO_EXP = -128;
__device__ __forceinline__ int h16_exponent(float amax) {
    if (amax == 0.f) return H16_ZERO_EXP;
    if (!(amax < 32768.f && amax >= 0.00390625f)) {
        if (amax != amax) return 0;
        const int e = (int)((__float_as_uint(amax) >> 23) & 0xFFu) - 141;
        return e < -127 ? -127 : (e > 127 ? 127 : e);
    }
    return 0;
}
// 8 activations of x (bf16, fp16 or fp32) starting at element 8c of row `row`, as fp32
template <int XDT>
__device__ __forceinline__ void load_x8(const void* row, int c, float v[8]) {
    if (XDT == MOE_DTYPE_F32) {
        const float4 a = reinterpret_cast<const float4*>(row)[2 * c], b = reinterpret_cast<const float4*>(row)[2 * c + 1];
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
        return;
    }
    const uint4 r = reinterpret_cast<const uint4*>(row)[c];
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (XDT == MOE_DTYPE_F16) {
            v[2 * q] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[q] & 0xFFFFu));
            v[2 * q + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[q] >> 16));
        } else {
            v[2 * q] = bf16lo(w[q]);
            v[2 * q + 1] = bf16hi(w[q]);
        }
    }
}

// One wave, token t: x [T, d] (bf16, fp16 or fp32) -> x16 = x 2^-E fp16 and E, E = h16_exponent of the row's largest |x|
// (bf16 and fp16 to fp16 are then exact except far below the row's largest, where fp16's subnormal range rounds); E goes to
// the gate/up epilogue. o.xsum (the exact-weight gate/up): also the sums of x16 over the 64-input groups, 16 bytes per
// token and 128-input slice in A-operand form: XS 2^-6 of its two groups as fp16 hi + lo, (hi0, hi1, hi0, hi1, lo0, lo1, 0,
// 0). x16 then takes the exponent that puts every row's largest at [2^14, 2^15), so that bf16 rows keep inputs down to
// 2^-38 of it.
template <int XDT>
__device__ __forceinline__ void x16_row(const void* __restrict__ x, int t, const X16Out& o, int d) {
    const int lane = threadIdx.x & 63;
    const void* row = reinterpret_cast<const uint8_t*>(x) + (size_t)t * d * (XDT == MOE_DTYPE_F32 ? 4 : 2);
    uint4* out = reinterpret_cast<uint4*>(o.x16 + (size_t)t * d);
    const int nch = d >> 3;   // 8-element chunks, a multiple of 8
    constexpr int CPT = 4;    // chunks per lane and round (one round up to d = 2048)
    const bool one = nch <= 64 * CPT;   // the row stays in registers
    float am = 0.f, v[CPT][8];
    for (int c0 = 0; c0 < nch; c0 += 64 * CPT) {
#pragma unroll
        for (int i = 0; i < CPT; ++i)
            if (c0 + i * 64 + lane < nch) load_x8<XDT>(row, c0 + i * 64 + lane, v[i]);
#pragma unroll
        for (int i = 0; i < CPT; ++i)
            if (c0 + i * 64 + lane < nch) {
#pragma unroll
                for (int q = 0; q < 8; ++q) am = fmaxf(am, fabsf(v[i][q]));
            }
    }
    const float amax = wave_max_dpp(am);
    int E = h16_exponent(amax);
    if (o.xsum && E == 0 && amax == amax) E = (int)((__float_as_uint(amax) >> 23) & 0xFFu) - 141;   // ordinary rows too
    if (lane == 0) o.xexp[t] = E;
    for (int c0 = 0; c0 < nch; c0 += 64 * CPT) {   // longer rows: read again (cache hits)
#pragma unroll
        for (int i = 0; i < CPT; ++i)
            if (!one && c0 + i * 64 + lane < nch) load_x8<XDT>(row, c0 + i * 64 + lane, v[i]);
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int c = c0 + i * 64 + lane;
            float sum = 0.f;
            if (c < nch) {
                uint32_t o4[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const _Float16 lo = (_Float16)__builtin_ldexpf(v[i][2 * q], -E), hi = (_Float16)__builtin_ldexpf(v[i][2 * q + 1], -E);
                    o4[q] = (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
                    sum += (float)lo + (float)hi;
                }
                out[c] = make_uint4(o4[0], o4[1], o4[2], o4[3]);
            }
            if (o.xsum) {   // 8 chunks per group, 16 per slice; a slice that ends at input 64 has a zero second group
                sum = sum_lanes<8>(sum);
                const float s1 = __shfl(sum, lane | 8, 64);
                if (c < nch && (c & 15) == 0) {
                    const float w0 = sum * 0x1p-6f, w1 = s1 * 0x1p-6f;
                    const _Float16 h0 = (_Float16)w0, h1 = (_Float16)w1;
                    const _Float16 l0 = (_Float16)(w0 - (float)h0), l1 = (_Float16)(w1 - (float)h1);
                    const uint32_t hh = (uint32_t)__builtin_bit_cast(uint16_t, h0) | ((uint32_t)__builtin_bit_cast(uint16_t, h1) << 16);
                    const uint32_t ll = (uint32_t)__builtin_bit_cast(uint16_t, l0) | ((uint32_t)__builtin_bit_cast(uint16_t, l1) << 16);
                    reinterpret_cast<uint4*>(o.xsum)[(size_t)t * ((d + 127) >> 7) + (c >> 4)] = make_uint4(hh, hh, ll, 0u);
                }
            }
        }
    }
}

}  // namespace moe
