// limbs.hpp — fp32 activations as two f16 limbs and quantisation codes as
// exact f16, the operands of the batched prefill's f16 MFMA (prefill.hip).
#pragma once

#include "device.hpp"

namespace nut {

// An activation the GEMMs read as two f16 limbs: hi = f16(v), lo =
// f16(v - hi), so hi + lo carries v to about 2^-22 relative.
// v as an fp32 value in a register, opaque to the optimiser: otherwise the
// multiply that produced v may be folded into either conversion (fma_mix
// from the unrounded product) but not the other, and hi + lo then misses v
// by an f16 ulp where the two roundings part (measured: rel-L2 5e-5 on the
// K/V rows of a batched prefill instead of 5e-7).
__device__ __forceinline__ float settle(float v)
{
    asm("" : "+v"(v));
    return v;
}

__device__ __forceinline__ void put_limbs(_Float16 *hi, _Float16 *lo, size_t i, float v)
{
    v = settle(v);
    const _Float16 a = (_Float16)v;
    hi[i] = a;
    lo[i] = (_Float16)(v - (float)a);
}

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));

// put_limbs of four consecutive values, i a multiple of 4: one 8-byte store
// per limb.
__device__ __forceinline__ void put_limbs4(_Float16 *hi, _Float16 *lo, size_t i, float4 v)
{
    v = make_float4(settle(v.x), settle(v.y), settle(v.z), settle(v.w));
    half4v a, b;
    a.x = (_Float16)v.x;
    a.y = (_Float16)v.y;
    a.z = (_Float16)v.z;
    a.w = (_Float16)v.w;
    b.x = (_Float16)(v.x - (float)a.x);
    b.y = (_Float16)(v.y - (float)a.y);
    b.z = (_Float16)(v.z - (float)a.z);
    b.w = (_Float16)(v.w - (float)a.w);
    *reinterpret_cast<half4v *>(hi + i) = a;
    *reinterpret_cast<half4v *>(lo + i) = b;
}

// put_limbs of two consecutive values, i even: one 4-byte store per limb.
__device__ __forceinline__ void put_limbs2(_Float16 *hi, _Float16 *lo, size_t i, float2 v)
{
    v = make_float2(settle(v.x), settle(v.y));
    half2v a, b;
    a.x = (_Float16)v.x;
    a.y = (_Float16)v.y;
    b.x = (_Float16)(v.x - (float)a.x);
    b.y = (_Float16)(v.y - (float)a.y);
    *reinterpret_cast<half2v *>(hi + i) = a;
    *reinterpret_cast<half2v *>(lo + i) = b;
}

typedef _Float16 half8 __attribute__((ext_vector_type(8)));

// Two quantisation codes as two f16 (exact): an offset-binary code u sits
// in the low byte of an f16 whose high byte is 0x64, which is the value
// 1024 + u; subtracting 1024 + bias gives the code. `pair` holds such a
// word for two codes.
__device__ __forceinline__ uint32_t codes_from_pair(uint32_t pair, float bias)
{
    const half2v v = __builtin_bit_cast(half2v, pair) -
                     half2v{(_Float16)(1024.0f + bias), (_Float16)(1024.0f + bias)};
    return __builtin_bit_cast(uint32_t, v);
}

// Eight codes (k = 8 g .. 8 g + 7 of one row) as f16: INT8 from 8 bytes,
// INT4 from 4 bytes (even k in the low nibble).
template <int QT>
__device__ __forceinline__ half8 codes8(uint2 raw)
{
    uint32_t out[4];
    if (QT == 1) {
        const uint32_t t = raw.x ^ 0x88888888u, s4 = t >> 4;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const uint32_t sel = 0x0c000c00u | uint32_t(4 + b) << 16 | uint32_t(b);
            out[b] = codes_from_pair((__builtin_amdgcn_perm(s4, t, sel) & 0x000f000fu) |
                                         0x64006400u,
                                     8.0f);
        }
    } else {
        const uint32_t words[2] = {raw.x, raw.y};
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t t = words[j] ^ 0x80808080u;
            out[2 * j] = codes_from_pair(__builtin_amdgcn_perm(0x64646464u, t, 0x04010400u), 128.0f);
            out[2 * j + 1] =
                codes_from_pair(__builtin_amdgcn_perm(0x64646464u, t, 0x04030402u), 128.0f);
        }
    }
    return __builtin_bit_cast(half8, make_uint4(out[0], out[1], out[2], out[3]));
}

} // namespace nut
