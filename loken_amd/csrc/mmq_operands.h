// Token rows as the f16 tiles (mmq_tile.h) take them: the Q8_1 quantization of a row, its codes as f16 in the order of the
// matrix instruction's operand, its scales as f32, and d8 * S (S: the sum of a sub-block's codes) for the minimums. Written
// once per call instead of by every workgroup that reads a row. Per (256-value block, row):
//   512 bytes of codes, 64 per sub-block as four atoms 2 hf + h of eight f16 (values 16 h + 8 hf + {0 2 1 3 4 6 5 7});
//    80 bytes of tables: eight f32 d8, then d8 * S as three planes (hi, mid, lo) of eight bf16 that add up to it exactly.
#pragma once

#include "lk_common.h"

constexpr int LK_OPERAND_CODES = 512, LK_OPERAND_TAB = 80;

struct LkTokenOperands {
    uint8_t* codes;   // [block][row][512]
    uint8_t* tabs;    // [block][row][80]
    int64_t rows;     // rows of a block: the tokens and LK_OPERAND_PAD more, which a last tile reads and drops (any bits)
};
constexpr int LK_OPERAND_PAD = 128;

static inline size_t lk_operand_bytes(int64_t tokens, int64_t blocks) {
    return (size_t)blocks * (tokens + LK_OPERAND_PAD) * (LK_OPERAND_CODES + LK_OPERAND_TAB);
}
static inline LkTokenOperands lk_operands_at(void* buffer, int64_t tokens, int64_t blocks) {
    const int64_t rows = tokens + LK_OPERAND_PAD;
    return {(uint8_t*)buffer, (uint8_t*)buffer + blocks * rows * LK_OPERAND_CODES, rows};
}

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
static __device__ __forceinline__ h2 as_h2(uint32_t bits) { return __builtin_bit_cast(h2, bits); }
static __device__ __forceinline__ uint32_t h2_bits(h2 v) { return __builtin_bit_cast(uint32_t, v); }

// Four int8 codes -> f16, as the pairs (0, 2) and (1, 3): byte ^ 0x80 = code + 128, OR-ed into the mantissa of 1024.0 (one
// XOR does both: the constants' bits do not overlap), then 1024 + 128 comes off.
static __device__ __forceinline__ void operand_codes(uint32_t u, uint32_t& even, uint32_t& odd) {
    const h2 bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    even = h2_bits(as_h2((u & 0x00FF00FFu) ^ 0x64806480u) - bias);
    odd = h2_bits(as_h2(((u >> 8) & 0x00FF00FFu) ^ 0x64806480u) - bias);
}

// The table entries of sub-block s: d8 and d8 * S as three bf16 (truncations of the running remainder: 8 bits each, 11 + 13 in all).
static __device__ __forceinline__ void operand_scales(uint8_t* tab, int s, float d8, int sum) {
    const float p0 = d8 * (float)sum;
    const uint32_t b0 = __float_as_uint(p0) & 0xFFFF0000u;
    const float p1 = p0 - __uint_as_float(b0);
    const uint32_t b1 = __float_as_uint(p1) & 0xFFFF0000u;
    const float p2 = p1 - __uint_as_float(b1);
    *(float*)(tab + 4 * s) = d8;
    *(uint16_t*)(tab + 32 + 2 * s) = (uint16_t)(b0 >> 16);
    *(uint16_t*)(tab + 48 + 2 * s) = (uint16_t)(b1 >> 16);
    *(uint16_t*)(tab + 64 + 2 * s) = (uint16_t)(__float_as_uint(p2) >> 16);
}

// Four consecutive values of a 32-value sub-block, from value 4 l8 on, by each of the eight lanes of an aligned group: the
// Q8_1 rule of the records' quantizer (d = amax / 127, codes = round_half_away(x * (1 / d)), d kept as f16), straight into
// the operands of its row.
static __device__ __forceinline__ void operand_quad(float4 v, uint8_t* codes, uint8_t* tab, int s, int l8) {
    float d;
    int sum;
    {
#pragma clang fp contract(off)
        const float amax = max8(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        d = amax / 127.0f;
        const float inv = d != 0.0f ? 1.0f / d : 0.0f;
        const int q0 = (int)roundf(v.x * inv), q1 = (int)roundf(v.y * inv), q2 = (int)roundf(v.z * inv), q3 = (int)roundf(v.w * inv);
        int quad_sum;
        sum = sum8(q0 + q1 + q2 + q3, quad_sum);
        uint2 o;
        operand_codes((uint32_t)(q0 & 0xFF) | (uint32_t)(q1 & 0xFF) << 8 | (uint32_t)(q2 & 0xFF) << 16 | (uint32_t)(q3 & 0xFF) << 24, o.x, o.y);
        // value 16 h + 8 hf + 4 i is half i of atom 2 hf + h
        *(uint2*)(codes + 64 * s + 32 * ((l8 >> 1) & 1) + 16 * (l8 >> 2) + 8 * (l8 & 1)) = o;
    }
    if (l8 == 0) operand_scales(tab, s, __half2float(__float2half_rn(d)), sum);
}
