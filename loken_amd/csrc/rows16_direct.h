// The activation of the short 16-row launches (rows16_short.hip, rows16_q6k_short.hip) straight from rows of values: a wave quantizes
// the super-blocks it multiplies.
#pragma once
#include "lk_common.h"

#include <type_traits>

namespace rows16_direct {

enum Src { Q81, ROWS_F32, ROWS_F16, ROWS_BF16 };   // the activation: Q8_1 rows, or rows of values that a wave quantizes itself
// Element, four of them as they lie in memory, and the load of these: rows start on any element (one load either way; 1024 x 4096 at 3 to
// 8 rows off a 16-byte boundary 5.7 us, by way of the quantizer 6.6).
template <int SRC> struct SrcOf {
    typedef float T;
    typedef uint32_t Raw __attribute__((ext_vector_type(4)));
    typedef Raw Load __attribute__((aligned(4)));
};
struct SrcOfHalf {
    typedef uint32_t Raw __attribute__((ext_vector_type(2)));
    typedef Raw Load __attribute__((aligned(2)));
};
template <> struct SrcOf<ROWS_F16> : SrcOfHalf { typedef __half T; };
template <> struct SrcOf<ROWS_BF16> : SrcOfHalf { typedef __hip_bfloat16 T; };
constexpr int CODE_BYTES = 8 * 8 * 32;   // a super-block's codes of eight rows, where the wave quantizes

// Eight rows of a super-block as the stand-alone quantizer codes them (the steps of lk_store_q8_1_block): lane (row lane / 8, piece lane % 8) brings values 4
// piece .. of every sub-block. The divisions are made once for all 64 (row, sub-block)s, each by the lane of the row that has the sub-block's number; rounding
// half away from zero adds the number below one half and cuts, which is roundf for every magnitude below 2^22.
template <typename T, typename Raw>
static __device__ __forceinline__ void quantize(const Raw (&raw)[8], int lane, int m_rows, float* table, uint32_t* codes) {
#pragma clang fp contract(off)
    const int row = lane >> 3, piece = lane & 7;
    float mine = 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const float4 v = Load4<T>::at((const T*)&raw[u]);
        const float amax = max8(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        mine = piece == u ? amax : mine;
    }
    const float d = mine / 127.0f, inv = d != 0.0f ? 1.0f / d : 0.0f;
    table[piece * 8 + row] = row < m_rows ? __half2float(__float2half_rn(d)) : 0.f;
    auto code = [](float x) { return (uint32_t)(int)(x + copysignf(0.49999997f, x)); };
    auto sub = [&](auto u_c) {
        constexpr int U = decltype(u_c)::value;
        const float s = __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(inv), U << 5 | 0x18));   // of lane (row, U)
        const float4 v = Load4<T>::at((const T*)&raw[U]);
        const uint32_t q0 = code(v.x * s), q1 = code(v.y * s), q2 = code(v.z * s), q3 = code(v.w * s);
        const uint32_t lo = __builtin_amdgcn_perm(q1, q0, 0x0C0C0400u), hi = __builtin_amdgcn_perm(q3, q2, 0x04000C0Cu);
        codes[U * 64 + lane] = lo | hi;
    };
    sub(std::integral_constant<int, 0>{}), sub(std::integral_constant<int, 1>{}), sub(std::integral_constant<int, 2>{}), sub(std::integral_constant<int, 3>{});
    sub(std::integral_constant<int, 4>{}), sub(std::integral_constant<int, 5>{}), sub(std::integral_constant<int, 6>{}), sub(std::integral_constant<int, 7>{});
}

}  // namespace rows16_direct
