// Q4_K, Q5_K, Q6_K, Q8_0 and Q4_0 weight rows against Q8_1 token rows: the sub-block dots on the f16 matrix unit.
//
//   out[token, n] = sum over 256-value blocks of
//        d[n] * sum_s d8_s[token] * D_s[n, token]  -  dmin[n] * sum_s m_s[n] * (d8_s * S_s)[token]
//   D_s[n, token] = sum over the 32 values of sub-block s of (sc[n] * q[n, k]) * a[token, k]
//
// The same integers as the int8 tiles form (sc * dot of the codes and the int8 codes: loken's BlockQ4K::dot_scalar,
// src/tensor/quant_cpu/format/q4_k.rs:138-153, q6_k.rs:137-160, combined as cuda/moe/gguf.cuh:664-713, 782-816 combine
// them), reached another way. An int8 matrix instruction leaves dot_s, which still has to meet two factors per output
// element, sc_s[n] and d8_s[token]: a convert and two multiplies on the vector unit per element and sub-block. Here the
// scale rides into the matrix unit with the weight: sc * q (at most 63 * 15, Q5_K 63 * 31) is exact in f16, so is an int8
// code, their products and the 32-term sums are exact in the f32 accumulator (< 2^24). D_s leaves the unit as a float that
// already carries the weight scale, and one fma by the lane's d8 finishes it.
// Q6_K's signed scales meet six-bit codes: |sc * q| <= 128 * 32 has one bit more than f16 holds. The operand is the
// product rounded to f16 and a second one carries what the rounding took (-1, 0 or 1, exact); both terms add up in the
// same accumulator, still exactly (128 * 32 * 127 * 32 < 2^24), four matrix instructions per sub-block instead of two.
// Q8_0, Q4_0, IQ4_NL and MXFP4 have no integer scale: their codes or levels are the operand (128 * 127 * 32 < 2^24), see TileSub.
//
// Shape: a wave owns 32 weight rows x TT token tiles of 32 (registers <-> weight rows, lanes <-> tokens,
// v_mfma_f32_32x32x16_f16 called as weights x tokens), so that the expansion of its rows is shared by TT items. Four waves
// and 80 KiB make a workgroup, two of them share a CU: its SIMDs then hold two waves that meet at no common barrier, and one
// tile's first loads and stores run under the other's products. Token operands come expanded (LkTokenOperands) and, like
// the weights of the 16-byte aligned formats, go to LDS without passing through registers.
// What bounds it: the issue of vector and matrix instructions (probe: two waves of [2 matrix + 16 fma] take 85 cycles an
// item, the whole item of Q4_K 143, of Q6_K 184 at TT = 4), and the clock with it, which falls from 2.4 GHz to 1.8 under
// this load: what a variant gains in cycles it gives back in clock. So fewer instructions and bytes per item count, stalls hardly:
// eight waves of one workgroup at twice the rows take 163 cycles at 1.91 GHz where two of four take 143 at 1.81.
// Measured (us, matmul alone, against the 64-token tiles that expanded the tokens in every workgroup, one workgroup a CU):
// Q6_K 4096 x 14336 at 2048 rows 545 -> 440 (TT = 2, 3, 4: 529, 504, 440), Q5_K 14336 x 4096 at 512 rows 128 -> 91, Q4_K 92 -> 88.
//
// K order inside a sub-block: lane half h (lane / 32) of matrix instruction hf holds values 16 h + 8 hf + i,
// i in the order 0 2 1 3 4 6 5 7 (what masking a dword's even and odd bytes yields); weights and
// tokens use the same order, which is all a dot product asks. (A lane half holds one of Q6_K's 16-value groups.)
#pragma once

#include "legacy_blocks.h"
#include "mmq_operands.h"
#include "mmq_problem.h"

#include <type_traits>
#include <utility>

namespace mmq_tile {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

constexpr uint32_t H1024 = 0x64006400u;   // two f16 1024.0: OR-ing an 8-bit integer into the mantissa adds it

// ------------------------------------------------------------------ weight formats
// A block reaches LDS in 16-byte pieces, in two regions per row that are each read once and free after that: A (AP pieces:
// header or scales and the first half of the codes) and B (BP pieces: the second half), so that one stage is enough and the
// next block's pieces have most of a block's time to arrive. a_src / b_src: where piece p lies in the block, place: its place in the
// row's region (formats through registers). UNIT: what `row_blocks` counts, in bytes. DMA: blocks are
// 16-byte aligned and go to LDS directly; else through registers. Row strides are an odd number of pieces, or the pieces of
// a row are exchanged by its number (B of Q4_K / Q5_K), so that 32 rows spread over the banks (Q6_K's six: two rows a bank).
// Codes: what a lane needs of half a block (four sub-blocks). Raw: its row's header as it lies, Header: what prepare() makes of it.
// operand(): the lane's eight values of matrix instruction hf of sub-block s, times the scale, as TERMS f16 operands; where
// that needs no offset the codes stay where they are in the f16's mantissa, q * 2^-24, and the scale is the larger power of two that keeps
// the product an f16 (Q4_K, Q5_K; D_UP takes it out of the products again with the row's d, exactly: the same bits as codes OR-ed into
// 1024.0 and an offset gave. With the scales unpacked four at a time a block of Q4_K takes 52 vector instructions less of 755 at TT = 4, of
// 368 at TT = 1: 14336 x 4096 at 512 rows 91.4 -> 89.3 us, 128 experts of 2048 -> 768 at 256 tokens, top-8, 139.5 -> 136.3).
struct Scale16 { h2 scale, offset; };
static __device__ __forceinline__ h2 both(h2 v, int half) { return half ? __builtin_shufflevector(v, v, 1, 1) : __builtin_shufflevector(v, v, 0, 0); }
// bytes 0 | 2 and 1 | 3 of a word as halves
static __device__ __forceinline__ uint32_t even_bytes(uint32_t w) { return __builtin_amdgcn_perm(0, w, 0x0C020C00u); }
static __device__ __forceinline__ uint32_t odd_bytes(uint32_t w) { return __builtin_amdgcn_perm(0, w, 0x0C030C01u); }

// A code of a format with a plane of high bits is put together as a byte, four to an instruction, and the bytes 0 | 2 and
// 1 | 3 leave for the mantissas of two 1024.0 in one v_perm_b32 each (masking and shifting the high bits per pair of
// halves instead took 312 vector instructions of a Q6_K block for 184).
static __device__ __forceinline__ uint32_t bits_from(uint32_t w, int up, uint32_t mask) {
    return (up >= 0 ? w << (up & 31) : w >> (-up & 31)) & mask;
}
static __device__ __forceinline__ uint32_t even_codes(uint32_t c, uint32_t h1024) { return __builtin_amdgcn_perm(h1024, c, 0x07020500u); }
static __device__ __forceinline__ uint32_t odd_codes(uint32_t c, uint32_t h1024) { return __builtin_amdgcn_perm(h1024, c, 0x07030501u); }

template <bool Q5>
struct TileQ45K {
    static constexpr int BYTES = Q5 ? Q5K_BYTES : Q4K_BYTES, UNIT = BYTES, ALIGN = 16, TERMS = 1;
    static constexpr bool HAS_MIN = true, D_PER_SUB = false;
    static constexpr int TT_MOST = 4;
    static constexpr int AP = Q5 ? 7 : 5, BP = 4;
    static constexpr bool DMA = true;
    static __host__ __device__ constexpr int a_src(int p) { return 16 * p; }
    static __device__ __forceinline__ int b_src(int p, int row) { return 16 * AP + 16 * (p ^ ((row >> 1) & 3)); }
    struct Raw { uint4 w; };
    struct Header { uint32_t dm, mins[2]; h2 sc[4]; };   // d | dmin; the eight minimums' bytes; scales 0 | 2, 1 | 3, 4 | 6, 5 | 7
    struct Codes { uint4 q[2], qh; uint32_t up[4]; };
    static __device__ __forceinline__ Raw raw_header(const uint8_t* ra) { return {*(const uint4*)ra}; }
    static __device__ __forceinline__ void codes0(Codes& c, const uint8_t* ra, int h, int row) {
        (void)row;
#pragma unroll
        for (int p = 0; p < 2; ++p) c.q[p] = *(const uint4*)(ra + (Q5 ? 48 : 16) + 32 * p + 16 * h);
        if (Q5) c.qh = *(const uint4*)(ra + 16 + 16 * h);
    }
    static __device__ __forceinline__ void codes1(Codes& c, const uint8_t* rb, int h, int row) {
#pragma unroll
        for (int p = 0; p < 2; ++p) c.q[p] = *(const uint4*)(rb + 16 * ((2 * p + h) ^ ((row >> 1) & 3)));
    }
    // The six-bit scales and minimums (get_scale_min_k4 of the format) four to a word, then two scales to a register:
    // 16 vector instructions a block for the eight scales, where one at a time took 44. A scale carries 2^10; Q4_K's odd sub-blocks, whose nibbles
    // stay four bits up, 2^6: products sc * q * 2^-14, every one but zero a normal f16.
    static constexpr float D_UP = 16384.0f;
    static __device__ __forceinline__ Header prepare(const Raw& r, int h) {
        (void)h;
        const uint32_t sc[2] = {r.w.y & 0x3F3F3F3Fu, (r.w.w & 0x0F0F0F0Fu) | ((r.w.y >> 2) & 0x30303030u)};
        Header hd{r.w.x, {r.w.z & 0x3F3F3F3Fu, ((r.w.w >> 4) & 0x0F0F0F0Fu) | ((r.w.z >> 2) & 0x30303030u)}, {}};
        const h2 base = {(_Float16)1024.0f, (_Float16)1024.0f};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const _Float16 up = (_Float16)(!Q5 && (i & 1) ? 64.0f : 1024.0f);
            hd.sc[i] = (as_h2(i & 1 ? odd_codes(sc[i >> 1], H1024) : even_codes(sc[i >> 1], H1024)) - base) * h2{up, up};
        }
        return hd;
    }
    static __device__ __forceinline__ uint32_t min_of(const Header& hd, int s) { return (hd.mins[s >> 2] >> (8 * (s & 3))) & 0xFFu; }
    static __device__ __forceinline__ Scale16 scale(const Header& hd, int s) { return {both(hd.sc[(s >> 2) * 2 + (s & 1)], (s >> 1) & 1), {}}; }
    static __device__ __forceinline__ void operand(Codes& cd, int s, int hf, const Scale16& sc, uint32_t h1024, v8h a[TERMS]) {
        (void)h1024;
        const uint4 q = cd.q[(s >> 1) & 1];
        const uint32_t u[4] = {q.x, q.y, q.z, q.w}, b[4] = {cd.qh.x, cd.qh.y, cd.qh.z, cd.qh.w};
        const bool high = (s & 1) != 0;
        uint32_t ab[4];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const uint32_t x = u[2 * hf + e];
            uint32_t even, odd;
            if constexpr (Q5) {   // bit s of the byte goes on top of the nibble
                const uint32_t c = bits_from(b[2 * hf + e], 4 - s, 0x10101010u) | ((high ? x >> 4 : x) & 0x0F0F0F0Fu);
                even = even_bytes(c);
                odd = odd_bytes(c);
            } else {
                const uint32_t mask = high ? 0x00F000F0u : 0x000F000Fu;
                if (!high) cd.up[2 * hf + e] = x >> 8;   // the odd sub-block of the pair takes it from here
                even = x & mask;
                odd = cd.up[2 * hf + e] & mask;
            }
            ab[2 * e] = h2_bits(as_h2(even) * sc.scale);
            ab[2 * e + 1] = h2_bits(as_h2(odd) * sc.scale);
        }
        a[0] = __builtin_bit_cast(v8h, make_uint4(ab[0], ab[1], ab[2], ab[3]));
    }
};

struct TileQ6K {
    static constexpr int BYTES = Q6K_BYTES, UNIT = BYTES, ALIGN = 2, TERMS = 2;   // its d, two bytes past the 13 pieces, travels by itself
    static constexpr bool HAS_MIN = false, D_PER_SUB = false;
    static constexpr int TT_MOST = 4;
    static constexpr int AP = 7, BP = 6;
    static constexpr bool DMA = false;
    static __host__ __device__ constexpr int a_src(int p) { return p < 4 ? 16 * p : p < 6 ? 128 + 16 * (p - 4) : 192; }
    static __device__ __forceinline__ int b_src(int p, int row) { (void)row; return p < 4 ? 64 + 16 * p : 160 + 16 * (p - 4); }
    static __device__ __forceinline__ int place(int p, int row) { (void)row; return p; }
    struct Raw { uint4 w; };
    struct Header { uint32_t sc[4]; };   // bytes 0 and 2 of word s / 2: the scales of the lane's 16 values of sub-blocks s and s + 1
    struct Codes { uint4 q[2], qh; };
    static constexpr float D_UP = 1.0f;
    static __device__ __forceinline__ Raw raw_header(const uint8_t* ra) { return {*(const uint4*)(ra + 96)}; }
    static __device__ __forceinline__ Header prepare(const Raw& r, int h) { return {{r.w.x >> (8 * h), r.w.y >> (8 * h), r.w.z >> (8 * h), r.w.w >> (8 * h)}}; }
    static __device__ __forceinline__ void codes0(Codes& c, const uint8_t* ra, int h, int row) {
        (void)row;
#pragma unroll
        for (int p = 0; p < 2; ++p) c.q[p] = *(const uint4*)(ra + 32 * p + 16 * h);
        c.qh = *(const uint4*)(ra + 64 + 16 * h);
    }
    static __device__ __forceinline__ void codes1(Codes& c, const uint8_t* rb, int h, int row) {
        codes0(c, rb, h, row);
    }
    // (The scale's even part and its last bit as the two operands, both on codes left where they lie, would be two vector instructions
    // a pair of codes instead of three, but a dense second operand: 4096 x 14336 at 2048 rows 525 us against 508. This one is zeros
    // but for odd products past 2048, and the matrix unit's power, which sets the clock here, follows its operands.)
    static __device__ __forceinline__ Scale16 scale(const Header& hd, int s) {
        const _Float16 a = (_Float16)(float)(int8_t)((hd.sc[s >> 1] >> (16 * (s & 1))) & 0xFFu);
        const _Float16 b = (_Float16)-1056.0f;
        return {{a, a}, {b, b}};
    }
    static __device__ __forceinline__ void operand(const Codes& cd, int s, int hf, const Scale16& sc, uint32_t h1024, v8h a[TERMS]) {
        const int g = s & 3;
        const uint4 q = cd.q[g & 1];
        const uint32_t u[4] = {q.x, q.y, q.z, q.w}, b[4] = {cd.qh.x, cd.qh.y, cd.qh.z, cd.qh.w};
        uint32_t t0[4], t1[4], c[2];
#pragma unroll
        for (int e = 0; e < 2; ++e)
            c[e] = bits_from(b[2 * hf + e], 4 - 2 * g, 0x30303030u) | ((g >= 2 ? u[2 * hf + e] >> 4 : u[2 * hf + e]) & 0x0F0F0F0Fu);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t x = e & 1 ? odd_codes(c[e >> 1], h1024) : even_codes(c[e >> 1], h1024);
            const h2 code = as_h2(x) + sc.offset;   // 1024 + code - 1056: -32 .. 31
            const h2 v = code * sc.scale;
            t0[e] = h2_bits(v);
            t1[e] = h2_bits(__builtin_elementwise_fma(code, sc.scale, -v));   // what the rounding took
        }
        a[0] = __builtin_bit_cast(v8h, make_uint4(t0[0], t0[1], t0[2], t0[3]));
        a[1] = __builtin_bit_cast(v8h, make_uint4(t1[0], t1[1], t1[2], t1[3]));
    }
};
using TileQ4K = TileQ45K<false>;
using TileQ5K = TileQ45K<true>;

// Q8_0, Q4_0, IQ4_NL and MXFP4: eight 32-value blocks make a block here, each with a d of its own that no integer scale takes into the matrix
// unit: the codes are the operand, and a sub-block's dots meet d8 and its rows' d (D_PER_SUB) on their way into the sums, two
// vector instructions an element, as f32. An item costs 32 of them and the two matrix instructions, and nothing folds at a block's end. Measured
// (us, a linear of f32 rows, against the int8 tiles): Q8_0 14336 x 4096 at 17 / 96 / 512 / 2048 rows 47 / 83 / 158 / 695 -> 32 / 52 / 146 / 521,
// 11003 x 4096 at 40 rows 97 -> 40, Q4_0 4096 x 14336 at 512 rows 184 -> 134, 2048 x 4096 at 17 rows 17.4 -> 16.1. Pieces are placed by the row's number (their rows in LDS are 128 and 64 bytes).
template <int ID>
struct TileSub {
    static constexpr bool Q4 = ID != LK_TYPE_Q8_0;   // 16 bytes of nibbles a sub-block
    using L = Legacy<Q4 ? ID : LK_TYPE_Q4_0>;
    static constexpr int UNIT = Q4 ? L::BYTES : Q80_BYTES, BYTES = 8 * UNIT, ALIGN = UNIT % 2 ? 1 : 2, TERMS = 1;
    static constexpr bool HAS_MIN = false, D_PER_SUB = true;
    static constexpr int TT_MOST = Q4 ? 4 : 3;   // what LDS has room for
    static constexpr int AP = Q4 ? 4 : 8, BP = AP;
    static constexpr bool DMA = false;
    static __host__ __device__ constexpr int a_src(int p) { return Q4 ? UNIT * p + L::QS_AT : UNIT * (p >> 1) + 2 + 16 * (p & 1); }
    static __device__ __forceinline__ int b_src(int p, int row) { (void)row; return 4 * UNIT + a_src(p); }
    // d as it lies (one byte of MXFP4's E8M0, else f16), and its value
    static __device__ __forceinline__ uint16_t scale_bits(const uint8_t* p) { return UNIT % 2 ? *p : *(const uint16_t*)p; }
    static __device__ __forceinline__ float scale_value(uint16_t bits) { return L::TABLE == 2 ? e8m0_half(bits) : f16_bits_to_f32(bits); }
    static __device__ __forceinline__ int place(int p, int row) { return Q4 ? p ^ ((row >> 1) & 3) : p ^ (row & 7); }
    struct Raw {};
    struct Header {};
    struct Codes { uint4 q[4]; };
    static constexpr float D_UP = 1.0f;
    static __device__ __forceinline__ Raw raw_header(const uint8_t* ra) { (void)ra; return {}; }
    static __device__ __forceinline__ Header prepare(const Raw& r, int h) { (void)r; (void)h; return {}; }
    static __device__ __forceinline__ void codes0(Codes& c, const uint8_t* ra, int h, int row) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            c.q[p] = *(const uint4*)(ra + 16 * place(Q4 ? p : 2 * p + h, row));
            if (Q4) {   // values 0 .. 15 are the low nibbles, 16 .. 31 the high ones
                c.q[p].x >>= 4 * h; c.q[p].y >>= 4 * h; c.q[p].z >>= 4 * h; c.q[p].w >>= 4 * h;
            }
        }
    }
    static __device__ __forceinline__ void codes1(Codes& c, const uint8_t* rb, int h, int row) { codes0(c, rb, h, row); }
    static __device__ __forceinline__ Scale16 scale(const Header& hd, int s) {
        (void)hd; (void)s;
        const _Float16 b = (_Float16)(Q4 && !L::TABLE ? -1032.0f : -1152.0f);   // levels and Q8_0's codes are int8
        return {{b, b}, {b, b}};
    }
    static __device__ __forceinline__ void operand(const Codes& cd, int s, int hf, const Scale16& sc, uint32_t h1024, v8h a[TERMS]) {
        const uint4 q = cd.q[s & 3];
        const uint32_t u[4] = {q.x, q.y, q.z, q.w};
        uint32_t ab[4];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            uint32_t c = u[2 * hf + e];
            if (Q4) c &= 0x0F0F0F0Fu;
            if (Q4 && L::TABLE) c = levels_of<L::TABLE>(c);
            if (!Q4 || L::TABLE) c ^= 0x80808080u;
            ab[2 * e] = h2_bits(as_h2(even_codes(c, h1024)) + sc.offset);
            ab[2 * e + 1] = h2_bits(as_h2(odd_codes(c, h1024)) + sc.offset);
        }
        a[0] = __builtin_bit_cast(v8h, make_uint4(ab[0], ab[1], ab[2], ab[3]));
    }
};
using TileQ80 = TileSub<LK_TYPE_Q8_0>;
using TileQ40 = TileSub<LK_TYPE_Q4_0>;
using TileIq4Nl = TileSub<LK_TYPE_IQ4_NL>;
using TileMxfp4 = TileSub<LK_TYPE_MXFP4>;

// ------------------------------------------------------------------ movement
// 64 lanes x 16 bytes from global memory straight into LDS: uniform base + the lane's 32-bit offset on the global side;
// lane i's bytes land at wave_base + 16 i. Written out, because for the builtin the compiler waits for every load in flight
// before each LDS access that it cannot tell apart from its target; here `meet` waits for what is needed.
static __device__ __forceinline__ void to_lds16(const uint8_t* base, uint32_t lane_off, uint32_t wave_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane((int)wave_base)),
                 "v"(lane_off), "s"(base)
                 : "m0");
}

// This wave's LDS accesses are done and of its loads at most the latest KEEP are in flight; then the workgroup's barrier.
// The memory clobber keeps the compiler from moving memory accesses across it.
template <int KEEP>
static __device__ __forceinline__ void meet() {
    static_assert(KEEP >= 0 && KEEP < 64, "the counter's range");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(KEEP) : "memory");
}

// What other lanes of this wave wrote to LDS before is read after, and the other way round: LDS serves a wave's
// accesses in order, so only the compiler has to keep them there.
static __device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The tile's plan, for TT token tiles and WAVES waves. Items (sub-block, token tile) of a block run in slots 0 .. NI - 1;
// a quarter is the two sub-blocks whose token codes travel together, one barrier each.
template <class F, int TT, int WAVES>
struct TileShape {
    static constexpr int THREADS = 64 * WAVES, ROWS = 32 * WAVES;
    static constexpr int NI = 8 * TT, QI = 2 * TT;
    // Quarters of token codes in LDS, and how far ahead they are loaded. Two where LDS has to leave room for a second
    // workgroup (80 KiB each).
    static constexpr int NQ = TT >= 3 && WAVES == 4 ? 2 : 4, LEAD = NQ - 1;
    static constexpr int QB = 4096 * TT;                                    // bytes of a quarter's codes
    static constexpr int CC = (4 * TT + WAVES - 1) / WAVES;                 // its 1 KiB chunks, per wave
    static constexpr int TCH = (5 * TT + 1) / 2, RC = (TCH + WAVES - 1) / WAVES, TABB = TCH * 1024;   // a block's token tables, likewise
    // wave loads of a block's weights, A then B; through registers a load takes eight rows, eight lanes (pieces) each
    static constexpr int AC = F::DMA ? (32 * F::AP + 63) / 64 : 4, BC = F::DMA ? (32 * F::BP + 63) / 64 : 4, CH = AC + BC;
    static constexpr int A_ROW = 16 * F::AP, B_ROW = 16 * F::BP;
    static constexpr int A_BYTES = F::DMA ? AC * 1024 : 32 * A_ROW, W_BYTES = A_BYTES + 32 * B_ROW;
    // LDS: ring of quarters, two blocks' tables, each wave's weights, each wave's d of its rows for two blocks (D_PER_SUB: of one)
    static constexpr int D_ROW = 36, D_BYTES = F::D_PER_SUB ? 8 * D_ROW * 4 : 256;   // d of a sub-block: 32 floats and 16 bytes to spread the banks
    static constexpr int T_AT = 0, TAB_AT = NQ * QB, W_AT = TAB_AT + 2 * TABB, D_AT = W_AT + WAVES * W_BYTES, LDS = D_AT + WAVES * D_BYTES;
    static_assert(LDS <= (WAVES == 4 ? 80 : 160) * 1024, "LDS of a workgroup");
    // Slots in which weights are loaded: directly, a region's next pieces right after the slot that has read it (A, read in slot
    // 7 TT - 1 for the next block: the block after that; B, in 3 TT - 1: the next block), so that they have almost a block's time.
    // Through registers, with few token tiles a piece is in flight for a whole block (LONG: the block after the next), with
    // many for 2 TT slots, which leaves registers; stored in commit_slot.
    static constexpr bool LONG = TT <= 2;
    static constexpr int commit_slot(int i) {
        const int c = (i < AC ? i + 2 : i + 1) * TT;
        return F::DMA ? -1 : c < NI ? c : NI - 1;
    }
    static constexpr int fetch_slot(int i) {
        return F::DMA ? (i < AC ? 7 * TT + i * TT / AC : 3 * TT + (i - AC) * TT / BC) : LONG ? commit_slot(i) : commit_slot(i) - 2 * TT;
    }
    // Direct loads a wave issues in slot I. (Loads into registers, which the compiler places, are left out: `keep` then asks
    // for more than it has to and never for less.)
    static constexpr int direct(int I) {
        I = (I % NI + NI) % NI;
        const int q = I / QI, r = I % QI;
        int n = (r < CC) + (q == 1 && r >= CC && r < CC + RC);
        for (int i = 0; F::DMA && i < CH; ++i) n += fetch_slot(i) == I;
        return n;
    }
    static constexpr int later(int a, int b) { return a > b ? a : b; }
    // Loads that may still be in flight at quarter q's barrier, in slot QI - 2 of the quarter: all issued after the last one
    // that the slots up to the next barrier read.
    static constexpr int keep(int q) {
        int last = (q + 1 - LEAD) * QI + CC - 1;                             // codes of quarter q + 1
        if (q == 3) last = later(last, QI + CC + RC - 1);                    // the next block's tables
        // the next block's A, read in slot 7 TT - 1, and this block's B, in 3 TT - 1: the last barriers before
        if (F::DMA && q == (TT == 1 ? 3 : 2)) last = later(last, fetch_slot(AC - 1) - NI);
        if (F::DMA && q == (TT == 1 ? 1 : 0)) last = later(last, fetch_slot(CH - 1) - NI);
        int n = 0;
        for (int I = last + 1; I < q * QI + QI - 2; ++I) n += direct(I);
        return n;
    }
};

// What a wave carries through the pipeline. Every index into the arrays is a compile-time constant (the slots are template
// instances), so all of it lives in registers.
template <class F, int TT, int WAVES, bool GATHER>
struct TileWave {
    using S = TileShape<F, TT, WAVES>;
    static constexpr int NI = S::NI, QI = S::QI, TERMS = F::TERMS;
    using piece = typename std::conditional<F::ALIGN == 16, uint4, typename std::conditional<F::ALIGN == 1, uint4_a1, uint4_a2>::type>::type;
    // global side: uniform bases, lane offsets
    const uint8_t *codes, *tabs, *w;
    int64_t code_slab, tab_slab, row_bytes8;   // bytes of a block's codes, of its tables, of eight weight rows
    uint32_t code_off[GATHER ? S::CC : 1], tab_off[GATHER ? S::RC : 1], from[F::DMA ? S::CH : 2], d_from;
    uint32_t lds_at;   // LDS address of the tile's memory
    int wave, h, j;
    // LDS side of this lane
    const uint8_t* tb[4];      // its token's atoms (sub-block parity, hf) in the first token tile
    const uint8_t *rp, *mp;    // its token's table record; the hi (lanes 0 .. 31) or mid plane in it
    const uint8_t *ra, *rb;    // its weight row's regions
    uint8_t* wstage;
    float* wd;

    v16f acc[TT], part[F::D_PER_SUB ? 1 : TT], dot[2];
    v8h a[2][TERMS], b[2][2];
    float d8v[4], dv[F::D_PER_SUB ? 2 : 1][16];
    uint4 data[S::CH];
    uint16_t d[F::D_PER_SUB ? 4 : 1];
    typename F::Raw raw;
    typename F::Header hd;
    typename F::Codes cd;
    uint32_t mh[4], mm[4];      // -dmin * min of the row's eight sub-blocks: two bf16 that add up to it exactly
    v8bf m_hi, m_mid, m_x;
    uint4 pb0, pb1;
    uint32_t h1024;

    __device__ __forceinline__ void load_codes(int kb, int q, int c) const {   // chunk wave + WAVES c of quarter q
        const int chunk = 4 * TT % WAVES == 0 ? wave + WAVES * c : min(wave + WAVES * c, 4 * TT - 1);
        to_lds16(codes + kb * code_slab + 128 * q + (GATHER ? 0 : chunk * (8 * LK_OPERAND_CODES)), code_off[GATHER ? c : 0],
                 lds_at + S::T_AT + (q % S::NQ) * S::QB + chunk * 1024);
    }
    __device__ __forceinline__ void load_tabs(int kb, int c) const {
        const int chunk = min(wave + WAVES * c, S::TCH - 1);
        to_lds16(tabs + kb * tab_slab + (GATHER ? 0 : chunk * 1024), tab_off[GATHER ? c : 0], lds_at + S::TAB_AT + (kb & 1) * S::TABB + chunk * 1024);
    }
    __device__ __forceinline__ void fetch(int kb, int i) {
        const uint8_t* block = w + (int64_t)kb * F::BYTES;
        if constexpr (F::DMA)
            to_lds16(block, from[i], lds_at + S::W_AT + wave * S::W_BYTES + (i < S::AC ? i * 1024 : S::A_BYTES + (i - S::AC) * 1024));
        else
            data[i] = *(const piece*)(block + (i & 3) * row_bytes8 + from[i / 4]);
    }
    __device__ __forceinline__ void fetch_d(int kb) {
        const uint8_t* block = w + (int64_t)kb * F::BYTES;
        if constexpr (F::D_PER_SUB) {   // eight rows a load, eight sub-blocks each
#pragma unroll
            for (int i = 0; i < 4; ++i) d[i] = F::scale_bits(block + i * row_bytes8 + d_from);
        } else if constexpr (!F::DMA) d[0] = *(const uint16_t*)(block + d_from);
    }
    __device__ __forceinline__ void commit(int i) const {
        const int lane = threadIdx.x & 63, row = 8 * (i & 3) + (lane >> 3);
        const int at = i < S::AC ? row * S::A_ROW + 16 * F::place(min(lane & 7, F::AP - 1), row)
                                : S::A_BYTES + row * S::B_ROW + 16 * F::place(min(lane & 7, F::BP - 1), row);
        *(uint4*)(wstage + at) = data[i];
    }
    template <int I, int HF>
    __device__ __forceinline__ void load_atom() {
        constexpr int s = I / TT, tt = I % TT;
        b[I & 1][HF] = *(const v8h*)(tb[(s & 1) * 2 + HF] + ((s >> 1) % S::NQ) * S::QB + tt * 4096);
    }
    template <int I>
    __device__ __forceinline__ void load_d8(int parity) {
        constexpr int s = I / TT, tt = I % TT;
        d8v[I & 3] = *(const float*)(rp + parity * S::TABB + tt * (32 * LK_OPERAND_TAB) + 4 * s);
    }
    template <int s>
    __device__ __forceinline__ void operands() {
        const auto sc = F::scale(hd, s);
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) F::operand(cd, s, hf, sc, h1024, a[hf]);
    }
    __device__ __forceinline__ void write_d(int parity) {
        if constexpr (F::D_PER_SUB) {
            const int lane = threadIdx.x & 63;
#pragma unroll
            for (int i = 0; i < 4; ++i) wd[(lane & 7) * S::D_ROW + 8 * i + (lane >> 3)] = F::scale_value(d[i]);
        } else if (h == 0) {
            if constexpr (F::HAS_MIN) wd[parity * 32 + j] = F::D_UP * f16_bits_to_f32(hd.dm & 0xFFFFu);
            else wd[parity * 32 + j] = F::D_UP * f16_bits_to_f32(d[0]);
        }
    }
    template <int TO = 0>
    __device__ __forceinline__ void read_dv(int at) {   // `at`: in rows' d
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const float4 t = *(const float4*)(wd + at + 8 * g + 4 * h);
            dv[TO][4 * g] = t.x; dv[TO][4 * g + 1] = t.y; dv[TO][4 * g + 2] = t.z; dv[TO][4 * g + 3] = t.w;
        }
    }
    // (11 + 6 bits: rounded to bf16 and what the rounding took, eight bits each)
    template <int Q>
    __device__ __forceinline__ void min_pair() {
        typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
        const float ndm = -f16_bits_to_f32(hd.dm >> 16);
        const float x = ndm * (float)F::min_of(hd, 2 * Q), y = ndm * (float)F::min_of(hd, 2 * Q + 1);
        const v2bf hi = {(__bf16)x, (__bf16)y};
        mh[Q] = __builtin_bit_cast(uint32_t, hi);
        const v2bf mid = {(__bf16)(x - __uint_as_float(mh[Q] << 16)), (__bf16)(y - __uint_as_float(mh[Q] & 0xFFFF0000u))};
        mm[Q] = __builtin_bit_cast(uint32_t, mid);
    }
    template <int FROM, int TO, int P>
    __device__ __forceinline__ void fix_up() {
        constexpr int pt = P % TT, ps = P / TT;
        const float d8p = d8v[P & 3];
#pragma unroll
        for (int v = FROM; v < TO; ++v) {
            if constexpr (F::D_PER_SUB) acc[pt][v] = fmaf(dv[ps & 1][v], dot[P & 1][v] * d8p, acc[pt][v]);
            else part[pt][v] = ps == 0 ? dot[P & 1][v] * d8p : fmaf(dot[P & 1][v], d8p, part[pt][v]);
        }
    }
    template <int T>
    __device__ __forceinline__ void fold() {
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[T][v] = fmaf(dv[0][v], part[T][v], acc[T][v]);
    }

    static __device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }
    // Slot I of block kb: the matrix instructions of item I, the 16 fmas of item I - 1 between them (a wave's vector
    // instructions do not issue past a matrix instruction that waits for the one before), the LDS reads of item I + 2 into the
    // operand registers just used, and this slot's share of everything else.
    template <int I>
    __device__ __forceinline__ void slot(int kb, int next, int next2) {
        constexpr int s = I / TT, tt = I % TT, q = I / QI, r = I % QI;
        constexpr int P = (I + NI - 1) % NI, N2 = (I + 2) % NI;
        const int par = kb & 1;
        if constexpr (r == QI - 2) meet<S::keep(q)>();
        if constexpr (r < S::CC) load_codes(q + S::LEAD < 4 ? kb : next, (q + S::LEAD) & 3, r);
        if constexpr (q == 1 && r >= S::CC && r < S::CC + S::RC) load_tabs(next, r - S::CC);
        const int npar = I + 2 >= NI ? par ^ 1 : par;
        {
            const v16f zero = {0.f};
            dot[I & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0][0], b[I & 1][0], zero, 0, 0, 0);
        }
        fence();
        if constexpr (TERMS == 1) {
            load_atom<N2, 0>();
            fix_up<0, 8, P>();
            fence();
            dot[I & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1][0], b[I & 1][1], dot[I & 1], 0, 0, 0);
            fence();
            load_atom<N2, 1>();
            load_d8<N2>(npar);
            fix_up<8, 16, P>();
        } else {
            fix_up<0, 5, P>();
            fence();
            dot[I & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0][1], b[I & 1][0], dot[I & 1], 0, 0, 0);
            fence();
            load_atom<N2, 0>();
            fix_up<5, 10, P>();
            fence();
            dot[I & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1][0], b[I & 1][1], dot[I & 1], 0, 0, 0);
            fence();
            fix_up<10, 16, P>();
            fence();
            dot[I & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1][1], b[I & 1][1], dot[I & 1], 0, 0, 0);
            fence();
            load_atom<N2, 1>();
            load_d8<N2>(npar);
        }
        if constexpr (I == 7 * TT) hd = F::prepare(raw, h);
        if constexpr (tt == TT - 1) operands<(s + 1) & 7>();
        if constexpr (I == 3 * TT - 1) { F::codes1(cd, rb, h, j); wave_order(); }
        // weights into the region that the slot before has read (those reads are over here)
        if constexpr (F::DMA && (I == 3 * TT || I == 7 * TT)) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        commits<I>(kb, next, next2, std::make_integer_sequence<int, S::CH>{});
        if constexpr (I == 7 * TT - 1) {
            wave_order();
            raw = F::raw_header(ra);
            F::codes0(cd, ra, h, j);
        }
        if constexpr (I == 7 * TT) { write_d(par ^ 1); fetch_d(next2); wave_order(); }
        // the block before: tile I is complete since slot I at the latest and starts again in slot I + 1
        if constexpr (I < TT && !F::D_PER_SUB) fold<I>();
        if constexpr (F::HAS_MIN) {
            mins<I>(std::make_integer_sequence<int, 4>{});
            if constexpr (I == 2 * TT - 1) {
                m_hi = __builtin_bit_cast(v8bf, make_uint4(mh[0], mh[1], mh[2], mh[3]));
                m_mid = __builtin_bit_cast(v8bf, make_uint4(mm[0], mm[1], mm[2], mm[3]));
                m_x = h ? m_mid : m_hi;
            }
            // The minimums of token tile J / 3, straight into its sums: (hi + mid) of the weights times (hi + mid + lo) of
            // d8 * S, six products of eight sub-blocks, two to an instruction (K slots 0 .. 7 and 8 .. 15)
            constexpr int J = I - 2 * TT;
            if constexpr (J >= 0 && J < 3 * TT)
                acc[J / 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(J % 3 == 0 ? m_hi : J % 3 == 1 ? m_mid : m_x,
                                                                    __builtin_bit_cast(v8bf, J % 3 == 2 ? pb1 : pb0), acc[J / 3], 0, 0, 0);
            if constexpr (J >= -1 && J < 3 * TT - 1 && (J + 1) % 3 == 0) pb0 = *(const uint4*)(mp + par * S::TABB + (J + 1) / 3 * (32 * LK_OPERAND_TAB));
            if constexpr (J >= 0 && J < 3 * TT && J % 3 == 1) pb1 = *(const uint4*)(rp + par * S::TABB + J / 3 * (32 * LK_OPERAND_TAB) + 64);
        }
        if constexpr (F::D_PER_SUB) {   // the next sub-block's, over those that this slot's fmas were the last to read
            if constexpr (tt == 0) read_dv<(s + 1) & 1>((s + 1) % 8 * S::D_ROW);
        } else if constexpr (I == NI - 1) read_dv(par * 32);
        // pins the slot's end for the instruction selector, which orders only what has side effects
        if constexpr (F::D_PER_SUB) asm volatile("" : "+v"(acc[P % TT]), "+v"(a[0][0]));
        else asm volatile("" : "+v"(part[P % TT]), "+v"(a[0][0]));
        if constexpr (I < TT && !F::D_PER_SUB) asm volatile("" : "+v"(acc[I % TT]));
        fence();
    }
    template <int I, int... C>
    __device__ __forceinline__ void commits(int kb, int next, int next2, std::integer_sequence<int, C...>) {
        ([&] {
            if constexpr (!F::DMA && S::commit_slot(C) == I) commit(C);
            if constexpr (S::fetch_slot(C) == I) fetch((F::DMA ? C < S::AC : S::LONG) ? next2 : next, C);
        }(), ...);
    }
    template <int I, int... Q>
    __device__ __forceinline__ void mins(std::integer_sequence<int, Q...>) {
        ([&] { if constexpr (I == TT + Q * TT / 4) min_pair<Q>(); }(), ...);
    }
    template <int... I>
    __device__ __forceinline__ void block(int kb, int last, std::integer_sequence<int, I...>) {
        const int next = min(kb + 1, last), next2 = min(kb + 2, last);
        (slot<I>(kb, next, next2), ...);
    }
};

// The products of a wave's 32 weight rows with tokens m0 .. m0 + 32 TT - 1, left in `t`: rows row0 .. row0 + 31 of the `live`
// rows from `weights` on (formats through registers: they all exist; others re-read the last one, whose results are never
// stored). Row m0 + i of the operands is token m0 + i, with GATHER row gather[m0 + i].
template <class F, int TT, int WAVES, bool GATHER>
static __device__ __forceinline__ void multiply(TileWave<F, TT, WAVES, GATHER>& t, const MmqProblem& pb, const LkTokenOperands& ops,
                                                const int32_t* gather, const uint8_t* weights, int row0, int live, int m0, uint8_t* lds) {
    using S = TileShape<F, TT, WAVES>;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // a caller's loop over tiles keeps none of what follows from it in registers meanwhile
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int last = (int)pb.nb - 1;
    const int64_t row_bytes = pb.row_blocks * F::UNIT;
    t.wave = wave;
    t.j = lane & 31;
    t.h = lane >> 5;
    t.lds_at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds);
    t.code_slab = ops.rows * LK_OPERAND_CODES;
    t.tab_slab = ops.rows * LK_OPERAND_TAB;
    t.codes = ops.codes;
    t.tabs = ops.tabs;
    t.w = weights;
    // a chunk is eight tokens x 128 bytes; atom p of token t lands in place p ^ (t % 8), so that 32 tokens spread over the banks
    const uint32_t swz = 16 * ((lane & 7) ^ (lane >> 3));
    if constexpr (GATHER) {
#pragma unroll
        for (int c = 0; c < S::CC; ++c) {
            const int token = 8 * min(wave + WAVES * c, 4 * TT - 1) + (lane >> 3);
            t.code_off[c] = (uint32_t)gather[min(m0 + token, pb.m_end - 1)] * LK_OPERAND_CODES + swz;
        }
#pragma unroll
        for (int c = 0; c < S::RC; ++c) {
            const int idx = 64 * min(wave + WAVES * c, S::TCH - 1) + lane;
            t.tab_off[c] = (uint32_t)gather[min(m0 + idx / 5, pb.m_end - 1)] * LK_OPERAND_TAB + 16 * (idx % 5);
        }
    } else {
        t.codes += (int64_t)m0 * LK_OPERAND_CODES;
        t.tabs += (int64_t)m0 * LK_OPERAND_TAB;
        t.code_off[0] = (lane >> 3) * LK_OPERAND_CODES + swz;
        t.tab_off[0] = 16 * lane;
    }
    if constexpr (F::DMA) {
#pragma unroll
        for (int i = 0; i < S::CH; ++i) {
            const bool in_a = i < S::AC;
            const int per = in_a ? F::AP : F::BP;
            const int idx = min(lane + 64 * (in_a ? i : i - S::AC), 32 * per - 1), row = idx / per, p = idx % per;
            t.from[i] = (uint32_t)min(row0 + row, live - 1) * (uint32_t)row_bytes + (in_a ? F::a_src(p) : F::b_src(p, row));
        }
    } else {
        const uint32_t row = (uint32_t)(row0 + (lane >> 3)) * (uint32_t)row_bytes;
        t.from[0] = row + F::a_src(min(lane & 7, F::AP - 1));
        t.from[1] = row + F::b_src(min(lane & 7, F::BP - 1), 0);
        t.row_bytes8 = 8 * row_bytes;
    }
    t.d_from = F::D_PER_SUB ? (uint32_t)(row0 + (lane >> 3)) * (uint32_t)row_bytes + F::UNIT * (lane & 7)
                            : (uint32_t)min(row0 + t.j, live - 1) * (uint32_t)row_bytes + F::BYTES - 2;
#pragma unroll
    for (int i = 0; i < (F::D_PER_SUB ? 4 : 1); ++i) t.d[i] = 0;
#pragma unroll
    for (int x = 0; x < 4; ++x) t.tb[x] = lds + S::T_AT + t.j * 128 + 16 * ((2 * x + t.h) ^ (t.j & 7));
    t.rp = lds + S::TAB_AT + t.j * LK_OPERAND_TAB;
    t.mp = t.rp + 32 + 16 * t.h;
    t.wstage = lds + S::W_AT + wave * S::W_BYTES;
    t.ra = t.wstage + t.j * S::A_ROW;
    t.rb = t.wstage + S::A_BYTES + t.j * S::B_ROW;
    t.wd = (float*)(lds + S::D_AT) + wave * (S::D_BYTES / 4);
    t.h1024 = H1024;   // in a vector register: (x & mask) | h1024 is then one v_and_or_b32 with the mask as its literal
    asm volatile("" : "+v"(t.h1024));
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int v = 0; v < 16; ++v) { t.acc[tt][v] = 0.f; t.part[F::D_PER_SUB ? 0 : tt][v] = 0.f; }
#pragma unroll
    for (int v = 0; v < 16; ++v) { t.dot[(S::NI - 1) & 1][v] = 0.f; t.dv[F::D_PER_SUB][v] = 0.f; }
    t.d8v[(S::NI - 1) & 3] = 0.f;   // "the item before the first": zeros times zero

#pragma unroll
    for (int i = 0; i < S::CH; ++i) t.fetch(0, i);
    t.fetch_d(0);
#pragma unroll
    for (int q = 0; q < S::LEAD; ++q)
#pragma unroll
        for (int c = 0; c < S::CC; ++c) t.load_codes(0, q, c);
#pragma unroll
    for (int c = 0; c < S::RC; ++c) t.load_tabs(0, c);
    if constexpr (!F::DMA)
#pragma unroll
        for (int i = 0; i < S::CH; ++i) t.commit(i);
    meet<0>();
    t.hd = F::prepare(F::raw_header(t.ra), t.h);
    F::codes0(t.cd, t.ra, t.h, t.j);
    t.write_d(0);
    wave_order();
    if constexpr (F::D_PER_SUB) t.template read_dv<0>(0);
    t.fetch_d(min(1, last));
    if constexpr (F::DMA) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if constexpr (F::DMA || S::LONG)
#pragma unroll
        for (int i = 0; i < (F::DMA ? S::AC : S::CH); ++i) t.fetch(min(1, last), i);
    t.template load_atom<0, 0>(); t.template load_atom<0, 1>(); t.template load_d8<0>(0);
    t.template load_atom<1, 0>(); t.template load_atom<1, 1>(); t.template load_d8<1>(0);
    t.template operands<0>();

    for (int kb = 0; kb <= last; ++kb) t.block(kb, last, std::make_integer_sequence<int, S::NI>{});

    t.template fix_up<0, 16, S::NI - 1>();
    if constexpr (!F::D_PER_SUB)
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int v = 0; v < 16; ++v) t.acc[tt][v] = fmaf(t.dv[0][v], t.part[tt][v], t.acc[tt][v]);
}

// A wave's results to dst[token][row], or dst[ids_dst[token]][row]; `first` its first weight row.
template <class F, int TT, int WAVES, bool GATHER>
static __device__ __forceinline__ void store_rows(const TileWave<F, TT, WAVES, GATHER>& t, const MmqProblem& pb, int first, int m0) {
    const bool vec_ok = pb.out_type == LK_TYPE_F32 && (uintptr_t)pb.dst % 16 == 0 && pb.ldd % 4 == 0 && first % 4 == 0;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
        const int col = m0 + 32 * tt + t.j;
        if (col >= pb.m_end) continue;
        const int64_t out = (pb.ids_dst ? pb.ids_dst[col] : col) * pb.ldd;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int row = first + 8 * g + 4 * t.h;
            if (row + 3 < pb.n) {
                mmq_store4(pb, out + row, make_float4(t.acc[tt][4 * g], t.acc[tt][4 * g + 1], t.acc[tt][4 * g + 2], t.acc[tt][4 * g + 3]), vec_ok);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (row + e < pb.n) lk_store_as(pb.dst, out + row + e, t.acc[tt][4 * g + e], pb.out_type);
            }
        }
    }
}

// silu(gate) * up of a token tile as the next product's operands. The 32 weight rows of a wave are one sub-block of them: lane
// (j, h) holds 16 of token j's values, lane (j, 1 - h) the others; `first` their first row. The steps of operand_quad.
static __device__ __forceinline__ void store_gated(const v16f& gate, const v16f& up, const LkTokenOperands& to, int first, int row, int h, bool live) {
    const int64_t at = (int64_t)(first / 256) * to.rows + row;
    const int s = (first / 32) & 7;
    float v[16], amax = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        v[i] = gate[i] / (1.0f + expf(-gate[i])) * up[i];
        amax = fmaxf(amax, fabsf(v[i]));
    }
    amax = fmaxf(amax, __shfl_xor(amax, 32));
    float d;
    int sum = 0;
    uint2 codes[4];
    {
#pragma clang fp contract(off)
        d = amax / 127.0f;
        const float inv = d != 0.0f ? 1.0f / d : 0.0f;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            uint32_t word = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int q = (int)roundf(v[4 * g + e] * inv);
                sum += q;
                word |= (uint32_t)(q & 0xFF) << (8 * e);
            }
            operand_codes(word, codes[g].x, codes[g].y);
        }
    }
    sum += __shfl_xor(sum, 32);
    if (!live) return;
    uint8_t* out = to.codes + at * LK_OPERAND_CODES + 64 * s + 8 * h;   // row 8 g + 4 h + e is value 4 h + e of atom (g % 2, g / 2)
#pragma unroll
    for (int g = 0; g < 4; ++g) *(uint2*)(out + 32 * (g & 1) + 16 * (g >> 1)) = codes[g];
    if (h == 0) operand_scales(to.tabs + at * LK_OPERAND_TAB, s, __half2float(__float2half_rn(d)), sum);
}

// Workgroup id -> (n tile, K range, m tile): the m tiles of one n tile re-read the same weight rows, so they are issued back
// to back on one XCD (ids are dealt round robin over the 8 XCDs). Each XCD takes an eighth of all tiles in that order, give or take one: dealt
// whole n tiles, those of 1213 rows, ten, left six XCDs with half the work of the other two. splits > 1: the tile over one of `splits`
// ranges of K, the partial tile to part[range].
template <class F, int TT, int WAVES>
__global__ __launch_bounds__(64 * WAVES, WAVES == 4 ? 2 : 1) void tile_dense_kernel(MmqProblem pb, LkTokenOperands ops, int n_tiles,
                                                                                    int m_tiles, int splits, float* part) {
    extern __shared__ __align__(16) uint8_t lds[];
    constexpr int ROWS = 32 * WAVES;
    const uint32_t xcd = blockIdx.x & 7, all = (uint32_t)n_tiles * m_tiles * splits;
    if (blockIdx.x >> 3 >= all / 8 + (xcd < all % 8)) return;
    uint32_t at = (blockIdx.x >> 3) + all / 8 * xcd + min(xcd, all % 8);
    const int m_tile = at % m_tiles;
    at /= m_tiles;
    const int split = at % splits, n_tile = at / splits;
    if (splits > 1) {
        const int64_t kb0 = pb.nb * split / splits, kb1 = pb.nb * (split + 1) / splits;
        pb.w += kb0 * F::BYTES;
        ops.codes += kb0 * ops.rows * LK_OPERAND_CODES;
        ops.tabs += kb0 * ops.rows * LK_OPERAND_TAB;
        pb.nb = kb1 - kb0;
        pb.ldd = mmq_part_stride(pb);
        pb.dst = part + split * (pb.m_end * pb.ldd);
        pb.out_type = LK_TYPE_F32;
    }
    int n0 = n_tile * ROWS;
    if (!F::DMA) n0 = min(n0, pb.n - ROWS);   // (the last tile slides back over the one before: same rows, same results)
    const int row0 = 32 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    TileWave<F, TT, WAVES, false> t;
    multiply(t, pb, ops, nullptr, pb.w + n0 * (pb.row_blocks * F::UNIT), row0, pb.n - n0, m_tile * 32 * TT, lds);
    store_rows(t, pb, n0 + row0, m_tile * 32 * TT);
}

// ------------------------------------------------------------------ experts
// One tile of an expert's run. GATED: waves 0 and 1 take 64 rows of the gate, 2 and 3 the same rows of the up matrix (pb.w,
// w_second), and the gated products leave as operands (`to`, a row per sorted row); else 128 rows of pb.w to pb.dst.
template <class F, int TT, bool GATED>
static __device__ __forceinline__ void expert_tile(const MmqProblem& pb, const LkTokenOperands& ops, const int32_t* gather, const uint8_t* w_second,
                                                   const LkTokenOperands& to, int n_tile, int m0, uint8_t* lds) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t row_bytes = pb.row_blocks * F::UNIT;
    TileWave<F, TT, 4, GATED> t;
    if constexpr (!GATED) {
        int n0 = n_tile * 128;
        if (!F::DMA) n0 = min(n0, pb.n - 128);
        multiply(t, pb, ops, gather, pb.w + n0 * row_bytes, 32 * wave, pb.n - n0, m0, lds);
        store_rows(t, pb, n0 + 32 * wave, m0);
    } else {
        const int n0 = n_tile * 64, row0 = 32 * (wave & 1);
        const bool is_up = wave >= 2;
        multiply(t, pb, ops, gather, (is_up ? w_second : pb.w) + n0 * row_bytes, row0, pb.n - n0, m0, lds);
        meet<0>();
        // the two waves of a row block trade token tiles through LDS: even ones are finished by the gate's wave, odd ones by the up's
        float* mine = (float*)lds + (threadIdx.x & 63) * 4;
        auto slab = [&](int tt) { return mine + ((wave & 1) * TT + tt) * 1024; };
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
            if ((tt & 1) != (int)is_up)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *(float4*)(slab(tt) + 256 * g) = make_float4(t.acc[tt][4 * g], t.acc[tt][4 * g + 1], t.acc[tt][4 * g + 2], t.acc[tt][4 * g + 3]);
        meet<0>();
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
            if ((tt & 1) == (int)is_up) {
                v16f other;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float4 o = *(const float4*)(slab(tt) + 256 * g);
                    other[4 * g] = o.x; other[4 * g + 1] = o.y; other[4 * g + 2] = o.z; other[4 * g + 3] = o.w;
                }
                const int row = m0 + 32 * tt + t.j;
                store_gated(is_up ? other : t.acc[tt], is_up ? t.acc[tt] : other, to, n0 + row0, row, t.h, row < pb.m_end);
            }
    }
}

// Expert e's slab against the sorted rows [bounds[e], bounds[e + 1]); grid: mmq_moe_grid. A run of c token tiles of 32 is cut
// into as few tiles of at most MAX as hold it, of equal length up to one (MAX = 3, four: two and two).
template <class F, bool GATED, int MAX>
__global__ __launch_bounds__(256, MAX == 1 && F::DMA ? 3 : 2) void tile_moe_kernel(MmqProblem pb, LkTokenOperands ops, const int32_t* __restrict__ gather,
                                                                         const uint8_t* w_second, int64_t dst_second, LkTokenOperands to,
                                                                         const int32_t* __restrict__ bounds, int64_t stride_expert,
                                                                         int n_experts, int group) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int stack = blockIdx.y / n_experts, e = blockIdx.y % n_experts;
    const int n_tiles = GATED ? pb.n / 64 : (pb.n + 127) / 128, n_tile = blockIdx.x % n_tiles;
    pb.m_begin = bounds[e];
    pb.m_end = bounds[e + 1];
    const int c = (pb.m_end - pb.m_begin + 31) / 32, tiles = (c + MAX - 1) / MAX;
    if (c <= 0) return;
    pb.w = (stack ? w_second : pb.w) + e * stride_expert;
    if (GATED) w_second += e * stride_expert;
    if (stack) pb.dst += dst_second;
    pb.out_type = LK_TYPE_F32;   // known here: the stores need no choice
    const int first = blockIdx.z * group + blockIdx.x / n_tiles, step = gridDim.z * group;
    for (int i = first; i < tiles; i += step) {
        if (i != first) meet<0>();   // the next tile's first loads go where this one's were
        const int from = c * i / tiles, count = c * (i + 1) / tiles - from, m0 = pb.m_begin + 32 * from;
        if (MAX == 1 || count == 1) expert_tile<F, 1, GATED>(pb, ops, gather, w_second, to, n_tile, m0, lds);
        if constexpr (MAX >= 2) if (count == 2) expert_tile<F, 2, GATED>(pb, ops, gather, w_second, to, n_tile, m0, lds);
        if constexpr (MAX >= 3) if (count == 3) expert_tile<F, 3, GATED>(pb, ops, gather, w_second, to, n_tile, m0, lds);
        if constexpr (MAX >= 4) if (count == 4) expert_tile<F, 4, GATED>(pb, ops, gather, w_second, to, n_tile, m0, lds);
    }
}

template <class F, int MAX>
static constexpr int moe_lds() {
    if constexpr (MAX == 1) return TileShape<F, 1, 4>::LDS;
    else return TileShape<F, MAX, 4>::LDS > moe_lds<F, MAX - 1>() ? TileShape<F, MAX, 4>::LDS : moe_lds<F, MAX - 1>();
}
template <class F, bool GATED, int MAX>
static int launch_moe(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTileExperts& ex, hipStream_t s) {
    auto kernel = tile_moe_kernel<F, GATED, MAX>;
    constexpr int LDS = moe_lds<F, MAX>();
    if (int rc = mmq_prepare_kernel(kernel, LDS)) return rc;
    // (MAX = 1: a second column tile for the runs that turn out longer than expected, which would double the launch's end)
    const MmqMoeGrid g = mmq_moe_grid(pb, GATED ? 64 : 128, 32 * MAX, !GATED && ex.w_second ? 2 : 1, ex.n_experts, ex.longest + (MAX == 1 ? 8 : 0));
    hipLaunchKernelGGL(kernel, g.grid, dim3(256), LDS, s, pb, ops, ex.gather, ex.w_second, ex.dst_second, ex.to ? *ex.to : LkTokenOperands{},
                       ex.bounds, ex.stride, ex.n_experts, g.group);
    return lk_launch_status();
}
// Tiles of at most three token tiles (a fourth costs Q6_K 35 spilled registers and no format gains: runs of 69 rows 246 us
// against 250, of 278 rows 118 against 120); runs of 32 rows and less leave registers for a third workgroup a CU (256 tokens over
// 128 experts 138 -> 126 us).
template <class F, bool GATED>
static int launch_moe(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTileExperts& ex, hipStream_t s) {
    return ex.longest <= 32 ? launch_moe<F, GATED, 1>(pb, ops, ex, s) : launch_moe<F, GATED, 3>(pb, ops, ex, s);
}

template <class F, int TT, int WAVES>
static int launch_dense(const MmqProblem& pb, const LkTokenOperands& ops, int splits, float* part, hipStream_t s) {
    constexpr int LDS = TileShape<F, TT, WAVES>::LDS;
    auto kernel = tile_dense_kernel<F, TT, WAVES>;
    if (int rc = mmq_prepare_kernel(kernel, LDS)) return rc;
    const int n_tiles = (pb.n + 32 * WAVES - 1) / (32 * WAVES), m_tiles = (pb.m_end + 32 * TT - 1) / (32 * TT);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(((int64_t)n_tiles * m_tiles * splits + 7) / 8 * 8)), dim3(64 * WAVES), LDS, s, pb, ops, n_tiles, m_tiles,
                       splits, part);
    return lk_launch_status();
}

template <class F>
static int launch_dense_plan(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTilePlan& plan, float* part, hipStream_t s) {
    if (plan.waves == 8) {
        if constexpr (F::DMA) return launch_dense<F, 4, 8>(pb, ops, plan.splits, part, s);
        return LK_ERR_ARG;
    }
    switch (plan.tt) {
        case 1: return launch_dense<F, 1, 4>(pb, ops, plan.splits, part, s);
        case 2: return launch_dense<F, 2, 4>(pb, ops, plan.splits, part, s);
        case 3: return launch_dense<F, 3, 4>(pb, ops, plan.splits, part, s);
        default:
            if constexpr (F::TT_MOST == 4) return launch_dense<F, 4, 4>(pb, ops, plan.splits, part, s);
            return LK_ERR_ARG;
    }
}

}  // namespace mmq_tile

#define LK_DEFINE_EXPERT_TILES(NAME, FORMAT)                                                                                      \
    int lk_tile_moe_##NAME(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTileExperts& ex, hipStream_t s) {           \
        return ex.to ? mmq_tile::launch_moe<FORMAT, true>(pb, ops, ex, s) : mmq_tile::launch_moe<FORMAT, false>(pb, ops, ex, s);  \
    }
#define LK_DEFINE_TILES(NAME, FORMAT)                                                                                             \
    LK_DEFINE_EXPERT_TILES(NAME, FORMAT)                                                                                          \
    int lk_tile_dense_##NAME(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTilePlan& plan, float* part, hipStream_t s) { \
        return mmq_tile::launch_dense_plan<FORMAT>(pb, ops, plan, part, s);                                                       \
    }
