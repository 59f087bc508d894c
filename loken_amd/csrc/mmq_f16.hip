// Q4_K, Q5_K and Q6_K weight rows against 33 or more Q8_1 token rows, a dense call's or those expected of an expert: the
// sub-block dots on the f16 matrix unit.
//
//   out[token, n] = sum over 256-value blocks of
//        d[n] * sum_s d8_s[token] * D_s[n, token]  -  dmin[n] * sum_s m_s[n] * (d8_s * S_s)[token]
//   D_s[n, token] = sum over the 32 values of sub-block s of (sc[n] * q[n, k]) * a[token, k]
//
// The same integers as the int8 tile kernel forms (sc * dot of the codes and the int8 codes: loken's
// BlockQ4K::dot_scalar, src/tensor/quant_cpu/format/q4_k.rs:138-153, q6_k.rs:137-160, combined as cuda/moe/gguf.cuh:
// 664-713, 782-816 combine them), reached another way. An int8 MFMA leaves dot_s, which still has to meet
// two factors per output element, sc_s[n] and d8_s[token]: a convert and two multiplies on the
// vector unit per element and sub-block, four to six times the cycles of the MFMA that fed them.
// Here the scale rides into the matrix unit with the weight: sc * q (at most 63 * 15, Q5_K 63 * 31) is exact in
// f16, so is an int8 code, their products and the 32-term sums are exact in the f32 accumulator
// (< 2^24). D_s leaves the unit as a float that already carries the weight scale, and one fma by
// the lane's d8 finishes it. Half the matrix rate of int8, a third of the vector work.
// Q6_K's signed scales meet six-bit codes: |sc * q| <= 128 * 32 has one bit more than f16 holds. The operand is the
// product rounded to f16 and a second one carries what the rounding took (-1, 0 or 1, exact); both terms add up in the
// same accumulator, still exactly (128 * 32 * 127 * 32 < 2^24). Four matrix instructions per sub-block instead of
// two, against eight vector instructions per two elements of the int8 form (two dots of 16 values, a scale each).
//
// Shape: a workgroup of eight waves takes 256 weight rows x 64 tokens; a wave owns 32 of the rows
// and both token tiles of 32; registers <-> weight rows, lanes <-> tokens (v_mfma_f32_32x32x16_f16
// called as weights x tokens). Per 256-value step a wave copies its 32 rows' blocks into
// LDS as they lie in memory (consecutive lanes read consecutive 16-byte pieces of a row's block:
// loading them lane-per-row instead touches 64 cache lines per instruction and was a fifth of
// the kernel's time), and each lane then picks its row's codes out of LDS in operand order and
// expands them in registers. A wave reads no rows but its own, so the weights need one stage and no barrier:
// the codes of a step are in registers by its fifth sub-block, and the next step's take their place. Token codes are
// expanded to f16 once per step into LDS, two stages deep, one barrier per step.
// The min term is a rank-8 update per block on the bf16 matrix unit, with d8 * S split into
// three bf16 pieces (24 bits, nothing lost).
// Bound by the issue of vector and matrix instructions, which do not overlap here (counters on Q6_K, 2048 rows of
// 14336 -> 4096: vector unit 62 % of the cycles, matrix unit 39 %; the wide kernel 65 and 36): 16 fmas per item, the
// expansion of a wave's weights shared by two token tiles, and twice the matrix instructions for Q6_K. 417 TFLOP/s
// there (int8 tiles 341). Half as many rows per workgroup, two workgroups a CU, took 622 us for 577 there and 453 for 429 on
// 128 experts at 1111 tokens (the token side is expanded twice as often), though few large tiles gain (8 experts 77 -> 67).
//
// K order inside a sub-block: lane half h (lane / 32) of MFMA hf holds values 16 h + 8 hf + i,
// i in the order 0 2 1 3 4 6 5 7 (what masking a dword's even and odd bytes yields); weights and
// tokens use the same order, which is all a dot product asks. (A lane half holds one of Q6_K's 16-value groups.)

#include "mmq_problem.h"

#include <type_traits>

namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

static __device__ __forceinline__ h2 as_h2(uint32_t bits) { return __builtin_bit_cast(h2, bits); }
static __device__ __forceinline__ uint32_t h2_bits(h2 v) { return __builtin_bit_cast(uint32_t, v); }

constexpr uint32_t H1024 = 0x64006400u;   // two f16 1024.0: OR-ing an 8-bit integer into the mantissa adds it

struct Wide {
    static constexpr int WAVES = 8;                   // along the weight rows
    static constexpr int THREADS = 64 * WAVES;
    static constexpr int TT = 2;                      // token tiles of 32 per wave
    static constexpr int TM = 32 * TT;                // tokens per workgroup tile
    static constexpr int TN = 32 * WAVES;             // weight rows per workgroup tile
    static constexpr int CCH = TM * 16 / THREADS;     // 16-code chunks per thread per step
    static constexpr int PARTS = THREADS / TM;        // threads sharing one token's scales
    static_assert(TM * 16 % THREADS == 0 && PARTS == 8, "one sub-block's scale per thread");
    // one token stage: f16 codes [plane = (s, hf, h)][token ^ swizzle][8 halves], d8 [s][token] f32,
    // pieces [hi, mid, lo, zero][token][8 bf16]
    static constexpr int CODES = TM * 512, D8 = TM * 32, PIECES = 4 * TM * 16;
    static constexpr int STAGE = CODES + D8 + PIECES;
    static constexpr int TABLE = WAVES * 256;   // per wave: d and -dmin of its 32 rows
};

// ------------------------------------------------------------------ weight formats
// A block in LDS is its first ROW bytes (16-byte pieces, an odd number of them: 32 rows then spread over the banks).
// Codes: what a lane needs of half a block (four sub-blocks). operand(): the lane's eight values of MFMA hf of
// sub-block s, times the scale, as TERMS f16 operands.
struct Scale16 { h2 scale, offset; };

// A code of a format with a plane of high bits is put together as a byte, four to an instruction, and the bytes 0 | 2 and
// 1 | 3 leave for the mantissas of two 1024.0 in one v_perm_b32 each (with the high bits masked and shifted per pair of
// halves instead, 312 of the 863 vector instructions of a Q6_K block went there, now 184 of 735: 4096 x 14336 at 2048
// rows 610 -> 577 us, Q5_K 11003 x 4096 at 77 rows 43.3 -> 40.5).
static __device__ __forceinline__ uint32_t bits_from(uint32_t w, int up, uint32_t mask) {
    return (up >= 0 ? w << (up & 31) : w >> (-up & 31)) & mask;
}
static __device__ __forceinline__ uint32_t even_codes(uint32_t c, uint32_t h1024) { return __builtin_amdgcn_perm(h1024, c, 0x07020500u); }
static __device__ __forceinline__ uint32_t odd_codes(uint32_t c, uint32_t h1024) { return __builtin_amdgcn_perm(h1024, c, 0x07030501u); }

template <bool Q5>
struct F16Q45K {
    static constexpr int BYTES = Q5 ? Q5K_BYTES : Q4K_BYTES, ROW = BYTES, ALIGN = 16, TERMS = 1;
    static constexpr bool HAS_MIN = true;
    struct Header { uint4 w; };
    struct Codes { uint4 q[2], qh; };
    static __device__ __forceinline__ Header header(const uint8_t* row, int h) { (void)h; return {*(const uint4*)row}; }
    static __device__ __forceinline__ void codes(Codes& c, const uint8_t* row, int half, int h) {
#pragma unroll
        for (int p = 0; p < 2; ++p) c.q[p] = *(const uint4*)(row + (Q5 ? 48 : 16) + 64 * half + 32 * p + 16 * h);
        if (Q5) c.qh = *(const uint4*)(row + 16 + 16 * h);
    }
    static __device__ __forceinline__ uint32_t scale_of(const Header& hd, int s) {   // get_scale_min_k4 of the format
        return s < 4 ? (hd.w.y >> (8 * s)) & 63u : ((hd.w.w >> (8 * (s - 4))) & 0xFu) | (((hd.w.y >> (8 * (s - 4) + 6)) & 3u) << 4);
    }
    static __device__ __forceinline__ uint32_t min_of(const Header& hd, int s) {
        return s < 4 ? (hd.w.z >> (8 * s)) & 63u : ((hd.w.w >> (8 * (s - 4) + 4)) & 0xFu) | (((hd.w.z >> (8 * (s - 4) + 6)) & 3u) << 4);
    }
    // (1024 + q) * sc - 1024 * sc; Q4_K's high nibbles stay four bits up, (1024 + 16 q) * (sc / 16) - 64 * sc.
    // Both exact in f16 (sc <= 63).
    static __device__ __forceinline__ Scale16 scale(const Header& hd, int s) {
        const float sc = (float)scale_of(hd, s);
        const bool up = !Q5 && (s & 1);
        const _Float16 a = (_Float16)(sc * (up ? 0.0625f : 1.0f)), b = (_Float16)(sc * (up ? -64.0f : -1024.0f));
        return {{a, a}, {b, b}};
    }
    static __device__ __forceinline__ void operand(const Codes& cd, int s, int hf, const Scale16& sc, uint32_t h1024, v8h a[TERMS]) {
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
                even = even_codes(c, h1024);
                odd = odd_codes(c, h1024);
            } else {
                const uint32_t mask = high ? 0x00F000F0u : 0x000F000Fu;
                even = (x & mask) | h1024;
                odd = ((x >> 8) & mask) | h1024;
            }
            ab[2 * e] = h2_bits(__builtin_elementwise_fma(as_h2(even), sc.scale, sc.offset));
            ab[2 * e + 1] = h2_bits(__builtin_elementwise_fma(as_h2(odd), sc.scale, sc.offset));
        }
        a[0] = __builtin_bit_cast(v8h, make_uint4(ab[0], ab[1], ab[2], ab[3]));
    }
};

struct F16Q6K {
    static constexpr int BYTES = Q6K_BYTES, ROW = 208, ALIGN = 2, TERMS = 2;   // its d, two bytes past the 13 pieces, travels by itself
    static constexpr bool HAS_MIN = false;
    struct Header { uint32_t sc[4]; };   // byte 2 * (s % 2) of word s / 2: the scale of the lane's 16 values of sub-block s
    struct Codes { uint4 q[2], qh; };
    static __device__ __forceinline__ Header header(const uint8_t* row, int h) {
        const uint4 w = *(const uint4*)(row + 192);
        return {{w.x >> (8 * h), w.y >> (8 * h), w.z >> (8 * h), w.w >> (8 * h)}};
    }
    static __device__ __forceinline__ void codes(Codes& c, const uint8_t* row, int half, int h) {
#pragma unroll
        for (int p = 0; p < 2; ++p) c.q[p] = *(const uint4*)(row + 64 * half + 32 * p + 16 * h);
        c.qh = *(const uint4*)(row + 128 + 32 * half + 16 * h);
    }
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
using F16Q4K = F16Q45K<false>;
using F16Q5K = F16Q45K<true>;

template <class F>
static constexpr int f16_lds_bytes() { return 2 * Wide::STAGE + Wide::TN * F::ROW + Wide::TABLE; }

// A wave's copy of one step's blocks of its 32 rows: piece q = lane + 64 i is 16-byte piece q % PIECES of row
// q / PIECES, and lands at byte 16 q of the wave's part of the stage. The last round may have pieces for some lanes
// only; the others repeat the last piece (same bytes to the same place), which keeps the step free of branches.
template <class F>
struct WeightCopy {
    static constexpr int PIECES = F::ROW / 16, CH = (32 * PIECES + 63) / 64;
    using piece = typename std::conditional<F::ALIGN == 16, uint4, uint4_a2>::type;
    const uint8_t* base;   // the tile's first row
    uint32_t from[CH], d_from;   // byte offsets in step 0 (rows past the end re-read the last row)
    uint4 data[CH];
    uint16_t d;            // Q6_K: row lane % 32's d

    __device__ __forceinline__ void place(const uint8_t* w, int64_t row_bytes, int n0, int n, int wave) {
        const int lane = threadIdx.x & 63;
        base = w + (int64_t)n0 * row_bytes;
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const int q = min(lane + 64 * i, 32 * PIECES - 1);
            from[i] = (uint32_t)min(32 * wave + q / PIECES, n - 1 - n0) * (uint32_t)row_bytes + 16 * (q % PIECES);
        }
        d_from = (uint32_t)min(32 * wave + (lane & 31), n - 1 - n0) * (uint32_t)row_bytes + F::ROW;
        d = 0;
    }
    __device__ __forceinline__ void fetch_part(int64_t step_bytes, int i) {
        data[i] = *(const piece*)(base + step_bytes + from[i]);
    }
    __device__ __forceinline__ void fetch_d(int64_t step_bytes) {
        if constexpr (F::BYTES != F::ROW) d = *(const uint16_t*)(base + step_bytes + d_from);
    }
    __device__ __forceinline__ void commit_part(uint8_t* stage, int i) const {
        *(uint4*)(stage + min((int)(threadIdx.x & 63) + 64 * i, 32 * PIECES - 1) * 16) = data[i];
    }
};

struct TokenFrag16 {
    using C = Wide;
    uint4 codes[C::CCH];
    uint16_t d8, sum;   // of sub-block tid / TM of token tid % TM

    // Byte offsets of this thread's loads inside one K step's slab of records (rows past the end
    // re-read the last row: their results are never stored).
    uint32_t code_at[C::CCH], scale_at;
    __device__ __forceinline__ void place(int m0, int m_end) {
        const int tid = threadIdx.x;
#pragma unroll
        for (int i = 0; i < C::CCH; ++i) {
            const int idx = tid + i * C::THREADS, r = idx >> 4, c = idx & 15;
            code_at[i] = (uint32_t)min(m0 + r, m_end - 1) * MMQ_REC_BYTES + 16 * c;
        }
        const int r = tid % C::TM, part = tid / C::TM;
        scale_at = (uint32_t)min(m0 + r, m_end - 1) * MMQ_REC_BYTES + 256 + 2 * part;
    }
    // Part i < CCH: a chunk of codes; part CCH: the scales and sums.
    static constexpr int FETCH_PARTS = C::CCH + 1;
    __device__ __forceinline__ void fetch_part(const uint8_t* __restrict__ slab, int i) {
        if (i < C::CCH) {
            codes[i] = *(const uint4*)(slab + code_at[i]);
        } else {
            d8 = *(const uint16_t*)(slab + scale_at);
            sum = *(const uint16_t*)(slab + scale_at + 16);
        }
    }
    __device__ __forceinline__ void fetch(const uint8_t* __restrict__ slab) {
#pragma unroll
        for (int i = 0; i < FETCH_PARTS; ++i) fetch_part(slab, i);
    }

    // four int8 codes -> f16, as the pairs (0, 2) and (1, 3)
    static __device__ __forceinline__ void expand(uint32_t u, uint32_t& even, uint32_t& odd) {
        // byte ^ 0x80 = code + 128 in 0..255; OR-ed into the mantissa of 1024.0 (one XOR does both:
        // the constants' bits do not overlap), then 1024 + 128 comes off
        const h2 bias = {(_Float16)1152.0f, (_Float16)1152.0f};
        even = h2_bits(as_h2((u & 0x00FF00FFu) ^ 0x64806480u) - bias);
        odd = h2_bits(as_h2(((u >> 8) & 0x00FF00FFu) ^ 0x64806480u) - bias);
    }

    // Part i of the registers into a stage (the parts of fetch_part).
    template <bool WITH_SUMS>
    __device__ __forceinline__ void commit(uint8_t* stage) const {
#pragma unroll
        for (int i = 0; i < FETCH_PARTS; ++i) commit_part<WITH_SUMS>(stage, i);
    }
    template <bool WITH_SUMS>
    __device__ __forceinline__ void commit_part(uint8_t* stage, int i) const {
        const int tid = threadIdx.x;
        if (i < C::CCH) {
            const int idx = tid + i * C::THREADS, r = idx >> 4, c = idx & 15;
            const int s = c >> 1, h = c & 1;
            const uint32_t u[4] = {codes[i].x, codes[i].y, codes[i].z, codes[i].w};
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                uint4 out;
                expand(u[2 * hf], out.x, out.y);
                expand(u[2 * hf + 1], out.z, out.w);
                const int plane = (s * 2 + hf) * 2 + h;
                // the 16 lanes that share a token write 16 planes: the token index is XOR-ed with
                // the plane's (s, h) so that they land in 16 different bank groups
                *(uint4*)(stage + (plane * C::TM + (r ^ c)) * 16) = out;
            }
            return;
        }
        float* ad8 = (float*)(stage + C::CODES);
        uint8_t* ap = stage + C::CODES + C::D8;
        const int r = tid % C::TM, s = tid / C::TM;
        const float d = f16_bits_to_f32(d8);
        ad8[s * C::TM + r] = d;
        if (!WITH_SUMS) return;
        // d8 * S as three bf16 (truncations of the running remainder: 8 bits each, exact)
        const float p0 = d * (float)(int)(int16_t)sum;
        const uint32_t b0 = __float_as_uint(p0) & 0xFFFF0000u;
        const float p1 = p0 - __uint_as_float(b0);
        const uint32_t b1 = __float_as_uint(p1) & 0xFFFF0000u;
        const float p2 = p1 - __uint_as_float(b1);
        const uint32_t b2 = __float_as_uint(p2) & 0xFFFF0000u;
        const int at = r * 16 + s * 2;
        *(uint16_t*)(ap + 0 * C::TM * 16 + at) = (uint16_t)(b0 >> 16);
        *(uint16_t*)(ap + 1 * C::TM * 16 + at) = (uint16_t)(b1 >> 16);
        *(uint16_t*)(ap + 2 * C::TM * 16 + at) = (uint16_t)(b2 >> 16);
    }
};

// The B operands and the token scale of item (s, tt). `ad8` already points at the lane's token.
static __device__ __forceinline__ void load_item(const uint8_t* stage, const uint8_t* ad8, int s, int tt, int token0,
                                                 int h, v8h b[2], float& d8) {
    // token0 ^ (2 s + h) only changes the low four bits, so the tile offset 32 tt adds on top
    using C = Wide;
    const uint8_t* at = stage + (token0 ^ (2 * s + h)) * 16 + h * C::TM * 16 + tt * 512;
    b[0] = *(const v8h*)(at + (s * 4 + 0) * C::TM * 16);
    b[1] = *(const v8h*)(at + (s * 4 + 2) * C::TM * 16);
    d8 = *(const float*)(ad8 + (s * C::TM + 32 * tt) * 4);
}

// Results [FROM, TO) of item `it` into the block's partial sums; TT: the token tiles that are walked.
template <int TT, int FROM, int TO>
static __device__ __forceinline__ void scale_item(int it, const v16f& dot, float d8, v16f part[TT]) {
    const int s = it / TT, tt = it % TT;
#pragma unroll
    for (int v = FROM; v < TO; ++v) part[tt][v] = s == 0 ? dot[v] * d8 : fmaf(dot[v], d8, part[tt][v]);
}

// What other lanes of this wave wrote to LDS before is read after, and the other way round: LDS serves a wave's
// accesses in order, so only the compiler has to keep them there.
static __device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// TT: 2, or 1 where the tile's second 32 tokens lie past the end.
template <class F, int TT>
static __device__ __forceinline__ void f16_tile_of(const MmqProblem& pb, int n0, int m0, uint8_t* lds) {
    using C = Wide;
    constexpr int TM = C::TM, TERMS = F::TERMS;
    using Copy = WeightCopy<F>;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, h = lane >> 5;
    uint8_t* wstage = lds + 2 * C::STAGE + wave * (32 * F::ROW);
    float* wd = (float*)(lds + 2 * C::STAGE + C::TN * F::ROW) + wave * 64;   // [0, 32) d, [32, 64) -dmin of the wave's rows
    const uint8_t* wrow = wstage + j * F::ROW;
    const int last = (int)pb.nb - 1;

    v16f acc[TT];
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[tt][v] = 0.f;

    if (F::HAS_MIN)   // the zero piece of both stages (the second bf16 MFMA of the min term has 8 spare K slots)
        for (int i = tid; i < 2 * TM; i += C::THREADS) {
            uint8_t* stage = lds + (i / TM) * C::STAGE;
            *(uint4*)(stage + C::CODES + C::D8 + (3 * TM + i % TM) * 16) = make_uint4(0, 0, 0, 0);
        }

    Copy wc;
    TokenFrag16 tf;
    const int64_t slab_bytes = pb.rows_total * MMQ_REC_BYTES;
    tf.place(m0, pb.m_end);
    wc.place(pb.w, pb.row_blocks * F::BYTES, n0, pb.n, wave);
    tf.fetch(pb.y);
#pragma unroll
    for (int i = 0; i < Copy::CH; ++i) wc.fetch_part(0, i);
    wc.fetch_d(0);
    tf.template commit<F::HAS_MIN>(lds);
#pragma unroll
    for (int i = 0; i < Copy::CH; ++i) wc.commit_part(wstage, i);
    uint16_t d_now = wc.d;
    tf.fetch(pb.y + min(1, last) * slab_bytes);
#pragma unroll
    for (int i = 0; i < Copy::CH; ++i) wc.fetch_part((int64_t)min(1, last) * F::BYTES, i);
    wc.fetch_d((int64_t)min(1, last) * F::BYTES);
    wave_order();
    typename F::Header hd = F::header(wrow, h);
    typename F::Codes codes;
    F::codes(codes, wrow, 0, h);
    __syncthreads();

    // 1024.0 | 1024.0 in a vector register: with the mask as the instruction's one literal,
    // (x & mask) | h1024 is a single v_and_or_b32
    uint32_t h1024 = H1024;
    asm volatile("" : "+v"(h1024));
    const int token0 = j;   // the lane's token in the first token tile

    for (int kb = 0; kb <= last; ++kb) {
        const uint8_t* stage = lds + (kb & 1) * C::STAGE;
        const uint8_t* ad8 = stage + C::CODES + token0 * 4;
        const uint8_t* ap = stage + C::CODES + C::D8 + token0 * 16;
        const uint8_t* next_slab = pb.y + min(kb + 2, last) * slab_bytes;
        const int64_t next_step = (int64_t)min(kb + 2, last) * F::BYTES;

        if (h == 0) {
            if constexpr (F::HAS_MIN) {
                wd[j] = f16_bits_to_f32(hd.w.x & 0xFFFFu);
                wd[32 + j] = -f16_bits_to_f32(hd.w.x >> 16);
            } else {
                wd[j] = f16_bits_to_f32(d_now);
            }
        }

        // Items (s, tt) run through a three-deep pipeline written out by hand: the LDS reads of
        // item i + 1, the matrix instructions of item i, the 16 fmas of item i - 1. Left to itself the
        // scheduler keeps one item in flight (read, wait, multiply, wait, scale).
        constexpr int NI = 8 * TT;
        v8h a[2][TERMS], b[2][2];   // a: [hf][term] of the current sub-block
        float d8v[3];   // read at item i + 1's loads, used at item i - 1's fmas: three alive
        v16f dot[2], part[TT];
        auto operands = [&](int s) {
            const Scale16 sc = F::scale(hd, s);
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) F::operand(codes, s, hf, sc, h1024, a[hf]);
        };
        operands(0);
        load_item(stage, ad8, 0, 0, token0, h, b[0], d8v[0]);
#pragma unroll
        for (int it = 0; it < NI; ++it) {
            const int s = it / TT, tt = it % TT;
            if (it + 1 < NI) load_item(stage, ad8, (it + 1) / TT, (it + 1) % TT, token0, h, b[(it + 1) & 1], d8v[(it + 1) % 3]);
            // A matrix instruction takes the one before's result as its accumulator and cannot issue
            // before that is written, and a wave's own vector instructions do not issue past a
            // waiting one: whatever should run meanwhile has to sit between them.
            v16f& now = dot[it & 1];
            const v16f& before = dot[(it - 1) & 1];
            const float d8p = d8v[(it + 2) % 3];
            {
                v16f zero = {0.f};
                now = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0][0], b[it & 1][0], zero, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (it >= 1) scale_item<TT, 0, TERMS == 2 ? 6 : 8>(it - 1, before, d8p, part);
            __builtin_amdgcn_sched_barrier(0);
            now = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1][0], b[it & 1][1], now, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (TERMS == 2) {
                if (it >= 1) scale_item<TT, 6, 11>(it - 1, before, d8p, part);
                __builtin_amdgcn_sched_barrier(0);
                now = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0][1], b[it & 1][0], now, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (it >= 1) scale_item<TT, 11, 16>(it - 1, before, d8p, part);
                __builtin_amdgcn_sched_barrier(0);
                now = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1][1], b[it & 1][1], now, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            } else {
                if (it >= 1) scale_item<TT, 8, 16>(it - 1, before, d8p, part);
            }
            if (tt == TT - 1 && s + 1 < 8) operands(s + 1);   // over the ones the sub-block's last item has just used
            if (tt == TT - 1 && s == 2) F::codes(codes, wrow, 1, h);   // the second half's codes; nothing of this step is read from the stage after them
            // The next step's tokens leave their registers for the other stage (whose last readers left at the
            // barrier that ended the previous step), its weights for the wave's own, one part per item, so
            // that eight waves' LDS writes do not arrive in one burst; each part's registers take
            // the load of the step after next. (One token tile: half the items, two weight parts each.)
            constexpr int W0 = 4 * TT, EACH = (Copy::CH + W0 - 1) / W0, T0 = W0 - TokenFrag16::FETCH_PARTS;
            if (it >= T0 && it < W0) {
                tf.template commit_part<F::HAS_MIN>(lds + ((kb + 1) & 1) * C::STAGE, it - T0);
                tf.fetch_part(next_slab, it - T0);
            }
            if (it == W0 - 1) wave_order();
            if (it >= W0) {
#pragma unroll
                for (int e = 0; e < EACH; ++e) {
                    const int c = (it - W0) * EACH + e;
                    if (c < Copy::CH) {
                        wc.commit_part(wstage, c);
                        wc.fetch_part(next_step, c);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        scale_item<TT, 0, 16>(NI - 1, dot[(NI - 1) & 1], d8v[(NI - 1) % 3], part);

        // the next block's header and first codes come out of the stage under the rest of this one
        const typename F::Header hd_now = hd;
        wave_order();
        hd = F::header(wrow, h);
        F::codes(codes, wrow, 0, h);

        // the block's per-row factors, for the 16 rows this lane's registers stand for
        float dv[16];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const float4 t = *(const float4*)(wd + 8 * g + 4 * h);
            dv[4 * g + 0] = t.x; dv[4 * g + 1] = t.y; dv[4 * g + 2] = t.z; dv[4 * g + 3] = t.w;
        }
        if constexpr (F::HAS_MIN) {
            float ndm[16];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float4 u = *(const float4*)(wd + 32 + 8 * g + 4 * h);
                ndm[4 * g + 0] = u.x; ndm[4 * g + 1] = u.y; ndm[4 * g + 2] = u.z; ndm[4 * g + 3] = u.w;
            }
            // small integers as bf16: the top half of their f32
            uint32_t mb[4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                mb[q] = (__float_as_uint((float)F::min_of(hd_now, 2 * q)) >> 16) |
                        (__float_as_uint((float)F::min_of(hd_now, 2 * q + 1)) & 0xFFFF0000u);
            const v8bf m_op = __builtin_bit_cast(v8bf, make_uint4(mb[0], mb[1], mb[2], mb[3]));
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) {
                const v8bf p0 = *(const v8bf*)(ap + (h * TM + 32 * tt) * 16);          // hi | mid
                const v8bf p1 = *(const v8bf*)(ap + ((2 + h) * TM + 32 * tt) * 16);    // lo | zero
                v16f mins = {0.f};
                mins = __builtin_amdgcn_mfma_f32_32x32x16_bf16(m_op, p0, mins, 0, 0, 0);
                mins = __builtin_amdgcn_mfma_f32_32x32x16_bf16(m_op, p1, mins, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    acc[tt][v] = fmaf(ndm[v], mins[v], fmaf(dv[v], part[tt][v], acc[tt][v]));
            }
        } else {
            d_now = wc.d;   // (fetched with the pieces that this step has committed)
            wc.fetch_d(next_step);
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[tt][v] = fmaf(dv[v], part[tt][v], acc[tt][v]);
        }
        wave_order();
        __syncthreads();
    }

    const bool vec_ok = pb.out_type == LK_TYPE_F32 && (uintptr_t)pb.dst % 16 == 0 && pb.ldd % 4 == 0;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
        const int col = m0 + 32 * tt + j;
        if (col >= pb.m_end) continue;
        const int64_t out = (pb.ids_dst ? pb.ids_dst[col] : col) * pb.ldd;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int gn0 = n0 + 32 * wave + 8 * g + 4 * h;
            if (gn0 + 3 < pb.n) {
                mmq_store4(pb, out + gn0, make_float4(acc[tt][4 * g], acc[tt][4 * g + 1], acc[tt][4 * g + 2], acc[tt][4 * g + 3]), vec_ok);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (gn0 + e < pb.n) lk_store_as(pb.dst, out + gn0 + e, acc[tt][4 * g + e], pb.out_type);
            }
        }
    }
}

// A tile of which 32 tokens or fewer exist walks one token tile instead of two: padding costs as much as live tokens
// (128 experts of 2048 -> 768 -> 2048 at 1111 tokens, runs of 69 rows on average, so a full tile and a few rows over:
// Q4_K block 400 -> 381 us, Q6_K down 464 -> 448). Same operations per output, same results.
template <class F>
static __device__ __forceinline__ void f16_tile(const MmqProblem& pb, int n0, int m0, uint8_t* lds) {
    if (pb.m_end - m0 <= 32) f16_tile_of<F, 1>(pb, n0, m0, lds);
    else f16_tile_of<F, 2>(pb, n0, m0, lds);
}

// Expert-batched: expert e's slab against the sorted rows [bounds[e], bounds[e+1]); grid: mmq_moe_grid.
template <class F>
__global__ __launch_bounds__(Wide::THREADS, 1) void f16_moe_kernel(MmqProblem pb, const uint8_t* w_second, int64_t dst_second,
                                                                  const int32_t* __restrict__ bounds, int64_t stride_expert,
                                                                  int n_experts, int group) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int stack = blockIdx.y / n_experts, e = blockIdx.y % n_experts;
    const int n_tiles = (pb.n + Wide::TN - 1) / Wide::TN, n_tile = blockIdx.x % n_tiles;
    pb.m_begin = bounds[e];
    pb.m_end = bounds[e + 1];
    if (pb.m_end <= pb.m_begin) return;
    pb.w = (stack ? w_second : pb.w) + (int64_t)e * stride_expert;
    if (stack) pb.dst += dst_second;
    pb.out_type = LK_TYPE_F32;   // known here: the tile's stores need no choice
    for (int m0 = pb.m_begin + (blockIdx.z * group + blockIdx.x / n_tiles) * Wide::TM; m0 < pb.m_end; m0 += gridDim.z * group * Wide::TM) {
        f16_tile<F>(pb, n_tile * Wide::TN, m0, lds);
        __syncthreads();   // the next tile's prologue rewrites the first stages
    }
}

// Record offsets inside a slab and row offsets inside a tile are 32-bit.
template <class F>
static bool f16_suits(const MmqProblem& pb) {
    return (uintptr_t)pb.w % F::ALIGN == 0 && (uintptr_t)pb.y % 16 == 0 && pb.rows_total <= (1 << 23) &&
           pb.row_blocks * F::BYTES * Wide::TN <= (int64_t)INT32_MAX;
}

template <class F>
static int f16_moe(const MmqProblem& pb, const uint8_t* w_second, int64_t dst_second, const int32_t* bounds,
                   int64_t stride_expert, int n_experts, int64_t ncols_max, hipStream_t s) {
    using C = Wide;
    constexpr int LDS = f16_lds_bytes<F>();
    if (!f16_suits<F>(pb) || (uintptr_t)w_second % F::ALIGN != 0 || stride_expert % F::ALIGN != 0) return -1;
    if (mmq_prepare_kernel(f16_moe_kernel<F>, LDS) != LK_OK) return 0;
    const MmqMoeGrid g = mmq_moe_grid(pb, C::TN, C::TM, w_second ? 2 : 1, n_experts, ncols_max);
    hipLaunchKernelGGL(f16_moe_kernel<F>, g.grid, dim3(C::THREADS), LDS, s, pb, w_second, dst_second, bounds,
                       stride_expert, n_experts, g.group);
    return hipGetLastError() == hipSuccess ? C::TM : 0;
}

}  // namespace

int lk_mmq_f16_moe(int wtype, const MmqProblem& pb, const uint8_t* w_second, int64_t dst_second, const int32_t* bounds,
                   int64_t stride_expert, int n_experts, int64_t ncols_max, hipStream_t s) {
    return wtype == LK_TYPE_Q4_K   ? f16_moe<F16Q4K>(pb, w_second, dst_second, bounds, stride_expert, n_experts, ncols_max, s)
           : wtype == LK_TYPE_Q5_K ? f16_moe<F16Q5K>(pb, w_second, dst_second, bounds, stride_expert, n_experts, ncols_max, s)
           : wtype == LK_TYPE_Q6_K ? f16_moe<F16Q6K>(pb, w_second, dst_second, bounds, stride_expert, n_experts, ncols_max, s)
                                   : -1;
}
