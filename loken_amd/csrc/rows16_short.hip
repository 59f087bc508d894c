// Q4_K / Q5_K weights x up to 128 Q8_1 activation rows, in sets of eight or sixteen, where there are few 16-row tiles: the short launch of the
// 16-row family (rows16_core.h has the arithmetic's layout, rows16_mfma.hip the launches for many tiles).
//
// What bounds it: the o projection of a small model (2048 x 2048, 2.4 MB) is 128 row tiles. rows16_mfma.hip gives a workgroup of
// eight waves two of them and stages the activation for both, so 64 CUs work, a barrier stands between the loads and the
// arithmetic, and a wave has two super-blocks to walk. Here a workgroup is one tile, its super-blocks spread over up to sixteen waves, one
// each up to k = 4096; a wave reads the activation codes of its own super-blocks itself, all its loads in flight at
// once, and forms the codes' sums from what it holds.

#include "lk_common.h"
#include "rows16.h"
#include "rows16_core.h"
#include "rows16_direct.h"

namespace {

using rows16::Blk;
using namespace rows16_direct;
using rows16::TILE;
using rows16::WFrag;

constexpr int SET = 16;                  // activation rows a workgroup takes at most; more are sets over grid.y
constexpr int GROUPS = 16;               // of a tile's super-blocks at most, each summed by one wave
constexpr int PART_BYTES = 4 * 64 * 4;   // a wave's partial tile; the first one holds its scales until then, [8][TOKS] floats
enum Out { F32, ANY, DUAL_F32, DUAL_Q81 };   // plain: f32 or p.out_type; act(gate) * up: f32 or the Q8_1 rows that the next linear reads

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 __attribute__((aligned(4))) u32x4_a4;

template <typename T>
static __device__ __forceinline__ T pick3(const T (&a)[3], int i) { return i == 0 ? a[0] : i == 1 ? a[1] : a[2]; }

struct TileRef {
    int mat, tile;
};
// Tile i of workgroup `wg`'s NT: plain: of the matrices' groups of NT tiles one after another (a matrix's last group may have tiles past its
// rows, which store nothing); dual: gate and up of the same rows by turns.
template <int OUT, int NT>
static __device__ __forceinline__ TileRef tile_of(const LkRows16& p, int wg, int i) {
    if (OUT >= DUAL_F32) return {i & 1, wg * (NT / 2) + (i >> 1)};
    int mat = 0;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        const int groups = (p.n[m] + NT * TILE - 1) / (NT * TILE);
        if (mat == m && m + 1 < p.count && wg >= groups) wg -= groups, mat = m + 1;
    }
    return {mat, wg * NT + i};
}

static __host__ __device__ constexpr int lds_bytes_for(int waves, int nt, bool q81, bool rows = false) {
    return waves * (nt * PART_BYTES + (rows ? CODE_BYTES : 0)) + (q81 ? SET * nt / 4 * 32 * 4 : 0);
}

// grid.x workgroups of NT row tiles each (one; two where one would be more workgroups than CUs, and for a gate and its up; four for
// the 32 rows of a Q8_1 block), 64 * waves threads: wave w takes super-blocks w, w + waves, ... of every one of them, against one reading of the
// activation.
template <bool Q5, int TOKS, int OUT, int NT, int SRC>
__global__ __launch_bounds__(64 * GROUPS, 1) void q4k_rows16_short_kernel(LkRows16 p, int groups) {
    static_assert(TOKS == 8 || TOKS == 16, "eight or sixteen activation rows");
    static_assert(SRC == Q81 || (TOKS == 8 && OUT <= ANY), "rows of values: eight at a time, dense");
    static_assert(NT == 1 || NT % 2 == 0, "tiles in turn through two sets of weight registers");
    constexpr bool T16 = TOKS == 16, DUAL = OUT >= DUAL_F32;
    extern __shared__ __align__(16) uint8_t lds[];
    const int lane = threadIdx.x & 63, l16 = lane & 15, grp = lane >> 4, half = grp & 1, par = grp >> 1;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = (int)blockDim.x >> 6;
    const int m0 = (int)blockIdx.y * TOKS, m_rows = min(TOKS, p.m - m0);
    float* part = (float*)(lds + wave * NT * PART_BYTES);
    float* table = part;   // d8 [8][TOKS] of the super-block in hand

    // The weights too are asked for in the order they lie in, four lanes to a row's 64 bytes, and handed to the operand's lanes, where the registers hold the
    // code before and after (8192 x 14336 at 8 rows 19.1 us -> 17.5, 5000 x 12288 14.9 -> 12.4; sixteen rows with four tiles spill and go 7.5 -> 9.8)
    constexpr bool IN_ORDER = !T16 || (NT == 2 && !Q5);
    const int w_tile_row = IN_ORDER ? lane >> 2 : l16, w_piece = IN_ORDER ? lane & 3 : grp;
    const uint8_t* w_base[NT];   // each tile's matrix, and the lane's row in it (past the last row: the last)
    // Sixteen rows with four tiles: a row's offset is made at each load from the matrix's (uniform) first row. Kept for the four tiles, they were what
    // spilled 28 registers: 8192 x 4096 at 48 rows 26.8 us -> 17.7.
    constexpr bool ROW_AT_LOAD = !DUAL && T16 && NT == 4;
    uint32_t w_row[ROW_AT_LOAD ? 1 : NT];
    int w_first = 0, w_last = 0;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        // (the minimum, which changes nothing, keeps what follows apart from the results' tiles at the end: without it a step's q + k + v and o take 0.1 to
        // 0.3 us longer at any row count)
        const TileRef r = tile_of<OUT, NT>(p, DUAL ? (int)blockIdx.x : min((int)blockIdx.x, groups - 1), i);
        w_base[i] = (const uint8_t*)to_gbytes(pick3(p.w, r.mat));
        if (i == 0) w_first = r.tile * TILE, w_last = pick3(p.n, r.mat) - 1;
        if (!ROW_AT_LOAD) w_row[i] = (uint32_t)min(r.tile * TILE + w_tile_row, pick3(p.n, r.mat) - 1) * (uint32_t)(p.nb * Blk<Q5>::BYTES);
    }
    const int tok = l16 & (TOKS - 1);
    // The activation is asked for in the order it lies in, a row's pieces by neighbouring lanes, and handed to the operand's lanes by a
    // permutation (in the operand's order, neighbouring rows by neighbouring lanes, a load is a line a lane). Sixteen rows: load u is the four pieces of
    // (row lane / 4, unit u), unit u = 2 c2 + nib being sub-blocks 4 c2 + nib and + 2; eight: load c2 the eight pieces of (row lane / 8, units
    // 2 c2 and 2 c2 + 1).
    constexpr int PER_ROW = 64 / TOKS, LOADS = 16 / PER_ROW;
    const int y_tok = lane / PER_ROW, y_piece = lane % PER_ROW;
    const uint8_t* y_codes = p.y + ((size_t)(m0 + min(y_tok, m_rows - 1)) * p.stride_y + (T16 ? 2 * (y_piece >> 1) : y_piece >> 1)) * Q81_BYTES + 4 + 16 * (y_piece & 1);
    int from[T16 ? 1 : 2];   // byte address of the lane that holds the operand's piece (eight rows: of units of nib 0 and 1)
#pragma unroll
    for (int nib = 0; nib < (T16 ? 1 : 2); ++nib) from[nib] = 4 * (tok * PER_ROW + (T16 ? grp : 2 * (nib + 2 * par) + half));
    // scales: (row h_tok + 8 j, sub-block h_sub)
    constexpr int HEADS = TOKS / 8;
    const int h_tok = lane >> 3, h_sub = lane & 7;
    const uint8_t* y_head[HEADS];
#pragma unroll
    for (int j = 0; j < HEADS; ++j) y_head[j] = p.y + ((size_t)(m0 + min(h_tok + 8 * j, m_rows - 1)) * p.stride_y + h_sub) * Q81_BYTES;
    // lanes the instruction sees: sixteen rows: sub-block s in lane groups 0, 1 and, by the second one, s + 2 in groups 2, 3;
    // eight: slots (sub-block, row)
    const bool live = T16 ? par == 0 : (l16 >> 3) == par;
    const float* t_lane = T16 ? table + 4 * grp : table + 2 * par * TOKS + 4 * half;
    const int sh16 = T16 ? 0 : 16 * par, sh2 = 2 * par;

    // Rows of values: load u is (row lane / 8, sub-block u, values 4 (lane % 8) ..), the quantizer's own layout.
    typedef typename SrcOf<SRC>::T T;
    const T* x_row = (const T*)p.x + (size_t)(m0 + min(lane >> 3, m_rows - 1)) * p.nb * 256 + 4 * (lane & 7);
    uint32_t* codes = (uint32_t*)(lds + waves * NT * PART_BYTES + wave * CODE_BYTES);   // [sub-block][row][8]
    struct Act {
        u32x4 raw[LOADS];
        uint32_t head[HEADS];
        typename SrcOf<SRC>::Raw v[SRC == Q81 ? 1 : 8];
    };
    auto load_act = [&](Act& b, int kb) {
        if constexpr (SRC != Q81) {
#pragma unroll
            for (int u = 0; u < 8; ++u) b.v[u] = *(const typename SrcOf<SRC>::Load*)(x_row + kb * 256 + 32 * u);
            return;
        }
        const uint32_t at = (uint32_t)(kb * 8 * Q81_BYTES);
#pragma unroll
        for (int j = 0; j < HEADS; ++j) b.head[j] = *(const uint32_t*)(y_head[j] + at);
#pragma unroll
        for (int u = 0; u < LOADS; ++u) b.raw[u] = *(const u32x4_a4*)(y_codes + at + (T16 ? 4 * (u >> 1) + (u & 1) : 4 * u) * Q81_BYTES);
    };
    auto load_w = [&](WFrag& w, int i, int kb) {
        int tile_row = w_tile_row;
        if (ROW_AT_LOAD) asm volatile("" : "+v"(tile_row));   // (or the compiler makes the four before the loop)
        const uint32_t row = ROW_AT_LOAD ? (uint32_t)min(w_first + TILE * i + tile_row, w_last) * (uint32_t)(p.nb * Blk<Q5>::BYTES) : w_row[i];
        const uint32_t at = row + (uint32_t)(kb * Blk<Q5>::BYTES), at_q = at + 16 * w_piece;
        w.hdr = *(const uint4*)(w_base[i] + at);
        if (Q5) w.qh = *(const uint4*)(w_base[i] + (at + 16 * (w_piece & 1)) + 16);
        w.q[0] = *(const uint4*)(w_base[i] + at_q + Blk<Q5>::QS);
        w.q[1] = *(const uint4*)(w_base[i] + at_q + Blk<Q5>::QS + 64);
    };

    // eight rows: the lane's sums of sub-blocks 0, 1, 4, 5 or 2, 3, 6, 7; sixteen: of both, apart, so that either form adds the same
    // numbers in the same order and a launch may choose
    float acc[NT][T16 ? 2 : 1][4] = {};
    float d8s[2];   // d8 * S of (row, sub-block 4 h + grp), for the minimums
    auto settle = [] {   // between the wave's writes to its table and its reads of other lanes' entries
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    u32x4 a[4];   // the lane's pieces: unit (c2, nib): row tok, sub-block 4 c2 + nib + 2 par, codes 16 half ..
    auto settle_act = [&](const Act& b) {
        settle();
        if constexpr (SRC != Q81) {
            quantize<T>(b.v, lane, m_rows, table, codes);
            settle();
#pragma unroll
            for (int u = 0; u < 4; ++u) a[u] = *(const u32x4*)(codes + ((4 * (u >> 1) + (u & 1) + 2 * par) * 8 + tok) * 8 + 4 * half);
        } else {
#pragma unroll
        for (int j = 0; j < HEADS; ++j) table[h_sub * TOKS + h_tok + 8 * j] = h_tok + 8 * j < m_rows ? f16_bits_to_f32(b.head[j] & 0xFFFFu) : 0.f;
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) a[u][e] = (uint32_t)__builtin_amdgcn_ds_bpermute(from[T16 ? 0 : u & 1], (int)b.raw[T16 ? u : u >> 1][e]);
        settle();
        }
        // the lane holds half the codes of sub-blocks 4 h + 2 par and + 1; its own is + half, the other half of whose codes is with the lane
        // sixteen on
        const uint4 ones = make_uint4(0x01010101u, 0x01010101u, 0x01010101u, 0x01010101u);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            int sums[2];
#pragma unroll
            for (int nib = 0; nib < 2; ++nib) {
                const u32x4 v = a[2 * h + nib];
                sums[nib] = dot16(ones, make_uint4(v[0], v[1], v[2], v[3]), 0);
            }
            const int other = __builtin_amdgcn_ds_swizzle(half ? sums[0] : sums[1], 0x401F);   // lane ^ 16
            d8s[h] = table[(4 * h + grp) * TOKS + tok] * (float)((half ? sums[1] : sums[0]) + other);
        }
    };
    auto to_lane = [&](const uint4& v) {
        if constexpr (!IN_ORDER) return v;
        const int w_from = 4 * (4 * l16 + grp);
        return make_uint4((uint32_t)__builtin_amdgcn_ds_bpermute(w_from, (int)v.x), (uint32_t)__builtin_amdgcn_ds_bpermute(w_from, (int)v.y),
                          (uint32_t)__builtin_amdgcn_ds_bpermute(w_from, (int)v.z), (uint32_t)__builtin_amdgcn_ds_bpermute(w_from, (int)v.w));
    };
    auto compute = [&](const WFrag& raw, float (&sum)[T16 ? 2 : 1][4]) {
        // (accumulators from the bit pattern of 1.5 * 2^23, the offset off again in the first fused multiply-add, exactly: rows16_core.h)
        constexpr int MAGIC_BITS = 0x4B400000;
        constexpr float MAGIC = 12582912.0f;
        const v4i magic = {MAGIC_BITS, MAGIC_BITS, MAGIC_BITS, MAGIC_BITS};
        auto fold = [&](float (&s)[4], const v4i& c, float dsc, int sub) {
            const float off = -MAGIC * dsc;
            const float4 t = *(const float4*)(t_lane + sub * TOKS);
            s[0] = fmaf(fmaf(__int_as_float(c[0]), dsc, off), t.x, s[0]);
            s[1] = fmaf(fmaf(__int_as_float(c[1]), dsc, off), t.y, s[1]);
            s[2] = fmaf(fmaf(__int_as_float(c[2]), dsc, off), t.z, s[2]);
            s[3] = fmaf(fmaf(__int_as_float(c[3]), dsc, off), t.w, s[3]);
        };
        WFrag w;
        w.hdr = to_lane(raw.hdr);
        if (Q5) w.qh = to_lane(raw.qh);
        w.q[0] = to_lane(raw.q[0]);
        w.q[1] = to_lane(raw.q[1]);
        const uint32_t w1 = w.hdr.y, w2 = w.hdr.z, w3 = w.hdr.w;
        const uint32_t sc_lo = (w1 & 0x3F3F3F3Fu) >> sh16, sc_hi = ((w3 & 0x0F0F0F0Fu) | ((w1 >> 2) & 0x30303030u)) >> sh16;
        const float d = f16_bits_to_f32(w.hdr.x & 0xFFFFu), dmin = f16_bits_to_f32(w.hdr.x >> 16);
        const uint32_t hp[4] = {w.qh.x >> sh2, w.qh.y >> sh2, w.qh.z >> sh2, w.qh.w >> sh2};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c2 = u >> 1, nib = u & 1;
            const uint32_t q[4] = {w.q[c2].x, w.q[c2].y, w.q[c2].z, w.q[c2].w};
            v4i codes, a0, a1;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                uint32_t x = (nib ? q[e] >> 4 : q[e]) & 0x0F0F0F0Fu;
                if (Q5) x |= ((hp[e] >> (4 * c2 + nib)) & 0x01010101u) << 4;
                codes[e] = (int)x;
                a0[e] = live ? (int)a[u][e] : 0;
                a1[e] = live ? 0 : (int)a[u][e];
            }
            const uint32_t scw = c2 ? sc_hi : sc_lo;
            fold(sum[0], __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, codes, magic, 0, 0, 0), d * (float)((scw >> (8 * nib)) & 0xFFu), 4 * c2 + nib);
            if constexpr (T16)
                fold(sum[1], __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, codes, magic, 0, 0, 0), d * (float)((scw >> (8 * nib + 16)) & 0xFFu),
                     4 * c2 + 2 + nib);
#pragma unroll
            for (int v = 0; v < 4; ++v) {   // (one unit's result tiles at a time: registers)
                asm volatile("" : "+v"(sum[0][v]));
                if constexpr (T16) asm volatile("" : "+v"(sum[1][v]));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // the minimums: d8 * S [row, sub-block] x (-dmin * min) [sub-block, weight row], four sub-blocks an instruction
        const uint32_t mins[2] = {w2 & 0x3F3F3F3Fu, ((w3 >> 4) & 0x0F0F0F0Fu) | ((w2 >> 2) & 0x30303030u)};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float bmin = -(dmin * (float)((mins[h] >> (8 * grp)) & 0xFFu));
            v4f c = {sum[0][0], sum[0][1], sum[0][2], sum[0][3]};
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(T16 || l16 < TOKS ? d8s[h] : 0.f, bmin, c, 0, 0, 0);
            sum[0][0] = c[0], sum[0][1] = c[1], sum[0][2] = c[2], sum[0][3] = c[3];
        }
    };

    WFrag w[2];   // NT 1: of two super-blocks; else of two tiles
    if constexpr (SRC != Q81) {   // (a super-block to a wave)
        Act act;
        load_act(act, wave);
        load_w(w[0], 0, wave);
        if constexpr (NT > 1) load_w(w[1], 1, wave);
        settle_act(act);
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            compute(w[i & 1], acc[i]);
            if (i + 2 < NT) load_w(w[i & 1], i + 2, wave);
        }
    } else if constexpr (NT == 1 && Q5 && T16) {   // (one activation set: registers. With two 4096 x 14336 takes 19.7 us against 17.5; the others lose 5 % with one)
        Act act;
        load_act(act, wave);
        load_w(w[0], 0, wave);
        if (wave + waves < p.nb) load_w(w[1], 0, wave + waves);
        for (int kb = wave; kb < p.nb; kb += 2 * waves) {
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                const int at = kb + d * waves;
                if (at >= p.nb) break;
                settle_act(act);
                if (at + waves < p.nb) load_act(act, at + waves);
                compute(w[d], acc[0]);
                if (at + 2 * waves < p.nb) load_w(w[d], 0, at + 2 * waves);
            }
        }
    } else if constexpr (NT == 1) {
        Act act[2];
        auto load = [&](int d, int kb) { load_act(act[d], kb), load_w(w[d], 0, kb); };
        auto step = [&](int d) { settle_act(act[d]), compute(w[d], acc[0]); };
        load(0, wave);
        if (wave + waves < p.nb) load(1, wave + waves);
        for (int kb = wave; kb < p.nb; kb += 2 * waves) {
            step(0);
            if (kb + 2 * waves < p.nb) load(0, kb + 2 * waves);
            if (kb + waves < p.nb) {
                step(1);
                if (kb + 3 * waves < p.nb) load(1, kb + 3 * waves);
            }
        }
    } else {
        Act act;
        load_act(act, wave);
        load_w(w[0], 0, wave);
        load_w(w[1], 1, wave);
        for (int kb = wave; kb < p.nb; kb += waves) {
            settle_act(act);
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                compute(w[i & 1], acc[i]);
                if (i + 2 < NT) load_w(w[i & 1], i + 2, kb);
                else if (kb + waves < p.nb) load_w(w[i & 1], i + 2 - NT, kb + waves);
            }
            if (kb + waves < p.nb) load_act(act, kb + waves);   // (not before: registers)
        }
    }

    settle();
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) part[(4 * i + v) * 64 + lane] = T16 ? acc[i][0][v] + acc[i][T16 ? 1 : 0][v] : acc[i][0][v];
    __syncthreads();
    // sixteen rows: output (register v, lane l < 64) adds the waves' lanes l; eight: (v, l < 32) lanes l and l + 32
    constexpr int LANES = 4 * TOKS, OUTS = DUAL ? NT / 2 : NT;
    float* meet = (float*)(lds + waves * NT * PART_BYTES);   // Q8_1 output: [TOKS][8 NT]
    for (int o = threadIdx.x; o < OUTS * 4 * LANES; o += (int)blockDim.x) {
        const int r = o / (4 * LANES), v = o / LANES & 3, l = o % LANES;
        auto total = [&](int i) {
            float sum = 0.f;
            for (int w = 0; w < waves; ++w) {
                const float* col = (const float*)(lds + (w * NT + i) * PART_BYTES) + v * 64 + l;
                sum += T16 ? col[0] : col[0] + col[32];
            }
            return sum;
        };
        float sum = total(DUAL ? 2 * r : r);
        if constexpr (DUAL) {
            LkGateAct act;
            act.kind = p.gelu ? LK_GATE_GELU : LK_GATE_SILU;
            sum = lk_gated(act, sum, total(2 * r + 1), 0);
        }
        const int t = 4 * (l >> 4) + v;
        if constexpr (OUT == DUAL_Q81) {
            meet[t * (8 * NT) + 16 * r + (l & 15)] = sum;
        } else {
            const TileRef at = tile_of<OUT, NT>(p, blockIdx.x, DUAL ? 2 * r : r);
            const int row = at.tile * TILE + (l & 15), mat = DUAL ? 0 : at.mat;
            if (t < m_rows && row < pick3(p.n, mat)) lk_store_as(pick3(p.dst, mat), (size_t)(m0 + t) * pick3(p.ldd, mat) + row, sum, OUT == ANY ? p.out_type : LK_TYPE_F32);
        }
    }
    if constexpr (OUT == DUAL_Q81) {
        __syncthreads();
        // eight lanes per (activation row, block of 32 results) write it (n is a multiple of 32: a block's two tiles are whole or both missing)
        constexpr int BLOCKS = NT / 4;
        const int l8 = threadIdx.x & 7;
        for (int o = (int)threadIdx.x >> 3; o < m_rows * BLOCKS; o += (int)blockDim.x / 8) {
            const int row = o / BLOCKS, at = o % BLOCKS, block = (int)blockIdx.x * BLOCKS + at;
            if (32 * block < p.n[0])
                lk_store_q8_1_block(*(const float4*)(meet + row * (8 * NT) + 32 * at + 4 * l8), l8,
                                    (uint32_t*)(p.q81_dst + ((size_t)(m0 + row) * p.q81_stride + block) * Q81_BYTES));
        }
    }
}

template <bool Q5, int TOKS, int OUT, int NT, int SRC = Q81>
int launch(const LkRows16& a, hipStream_t stream) {
    static const bool ok = hipFuncSetAttribute((const void*)q4k_rows16_short_kernel<Q5, TOKS, OUT, NT, SRC>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                               lds_bytes_for(GROUPS, NT, OUT == DUAL_Q81, SRC != Q81)) == hipSuccess;
    if (!ok) return LK_ERR_ARG;
    const int steps = (a.nb + GROUPS - 1) / GROUPS, waves = (a.nb + steps - 1) / steps;   // as equal a share of super-blocks as they allow
    constexpr int ROWS = (OUT >= DUAL_F32 ? NT / 2 : NT) * TILE;   // of a matrix, to a workgroup
    int groups = 0;
    for (int i = 0; i < (OUT >= DUAL_F32 ? 1 : a.count); ++i) groups += (a.n[i] + ROWS - 1) / ROWS;
    const int sets = (a.m + TOKS - 1) / TOKS;
    if (sets > 65535) return LK_ERR_ARG;
    hipLaunchKernelGGL((q4k_rows16_short_kernel<Q5, TOKS, OUT, NT, SRC>), dim3(groups, sets), dim3(64 * waves),
                       lds_bytes_for(waves, NT, OUT == DUAL_Q81, SRC != Q81), stream, a, groups);
    return lk_launch_status();
}

template <bool Q5, int TOKS, int NT>
int launch_plain(const LkRows16& a, hipStream_t stream) {
    return a.out_type == LK_TYPE_F32 ? launch<Q5, TOKS, F32, NT>(a, stream) : launch<Q5, TOKS, ANY, NT>(a, stream);
}

// Time of a launch of sets of sixteen rows, us, with `nt` tiles to a workgroup: a workgroup of one, two, four tiles is there for 3.5, 4.8, 6.6 us of 2048
// values, 4.5, 6.8, 9.6 of 4096, 7.5, 8.8, 13.4 of 6144, and each further one of its CU adds what the fit says. (Five to seven super-blocks take the time
// of eight: waves come four to the CU. 14592 x 1280 at 64 rows 20.2 us with two tiles, 14592 x 2048 18.8.)
float set_us(int nt, int tiles, int sets, int nb) {
    const int cus = lk_device().cus;
    const float base = nb <= 4 ? 1.6f + 1.2f * (float)(nt == 4 ? 3 : nt) : 1.6f + 0.6f * (float)(nt == 4 ? 3 : nt), block = nt == 1 ? 0.2f : nt == 2 ? 0.255f : 0.435f;
    const int64_t wgs = (int64_t)((tiles + nt - 1) / nt) * sets;
    return base + block * (float)((nb > 4 && nb < 8 ? 8 : nb) * ((wgs + cus - 1) / cus));
}

// Tiles to a workgroup of sets of sixteen: the least of the three (Q5_K has no registers for four: 13 spilled, level with two).
int set_tiles(int tiles, int sets, int nb, bool q5) {
    const float one = set_us(1, tiles, sets, nb), two = set_us(2, tiles, sets, nb);
    if (!q5 && set_us(4, tiles, sets, nb) < (one < two ? one : two)) return 4;
    return two < one ? 2 : 1;
}

// Tiles to a workgroup: up to eight rows as many as bring the launch to a workgroup to the CU, and so for a gate and its up.
template <bool Q5, int TOKS>
int launch_out(const LkRows16& a, bool dual, int tiles, hipStream_t stream) {
    const int cus = lk_device().cus, sets = (a.m + TOKS - 1) / TOKS;
    if constexpr (TOKS == 8) {
        if (tiles > 2 * cus) {
            if (a.q81_dst) return launch<Q5, TOKS, DUAL_Q81, 8>(a, stream);
            return dual ? launch<Q5, TOKS, DUAL_F32, 8>(a, stream) : launch_plain<Q5, TOKS, 4>(a, stream);
        }
    }
    if (a.q81_dst) return launch<Q5, TOKS, DUAL_Q81, 4>(a, stream);
    if (dual) return (int64_t)tiles * sets > cus ? launch<Q5, TOKS, DUAL_F32, 4>(a, stream) : launch<Q5, TOKS, DUAL_F32, 2>(a, stream);
    if constexpr (TOKS == 8) return tiles > cus ? launch_plain<Q5, TOKS, 2>(a, stream) : launch_plain<Q5, TOKS, 1>(a, stream);
    const int nt = set_tiles(tiles, sets, a.nb, Q5);
    if constexpr (!Q5)
        if (nt == 4) return launch_plain<Q5, TOKS, 4>(a, stream);
    return nt == 2 ? launch_plain<Q5, TOKS, 2>(a, stream) : launch_plain<Q5, TOKS, 1>(a, stream);
}

template <bool Q5, int OUT, int SRC>
int launch_rows(const LkRows16& a, int tiles, hipStream_t stream) {
    const int cus = lk_device().cus;
    return tiles > 2 * cus ? launch<Q5, 8, OUT, 4, SRC>(a, stream) : tiles > cus ? launch<Q5, 8, OUT, 2, SRC>(a, stream) : launch<Q5, 8, OUT, 1, SRC>(a, stream);
}

}  // namespace

int lk_rows16_short(const LkRows16& a, bool dual, bool q5, hipStream_t stream) {
    if (a.m < 1 || a.nb < 1 || a.count < 1 || a.count > 3) return LK_ERR_ARG;
    if ((dual && (a.count != 2 || a.n[0] != a.n[1])) || (a.q81_dst && (!dual || a.n[0] % 32 != 0 || a.q81_stride < a.n[0] / 32))) return LK_ERR_ARG;
    int tiles = 0;
    for (int i = 0; i < (dual ? 1 : a.count); ++i) tiles += (a.n[i] + TILE - 1) / TILE;
    if (tiles == 0) return LK_OK;
    // nine to sixteen rows: two sets of eight where both are resident at once (Q4_K 1024 x 2048 at 16 rows 4.2 us against 4.4 with sixteen)
    const bool eight = a.m <= 8 || (a.m <= 16 && !dual && 2 * tiles <= lk_device().cus);
    if (eight) return q5 ? launch_out<true, 8>(a, dual, tiles, stream) : launch_out<false, 8>(a, dual, tiles, stream);
    return q5 ? launch_out<true, 16>(a, dual, tiles, stream) : launch_out<false, 16>(a, dual, tiles, stream);
}

// Matrices of up to four row tiles to the CU, fewer or more by the class of row counts: beyond, the launches that stage the activation once and walk
// many tiles are level or ahead; above a tile to the CU rows of 2048 values or more. A choice by the matrix and the class of row counts alone (up to
// 8, 16, 32, 48, 64, 96, 128), so that several matrices in one launch carry the bits of one launch each and a row carries the same bits whatever rides
// with it in its class. Measured in a graph, Q4_K, us, staged launches against this:
//   3 / 8 rows   1024 x 2048 5.1, 5.2 / 3.7, 3.7; 4096 x 4096 7.7, 8.1 / 5.1, 5.0; 4096 x 14336 17.9, 19.4 / 12.0, 11.9; 6144 x 2048 5.5, 5.5 / 4.9, 4.9;
//                8192 x 4096 8.8, 9.1 / 7.3, 7.2; 5000 x 12288 16.7, 17.8 / 14.7, 15.0; 14336 x 4096 12.6, 13.3 / 10.6, 10.5; 8192 x 1024 4.2, 4.1 / 4.0, 4.2;
//                18944 x 3584 (five to the CU) 14.1, 14.4 / 15.2, 15.4
//   9 / 16 rows  2048 x 2048 5.9, 6.4 / 4.0, 3.9; 4096 x 4096 9.4, 10.2 / 5.6, 5.6; 2048 x 6144 12.1, 13.2 / 6.4, 6.4; 4096 x 14336 28.8, 32.2 / 13.6, 14.7;
//                8192 x 4096 10.3, 11.0 / 7.9, 8.0; 5000 x 12288 25.9, 28.6 / 16.9, 16.9; 8192 x 1024 4.2, 4.3 / 4.9, 5.1; 14336 x 4096 14.4, 15.4 / 16.0, 16.6
//   (with the weights from HBM, which the figures above have in a cache; in brackets gate and up to Q8_1 rows) 12288 x 2048 9.0, 9.7 / 7.9, 8.1 (12.6, 12.7 /
//                11.1, 11.4); 24576 x 2048 13.4, 12.9 / 10.9, 11.3 (17.2, 16.7 / 15.6, 16.5); 9216 x 4096 14.1, 14.9 / 10.7, 11.6 (20.4, 21.3 / 19.5,
//                20.8); 14336 x 4096 14.9, 15.7 / 11.4, 12.2 (20.7, 21.7 / 20.3, 21.8, and 1.2 more than that between a step's other launches);
//                10240 x 8192 28.6, 34.6 / 18.9, 20.1; 28672 x 8192 48.6, 56.8 / 38.0, 40.1. Q5_K, four tiles to the CU, is level (16, 27 / 14, 29)
// Above sixteen rows against the 32-row tiles, where a wave's share of a tile's super-blocks is a chain of matrix instructions and fix-up (1 us a super-
// block) behind a table that is built first, on a chip that a layer's 64 to 400 tiles do not fill. Weights from HBM:
//   17 / 32 rows    2048 x 2048 7.5, 8.4 / 4.1, 4.1 (13.0, 14.0 / 6.6, 6.7); 4096 x 4096 12.4, 13.9 / 7.4, 7.7 (21.7, 23.3 / 10.8, 11.6); 8192 x 4096
//                   12.9, 14.7 / 10.7, 11.2 (22.1, 24.0 / 20.4, 20.5); 4096 x 14336 35.2, 39.4 / 18.0, 19.4; 12288 x 2048 11.5, 13.3 / 10.0, 10.1
//                   (19.8, 22.9 / 15.1, 15.4); 14336 x 4096 18.7, 23.7 / 19.6, 20.0 (31.4, 38.6 / 38.2, 38.6)
//   48 / 64         2048 x 2048 8.3, 8.4 / 5.1, 5.2; 4096 x 4096 13.3, 14.3 / 11.1, 11.1 (22.6, 23.8 / 19.2, 19.6); 8192 x 4096 20.6, 23.2 / 17.7, 19.3
//                   (34.3, 37.9 / 29.2, 37.9); 14336 x 4096 34.1, 37.7 / 27.9, 35.7 (60.1, 65.7 / 55.5, 65.5); 32768 x 2048 34.9, 37.3 / 26.6, 33.1;
//                   at 49 to 64 rows past three tiles to the CU not those of more than 4096 values: 15880 x 5632 at 56 41.2 / 46.2, 13850 x 13568 at 51
//                   82.5 / 89.4 (8342 x 13568 at 60 85.6 / 67.9; at 38 rows 9304 x 11776 70.1 / 41.5)
//   96 / 128        2048 x 2048 8.6, 8.7 / 6.7, 6.7; 4096 x 4096 21.1, 22.9 / 17.0, 19.0 (35.1, 37.5 / 27.9, 36.3); 8192 x 4096 34.3, 36.9 / 27.1, 35.0
//                   (62.0, 64.6 / 55.3, 72.5); 14336 x 4096 51.2, 63.3 / 51.5, 60.1 (93.1, 118.6 / 99.3, 126.6)
//   Q5_K, 32 / 64   2048 x 2048 8.8, 8.8 / 4.6, 5.8; 4096 x 4096 14.7, 15.1 / 9.3, 15.2 (24.8, 25.2 / 17.9, 30.2); 8192 x 2048 10.0, 14.2 / 9.2, 13.9 (16.3,
//                   23.9 / 17.2, 28.3)
// (Rows of up to 32768 values: longer ones are the other launches' to take or refuse.)
bool lk_rows16_short_pays(int m, int n, int nb, bool q5) {
    const int tiles = (n + TILE - 1) / TILE, cus = lk_device().cus;
    if (m < 1 || lk_rows16_off(m) || nb > 128) return false;
    if (m <= 16) return tiles <= cus || (nb >= 8 && tiles <= (m <= 8 ? 4 : q5 ? 2 : nb <= 8 ? 6 : nb <= 16 ? 3 : 8) * cus);
    if (m > 128) return false;
    if (q5) return (int64_t)tiles * (m <= 32 ? 2 : m <= 64 ? 4 : 8) <= 2 * cus;
    // (five and six super-blocks: 14592 x 1280 at 48 / 64 / 128 rows 14.9, 15.3, 24.3 / 13.6, 19.5, 30.0; 8192 x 1280 8.5, 8.8, 13.7 / 8.5, 8.7, 19.0;
    // with the quantizer 2767 x 1280 at 113 11.2 / 12.1)
    if (nb == 5 || nb == 6) return (int64_t)tiles * (m <= 32 ? 2 : m <= 64 ? 4 : m <= 96 ? 6 : 8) <= (m <= 64 ? 12 : 4) * cus;
    if (nb <= 8) return tiles <= 16 * cus;
    return tiles <= (m <= 32 ? 2 : m <= 48 ? 4 : m <= 64 ? (nb <= 16 ? 4 : 3) : m <= 96 ? 2 : 1) * cus;
}

float lk_rows16_short_us(int m, int n, int nb, bool q5) {
    if (m <= 16 || !lk_rows16_short_pays(m, n, nb, q5)) return -1.f;
    const int tiles = (n + TILE - 1) / TILE, sets = (m + SET - 1) / SET;
    return set_us(set_tiles(tiles, sets, nb, q5), tiles, sets, nb);
}

// Rows of up to 4096 values, a super-block to a wave: up to eight rows, and more as sets of eight where these are a workgroup to the CU, two of rows of up
// to 2048 values, three of up to 1024. Every workgroup makes the codes again, in less time than a quantizer launch takes on the chip (2 us), and the host is
// through with one launch where it was with two: up to 8192 x 4096 9.4 us a call -> 6.8, 14336 x 4096 11.1 -> 9.4. Above sixteen rows, called eagerly and on the
// chip, with a quantizer / without: 690 x 3584 at 22 9.2, 7.0 / 6.7, 6.2; 806 x 1536 at 47 9.0, 6.2 / 6.6, 6.0; 536 x 512 at 89 9.0, 5.7 / 6.7, 4.4. Past
// the lines the chip is behind: 1222 x 3328 at 28 9.5, 7.2 / 8.6, 8.7; 1120 x 2816 at 41 8.9, 6.8 / 7.6, 7.8.
int lk_rows16_short_rows(const LkRows16& a, bool q5, hipStream_t stream) {
    const int tiles = (a.n[0] + TILE - 1) / TILE;
    if (a.count != 1 || a.nb < 1 || a.nb > GROUPS || !lk_rows16_short_pays(a.m, a.n[0], a.nb, q5)) return -1;
    // Fewer than 512 matrix rows keep the quantizer's launch above sixteen rows though one launch is faster (a call of 17 to 48 rows 6.8 us, 4.0 to 5.8): a
    // program that records such a call with nothing reserved is refused, and goes on being refused.
    if (a.m > 16 && a.n[0] < 512) return -1;
    if (a.m > 8 && tiles * ((a.m + 7) / 8) > (a.nb <= 4 ? 3 : a.nb <= 8 ? 2 : 1) * lk_device().cus) return -1;
    if (a.x_type == LK_TYPE_F32) return q5 ? launch_rows<true, F32, ROWS_F32>(a, tiles, stream) : launch_rows<false, F32, ROWS_F32>(a, tiles, stream);
    if (a.x_type == LK_TYPE_F16) return q5 ? launch_rows<true, ANY, ROWS_F16>(a, tiles, stream) : launch_rows<false, ANY, ROWS_F16>(a, tiles, stream);
    return q5 ? launch_rows<true, ANY, ROWS_BF16>(a, tiles, stream) : launch_rows<false, ANY, ROWS_BF16>(a, tiles, stream);
}
