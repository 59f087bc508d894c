// Q6_K weights x up to 128 Q8_1 activation rows, in sets of eight, sixteen or twice sixteen, where there are few 16-row tiles: the short launch of the
// 16-row family (rows16_q6k.hip has the arithmetic's description: one instruction's four lane groups hold four 16-value groups
// of a row, the activation live in the lanes of one group or of one of two).
//
// What bounds it: a `down` projection of a small model (2048 x 6144, 10 MB) is 128 row tiles, so a launch is over in about the
// time of one load, one wave's arithmetic and one reduction, whatever the bytes. rows16_q6k.hip hands a wave a granule of eight
// super-blocks, which makes that arithmetic eight steps long with three waves on a CU (11.1 us a launch at 16 rows in a
// graph, of which 2 are a launch that does nothing; now 7.8). Here a tile's super-blocks go to up to twelve waves (168 registers each), every load of the first two in flight at once; nothing is staged for the workgroup, so no barrier stands before the
// arithmetic: a wave reads the activation codes of its own super-blocks itself, and turns the weights and the eight scales per row through a buffer of its own.
//
// Any super-block may be a wave's, so its bytes start at any even phase of a 16-byte piece, another one for each row: the row's
// fourteen pieces are written to the buffer so that the block starts at byte 16 or 18, and a lane shifts what it reads by its row's
// zero or two bytes. Rows of any number of super-blocks are served.

#include "lk_common.h"
#include "rows16.h"
#include "rows16_direct.h"

namespace {

using namespace rows16_direct;

constexpr int TILE = 16, MAX_WAVES = 12;
constexpr int BLOCK_PIECES = 14;              // 16-byte pieces that hold a super-block, at any even phase
constexpr int PITCH = 16 + 16 * BLOCK_PIECES + 32;   // bytes between the rows of a wave's buffer: 16 rows on 16 bank groups
constexpr int ROWS_BYTES = TILE * PITCH;
static __host__ __device__ constexpr int wave_bytes(int sets) { return ROWS_BYTES + sets * 8 * 16 * 4; }   // and d8 [8][TOKS] of the super-block

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 __attribute__((aligned(4))) u32x4_a4;

struct Args {
    const uint8_t* w;     // 16-byte aligned
    const uint8_t* y;     // Q8_1 rows (rows of values: SRC's elements, nb * 256 of them each)
    float* dst;
    int nb, n, m;         // super-blocks per weight row, weight rows, activation rows
    int stride_y;         // Q8_1 blocks between activation rows
    int ldd;              // elements between output rows
    int out_type;         // element type of `dst` (lk_store_as)
};

// grid (row tiles, groups of SETS sets of TOKS activation rows), 64 * waves threads: wave w takes super-blocks w, w + waves, ...
// Two sets of sixteen to a workgroup: the weights go through the buffer, are unpacked and set apart by groups once for both, which makes the second
// set a quarter to a third of the first one's time (4096 x 14336: 17 us a round of workgroups with one, 23 with two).
template <int TOKS, int SETS, bool HALF, int SRC>
__global__ __launch_bounds__(64 * MAX_WAVES, 1) void q6k_rows16_short_kernel(Args p) {
    static_assert(TOKS == 8 || TOKS == 16, "sets of eight or sixteen activation rows");
    constexpr bool T16 = TOKS == 16;
    extern __shared__ __align__(16) uint8_t lds[];
    static_assert(SRC == Q81 || TOKS == 8, "rows of values: eight at a time");
    static_assert(SETS == 1 || (SETS == 2 && TOKS == 16), "two sets: of sixteen rows");
    constexpr int WAVE_BYTES = wave_bytes(SETS);
    const int lane = threadIdx.x & 63, l16 = lane & 15, grp = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = (int)blockDim.x >> 6;
    const int tile = (int)blockIdx.x, m0 = (int)blockIdx.y * SETS * TOKS, m_rows = min(SETS * TOKS, p.m - m0);
    const int last_row = min(TILE, p.n - tile * TILE) - 1;
    const int row_bytes = p.nb * Q6K_BYTES;
    uint8_t* buf = lds + wave * WAVE_BYTES;
    float* table = (float*)(buf + ROWS_BYTES);

    // ---- the weights: load u of a super-block is piece 64 u + lane of its 16 x 14 (sixteen rows are whole pieces: a tile is aligned)
    constexpr int LOADS = (TILE * BLOCK_PIECES + 63) / 64;   // 4, the last half used
    const uint8_t* w_tile = (const uint8_t*)(to_gbytes(p.w) + (size_t)tile * TILE * row_bytes);
    // (w_at with the piece's offset in it, a register a load. With the two apart the kernel over f16 rows took 91 registers for 78 and the compiler
    // waited for each of its activation loads before the next: 9136 x 2304 at 5 rows 16.8 us, 11.3; sixteen rows spilled one: 3 % at 13 rows.)
    uint32_t w_at[LOADS];
    int w_to[LOADS];
#pragma unroll
    for (int u = 0; u < LOADS; ++u) {
        const int id = min(64 * u + lane, TILE * BLOCK_PIECES - 1), row = id / BLOCK_PIECES;
        w_at[u] = (uint32_t)(min(row, last_row) * row_bytes + 16 * (id % BLOCK_PIECES));
        w_to[u] = row * PITCH + 16 * (id % BLOCK_PIECES) + 16;
    }
    const uint32_t my_at = (uint32_t)(min(l16, last_row) * row_bytes);   // of the lane's own row
    // ---- the activation, asked for in the order it lies in, a row's pieces by neighbouring lanes, and handed to the operand's lanes by a permutation
    // (in the operand's order, neighbouring rows by neighbouring lanes, a load is a line a lane). Sixteen rows: load u is the four pieces of (row
    // lane / 4, unit u: values 64 u ..); eight: load v the eight pieces of (row lane / 8, units 2 v and 2 v + 1)
    const int tok = l16 & (TOKS - 1), sel = l16 / TOKS;
    constexpr int PER_ROW = 64 / TOKS, Y_LOADS = 16 / PER_ROW, HEADS = TOKS / 8;
    const int y_tok = lane / PER_ROW, y_piece = lane % PER_ROW, h_tok = lane >> 3, h_sub = lane & 7;
    const uint8_t* y0 = p.y + (size_t)m0 * p.stride_y * Q81_BYTES;
    uint32_t y_codes[SETS], y_head[SETS][HEADS];   // scales: (row h_tok + 8 j, sub-block h_sub)
#pragma unroll
    for (int i = 0; i < SETS; ++i) {
        y_codes[i] = (uint32_t)((min(TOKS * i + y_tok, m_rows - 1) * p.stride_y + (y_piece >> 1)) * Q81_BYTES + 4 + 16 * (y_piece & 1));
#pragma unroll
        for (int j = 0; j < HEADS; ++j) y_head[i][j] = (uint32_t)((min(TOKS * i + h_tok + 8 * j, m_rows - 1) * p.stride_y + h_sub) * Q81_BYTES);
    }
    const int from = 4 * (tok * PER_ROW + grp);   // byte address of the lane that holds the operand's piece (eight rows: of even units)
    // eight rows: the lanes whose codes the first and the second instruction see
    const uint32_t keep0 = grp == sel ? ~0u : 0u, keep1 = grp == sel + 2 ? ~0u : 0u;
    // the lane's results: eight rows: groups grp / 2 and 2 + grp / 2, rows 4 (grp % 2) + v; sixteen: every group, rows 4 grp + v
    const float* t_lane = T16 ? table + 4 * grp : table + 4 * (grp & 1);
    const int sh_sc = T16 ? 0 : 8 * (grp >> 1), sh_qh = 2 * (grp >> 1);

    // rows of values: load u is (row lane / 8, sub-block u, values 4 (lane % 8) ..), the quantizer's own layout
    typedef typename SrcOf<SRC>::T T;
    typedef typename SrcOf<SRC>::Raw Raw;
    const T* x_row = (const T*)p.y + (size_t)(m0 + min(lane >> 3, m_rows - 1)) * p.nb * 256 + 4 * (lane & 7);
    uint32_t* codes_of_rows = (uint32_t*)(lds + waves * WAVE_BYTES + wave * CODE_BYTES);   // [sub-block][row][8]
    struct Weights {
        u32x4 w[LOADS];
    };
    struct Act {
        u32x4 y[Y_LOADS];
        uint32_t head[HEADS];
        Raw v[SRC == Q81 ? 1 : 8];
    };
    auto load_act = [&](Act& b, int i, int kb) {
        const uint32_t ya = (uint32_t)(kb * 8 * Q81_BYTES);
        if constexpr (SRC != Q81) {
#pragma unroll
            for (int u = 0; u < 8; ++u) b.v[u] = *(const typename SrcOf<SRC>::Load*)(x_row + kb * 256 + 32 * u);
        } else {
#pragma unroll
            for (int j = 0; j < HEADS; ++j) b.head[j] = *(const uint32_t*)(y0 + (y_head[i][j] + ya));
#pragma unroll
            for (int u = 0; u < Y_LOADS; ++u) b.y[u] = *(const u32x4_a4*)(y0 + (y_codes[i] + ya) + u * (8 / Y_LOADS) * Q81_BYTES);
        }
    };
    auto load_w = [&](Weights& b, int kb) {
        const uint32_t at = (uint32_t)(kb * Q6K_BYTES);
#pragma unroll
        for (int u = 0; u < LOADS; ++u) b.w[u] = *(const u32x4*)(w_tile + ((w_at[u] + at) & ~15u));
    };

    auto settle = [] {   // the wave's own LDS writes before its reads of other lanes' data
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto put_scales = [&](const Act& b, int i) {
#pragma unroll
        for (int j = 0; j < HEADS; ++j)
            table[i * 8 * TOKS + h_sub * TOKS + h_tok + 8 * j] = TOKS * i + h_tok + 8 * j < m_rows ? f16_bits_to_f32(b.head[j] & 0xFFFFu) : 0.f;
    };
    auto turn = [&](const Act& b, u32x4 (&act)[4]) {   // the lane's sixteen codes of unit u: values 64 u + 16 grp ..
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                act[u][e] = (uint32_t)__builtin_amdgcn_ds_bpermute(from + (T16 ? 0 : 16 * (u & 1)), (int)b.y[T16 ? u : u >> 1][e]);
    };
    auto put_w = [&](const Weights& b, int kb) {
        const uint32_t at = (uint32_t)(kb * Q6K_BYTES);
#pragma unroll
        for (int u = 0; u < LOADS; ++u)
            if (64 * u + lane < TILE * BLOCK_PIECES) *(u32x4_a4*)(buf + (w_to[u] - (int)((w_at[u] + at) & 12u))) = b.w[u];
    };
    auto piece_at = [&](int c, uint32_t sh, uint32_t& past) {   // sixteen bytes at byte c of the super-block; the four after them, unshifted
        const uint8_t* mine = buf + l16 * PITCH + 16;
        const u32x4 lo = *(const u32x4*)(mine + c);
        past = *(const uint32_t*)(mine + c + 16);
        return u32x4{__builtin_amdgcn_alignbyte(lo[1], lo[0], sh), __builtin_amdgcn_alignbyte(lo[2], lo[1], sh),
                     __builtin_amdgcn_alignbyte(lo[3], lo[2], sh), __builtin_amdgcn_alignbyte(past, lo[3], sh)};
    };
    auto codes_of = [&](int unit, uint32_t sh, u32x4& ql, u32x4& qhp) {   // the lane's sixteen signed codes: group 4 unit + grp of the row (units in turn)
        uint32_t past;
        if (unit % 2 == 0) {
            ql = piece_at(32 * unit + 16 * grp, sh, past);
            qhp = piece_at(128 + 16 * unit + 16 * (grp & 1), sh, past) >> (uint32_t)sh_qh;
        }
        v4i codes;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t nib = (unit & 1 ? ql[e] >> 4 : ql[e]) & 0x0F0F0F0Fu;
            const uint32_t up = (unit & 1 ? qhp[e] : qhp[e] << 4) & 0x30303030u;
            codes[e] = (int)(((nib | up) + 0x60606060u) ^ 0x80808080u);
        }
        return codes;
    };

    // eight rows: the lane's sums of groups 0 and 2 or 1 and 3 of each four; sixteen: of both, apart, so that either form adds the same
    // numbers in the same order and a launch may choose
    float acc[SETS][T16 ? 2 : 1][4] = {};
    // (accumulators from the bit pattern of 1.5 * 2^23, the offset off again in the first fused multiply-add, exactly: rows16_q6k.hip)
    constexpr int MAGIC_BITS = 0x4B400000;
    constexpr float MAGIC = 12582912.0f;
    const v4i magic = {MAGIC_BITS, MAGIC_BITS, MAGIC_BITS, MAGIC_BITS};
    auto fold = [&](float (&sum)[4], const v4i& c, float dsc, int i, int sub) {
        const float off = -MAGIC * dsc;
        const float4 t = *(const float4*)(t_lane + i * 8 * TOKS + sub * TOKS);
        sum[0] = fmaf(fmaf(__int_as_float(c[0]), dsc, off), t.x, sum[0]);
        sum[1] = fmaf(fmaf(__int_as_float(c[1]), dsc, off), t.y, sum[1]);
        sum[2] = fmaf(fmaf(__int_as_float(c[2]), dsc, off), t.z, sum[2]);
        sum[3] = fmaf(fmaf(__int_as_float(c[3]), dsc, off), t.w, sum[3]);
    };
    // sums of one unit, of every set
    auto unit_of = [&](int unit, const u32x4 (&act)[SETS][4], const v4i& codes, float d, uint32_t scs) {
        const uint32_t scw = scs >> (uint32_t)sh_sc;
        if constexpr (SETS == 2) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {   // the codes of group g alone, for both sets
                v4i mine;
#pragma unroll
                for (int e = 0; e < 4; ++e) mine[e] = grp == g ? codes[e] : 0;
                const float dsc = d * (float)(int)__builtin_amdgcn_sbfe(scw, 8 * g, 8);
#pragma unroll
                for (int i = 0; i < SETS; ++i) {
                    const v4i a = {(int)act[i][unit][0], (int)act[i][unit][1], (int)act[i][unit][2], (int)act[i][unit][3]};
                    fold(acc[i][T16 ? g & 1 : 0], __builtin_amdgcn_mfma_i32_16x16x64_i8(a, mine, magic, 0, 0, 0), dsc, i, 2 * unit + (g >> 1));
                }
            }
        } else if constexpr (T16) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {   // the activation of group g alone
                v4i a;
#pragma unroll
                for (int e = 0; e < 4; ++e) a[e] = grp == g ? (int)act[0][unit][e] : 0;
                const v4i c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, codes, magic, 0, 0, 0);
                fold(acc[0][T16 ? g & 1 : 0], c, d * (float)(int)__builtin_amdgcn_sbfe(scw, 8 * g, 8), 0, 2 * unit + (g >> 1));
            }
        } else {
            v4i a0, a1;
#pragma unroll
            for (int e = 0; e < 4; ++e) a0[e] = (int)(act[0][unit][e] & keep0), a1[e] = (int)(act[0][unit][e] & keep1);
            fold(acc[0][0], __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, codes, magic, 0, 0, 0), d * (float)(int)__builtin_amdgcn_sbfe(scw, 0, 8), 0, 2 * unit);
            fold(acc[0][0], __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, codes, magic, 0, 0, 0), d * (float)(int)__builtin_amdgcn_sbfe(scw, 16, 8), 0, 2 * unit + 1);
        }
        // one unit at a time (left free, the compiler keeps all the result tiles alive and runs out of registers)
#pragma unroll
        for (int i = 0; i < SETS; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                asm volatile("" : "+v"(acc[i][0][v]));
                if constexpr (T16) asm volatile("" : "+v"(acc[i][1][v]));
            }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto compute = [&](const Weights& w, const Act& b, int kb) {   // one set
        u32x4 act[SETS][4];
        if constexpr (SRC != Q81) {
            quantize<T>(b.v, lane, m_rows, table, codes_of_rows);
        } else {
            put_scales(b, 0);
            turn(b, act[0]);
        }
        put_w(w, kb);
        settle();
        if constexpr (SRC != Q81) {
#pragma unroll
            for (int u = 0; u < 4; ++u) act[0][u] = *(const u32x4*)(codes_of_rows + ((2 * u + (grp >> 1)) * 8 + tok) * 8 + 4 * (grp & 1));
        }
        const uint32_t sh = (my_at + (uint32_t)(kb * Q6K_BYTES)) & 2u;
        uint32_t past;
        u32x4 ql, qhp;
        const u32x4 sc = piece_at(192, sh, past);
        const float d = f16_bits_to_f32((past >> (8 * sh)) & 0xFFFFu);
#pragma unroll
        for (int unit = 0; unit < 4; ++unit) unit_of(unit, act, codes_of(unit, sh, ql, qhp), d, sc[unit]);
        settle();
    };

    if constexpr (SETS == 2) {
        // one super-block's loads in flight: each set of registers is asked for again as soon as it has been read (two would not fit)
        Weights w;
        Act act_of[SETS];
#pragma unroll
        for (int i = 0; i < SETS; ++i) load_act(act_of[i], i, wave);
        load_w(w, wave);
        for (int kb = wave; kb < p.nb; kb += waves) {
#pragma unroll
            for (int i = 0; i < SETS; ++i) put_scales(act_of[i], i);
            put_w(w, kb);
            settle();
            const int next = min(kb + waves, p.nb - 1);   // (past the last one it is read again)
            load_w(w, next);
            const uint32_t sh = (my_at + (uint32_t)(kb * Q6K_BYTES)) & 2u;
            uint32_t past;
            u32x4 ql, qhp;
            const u32x4 sc = piece_at(192, sh, past);
            const float d = f16_bits_to_f32((past >> (8 * sh)) & 0xFFFFu);
            u32x4 act[SETS][4];
#pragma unroll
            for (int i = 0; i < SETS; ++i) turn(act_of[i], act[i]), load_act(act_of[i], i, next);
#pragma unroll
            for (int unit = 0; unit < 4; ++unit) unit_of(unit, act, codes_of(unit, sh, ql, qhp), d, sc[unit]);
            settle();
        }
    } else if constexpr (SRC != Q81) {   // one in flight (registers)
        Weights w;
        Act act;
        for (int kb = wave; kb < p.nb; kb += waves) load_act(act, 0, kb), load_w(w, kb), compute(w, act, kb);
    } else {
        Weights w[2];
        Act act[2];
        auto load = [&](int i, int kb) { load_act(act[i], 0, kb), load_w(w[i], kb); };
        load(0, wave);
        if (wave + waves < p.nb) load(1, wave + waves);
        for (int kb = wave; kb < p.nb; kb += 2 * waves) {
            compute(w[0], act[0], kb);
            if (kb + 2 * waves < p.nb) load(0, kb + 2 * waves);
            if (kb + waves < p.nb) {
                compute(w[1], act[1], kb + waves);
                if (kb + 3 * waves < p.nb) load(1, kb + 3 * waves);
            }
        }
    }

    // the partial tiles, [SETS][4][64] floats at the start of each wave's buffer
    float* part = (float*)buf;
#pragma unroll
    for (int i = 0; i < SETS; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) part[(4 * i + v) * 64 + lane] = T16 ? acc[i][0][v] + acc[i][T16 ? 1 : 0][v] : acc[i][0][v];
    __syncthreads();
    // sixteen rows: output (register v, lane l < 64) adds the waves' lanes l; eight: (v, l < 32) lanes l and l + 32
    constexpr int LANES = 4 * TOKS;
    for (int o = threadIdx.x; o < SETS * 4 * LANES; o += (int)blockDim.x) {
        const int iv = o / LANES, l = o % LANES;
        float sum = 0.f;
        for (int w = 0; w < waves; ++w) {
            const float* col = (const float*)(lds + w * WAVE_BYTES) + iv * 64 + l;
            sum += T16 ? col[0] : col[0] + col[32];
        }
        const int t = (iv >> 2) * TOKS + 4 * (l >> 4) + (iv & 3), row = l & 15;
        if (t < m_rows && row <= last_row) lk_store_as(p.dst, (size_t)(m0 + t) * p.ldd + tile * TILE + row, sum, HALF ? p.out_type : LK_TYPE_F32);
    }
}

template <int TOKS, bool HALF, int SRC = Q81, int SETS = 1>
int launch(const Args& a, hipStream_t stream) {
    constexpr int bytes = wave_bytes(SETS) + (SRC == Q81 ? 0 : CODE_BYTES);
    static const bool ok = hipFuncSetAttribute((const void*)q6k_rows16_short_kernel<TOKS, SETS, HALF, SRC>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                               MAX_WAVES * bytes) == hipSuccess;
    if (!ok) return -1;
    const int steps = (a.nb + MAX_WAVES - 1) / MAX_WAVES, waves = (a.nb + steps - 1) / steps;   // as equal a share of super-blocks as they allow
    hipLaunchKernelGGL((q6k_rows16_short_kernel<TOKS, SETS, HALF, SRC>), dim3((a.n + TILE - 1) / TILE, (a.m + SETS * TOKS - 1) / (SETS * TOKS)), dim3(64 * waves),
                       waves * bytes, stream, a);
    return lk_launch_status();
}

// Whether the short launch takes the call, and the rows of a workgroup. Whether, by the matrix and the class of row counts alone (up to 8, 16, 32, 48,
// 64, 96, 128): its sums are of another order than the other launches', and a row carries the same bits whatever rides with it in its class.
int set_rows(int size_m, int size_n, int size_k) {
    // One workgroup fits a CU (registers), and a second round of them costs what the first did, so the line is the number of
    // workgroups. Eight rows to a workgroup where that is one round, else sixteen or two sets of sixteen, whose rounds are a third longer. Measured in a graph, us, the granules
    // of rows16_q6k.hip (rows of a multiple of 2048 values; more rows than it takes: the 32-row tiles) against this:
    //   3 / 8 rows      1024 x 2048 7.4, 7.4 / 4.3, 4.3; 2048 x 6144 8.8, 9.1 / 7.8, 7.8; 4096 x 4096 8.9, 9.5 / 7.2, 7.2; 4096 x 14336 15.4, 19.3 / 16.2, 16.3;
    //                   6144 x 2048 8.3, 9.8 / 7.0, 7.1; 8192 x 4096 10.5, 12.2 / 12.0, 12.3. Few tiles of long rows stay with the granules, whose waves have
    //                   less to do in LDS a super-block (it is what a CU of twelve waves waits for here): 1024 x 8192 8.9, 9.2 / 9.4, 9.5; 2048 x 14336
    //                   12.6, 13.4 / 14.1, 14.0
    //   9 / 16          1024 x 2048 9.2, 9.3 / 4.3, 4.4; 2048 x 6144 11.0, 11.0 / 8.0, 7.8; 4096 x 4096 10.4, 10.8 / 8.2, 8.2; 4096 x 14336 26.1, 25.8 / 19.1, 19.1;
    //                   2048 x 14336 16.7, 16.7 / 14.6, 14.3; 8192 x 4096 14.4, 15.0 / 14.4, 15.0
    //   24 / 32         1024 x 2048 9.2, 9.3 / 4.4, 4.4; 2048 x 6144 14.6, 12.9 / 9.3, 9.4; 2048 x 14336 24.3, 24.7 / 17.4, 17.3; 4096 x 4096 13.9, 13.7 / 12.9, 14.3
    //   48              1024 x 2048 10.1 / 5.0, 2048 x 6144 22.2 / 16.8, 2048 x 14336 46.0 / 31.2, 4096 x 4096 17.5 / 20.1
    // and against the 32-row tiles where rows are no granules: 700 x 11008 at 8 / 16 / 32 / 64 rows 32, 37, 43, 43 / 10, 11, 11, 14;
    // 10000 x 5120 at 8 / 16 / 32 25.3, 31.6, 36.7 / 19.9, 24.4, 41; 16384 x 3072 at 8 / 16 17.1, 20.2 / 17.9, 20.9; 3000 x 5120 at 32 / 48 20.0, 20.2 / 16.1, 24.1
    const int nb = size_k / 256, tiles = (size_n + TILE - 1) / TILE, cus = lk_device().cus;
    const bool granules = nb % 8 == 0;
    // More than a tile to the CU of rows longer than 4096 values stay too: 3 / 5 / 8 rows 5120 x 8192 15.4, 18.2, 18.7 / 19.3, 19.6, 20.3; 4608 x
    // 14336 21.0, 24.5, 25.7 / 27.4, 27.9, 28.1; 6144 x 10240 23.1, 22.6, 23.2 / 23.0, 23.3, 23.6; 6144 x 6144 13.0, 15.7, 16.6 / 15.5, 15.6, 15.8
    // (at 4096 values 6144 x 4096 11.3, 12.5, 13.0 / 12.3, 12.4, 12.5, and one launch with the quantizer in it).
    if (granules && size_m <= 8 && (2 * tiles <= cus ? nb >= 32 : tiles > cus && nb > 16)) return 0;
    // Two sets of sixteen, with the weights from HBM, others / one set / two: 17 and 32 rows 4096 x 2048 11.2, 10.2 / 8.5, 8.5 / 6.6, 7.3; 4096 x 4096 13.6,
    // 14.3 / 14.4, 14.5 / 9.9, 11.3; 4096 x 6144 23.3, 19.3 / 18.1, 18.3 / 13.1, 14.6; 4096 x 14336 40.1, 40.5 / 34.3, 35.4 / 23.0, 27.0; 8192 x 4096 17.7,
    // 18.4 / 26.8, 27.4 / 18.0, 20.5; 40 and 64 rows 2048 x 2048 11.3, 11.5 / 8.0, 8.3 / 6.5, 6.7; 2048 x 6144 19.5, 21.2 / 17.6, 18.0 / 12.9, 14.0;
    // 2048 x 14336 39.2, 43.1 / 31.5, 32.8 / 22.3, 24.1; 4096 x 6144 19.8, 21.5 / 25.6, 33.4 / 23.7, 24.5; above 64 rows, others / two: 1024 x 2048 at
    // 80 11.4 / 6.4; 1024 x 14336 at 96 42 / 25.
    const int eights = (size_m + 7) / 8, sixteens = (size_m + 15) / 16, pairs = (size_m + 31) / 32;
    if (size_m <= 16) {
        const bool by_eight = size_m <= 8 || (int64_t)tiles * eights <= cus;
        if ((int64_t)tiles * (by_eight ? eights : sixteens) > (granules ? 3 * cus / 2 : 3 * cus)) return 0;
        return by_eight ? 8 : 16;
    }
    const bool pays = size_m <= 32 ? tiles <= (granules ? cus : 3 * cus / 2)
                      : size_m <= 64 ? tiles * (size_m <= 48 ? 3 : 4) <= 2 * cus
                                     : tiles * (size_m <= 96 ? 3 : 4) <= cus;
    if (!pays) return 0;
    if (tiles * eights <= cus) return 8;
    const int steps = (nb + MAX_WAVES - 1) / MAX_WAVES, resident = cus * (MAX_WAVES / ((nb + steps - 1) / steps));
    // a workgroup of two sets takes 4 / 3 of one with one, of short rows 3 / 2 (5000 x 2304 at 32 rows 13.8 us with one, 14.7 with two; 6000 x 5120 24.8, 24.7)
    const int rounds_two = (tiles * pairs + resident - 1) / resident, rounds_one = (tiles * sixteens + resident - 1) / resident;
    return (nb < 16 ? 3 * rounds_two < 2 * rounds_one : 4 * rounds_two < 3 * rounds_one) ? 32 : 16;
}

}  // namespace

bool lk_rows16_q6k_short_pays(int size_m, int size_n, int size_k) {
    // (rows of more than 32768 values: the others' to take or refuse)
    return size_m >= 1 && size_m <= 128 && size_n >= 1 && size_k >= 256 && size_k <= 32768 && !lk_rows16_off(size_m) && set_rows(size_m, size_n, size_k) != 0;
}

int lk_rows16_q6k_short(const void* w, const void* q8_1, float* output, int size_m, int size_n, int size_k, int stride_y, int ldd,
                        hipStream_t stream, int out_type) {
    if ((((uintptr_t)w) & 15) != 0 || !lk_rows16_q6k_short_pays(size_m, size_n, size_k)) return -1;
    const int rows = set_rows(size_m, size_n, size_k);
    const Args a{(const uint8_t*)w, (const uint8_t*)q8_1, output, size_k / 256, size_n, size_m, stride_y, ldd, out_type};
    if (rows == 32) return out_type == LK_TYPE_F32 ? launch<16, false, Q81, 2>(a, stream) : launch<16, true, Q81, 2>(a, stream);
    if (rows == 8) return out_type == LK_TYPE_F32 ? launch<8, false>(a, stream) : launch<8, true>(a, stream);
    return out_type == LK_TYPE_F32 ? launch<16, false>(a, stream) : launch<16, true>(a, stream);
}

// Rows of up to 4096 values straight from them where sets of eight are a workgroup to the CU, as lk_rows16_short_rows (672 x 1024 at 18 rows 9.6 us a call,
// 5.8 on the chip / 6.3, 4.2; 640 x 3584 at 44 9.2, 7.9 / 7.4, 7.5).
int lk_rows16_q6k_short_rows(const void* w, const void* x, float* output, int size_m, int size_n, int size_k, int x_type, hipStream_t stream) {
    if (size_k > 4096 || (((uintptr_t)w) & 15) != 0 || !lk_rows16_q6k_short_pays(size_m, size_n, size_k) || set_rows(size_m, size_n, size_k) != 8) return -1;
    if (size_m > 16 && size_n < 512) return -1;   // (a call recorded with nothing reserved stays refused, as in rows16_short.hip: 6.7 to 7.0 us, one launch 4.9 to 6.1)
    const Args a{(const uint8_t*)w, (const uint8_t*)x, output, size_k / 256, size_n, size_m, 0, size_n, x_type};
    if (x_type == LK_TYPE_F32) return launch<8, false, ROWS_F32>(a, stream);
    return x_type == LK_TYPE_F16 ? launch<8, true, ROWS_F16>(a, stream) : launch<8, true, ROWS_BF16>(a, stream);
}
