// Products of Q4_K, Q5_K, Q6_K, Q8_0 and Q4_0 weights on the f16 tiles (mmq_tile.h): which tile a call takes, and the token operands.

#include "mmq_operands.h"
#include "mmq_problem.h"
#include "stream_scratch.h"

#include <algorithm>

namespace {

// A sub-block's 32 codes as its four atoms; Vec: sixteen bytes as `codes` is aligned.
template <class Vec>
static __device__ __forceinline__ void operand_atoms(const uint8_t* codes, uint8_t* to) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const Vec c = *(const Vec*)(codes + 16 * h);
        uint4 lo, hi;
        operand_codes(c.x, lo.x, lo.y);
        operand_codes(c.y, lo.z, lo.w);
        operand_codes(c.z, hi.x, hi.y);
        operand_codes(c.w, hi.z, hi.w);
        *(uint4*)(to + 16 * h) = lo;
        *(uint4*)(to + 32 + 16 * h) = hi;
    }
}

// Workspace records -> operands. grid (blocks, rows / 32), 256 threads: eight threads a row, a sub-block each.
__global__ __launch_bounds__(256) void operands_from_records_kernel(const uint8_t* __restrict__ y, LkTokenOperands ops, int64_t rec_rows,
                                                                    int row0, int rows) {
    const int kb = blockIdx.x, s = threadIdx.x & 7;
    const int r = blockIdx.y * 32 + (threadIdx.x >> 3);
    if (r >= rows) return;
    const uint8_t* rec = y + ((int64_t)kb * rec_rows + row0 + r) * MMQ_REC_BYTES;
    operand_atoms<uint4>(rec + 32 * s, ops.codes + ((int64_t)kb * ops.rows + r) * LK_OPERAND_CODES + 64 * s);
    operand_scales(ops.tabs + ((int64_t)kb * ops.rows + r) * LK_OPERAND_TAB, s, f16_bits_to_f32(*(const uint16_t*)(rec + 256 + 2 * s)),
                   (int)*(const int16_t*)(rec + 272 + 2 * s));
}

// The runs' share of the sorted rows [from, to), counted from `from`.
__global__ __launch_bounds__(256) void bounds_of_pass_kernel(const int32_t* __restrict__ bounds, int32_t* __restrict__ pass, int count, int from, int to) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e < count) pass[e] = min(max(bounds[e], from), to) - from;
}

// Q8_1 rows, `stride` blocks apart -> operands, on the same grid: the codes and scales the quantizer below makes of the rows
// they came from, so the products carry its bits. A few rows a call: a launch's time, whatever the bytes.
__global__ __launch_bounds__(256) void operands_from_q8_1_kernel(const uint8_t* __restrict__ y, LkTokenOperands ops, int stride, int rows) {
    const int kb = blockIdx.x, s = threadIdx.x & 7;
    const int r = blockIdx.y * 32 + (threadIdx.x >> 3);
    if (r >= rows) return;
    const uint8_t* block = y + ((int64_t)r * stride + 8 * kb + s) * Q81_BYTES;
    operand_atoms<uint4_a4>(block + 4, ops.codes + ((int64_t)kb * ops.rows + r) * LK_OPERAND_CODES + 64 * s);
    int sum = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) sum = __builtin_amdgcn_sdot4(*(const int*)(block + 4 + 4 * i), 0x01010101, sum, false);
    operand_scales(ops.tabs + ((int64_t)kb * ops.rows + r) * LK_OPERAND_TAB, s, f16_bits_to_f32(*(const uint16_t*)block), sum);
}

// Rows of x -> operands, the quantizer and the expansion in one pass: grid (rows, k / 1024), four values a thread. Bound by
// its bytes (2048 x 14336 f32: 185 MB); the records' quantizer and the expansion after it move 285.
template <typename T>
__global__ __launch_bounds__(256) void operands_quantize_kernel(const T* __restrict__ x, LkTokenOperands ops, int k) {
    const int i0 = (blockIdx.y * 256 + threadIdx.x) * 4;
    if (i0 >= k) return;
    const int64_t row = blockIdx.x, at = (int64_t)(i0 / 256) * ops.rows + row;
    const T* from = x + row * k + i0;
    const float4 v = ((uintptr_t)from & (4 * sizeof(T) - 1)) == 0
                         ? Load4<T>::at(from)
                         : make_float4(to_f32<T>(from[0]), to_f32<T>(from[1]), to_f32<T>(from[2]), to_f32<T>(from[3]));
    operand_quad(v, ops.codes + at * LK_OPERAND_CODES, ops.tabs + at * LK_OPERAND_TAB, (i0 / 32) & 7, (i0 / 4) & 7);
}

// The formats' kernels; unit: bytes that `row_blocks` counts, of `values` values; align: of the weights.
struct Tiles {
    int type, unit, values, align, tt_most;
    int (*dense)(const MmqProblem&, const LkTokenOperands&, const MmqTilePlan&, float*, hipStream_t);
    int (*moe)(const MmqProblem&, const LkTokenOperands&, const MmqTileExperts&, hipStream_t);
};
constexpr Tiles TILES[] = {{LK_TYPE_Q4_K, Q4K_BYTES, 256, 16, 4, lk_tile_dense_q4k, lk_tile_moe_q4k},
                           {LK_TYPE_Q5_K, Q5K_BYTES, 256, 16, 4, lk_tile_dense_q5k, lk_tile_moe_q5k},
                           {LK_TYPE_Q6_K, Q6K_BYTES, 256, 2, 4, lk_tile_dense_q6k, lk_tile_moe_q6k},
                           {LK_TYPE_Q8_0, Q80_BYTES, 32, 2, 3, lk_tile_dense_q80, lk_tile_moe_q80},
                           {LK_TYPE_Q4_0, Q40_BYTES, 32, 2, 4, lk_tile_dense_q40, lk_tile_moe_q40},
                           {LK_TYPE_IQ4_NL, 18, 32, 2, 4, nullptr, lk_tile_moe_iq4nl},   // experts only
                           {LK_TYPE_MXFP4, 17, 32, 1, 4, nullptr, lk_tile_moe_mxfp4}};
const Tiles* tiles_of(int wtype) {
    for (const Tiles& t : TILES)
        if (t.type == wtype) return &t;
    return nullptr;
}

// What a launch takes, fitted to 2200 shapes on MI355X (those of the benchmark's models and drawn ones of 512 to 16384 x 1024 to 14336, 9 to 2048 rows, each at
// every tile width with K whole and cut into 2 to 12 ranges) for the plan it picks: 0.7 % longer in the mean than the best one of the sweep (the items' times
// are what makes it pick well, no more: a plan of each kind measured alone gives others). alone /
// full: nanoseconds an item (32 x 32 x 32 product) takes a SIMD with one workgroup on its CU or two, by token
// tiles; wide: with eight waves and tt = 4. start: microseconds of a workgroup beside its items. whole: how far rounds of workgroups stay apart
// (1: whole rounds). (As fitted to whole launches whose workgroups were dealt unevenly to the XCDs, with K cut into even ranges only, the picks were
// 3.8 % behind.) Q8_0 and Q4_0, whose items are longer, from 3100 shapes of their own (0.5 and 0.3 % behind the best; with the K-quants' blurred rounds 0.8 and 0.4, by more where a
// vocabulary meets a few rows, as K was left whole: Q8_0 79538 x 3328 at 14 129 us against 116 in two ranges, Q4_0 80340 x 3840 at 13 109 / 101, and in rounds that
// are just full: Q8_0 16060 x 7424 at 23 65 in two ranges, 56 in four).
struct ItemTimes {
    double alone[4], full[4], wide, start, whole;
};
constexpr ItemTimes ONE_TERM = {{162, 111, 121, 93.8}, {137, 93.6, 82.2, 75.7}, 67.4, 0.357, 0.655}, TWO_TERMS = {{239, 146, 166, 152}, {221, 140, 124, 122}, 0, 1.30, 0.655},
                    Q8_ITEM = {{267, 164, 179, 0}, {218, 150, 123, 0}, 0, 0.98, 1}, Q4_ITEM = {{249, 164, 180, 145}, {217, 145, 128, 114}, 0, 0.06, 1};

// The tile and the cut of K with the shortest estimated launch. Up to 2 * cus workgroups run at once, and a CU that holds two takes
// nearly the time of a full chip; past that the rounds blur (K-quants: two thirds of whole rounds, one of their share)
// but for the start of each, without which Q6_K 9675 x 9728 at 23 rows was cut into ten (52 us; into six, the most that is one round, 42). Of two workgroups on a CU with ranges
// of unequal length not both are the longest: two thirds of it, one of the mean. A cut costs a launch and its
// partial products, written, read and added.
MmqTilePlan plan_dense(const Tiles& f, const MmqProblem& pb, const void* fixup, int64_t fixup_bytes) {
    const ItemTimes& t = f.type == LK_TYPE_Q6_K ? TWO_TERMS : f.type == LK_TYPE_Q8_0 ? Q8_ITEM : f.type == LK_TYPE_Q4_0 ? Q4_ITEM : ONE_TERM;
    const int cus = lk_device().cus;
    const int forced_tt = lk_tune_env("LK_TUNE_MMQ_TT"), forced_splits = lk_tune_env("LK_TUNE_MMQ_SPLITS");   // measurement runs
    const int most = forced_splits < 0 ? 1 : std::min(mmq_splits_most(pb, fixup, true, fixup_bytes), 12);
    MmqTilePlan best{f.tt_most, 4, 1};
    double least = 1e30;
    for (int tt = 1; tt <= f.tt_most; ++tt) {
        if (forced_tt > 0 && tt != forced_tt) continue;
        const int64_t tiles = ((pb.n + 127ll) / 128) * ((pb.m_end + 32ll * tt - 1) / (32 * tt));
        for (int splits = forced_splits > 0 ? std::min(forced_splits, most) : 1; splits <= most; ++splits) {
            const double longest = (double)((pb.nb + splits - 1) / splits), mean = (double)pb.nb / splits, block = 8e-3 * tt;   // blocks; thousands of items
            const double one = t.start + block * longest * t.alone[tt - 1], two = t.start + 2 * block * (0.639 * longest + 0.361 * mean) * t.full[tt - 1];
            const int64_t groups = tiles * splits, rounds = groups / (2 * cus), rest = groups % (2 * cus);
            double us = rounds * two;
            if (rest > 0) us += rest <= cus ? one : one + (two - one) * (0.779 + 0.221 * (rest - cus) / cus);
            if (rounds > 0) us = t.whole * us + (1 - t.whole) * two * groups / (2 * cus);
            us += 2.38 * (double)((groups - 1) / (2 * cus));
            if (splits > 1) us += 1.85 + 0.227e-6 * (splits + 1) * pb.m_end * pb.n * 4;
            if (us < least) least = us, best = {tt, 4, splits};
            if (forced_splits > 0) break;
        }
    }
    if (t.wide > 0 && forced_splits <= 0 && (forced_tt <= 0 || forced_tt == 8)) {
        const int64_t tiles = ((pb.n + 255ll) / 256) * ((pb.m_end + 127ll) / 128), rest = tiles % cus;
        const double round = 64e-3 * pb.nb * t.wide;
        // (4.5 us the start of a round: without it short rows were taken here too, 13367 x 1536 of Q5_K at 1573 rows 131 us, with four waves 125)
        if (round * (tiles / cus + (rest > 0 ? 0.8 + 0.2 * rest / cus : 0.0)) + 4.5 * ((tiles + cus - 1) / cus) < least) best = {4, 8, 1};
    }
    return best;
}

// What the operands of one pass may take; a call with more goes in passes of token rows over the same buffer (stream order
// keeps them apart).
constexpr int64_t OPERANDS_CAP = 256ll << 20;

// Rows of a pass over `blocks` 256-value blocks each; less than 128: rows too long for these kernels.
int64_t rows_of_pass(int64_t blocks) { return OPERANDS_CAP / (blocks * (LK_OPERAND_CODES + LK_OPERAND_TAB)) / 128 * 128 - LK_OPERAND_PAD; }

// The product in passes; fill(operands, first row, rows) launches what writes a pass's operands. Returns as lk_mmq_tiles_dense.
template <class Fill>
int run_dense(const Tiles& f, const MmqProblem& pb, hipStream_t s, void* fixup, int64_t fixup_bytes, Fill fill) {
    if ((uintptr_t)pb.w % f.align != 0 || (f.align != 16 && pb.n < 128)) return -1;
    // lane offsets inside a tile are 32-bit
    if (pb.row_blocks * f.unit * 256 > (int64_t)INT32_MAX || pb.m_begin != 0) return -1;
    const int64_t fit = rows_of_pass(pb.nb);
    if (fit < 128 || pb.nb > INT32_MAX / 2) return -1;
    const int per_pass = (int)std::min<int64_t>(pb.m_end, fit);
    LkScratch scratch(s);
    void* buffer = scratch.get(LK_SCRATCH_TOKENS, lk_operand_bytes(per_pass, pb.nb));
    if (!buffer) return -1;
    int width = 0;
    for (int m0 = 0; m0 < pb.m_end; m0 += per_pass) {
        MmqProblem pass = pb;
        pass.m_end = std::min(per_pass, pb.m_end - m0);
        pass.dst = (float*)((uint8_t*)pb.dst + (int64_t)m0 * pb.ldd * (pb.out_type == LK_TYPE_F32 ? 4 : 2));
        const LkTokenOperands ops = lk_operands_at(buffer, pass.m_end, pb.nb);
        const MmqTilePlan plan = plan_dense(f, pass, fixup, fixup_bytes);
        fill(ops, m0, pass.m_end);
        if (f.dense(pass, ops, plan, (float*)fixup, s) != LK_OK) return 0;
        if (plan.splits > 1 && lk_mmq_split_sum((const float*)fixup, plan.splits, pass, s) != LK_OK) return 0;
        width = std::max(width, 32 * plan.tt);
    }
    return width;
}

}  // namespace

int lk_mmq_tiles_dense(int wtype, const MmqProblem& pb, hipStream_t s, void* fixup) {
    const Tiles* f = tiles_of(wtype);
    if (!f || !f->dense || (uintptr_t)pb.y % 16 != 0) return -1;
    return run_dense(*f, pb, s, fixup, MMQ_FIXUP_BYTES, [&](const LkTokenOperands& ops, int m0, int rows) {
        hipLaunchKernelGGL(operands_from_records_kernel, dim3((unsigned)pb.nb, (unsigned)((rows + 31) / 32)), dim3(256), 0, s, pb.y, ops,
                           pb.rows_total, m0, rows);
    });
}

extern "C" int lk_mmq_f16_tiles(int wtype, int64_t n, int64_t rows) {
    const Tiles* f = tiles_of(wtype);
    return f && f->dense && rows > 8 && n >= 512 && !lk_env_flag("LK_MMQ_I8");
}

int64_t lk_mmq_tiles_parts(int wtype, int k, int n, int rows) {
    if (!lk_mmq_f16_tiles(wtype, n, rows) || k % 256 != 0) return 0;
    MmqProblem pb{};
    pb.nb = k / 256, pb.m_end = rows, pb.n = n;
    if (rows > rows_of_pass(pb.nb)) return MMQ_HOST_FIXUP_BYTES;   // several passes: the last one's plan is another
    const int splits = plan_dense(*tiles_of(wtype), pb, (void*)256, MMQ_HOST_FIXUP_BYTES).splits;
    return splits > 1 ? splits * (int64_t)rows * mmq_part_stride(pb) * 4 : 0;
}

int lk_mmq_tiles_linear(int wtype, void* fixup, int64_t fixup_bytes, const void* w, const void* x, int type, void* out, int k, int n, int rows, hipStream_t s) {
    if (!lk_mmq_f16_tiles(wtype, n, rows) || k % 256 != 0) return -1;
    const MmqProblem pb{(const uint8_t*)w, nullptr, (float*)out, nullptr, k / 256, k / tiles_of(wtype)->values, rows, n, n, 0, rows, type};
    return run_dense(*tiles_of(wtype), pb, s, fixup, fixup_bytes, [&](const LkTokenOperands& ops, int m0, int count) {
        (void)lk_operands_quantize((const uint8_t*)x + (int64_t)m0 * k * (type == LK_TYPE_F32 ? 4 : 2), type, ops, k, count, s);
    });
}

int lk_mmq_tiles_linear_q8_1(int wtype, void* fixup, int64_t fixup_bytes, const void* w, const void* q8_1, int stride, int type, void* out, int k, int n, int rows,
                             hipStream_t s) {
    if (!lk_mmq_f16_tiles(wtype, n, rows) || k % 256 != 0) return -1;
    const MmqProblem pb{(const uint8_t*)w, nullptr, (float*)out, nullptr, k / 256, k / tiles_of(wtype)->values, rows, n, n, 0, rows, type};
    return run_dense(*tiles_of(wtype), pb, s, fixup, fixup_bytes, [&](const LkTokenOperands& ops, int m0, int count) {
        hipLaunchKernelGGL(operands_from_q8_1_kernel, dim3((unsigned)pb.nb, (unsigned)((count + 31) / 32)), dim3(256), 0, s,
                           (const uint8_t*)q8_1 + (int64_t)m0 * stride * Q81_BYTES, ops, stride, count);
    });
}

int lk_operands_quantize(const void* x, int type, const LkTokenOperands& ops, int k, int rows, hipStream_t s) {
    const dim3 grid((unsigned)rows, (unsigned)((k + 1023) / 1024));
    if (type == LK_TYPE_F16) hipLaunchKernelGGL(operands_quantize_kernel<__half>, grid, dim3(256), 0, s, (const __half*)x, ops, k);
    else if (type == LK_TYPE_BF16) hipLaunchKernelGGL(operands_quantize_kernel<__hip_bfloat16>, grid, dim3(256), 0, s, (const __hip_bfloat16*)x, ops, k);
    else hipLaunchKernelGGL(operands_quantize_kernel<float>, grid, dim3(256), 0, s, (const float*)x, ops, k);
    return lk_launch_status();
}

bool lk_mmq_tiles_moe_fit(int wtype, const void* w, const void* w_second, int64_t stride, int64_t n, int64_t k, int64_t rows, bool gated) {
    const Tiles* f = tiles_of(wtype);
    if (!f || k % 256 != 0 || n > INT32_MAX || n < 128 || (gated && n % 64 != 0)) return false;
    // operand row offsets inside a block, and row offsets inside a tile, are 32-bit
    return ((uintptr_t)w | (uintptr_t)w_second | (uintptr_t)stride) % f->align == 0 && rows < (1 << 23) && k / f->values * f->unit * 128 <= (int64_t)INT32_MAX;
}

int lk_mmq_tiles_moe(int wtype, const MmqProblem& pb, const LkTokenOperands& ops, const MmqTileExperts& ex, hipStream_t s) {
    return tiles_of(wtype)->moe(pb, ops, ex, s);
}

int lk_mmq_tiles_moe_records(int wtype, const MmqProblem& pb, const uint8_t* w_second, int64_t dst_second, const int32_t* bounds,
                             int64_t stride_expert, int n_experts, int64_t ncols_max, hipStream_t s) {
    if ((uintptr_t)pb.y % 16 != 0 || pb.row_blocks > INT32_MAX / 256 || pb.nb > INT32_MAX / 256 ||
        !lk_mmq_tiles_moe_fit(wtype, pb.w, w_second, stride_expert, pb.n, tiles_of(wtype)->values * pb.row_blocks, pb.rows_total, false))
        return -1;
    // More sorted rows than a pass holds: pass by pass, every expert's run cut at the pass's ends (its weights are read again by the
    // pass that goes on with it)
    const int64_t fit = rows_of_pass(pb.nb);
    if (fit < 128) return -1;
    const int64_t per_pass = std::min(pb.rows_total, fit);
    const size_t operand_bytes = lk_operand_bytes(per_pass, pb.nb);
    const bool whole = per_pass == pb.rows_total;
    LkScratch scratch(s);
    uint8_t* buffer = (uint8_t*)scratch.get(LK_SCRATCH_TOKENS, operand_bytes + (whole ? 0 : (size_t)(n_experts + 1) * 4));
    if (!buffer) return -1;
    int32_t* cut = (int32_t*)(buffer + operand_bytes);
    for (int64_t m0 = 0; m0 < pb.rows_total; m0 += per_pass) {
        MmqProblem pass = pb;
        pass.rows_total = std::min(per_pass, pb.rows_total - m0);
        if (pass.ids_dst) pass.ids_dst += m0;
        else pass.dst += m0 * pb.ldd;
        const LkTokenOperands ops = lk_operands_at(buffer, pass.rows_total, pb.nb);
        hipLaunchKernelGGL(operands_from_records_kernel, dim3((unsigned)pb.nb, (unsigned)((pass.rows_total + 31) / 32)), dim3(256), 0, s, pb.y, ops,
                           pb.rows_total, (int)m0, (int)pass.rows_total);
        if (!whole)
            hipLaunchKernelGGL(bounds_of_pass_kernel, dim3((unsigned)(n_experts / 256 + 1)), dim3(256), 0, s, bounds, cut, n_experts + 1, (int)m0,
                               (int)(m0 + pass.rows_total));
        const MmqTileExperts ex{whole ? bounds : cut, nullptr, w_second, dst_second, stride_expert, std::min(ncols_max, pass.rows_total), n_experts, nullptr};
        if (lk_mmq_tiles_moe(wtype, pass, ops, ex, s) != LK_OK) return 0;
    }
    return 128;
}
