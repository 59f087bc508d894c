// What the tiled-matmul kernels share: the problem record and the one-time kernel set-up.
#pragma once

#include "lk_common.h"

#include <mutex>
#include <unordered_map>

constexpr int MMQ_REC_BYTES = 288;   // workspace record: 256 codes + 8 f16 scales + 8 i16 sums

// One problem = one weight slab against a contiguous run of workspace rows.
struct MmqProblem {
    const uint8_t* w;      // [n][nb] blocks
    const uint8_t* y;      // workspace records
    float* dst;
    const int32_t* ids_dst;  // nullable: destination row of workspace row c
    int64_t nb;            // K steps: 256-value blocks per weight row
    int64_t row_blocks;    // format blocks between consecutive weight rows
    int64_t rows_total;    // rows the workspace was quantized with (record stride)
    int64_t ldd;           // floats between destination rows
    int n, m_begin, m_end;
    int out_type = LK_TYPE_F32;   // element type of `dst` (lk_store_as)
};

// Four results of one row from element `at` of the destination on; `vec`: f32 and 16-byte pieces allowed.
static __device__ __forceinline__ void mmq_store4(const MmqProblem& pb, int64_t at, const float4& v, bool vec) {
    if (vec) {
        *(float4*)(pb.dst + at) = v;
    } else if (pb.out_type == LK_TYPE_F32) {
        pb.dst[at] = v.x; pb.dst[at + 1] = v.y; pb.dst[at + 2] = v.z; pb.dst[at + 3] = v.w;
    } else {
        uint16_t h[4];
        const float f[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
            h[e] = pb.out_type == LK_TYPE_F16 ? __half_as_ushort(__float2half_rn(f[e])) : __bfloat16_as_ushort(__float2bfloat16(f[e]));
        uint16_t* out = (uint16_t*)pb.dst + at;
        if (((uintptr_t)out & 7) == 0) {
            *(uint2*)out = make_uint2(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) out[e] = h[e];
        }
    }
}

// Raises a kernel's dynamic LDS limit once per process; LK_ERR_ARG when the device has less.
template <typename K>
static int mmq_prepare_kernel(K kernel, int lds_bytes) {
    static std::mutex mu;
    static std::unordered_map<const void*, bool> done;
    std::lock_guard<std::mutex> lock(mu);
    if (done.count((const void*)kernel)) return LK_OK;
    if (lds_bytes > lk_device().lds_bytes) return LK_ERR_ARG;
    if (lds_bytes > 48 * 1024 &&
        hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) != hipSuccess) {
        (void)hipGetLastError();
        return LK_ERR_LAUNCH;
    }
    done[(const void*)kernel] = true;
    return LK_OK;
}

// What the caller's tmp_fixup holds (FIXUP_BYTES, src/tensor/quantized/kernel_matmul/mmq.rs:42): the
// reference's kernels keep their stream-k partial tiles there, these the partial products of a cut K.
constexpr int64_t MMQ_FIXUP_BYTES = 256ll * 128 * 128 * 4;

// A dense product whose tiles alone leave most of the chip idle is launched with K cut into ranges of
// blocks: a workgroup walks one range and writes its partial tile to part[range] ([token][n rounded up to four] floats
// in the caller's tmp_fixup), and lk_mmq_split_sum adds the ranges in ascending order, so a result does
// not depend on which workgroup finished when. mmq_splits: how many ranges, for `tiles` tiles on a chip
// that holds `slots` workgroups of the kernel at once: as many as bring tiles x ranges to the slots,
// while a range keeps at least two blocks and every partial product fits the buffer. 1 = the plain launch.
// Rows of a partial product are mmq_part_stride floats apart, so that the sum reads whole 16-byte pieces; `ragged`:
// the kernel cuts K of a matrix whose row count is no multiple of four, or into a destination of any alignment, too
// (11003 x 4096 at 77 rows, quantizer included: Q4_K 63 -> 40 us, Q5_K 73 -> 44, Q6_K 89 -> 51).
__host__ __device__ static inline int64_t mmq_part_stride(const MmqProblem& pb) { return ((int64_t)pb.n + 3) / 4 * 4; }
// What the host linear keeps for its own products: a product of many rows and columns has too few tiles for the chip at twice the
// partial products (1186 x 10240 at 1661 rows of Q6_K: 16 MiB leave it whole, 32 allow three ranges; 64 give no call of 1300 more). A recorded call
// whose plan has no use for more takes MMQ_FIXUP_BYTES, and so does one that cannot have this much.
constexpr int64_t MMQ_HOST_FIXUP_BYTES = 2 * MMQ_FIXUP_BYTES;
// The most ranges K may be cut into: two blocks each, their partial products in the buffer; 1 where it stays whole.
static inline int mmq_splits_most(const MmqProblem& pb, const void* fixup, bool ragged = false, int64_t fixup_bytes = MMQ_FIXUP_BYTES) {
    if (!fixup || pb.ids_dst || pb.m_begin != 0) return 1;
    const bool f32 = pb.out_type == LK_TYPE_F32;
    if (!ragged && (pb.n % 4 != 0 || (f32 && (pb.ldd % 4 != 0 || (uintptr_t)pb.dst % 16 != 0)))) return 1;
    if ((uintptr_t)fixup % 16 != 0) return 1;
    int64_t most = fixup_bytes / ((int64_t)pb.m_end * mmq_part_stride(pb) * 4);
    if (most > pb.nb / 2) most = pb.nb / 2;
    return most < 2 ? 1 : (int)most;
}
static inline int mmq_splits(const MmqProblem& pb, int64_t tiles, int64_t slots, const void* fixup) {
    const int forced = lk_tune_env("LK_TUNE_MMQ_SPLITS");   // measurement runs: -1 never, n > 0 that many where they fit
    if (forced < 0) return 1;
    const int64_t want = forced > 0 ? forced : slots / tiles, most = mmq_splits_most(pb, fixup);
    return want < 2 ? 1 : (int)(want < most ? want : most);
}
// dst[token][c] = part[0][token][c] + part[1][token][c] + ..., part[i] m_end x mmq_part_stride floats; LK_* status.
int lk_mmq_split_sum(const float* part, int splits, const MmqProblem& pb, hipStream_t s);

// Expert-batched launches: workgroup (x, y, z) = (n tile + n_tiles * (column tile % group), stack * experts + expert,
// column tile / group). The full tiles of a run of average length are issued together (they share the expert's weights
// in the caches); what lies past them comes after every expert's, so that the launch ends on the short tiles instead of
// paying a whole round of workgroups for them, and the workgroups of experts without such a tile do not skew the
// round robin over the XCDs. All of an expert's tiles together against this order: 128 experts, top-8, average run 50
// (longest expected 72), Q6_K block 477 us against 371, Q4_K 315 against 270; 32 experts of 3072 -> 512, average 70,
// Q6_K 151 against 141; 128 experts at 1111 tokens (average 69, Q6_K down) 447 against 427.
struct MmqMoeGrid {
    dim3 grid;
    int group;
};
static inline MmqMoeGrid mmq_moe_grid(const MmqProblem& pb, int tn, int tm, int stacks, int n_experts, int64_t ncols_max) {
    const int64_t n_tiles = ((int64_t)pb.n + tn - 1) / tn;
    int64_t col_tiles = (ncols_max + tm - 1) / tm;
    col_tiles = col_tiles < 1 ? 1 : col_tiles > 65535 ? 65535 : col_tiles;
    int64_t group = pb.rows_total / n_experts / tm;
    group = group < 1 ? 1 : group > col_tiles ? col_tiles : group;
    return {dim3((unsigned)(n_tiles * group), (unsigned)(stacks * n_experts), (unsigned)((col_tiles + group - 1) / group)), (int)group};
}

// Q4_K, Q5_K, Q6_K, Q8_0 and Q4_0 on the f16 tiles of mmq_tile.h. tt: token tiles of 32 a wave takes; waves: 4 (two workgroups a CU) or
// 8 (tt = 4, one); splits: ranges of K, partial products as above.
struct MmqTilePlan {
    int tt, waves, splits;
};
struct LkTokenOperands;
int lk_tile_dense_q4k(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTilePlan& plan, float* part, hipStream_t s);
int lk_tile_dense_q5k(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTilePlan& plan, float* part, hipStream_t s);
int lk_tile_dense_q6k(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTilePlan& plan, float* part, hipStream_t s);
int lk_tile_dense_q80(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTilePlan& plan, float* part, hipStream_t s);
int lk_tile_dense_q40(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTilePlan& plan, float* part, hipStream_t s);
// Expert-batched: expert e's slab, `stride` bytes after the one before, against the sorted rows [bounds[e], bounds[e + 1]).
// With `to`: gate (the problem's weights) and up (w_second) products of operand rows gather[sorted row], and silu(gate) * up as
// the operands `to` of the next product, a row per sorted row. Else the products to dst, w_second's dst_second floats further.
struct MmqTileExperts {
    const int32_t *bounds, *gather;
    const uint8_t* w_second;
    int64_t dst_second, stride, longest;   // longest: expected longest run
    int n_experts;
    const LkTokenOperands* to;
};
int lk_tile_moe_q4k(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTileExperts& ex, hipStream_t s);
int lk_tile_moe_q5k(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTileExperts& ex, hipStream_t s);
int lk_tile_moe_q6k(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTileExperts& ex, hipStream_t s);
int lk_tile_moe_q80(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTileExperts& ex, hipStream_t s);
int lk_tile_moe_q40(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTileExperts& ex, hipStream_t s);
int lk_tile_moe_iq4nl(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTileExperts& ex, hipStream_t s);
int lk_tile_moe_mxfp4(const MmqProblem& pb, const LkTokenOperands& ops, const MmqTileExperts& ex, hipStream_t s);
// Whether an expert-batched product can take them (alignment, sizes); `gated`: as lk_tile_moe_* with `to`.
bool lk_mmq_tiles_moe_fit(int wtype, const void* w, const void* w_second, int64_t stride, int64_t n, int64_t k, int64_t rows, bool gated);
int lk_mmq_tiles_moe(int wtype, const MmqProblem& pb, const LkTokenOperands& ops, const MmqTileExperts& ex, hipStream_t s);
// `rows` rows of x (k values each) as token operands.
int lk_operands_quantize(const void* x, int type, const LkTokenOperands& ops, int k, int rows, hipStream_t s);
// A dense product on them (mmq_tiles.hip), operands made from the workspace records; `fixup`: the caller's tmp_fixup or null.
// Returns the token-tile width launched, 0 when the launch failed, -1 when the operands do not suit these kernels (alignment,
// 32-bit offsets, no scratch) and the caller should take the int8 tiles.
int lk_mmq_tiles_dense(int wtype, const MmqProblem& pb, hipStream_t s, void* fixup);
// lk_mmq_f16_tiles: whether a dense product takes them: 9 token rows or more and 512 weight rows or more (LK_MMQ_I8 unset).
// Bytes of partial products that the plan of such a product writes, given MMQ_HOST_FIXUP_BYTES.
int64_t lk_mmq_tiles_parts(int wtype, int k, int n, int rows);
// The same for `rows` rows of x, k values each, results in x's type: nothing between x and the operands.
int lk_mmq_tiles_linear(int wtype, void* fixup, int64_t fixup_bytes, const void* w, const void* x, int type, void* out, int k, int n, int rows, hipStream_t s);
// The same from the rows' Q8_1 blocks, `stride` blocks between rows, with the same bits.
int lk_mmq_tiles_linear_q8_1(int wtype, void* fixup, int64_t fixup_bytes, const void* w, const void* q8_1, int stride, int type, void* out, int k, int n, int rows,
                             hipStream_t s);
// The expert-batched product over workspace records, same returns as the dense one.
int lk_mmq_tiles_moe_records(int wtype, const MmqProblem& pb, const uint8_t* w_second, int64_t dst_second, const int32_t* bounds,
                             int64_t stride_expert, int n_experts, int64_t ncols_max, hipStream_t s);
