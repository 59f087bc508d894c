// The steps of a mixture layer's expert block as lk_moe_forward (moe_forward.hip) puts them together: the
// same launches the exported entry points make, with what only a caller of both halves can ask for.
#pragma once

#include "mmq_operands.h"

// loken_moe_gemm_gguf_gate_up_silu_mul / loken_moe_gemm_gguf_down_reduce over pairs in slot order: pair i is
// slot i of expert choices[i], so no sorted routing is needed, and the down side writes `out` instead of
// adding to it. `wire`: the format's id of the reference's table.
int lk_moe_pairs_gate_up(int wire, const float* x, const void* gate, const void* up, const int32_t* choices, float* h, int experts,
                         int topk, int pairs, int ffn, int hidden, hipStream_t s);
int lk_moe_pairs_down(int wire, const float* h, const void* down, const int32_t* choices, const float* weights, float* out,
                      int experts, int topk, int pairs, int hidden, int ffn, hipStream_t s);
// What the two work in besides `h` (LK_SCRATCH_LAUNCHER), bytes.
size_t lk_moe_pairs_scratch(int wire_gu, int wire_down, const float* x, const float* h, const void* down, int topk, int pairs, int hidden, int ffn);

// Groups the router's choices by expert (moe_mmq.hip): counts [experts] (nullable), bounds [experts + 1], slots and src_rows [n].
// With `rows` the launch also quantizes `count` rows of k values, k a multiple of 32: to Q8_1 rows of k / 32 blocks where q81 is set,
// else to token operands (k a multiple of 256), the bytes of lk_quantize_q8_1 and lk_operands_quantize.
struct LkMoeRows {
    const float* x;
    int64_t count;
    int k;
    void* q81;
    LkTokenOperands operands;
};
int lk_moe_route(const int32_t* choices, int n, int topk, int experts, int32_t* counts, int32_t* bounds, int32_t* slots,
                 int32_t* src_rows, const LkMoeRows* rows, hipStream_t s);
// silu(gu[:, :width]) * gu[:, width:] of every row into the tile kernels' workspace (mmq.hip): the activation
// and the quantizer in one pass, same bytes as the two one after the other.
int lk_mmq_quantize_gated(const float* gu, void* y, int64_t rows, int width, hipStream_t s);
