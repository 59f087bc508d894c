// The expert block of a mixture layer as one call: every launch from the router's choices to the block's
// output, chosen by size as the reference's layer code chooses (src/inference/generic_transformer/
// moe_weights.rs:2118-2152; MmqRouting, src/inference/moe_cuda/mmq_experts.rs:108-736): expert-batched
// products over a grouped routing from about a routed row per expert on, a mat-vec per routed pair below.
//
// What it adds to the entry points it is made of: nothing is sorted, copied or cleared that the kernels do not
// read (pairs stay in slot order, sums are written instead of added to zeros), the activation between the two
// tiled products is quantized where it is computed, and the host does one call instead of eight to fifteen
// (a one-token block of 128 experts: 80 us with torch's sort, copies and fills around the two kernels).

#include "mmq_operands.h"
#include "mmq_problem.h"
#include "moe_block.h"
#include "stream_scratch.h"

#include <math.h>

namespace {

struct Format {
    int type, block_len, block_bytes, wire;   // wire: id of the per-pair launchers, -1: they do not take it
    int (*grouped)(const void*, const void*, int64_t, const void*, void*, const int*, const int*, int64_t, int64_t, int64_t, int64_t,
                   int64_t, int64_t, int, int64_t, int64_t, int, int, int64_t, int, void*);
};
constexpr Format FORMATS[] = {
    {LK_TYPE_Q8_0, 32, 34, 0, launch_mmq_moe_gguf_q8_0},       {LK_TYPE_Q4_K, 256, 144, 1, launch_mmq_moe_gguf_q4_k},
    {LK_TYPE_Q2_K, 256, 84, 2, launch_mmq_moe_gguf_q2_k},      {LK_TYPE_Q3_K, 256, 110, 3, launch_mmq_moe_gguf_q3_k},
    {LK_TYPE_Q5_K, 256, 176, 4, launch_mmq_moe_gguf_q5_k},     {LK_TYPE_Q6_K, 256, 210, 5, launch_mmq_moe_gguf_q6_k},
    {LK_TYPE_Q5_0, 32, 22, 6, launch_mmq_moe_gguf_q5_0},       {LK_TYPE_MXFP4, 32, 17, 7, launch_mmq_moe_gguf_mxfp4},
    {LK_TYPE_Q5_1, 32, 24, 8, launch_mmq_moe_gguf_q5_1},       {LK_TYPE_IQ4_NL, 32, 18, 9, launch_mmq_moe_gguf_iq4_nl},
    {LK_TYPE_IQ4_XS, 256, 136, 10, launch_mmq_moe_gguf_iq4_xs}, {LK_TYPE_IQ3_XXS, 256, 98, 11, launch_mmq_moe_gguf_iq3_xxs},
    {LK_TYPE_IQ3_S, 256, 110, 12, launch_mmq_moe_gguf_iq3_s},  {LK_TYPE_IQ2_S, 256, 82, 13, launch_mmq_moe_gguf_iq2_s},
    {LK_TYPE_Q2_0, 64, 18, 14, launch_mmq_moe_gguf_q2_0},      {LK_TYPE_IQ2_XXS, 256, 66, 15, nullptr},
    {LK_TYPE_Q4_0, 32, 18, -1, launch_mmq_moe_gguf_q4_0},      {LK_TYPE_Q4_1, 32, 20, -1, launch_mmq_moe_gguf_q4_1},
};
const Format* format_of(int type) {
    for (const Format& f : FORMATS)
        if (f.type == type) return &f;
    return nullptr;
}

int64_t stack_bytes(const Format& f, int n, int k) { return (int64_t)n * (k / f.block_len) * f.block_bytes; }   // of one expert
bool grouped_serves(const Format& f, int k) { return f.grouped && k % 256 == 0; }

size_t up256(size_t v) { return (v + 255) & ~(size_t)255; }
size_t workspace_bytes(int64_t rows, int k) { return (size_t)rows * ((k + 511) / 512 * 4) * 144 + 128 * 144; }

// The grouped block on the f16 tiles: the tokens quantized once, as operands (not once per routed pair), gathered by the gate +
// up launch, which leaves silu(gate) * up as the operands of the down launch. 128 experts of 2048 -> 768 -> 2048, top-8, 1111
// tokens, Q6_K down: 275 us, where records per pair, f32 products, a gated quantizer and tiles of 64 took 412.
int block_on_tiles(const Format& fg, const Format& fd, const float* x, const void* gate, const void* up, const void* down,
                   const int32_t* choices, const float* topk_weights, float* out, int tokens, int topk, int n_experts, int hidden, int ffn,
                   int longest, LkScratch& scratch, hipStream_t s) {
    const int rows = tokens * topk, nb = hidden / 256, nb2 = ffn / 256;
    size_t at = 0;
    auto take = [&](size_t bytes) { const size_t p = at; at += up256(bytes); return p; };
    const size_t bounds_at = take((size_t)(n_experts + 1) * 4), slots_at = take((size_t)rows * 4), src_at = take((size_t)rows * 4);
    const size_t x_at = take(lk_operand_bytes(tokens, nb)), h_at = take(lk_operand_bytes(rows, nb2)), pairs_at = take((size_t)rows * hidden * 4);
    uint8_t* base = (uint8_t*)scratch.get(LK_SCRATCH_BLOCK, at);
    if (!base) return LK_ERR_NOMEM;
    int32_t *bounds = (int32_t*)(base + bounds_at), *slots = (int32_t*)(base + slots_at), *src = (int32_t*)(base + src_at);
    float* pairs = (float*)(base + pairs_at);
    const LkTokenOperands tokens_in = lk_operands_at(base + x_at, tokens, nb), h = lk_operands_at(base + h_at, rows, nb2);

    const LkMoeRows quantized{x, tokens, hidden, nullptr, tokens_in};
    if (int rc = lk_moe_route(choices, rows, topk, n_experts, nullptr, bounds, slots, src, &quantized, s)) return rc;
    MmqProblem gu{(const uint8_t*)gate, nullptr, nullptr, nullptr, nb, hidden / fg.block_len, rows, 0, ffn, 0, 0};
    const MmqTileExperts first{bounds, src, (const uint8_t*)up, 0, stack_bytes(fg, ffn, hidden), longest, n_experts, &h};
    if (int rc = lk_mmq_tiles_moe(fg.type, gu, tokens_in, first, s)) return rc;
    MmqProblem dn{(const uint8_t*)down, nullptr, pairs, slots, nb2, ffn / fd.block_len, rows, hidden, hidden, 0, 0};
    const MmqTileExperts second{bounds, nullptr, nullptr, 0, stack_bytes(fd, hidden, ffn), longest, n_experts, nullptr};
    if (int rc = lk_mmq_tiles_moe(fd.type, dn, h, second, s)) return rc;
    return lk_moe_fold(pairs, topk_weights, choices, n_experts, out, tokens, topk, hidden, 0, s);
}

}  // namespace

// Routed rows from which the expert-batched launches beat a mat-vec per routed pair. The reference breaks even
// at one routed row per expert (mmq_experts.rs:72-86); here, measured on MI355X (128 experts of 2048 -> 768 -> 2048, top-8), the
// mat-vec per routed pair stays ahead of the int8 tiles up to three rows per expert, of the matrix-unit rows launch that
// Q4_K stacks take at short runs up to 1.625 (16 tokens: 51 us against 74; 24: 81 against 83; 32: 92 against 88; 48: 139 against
// 106), and of the f16 tiles up to two (Q5_K, 1.8 / 2.1 rows: 138 / 174 against 125 / 134) or two and a half (Q6_K, 2.4 / 2.9
// rows: 55 / 227 against 60 / 199), three of Q8_0 (2 / 4 rows: 226 / 399 against 257 / 266). MXFP4's mat-vec is slower (2.5 rows: 270
// against 191, 64 experts 142 against 121, 32 of 3072 -> 512 98 against 84); 8 experts, whose launches do not fill the chip, stay (54 against 70). `wtype`: the stacks' type where both have the same, else -1.
extern "C" int lk_moe_grouped_pays(int64_t rows, int n_experts, int wtype) {
    const int64_t experts = n_experts > 1 ? n_experts : 1;
    return wtype == LK_TYPE_Q4_K   ? 8 * rows >= 13 * experts
           : wtype == LK_TYPE_Q5_K ? rows >= 2 * experts
           : wtype == LK_TYPE_Q6_K || (wtype == LK_TYPE_MXFP4 && experts >= 32) ? 2 * rows >= 5 * experts
                                   : rows >= 3 * experts;
}

// The longest run of rows an expert is expected to own, every choice equally likely: mean + sqrt(2 ln experts)
// deviations of a binomial count (mmq_experts.rs:215-227).
extern "C" int lk_moe_longest_run(int tokens, int topk, int n_experts) {
    const double experts = n_experts > 1 ? n_experts : 1;
    const double p = topk / experts < 1.0 ? topk / experts : 1.0;
    const double mean = tokens * p, dev = sqrt(mean * (1.0 - p));
    const double longest = ceil(n_experts > 1 ? mean + dev * sqrt(2.0 * log(experts)) : mean);
    const double most = tokens > 1 ? tokens : 1;
    return (int)(longest < 1.0 ? 1.0 : longest > most ? most : longest);
}

// Whether a stack takes the matrix-unit rows launch (weights straight from HBM into the operand, a wave per
// 16-row tile, a pass per 8, 16 or 48 rows) rather than the tiled ones (weights expanded into LDS per 32 or 64 tokens),
// by the longest expected run. Measured on MI355X, whole Q4_K block, rows launches against tiles: 128 experts of
// 2048 -> 768 -> 2048, top-8, at 17 / 34 / 42 / 50 / 60 / 84 rows 113 / 154 / 179 / 210 / 287 / 349 us against 172 / 177 /
// 186 / 206 / 230 / 323; rows of more than eight super-blocks (32-row tiles, four waves a tile): 32 experts of
// 3072 -> 512, top-4, at 24 / 32 / 39 / 46 rows 55 / 64 / 82 / 92 against 69 / 72 / 82 / 84.
extern "C" int lk_moe_rows_launch_pays(int wtype, int k, int longest_run) {
    return wtype == LK_TYPE_Q4_K && k % 256 == 0 && longest_run <= (k <= 2048 ? 44 : 40);
}

// Whether the block goes on the f16 tiles with nothing but operands between its launches (block_on_tiles), for two stacks of
// Q4_K, Q5_K, Q6_K, Q8_0, Q4_0, IQ4_NL or MXFP4. Measured on MI355X, whole block, by the longest expected run, against the launches it replaces:
//   Q5_K always (128 experts of 2048 -> 768 at 11 / 31 / 50 rows 137 / 147 / 182 us against 167 / 186 / 216)
//   Q8_0 and Q4_0 likewise (Q8_0, 128 of 2048 -> 768, average run 4 / 16 / 64 rows: 266 / 274 / 365 us against 447 / 468 / 702, 8 of
//     2560 -> 1536 at 8 / 32 / 256 rows 75 / 77 / 204 against 104 / 126 / 356)
//   IQ4_NL and MXFP4 from 33 rows, or over fewer than 60 experts (MXFP4, 128 of 2048 -> 768, average run 16 / 32 / 64 rows: 221 / 245 / 327 us against 206 /
//     307 / 482, 64 of 1536 -> 1024 at 16 / 32 125 / 138 against 122 / 174, 8 of 2560 -> 1536 at 3 / 32 70 / 85 against 81 / 109; IQ4_NL alike)
//   Q6_K likewise (64 of 1536 -> 1024 at 9 / 26 / 50 rows 99 / 105 / 125 against 104 / 112 / 150), but for short runs over 60 experts and
//     more, whose int8 tiles of 32 tokens run two more workgroups a CU (128 of 2048 -> 768 at 11 / 22 rows 202 / 208 against 193 / 205)
//   Q4_K, whose short runs have the rows launch, from 20 rows (128 of 2048 -> 768 at 19 / 26 / 42 rows 123 / 128 / 152 against 117 / 145 / 202,
//     64 of 1536 -> 1024 at 15 / 22 / 42 rows 64 / 66 / 82 against 59 / 81 / 138); from 9 where that launch reads rows of more than
//     eight super-blocks and the tiles fill the chip (60 of 2560 -> 1280 at 7 / 9 / 17 / 26 rows 116 / 120 / 117 / 123 against 114 / 141 / 195 / 182)
//     Rows of one, five to seven or more than eight super-blocks have no wave-per-tile launch (rows16_moe.hip) and go through the 32-row tiles: gate and up of such
//     rows leave from 9 rows where down's are such too, from 14 up to 2048 values where down's are of two or three (8 of 1792 -> 512 at 19 rows 35 against 60, 8 of
//     1536 -> 1536 at 16 41 / 58, 8 of 1792 -> 1280 at 12 40 / 50, 60 of 1792 -> 512 at 19 56 / 72; past the lines 60 of 1280 -> 1024 at 14 70 / 64, 8 of
//     2816 -> 512 at 14 41 / 36, 128 of 1536 -> 512 at 13 77 / 72). Where the rows launch reads so few super-blocks that its 32-row tiles are through as soon, the
//     line is later or none: 1792 of down from 12 rows (64 of 1792 -> 1792 at 9 128 / 119), hidden 256 up to 1280 (128 of 256 -> 1792 at 12 65 / 57), longer rows
//     than 2048 from eight experts on and down's of more than one super-block (4 of 3072 -> 1536 at 9 46 / 41, 16 of 3072 -> 256 at 10 38 / 34). Over 408 drawn
//     blocks past these lines 0.80 of the time in the mean, 1.05 at most
// and with workgroups of 64 gate and up rows for a quarter of the CUs at least.
static bool block_takes_tiles(int gu, int down, int longest, int n_experts, int hidden, int ffn) {
    auto always = [](int type) { return type == LK_TYPE_Q5_K || type == LK_TYPE_Q8_0 || type == LK_TYPE_Q4_0; };
    auto of_levels = [](int type) { return type == LK_TYPE_IQ4_NL || type == LK_TYPE_MXFP4; };
    auto has_tiles = [&](int type) { return type == LK_TYPE_Q4_K || type == LK_TYPE_Q6_K || always(type) || of_levels(type); };
    if (!has_tiles(gu) || !has_tiles(down) || lk_env_flag("LK_MMQ_I8") || (int64_t)n_experts * (ffn / 64) < lk_device().cus / 4) return false;
    if (always(gu) || always(down)) return true;
    if (of_levels(gu) || of_levels(down)) return longest > 32 || n_experts < 60;
    if (gu == LK_TYPE_Q6_K && down == LK_TYPE_Q6_K) return longest > 22 || n_experts < 60;
    auto wave_a_tile = [](int k) { return k == 512 || k == 768 || k == 1024 || k == 2048; };
    if (gu == down && !wave_a_tile(hidden)) {
        if (wave_a_tile(ffn) ? longest >= 14 && hidden <= 2048 && ffn < 1024
                             : longest >= (hidden > 256 && hidden <= 2048 && ffn > 1536 ? 12 : 9) && (hidden == 256 ? ffn <= 1280 : hidden <= 2048 || (n_experts >= 8 && ffn > 256)))
            return true;
    }
    return longest >= 20 || (longest >= 9 && hidden > 2048 && 2ll * n_experts * ((ffn + 255) / 256) >= lk_device().cus);
}

// lk_moe_grouped_pays by the weights as well: the expert-batched launches take 28 to 50 us however little there is to read, a mat-vec per pair the time
// of the pairs' matrices (`bytes`, of which the L2s and the last cache hold what other pairs read). Whole block, pairs / batched, us, 8 experts unless said, at
// up to six rows each:
//   Q4_K 1.77 MB an expert, 24 pairs 19.3 / 28.4; 2.65, 26 24.6 / 31.6; 1.99, 44 27.1 / 39.6; (3.32, 48 35.0 / 32.5); Q4_K and Q6_K 2.55, 22 25.6 / 38.8; 3.44,
//   24 27.9 / 37.9; MXFP4 0.8 to 0.9 of the time under 100 MB; Q5_K under 80 MB 0.73; Q8_0 under 250 MB 0.64 to 0.75
// Only while there are few pairs: many of short rows take their own time however few their bytes (batched / pairs: 64 experts of 512 -> 256 in Q4_K, 304 pairs 22 /
// 33; 128 of 256 -> 256 in IQ3_S, 706 pairs 30 / 154; 60 of 512 -> 512 in IQ2_S, 314 39 / 127; 128 of 256 -> 256 in Q8_0, 760 34 / 74). Over drawn blocks of
// fifteen formats, 4 to 128 experts, the pairs are ahead or level (one block of 4000 drawn ones was 9 % behind) up to 40 of the K-quants Q4_K to Q6_K, 64 of Q8_0 and 20 of the others, at
// 1.4 to 2.2 times the batched speed in the mean.
// And where there is much to read the batched ones pay sooner: Q5_K from 1.25 rows past 600 MB and from 1.75 past 300 (0.83 of the time over 409 drawn blocks,
// 1.09 at most; fewer of either 0.95, up to 1.24: 32 experts of 2048 -> 1792, 40 pairs, 63.3 / 78.3), Q8_0 from 2.25 past 400 and 160 pairs (0.84 over
// 418, 1.10 at most; fewer pairs 1.03, up to 1.35: 32 of 2560 -> 1280, 72 pairs, 139 / 183).
static bool grouped_pays_over(int64_t pairs, int n_experts, int gu, int down, int line, int64_t bytes) {
    const int64_t experts = n_experts > 1 ? n_experts : 1, mb = 1000000;
    auto large_blocks = [](int type) { return type == LK_TYPE_Q4_K || type == LK_TYPE_Q5_K || type == LK_TYPE_Q6_K || type == LK_TYPE_Q8_0; };
    const int64_t few = line == LK_TYPE_Q8_0 ? 64 : large_blocks(gu) && large_blocks(down) ? 40 : 20;
    if (pairs <= 6 * experts && pairs <= few && bytes < (line == LK_TYPE_Q8_0 ? 250 : line == LK_TYPE_Q5_K ? 80 : 100) * mb) return false;
    if (line == LK_TYPE_Q5_K && ((4 * pairs >= 5 * experts && bytes > 600 * mb) || (4 * pairs >= 7 * experts && bytes > 300 * mb))) return true;
    if (line == LK_TYPE_Q8_0 && 4 * pairs >= 9 * experts && bytes > 400 * mb && pairs >= 160) return true;
    return lk_moe_grouped_pays(pairs, n_experts, line);
}

// What a batched block is made of, as lk_moe_block_path's bits.
static int batched_path(int wtype_gu, int wtype_down, int tokens, int topk, int n_experts, int hidden, int ffn) {
    const int longest = lk_moe_longest_run(tokens, topk, n_experts);
    if (block_takes_tiles(wtype_gu, wtype_down, longest, n_experts, hidden, ffn)) return LK_MOE_GROUPED | LK_MOE_TILES;
    const bool rows_down = lk_moe_rows_launch_pays(wtype_down, ffn, longest);
    const bool tiles_fill = 2ll * n_experts * ((ffn + 255) / 256) >= lk_device().cus;
    const bool rows_gu = lk_moe_rows_launch_pays(wtype_gu, hidden, longest) && (rows_down || longest <= 36) &&
                         (hidden <= 2048 || !tiles_fill || longest <= 20);
    return LK_MOE_GROUPED | (rows_gu ? LK_MOE_ROWS_GATE_UP : 0) | (rows_down ? LK_MOE_ROWS_DOWN : 0);
}

// Which launches the block is made of: LK_MOE_GROUPED (expert-batched products; else a mat-vec per routed pair),
// and in it LK_MOE_TILES (both products on the f16 tiles), or LK_MOE_ROWS_GATE_UP / LK_MOE_ROWS_DOWN
// (lk_moe_q4k_rows_grouped; else the tiled launch). The one place that decides: lk_moe_forward and a caller that issues the
// launches itself both ask here.
// Gate and up also leave the rows launch where
//   * down is tiled, past 36 rows: tiles for both keep the rows between them in the tiles' layout and the activation in
//     their quantizer
//   * their rows are long and their tiles fill the chip, past 20 rows
extern "C" int lk_moe_block_path(int wtype_gu, int wtype_down, int tokens, int topk, int n_experts, int hidden, int ffn) {
    const Format *fg = format_of(wtype_gu), *fd = format_of(wtype_down);
    if (!fg || !fd || tokens <= 0 || topk <= 0 || n_experts <= 0) return 0;
    auto has_tiles = [](int type) { return type == LK_TYPE_Q4_K || type == LK_TYPE_Q5_K || type == LK_TYPE_Q6_K; };
    const int line = wtype_gu == wtype_down ? wtype_gu : has_tiles(wtype_gu) && has_tiles(wtype_down) ? LK_TYPE_Q6_K : -1;
    const int64_t pairs = (int64_t)tokens * topk;
    // (Q4_0 and Q4_1 have no mat-vec per pair: no choice by the weights)
    const bool grouped = fg->wire < 0 || fd->wire < 0 ? lk_moe_grouped_pays(pairs, n_experts, line)
                                                      : grouped_pays_over(pairs, n_experts, wtype_gu, wtype_down, line, pairs * (2 * stack_bytes(*fg, ffn, hidden) + stack_bytes(*fd, hidden, ffn)));
    if (!grouped || !grouped_serves(*fg, hidden) || !grouped_serves(*fd, ffn)) return 0;
    return batched_path(wtype_gu, wtype_down, tokens, topk, n_experts, hidden, ffn);
}

extern "C" int lk_moe_forward(int wtype_gu, int wtype_down, const float* x, const void* gate, const void* up, const void* down,
                              const int32_t* choices, const float* topk_weights, float* out, int tokens, int topk, int n_experts,
                              int hidden, int ffn, void* stream) {
    const Format *fg = format_of(wtype_gu), *fd = format_of(wtype_down);
    if (!fg || !fd) return LK_ERR_TYPE;
    if (tokens == 0) return LK_OK;
    if (!x || !gate || !up || !down || !choices || !topk_weights || !out || tokens < 0 || topk <= 0 || n_experts <= 0 || hidden <= 0 ||
        ffn <= 0 || hidden % fg->block_len != 0 || ffn % fd->block_len != 0 || (int64_t)tokens * topk > INT32_MAX)
        return LK_ERR_ARG;
    hipStream_t s = (hipStream_t)stream;
    const int rows = tokens * topk;
    LkScratch scratch(s);

    int path = lk_moe_block_path(wtype_gu, wtype_down, tokens, topk, n_experts, hidden, ffn);
    if (!(path & LK_MOE_GROUPED)) {
        if (fg->wire < 0 || fd->wire < 0) return LK_ERR_TYPE;
        float* h = (float*)scratch.get(LK_SCRATCH_BLOCK, (size_t)rows * ffn * 4);
        // (asked for ahead only where it may be refused for good: a block of one token is bound by the host)
        const size_t more = scratch.recording() ? lk_moe_pairs_scratch(fg->wire, fd->wire, x, h, down, topk, rows, hidden, ffn) : 0;
        if (h && (more == 0 || scratch.get(LK_SCRATCH_LAUNCHER, more))) {
            if (int rc = lk_moe_pairs_gate_up(fg->wire, x, gate, up, choices, h, n_experts, topk, rows, ffn, hidden, s)) return rc;
            return lk_moe_pairs_down(fd->wire, h, down, choices, topk_weights, out, n_experts, topk, rows, hidden, ffn, s);
        }
        // Without that memory (a recorded call of which only larger ones, batched, ran before) the batched launches where these
        // serve: they work in the block's buffer alone.
        if (!grouped_serves(*fg, hidden) || !grouped_serves(*fd, ffn)) return LK_ERR_NOMEM;
        path = batched_path(wtype_gu, wtype_down, tokens, topk, n_experts, hidden, ffn);
    }

    const int longest = lk_moe_longest_run(tokens, topk, n_experts);
    const bool rows_gu = path & LK_MOE_ROWS_GATE_UP, rows_down = path & LK_MOE_ROWS_DOWN;
    if ((path & LK_MOE_TILES) &&
        lk_mmq_tiles_moe_fit(wtype_gu, gate, up, stack_bytes(*fg, ffn, hidden), ffn, hidden, tokens, true) &&
        lk_mmq_tiles_moe_fit(wtype_down, down, nullptr, stack_bytes(*fd, hidden, ffn), hidden, ffn, rows, false))
        return block_on_tiles(*fg, *fd, x, gate, up, down, choices, topk_weights, out, tokens, topk, n_experts, hidden, ffn, longest, scratch, s);
    const bool gated_later = !rows_gu && !rows_down && ffn % 32 == 0;   // the activation rides the second product's quantizer
    // the buffer's pieces
    size_t at = 0;
    auto take = [&](size_t bytes) { const size_t p = at; at += up256(bytes); return p; };
    const size_t bounds_at = take((size_t)(n_experts + 1) * 4), slots_at = take((size_t)rows * 4), src_at = take((size_t)rows * 4);
    const size_t y_at = take(rows_gu ? (size_t)tokens * (hidden / 32) * Q81_BYTES : workspace_bytes(rows, hidden));
    const size_t gu_at = take(rows_gu ? 0 : (size_t)rows * 2 * ffn * 4);
    const size_t h_at = take(gated_later ? 0 : (size_t)rows * ffn * 4);
    const size_t y2_at = take(rows_down ? (size_t)rows * (ffn / 32) * Q81_BYTES : workspace_bytes(rows, ffn));
    const size_t pairs_at = take((size_t)rows * hidden * 4);
    uint8_t* base = (uint8_t*)scratch.get(LK_SCRATCH_BLOCK, at);
    if (!base) return LK_ERR_NOMEM;
    int32_t *bounds = (int32_t*)(base + bounds_at), *slots = (int32_t*)(base + slots_at), *src = (int32_t*)(base + src_at);
    float *gu = (float*)(base + gu_at), *h = (float*)(base + h_at), *pairs = (float*)(base + pairs_at);
    uint8_t *y = base + y_at, *y2 = base + y2_at;

    auto grouped = [&](const Format& f, const void* w, const void* w2, int64_t second_at, const uint8_t* acts, float* dst, const int32_t* ids,
                       int n, int k, int stride) {
        const int64_t blocks = k / f.block_len;
        return f.grouped(w, w2, second_at, acts, dst, bounds, ids, n * blocks * f.block_bytes, k, n, rows, blocks, stride, n_experts, longest,
                         longest, 0, 0, 0, 0, stream) != 0
                   ? LK_OK
                   : LK_ERR_ARG;
    };
    auto quantize = [&](const float* from, const int32_t* gather, uint8_t* to, int k) {   // (one record layout serves every format)
        launch_mmq_quantize_q8_1_DS4(from, gather, to, LK_TYPE_F32, k, k, 0, 0, (k + 511) / 512 * 512, rows, 1, 1, stream);
    };

    const LkMoeRows quantized{x, tokens, hidden, y, {}};
    if (int rc = lk_moe_route(choices, rows, topk, n_experts, nullptr, bounds, slots, src, rows_gu ? &quantized : nullptr, s)) return rc;
    if (rows_gu) {
        if (int rc = lk_moe_q4k_rows_grouped(gate, up, 0, y, hidden / 32, bounds, src, nullptr, h, ffn, n_experts,
                                             (int64_t)ffn * (hidden / 256) * Q4K_BYTES, ffn, hidden, longest, stream)) return rc;
    } else {
        quantize(x, src, y, hidden);
        if (int rc = grouped(*fg, gate, up, ffn, y, gu, nullptr, ffn, hidden, 2 * ffn)) return rc;
        if (gated_later) {
            if (int rc = lk_mmq_quantize_gated(gu, y2, rows, ffn, s)) return rc;
        } else {
            loken_moe_mmq_silu_mul(gu, h, rows, ffn, stream);
        }
    }
    if (rows_down) {
        if (int rc = lk_quantize_q8_1(h, LK_TYPE_F32, y2, ffn, ffn, rows, stream)) return rc;
        if (int rc = lk_moe_q4k_rows_grouped(down, nullptr, 0, y2, ffn / 32, bounds, nullptr, slots, pairs, hidden, n_experts,
                                             (int64_t)hidden * (ffn / 256) * Q4K_BYTES, hidden, ffn, longest, stream)) return rc;
    } else {
        if (!gated_later) quantize(h, nullptr, y2, ffn);
        if (int rc = grouped(*fd, down, nullptr, 0, y2, pairs, slots, hidden, ffn, hidden)) return rc;
    }
    return lk_moe_fold(pairs, topk_weights, choices, n_experts, out, tokens, topk, hidden, 0, stream);
}
