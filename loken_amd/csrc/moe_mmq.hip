// The small steps around the expert-batched tiled matmul of a MoE prefill: where each expert's
// run of sorted rows starts (plan / route), the gated activation between the two matmuls, and
// the weighted fold of a token's routed rows. Same entry points and arguments as loken's
// cuda/moe/moe_mmq.cu:180-218 (declared at src/inference/moe_cuda/mmq_experts.rs:42-56).
//
// Differences by design:
//   * route places rows in a stable order (ascending pair index inside an expert) by ranking
//     instead of atomics, so a launch is reproducible run to run, and is one launch instead of three;
//   * SiLU uses the accurate expf, as the host path does (src/inference/moe_cuda_cpu/mod.rs:598).
#include "mmq_operands.h"
#include "moe_block.h"

namespace {

constexpr int THREADS = 256;
constexpr int ROW_WAVES = THREADS / 64;   // the row-wise kernels give every wave a row

// A sorted routing -> where each expert's run starts. Entry i looks at the experts on both sides
// of position i (the one before position 0 counts as -1, the one at position n as n_experts) and
// writes i into bounds[e] for every e in (before, at]: exactly the experts whose first row, or
// whose empty run, sits at i. Every bounds entry is written once and nothing is searched.
__global__ __launch_bounds__(THREADS) void plan_kernel(const int32_t* __restrict__ experts,
                                                       const int32_t* __restrict__ slots, int n, int topk,
                                                       int n_experts, int32_t* __restrict__ bounds,
                                                       int32_t* __restrict__ slots_out, int32_t* __restrict__ src_rows) {
    const int i = blockIdx.x * THREADS + threadIdx.x;
    if (i > n) return;
    const int before = i > 0 ? min(max(experts[i - 1], -1), n_experts) : -1;
    const int at = i < n ? min(max(experts[i], -1), n_experts) : n_experts;
    for (int e = before + 1; e <= at; ++e) bounds[e] = i;
    if (i < n) {
        const int slot = slots[i];
        slots_out[i] = slot;
        src_rows[i] = slot / topk;
    }
}

// The router's choices grouped by expert, in one launch. One workgroup per expert e: a thread takes a run
// of consecutive pairs and counts those that chose e and those that chose an expert before it; a block-wide
// scan turns the first into ranks (pairs keep their order inside an expert), the sum of the second is where
// e's rows start. Every workgroup reads all the choices (at most some tens of KB, from the caches), which is
// what makes the counting, the scan over experts and the placing of rows independent of one another: as three
// launches, the middle one a single thread walking the experts, they took 17 us at 2048 pairs and 30 at 8888
// over 128 experts.
// A choice that names no expert (negative, or n_experts and more: what a router leaves for a token whose logits
// are not numbers) counts as expert n_experts, whose workgroup puts those pairs behind all others. So `slots` is
// always a permutation and every entry of `src_rows` a token: quantizers walk all n of them.
// ROWS: the workgroups after those of the experts quantize the tokens that the block's first product reads, four to a thread, as
// operands of the f16 tiles or as Q8_1 rows: neither waits for the other, and a launch less (2048 pairs over 256 tokens of 2048: 4.9 and
// 4.9 us one after the other, 4.7 together; 8888 over 1111 5.1 + 5.3, 7.0).
constexpr int ROUTE_THREADS = 1024;
enum class Rows { NONE, OPERANDS, Q8_1 };
template <Rows ROWS>
__global__ __launch_bounds__(ROUTE_THREADS) void route_kernel(const int32_t* __restrict__ choices, int n, int topk, int run,
                                                              int n_experts, int32_t* __restrict__ counts,
                                                              int32_t* __restrict__ bounds, int32_t* __restrict__ slots,
                                                              int32_t* __restrict__ src_rows, LkMoeRows rows) {
    constexpr int W = ROUTE_THREADS / 64;
    if (ROWS != Rows::NONE && blockIdx.x > (unsigned)n_experts) {
        const uint32_t quads = rows.k / 4;
        const uint64_t start = (uint64_t)(blockIdx.x - n_experts - 1) * ROUTE_THREADS;   // (uniform: the long division is the scalar unit's)
        const uint32_t at = (uint32_t)(start % quads) + threadIdx.x;
        const int64_t row = (int64_t)(start / quads) + at / quads;
        if (row >= rows.count) return;   // (whole groups of eight: k is a multiple of 32)
        const int i0 = 4 * (int)(at % quads);
        const float* from = rows.x + row * rows.k + i0;
        const float4 v = ((uintptr_t)from & 15) == 0 ? *(const float4*)from : make_float4(from[0], from[1], from[2], from[3]);
        if (ROWS == Rows::OPERANDS) {
            const int64_t block = (int64_t)(i0 / 256) * rows.operands.rows + row;
            operand_quad(v, rows.operands.codes + block * LK_OPERAND_CODES, rows.operands.tabs + block * LK_OPERAND_TAB, (i0 / 32) & 7, (i0 / 4) & 7);
        } else {
            lk_store_q8_1_block(v, (i0 / 4) & 7, (uint32_t*)rows.q81 + (row * (rows.k / 32) + i0 / 32) * 9);
        }
        return;
    }
    __shared__ int wave_own[W], wave_less[W];
    const int e = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // `run` is a multiple of four: whole 16-byte pieces but for the last thread with pairs
    const int first = threadIdx.x * run, end = min(first + run, n);
    const bool vec = ((uintptr_t)choices & 15) == 0;
    auto expert_of = [&](int c) { return (int)min((unsigned)c, (unsigned)n_experts); };
    int own = 0, less = 0;
    auto look = [&](int c) {
        own += expert_of(c) == e;
        less += expert_of(c) < e;
    };
    int i = first;
    if (vec)
        for (; i + 4 <= end; i += 4) {
            const int4 c = *(const int4*)(choices + i);
            look(c.x); look(c.y); look(c.z); look(c.w);
        }
    for (; i < end; ++i) look(choices[i]);
    int upto = own;   // inclusive scan over the wave
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(upto, o);
        if (lane >= o) upto += t;
    }
    less = wave_sum_i32(less);
    if (lane == 63) { wave_own[wave] = upto; wave_less[wave] = less; }
    __syncthreads();
    int base = 0, before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        base += wave_less[w];
        total += wave_own[w];
        before += w < wave ? wave_own[w] : 0;
    }
    if (threadIdx.x == 0) {
        bounds[e] = base;   // bounds[n_experts]: the rows that have an expert
        if (counts && e < n_experts) counts[e] = total;
    }
    int row = base + before + upto - own;
    if (own == 0) return;
    auto place = [&](int c, int at) {
        if (expert_of(c) != e) return;
        slots[row] = at;
        src_rows[row] = at / topk;
        ++row;
    };
    i = first;
    if (vec)
        for (; i + 4 <= end; i += 4) {
            const int4 c = *(const int4*)(choices + i);
            place(c.x, i); place(c.y, i + 1); place(c.z, i + 2); place(c.w, i + 3);
        }
    for (; i < end; ++i) place(choices[i], i);
}

// The gated activations between the two expert matmuls. A wave takes one row of gu = [gate | up]
// and walks it in 16-byte pieces (both halves of a row are 16-byte aligned when width is a
// multiple of 4 and the buffers are; otherwise the wave falls back to single floats), so no
// element pays a division and a row's expert is found once, by the whole wave at a time.
struct GuRow {
    const float* gate;
    const float* up;
    float* out;
    bool vec;
};
static __device__ __forceinline__ GuRow gu_row(const float* gu, float* out, int64_t row, int width) {
    const float* g = gu + row * 2 * (int64_t)width;
    float* o = out + row * (int64_t)width;
    return GuRow{g, g + width, o, width % 4 == 0 && (((uintptr_t)g | (uintptr_t)o) & 15) == 0};
}
template <class F>
static __device__ __forceinline__ void for_row(const GuRow& r, int width, int lane, F&& f) {
    if (r.vec) {
        for (int c = 4 * lane; c < width; c += 256) {
            const float4 g = *(const float4*)(r.gate + c), u = *(const float4*)(r.up + c);
            *(float4*)(r.out + c) = make_float4(f(g.x, u.x, c), f(g.y, u.y, c + 1), f(g.z, u.z, c + 2), f(g.w, u.w, c + 3));
        }
    } else {
        for (int c = lane; c < width; c += 64) r.out[c] = f(r.gate[c], r.up[c], c);
    }
}

__global__ __launch_bounds__(THREADS) void silu_mul_kernel(const float* __restrict__ gu, float* __restrict__ out,
                                                           int64_t rows, int width) {
    const int64_t row = (int64_t)blockIdx.x * ROW_WAVES + (threadIdx.x >> 6);
    if (row >= rows) return;
    for_row(gu_row(gu, out, row, width), width, threadIdx.x & 63,
            [](float g, float u, int) { return g / (1.0f + expf(-g)) * u; });
}

// x = min(g + gb, limit), u' = clamp(u + ub, -limit, limit), out = x * sigmoid(alpha x) * (1 + u').
// The row's expert is the last one whose run starts at or before the row: the wave counts the
// starts that do, 64 at a time.
__global__ __launch_bounds__(THREADS) void swiglu_oai_kernel(const float* __restrict__ gu, float* __restrict__ out,
                                                             int64_t rows, int width, const int32_t* __restrict__ bounds,
                                                             int n_experts, const float* __restrict__ gate_bias,
                                                             const float* __restrict__ up_bias, float alpha, float limit) {
    const int64_t row = (int64_t)blockIdx.x * ROW_WAVES + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int lane = threadIdx.x & 63;
    const float* gb = nullptr;
    const float* ub = nullptr;
    if (gate_bias != nullptr || up_bias != nullptr) {
        int started = 0;
        for (int e0 = 0; e0 < n_experts; e0 += 64)
            started += __popcll(__ballot(e0 + lane < n_experts && bounds[e0 + lane] <= row));
        const int64_t e = started > 0 ? started - 1 : 0;
        if (gate_bias != nullptr) gb = gate_bias + e * width;
        if (up_bias != nullptr) ub = up_bias + e * width;
    }
    for_row(gu_row(gu, out, row, width), width, lane, [=](float g, float u, int c) {
        if (gb) g += gb[c];
        if (ub) u += ub[c];
        const float x = fminf(g, limit);
        const float clamped = fminf(fmaxf(u, -limit), limit);
        return (x * (1.0f / (1.0f + expf(-alpha * x)))) * (1.0f + clamped);
    });
}

// out[t, c] += (`write`: =) sum over k ascending of weights[p] * (pairs[p, c] + down_bias[choices[p], c]),
// p = t * topk + k, over the pairs whose choice names an expert (all of them without `choices`): the rows of
// the others were written by nobody. A workgroup column of the grid is one token; a thread owns four columns
// and keeps four routed rows' loads in flight, adding them in k order.
constexpr int FOLD_AHEAD = 4;
template <bool VEC>
__global__ __launch_bounds__(THREADS) void fold_kernel(const float* __restrict__ pairs, const float* __restrict__ weights,
                                                       const int32_t* __restrict__ choices, int n_experts,
                                                       const float* __restrict__ down_bias, float* __restrict__ out,
                                                       int topk, int cols, int write) {
    constexpr int W = VEC ? 4 : 1;
    const int c = (blockIdx.x * THREADS + threadIdx.x) * W;
    if (c >= cols) return;
    const int64_t t = blockIdx.y, p0 = t * topk;
    float* o = out + t * cols + c;
    float acc[W];
    if (write) {
#pragma unroll
        for (int e = 0; e < W; ++e) acc[e] = 0.f;
    } else if (VEC) {
        const float4 v = *(const float4*)o;
        acc[0] = v.x; acc[W > 1 ? 1 : 0] = v.y; acc[W > 2 ? 2 : 0] = v.z; acc[W > 3 ? 3 : 0] = v.w;
    } else {
        acc[0] = *o;
    }
    auto row_at = [&](const float* base, int64_t r, float (&v)[W]) {
        const float* src = base + r * cols + c;
        if (VEC) {
            const float4 x = *(const float4*)src;
            v[0] = x.x; v[W > 1 ? 1 : 0] = x.y; v[W > 2 ? 2 : 0] = x.z; v[W > 3 ? 3 : 0] = x.w;
        } else {
            v[0] = *src;
        }
    };
    for (int k0 = 0; k0 < topk; k0 += FOLD_AHEAD) {
        float v[FOLD_AHEAD][W], b[FOLD_AHEAD][W], w[FOLD_AHEAD];
        bool routed[FOLD_AHEAD];
#pragma unroll
        for (int j = 0; j < FOLD_AHEAD; ++j) {
            const int64_t p = p0 + min(k0 + j, topk - 1);   // past the end: a repeat, dropped below
            row_at(pairs, p, v[j]);
            w[j] = weights[p];
            const int e = choices != nullptr ? choices[p] : 0;
            routed[j] = choices == nullptr || (unsigned)e < (unsigned)n_experts;
            if (down_bias != nullptr && routed[j]) row_at(down_bias, e, b[j]);
        }
#pragma unroll
        for (int j = 0; j < FOLD_AHEAD; ++j) {
            if (k0 + j >= topk) break;
            if (!routed[j]) continue;
#pragma unroll
            for (int e = 0; e < W; ++e) acc[e] += w[j] * (down_bias != nullptr ? v[j][e] + b[j][e] : v[j][e]);
        }
    }
    if (VEC) *(float4*)o = make_float4(acc[0], acc[W > 1 ? 1 : 0], acc[W > 2 ? 2 : 0], acc[W > 3 ? 3 : 0]);
    else *o = acc[0];
}

}  // namespace

static inline unsigned row_groups(int64_t rows) { return (unsigned)((rows + ROW_WAVES - 1) / ROW_WAVES); }

extern "C" void loken_moe_mmq_plan(const int32_t* experts, const int32_t* slots, int n, int topk, int n_experts,
                                   int32_t* bounds, int32_t* slots_out, int32_t* src_rows, void* stream) {
    if (n < 0 || n_experts < 0 || topk <= 0) return;
    // positions 0 .. n inclusive: the one past the end closes the last runs
    hipLaunchKernelGGL(plan_kernel, dim3((unsigned)(n / THREADS + 1)), dim3(THREADS), 0, (hipStream_t)stream, experts,
                       slots, n, topk, n_experts, bounds, slots_out, src_rows);
    (void)hipGetLastError();
}

int lk_moe_route(const int32_t* choices, int n, int topk, int experts, int32_t* counts, int32_t* bounds, int32_t* slots,
                 int32_t* src_rows, const LkMoeRows* rows, hipStream_t s) {
    if (experts <= 0 || n < 0 || topk <= 0 || (rows && (rows->k <= 0 || rows->k % 32 != 0))) return LK_ERR_ARG;
    const int run = ((n + ROUTE_THREADS - 1) / ROUTE_THREADS + 3) / 4 * 4;
    const int64_t quantizers = rows ? (rows->count * (rows->k / 4) + ROUTE_THREADS - 1) / ROUTE_THREADS : 0;
    if (quantizers > INT32_MAX / 2) return LK_ERR_ARG;
    auto kernel = !rows ? route_kernel<Rows::NONE> : rows->q81 ? route_kernel<Rows::Q8_1> : route_kernel<Rows::OPERANDS>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(experts + 1 + quantizers)), dim3(ROUTE_THREADS), 0, s, choices, n, topk, run, experts, counts, bounds,
                       slots, src_rows, rows ? *rows : LkMoeRows{});
    return lk_launch_status();
}

extern "C" void loken_moe_mmq_route(const int32_t* choices, int n, int topk, int n_experts, int32_t* counts,
                                    int32_t* bounds, int32_t* slots, int32_t* src_rows, void* stream) {
    (void)lk_moe_route(choices, n, topk, n_experts, counts, bounds, slots, src_rows, nullptr, (hipStream_t)stream);
}

extern "C" void loken_moe_mmq_silu_mul(const float* gu, float* out, int64_t rows, int width, void* stream) {
    if (rows <= 0 || width <= 0) return;
    hipLaunchKernelGGL(silu_mul_kernel, dim3(row_groups(rows)), dim3(THREADS), 0, (hipStream_t)stream, gu, out, rows, width);
    (void)hipGetLastError();
}

extern "C" void loken_moe_mmq_swiglu_oai(const float* gu, float* out, int64_t rows, int width, const int32_t* bounds,
                                         int n_experts, const float* gate_bias, const float* up_bias, float alpha,
                                         float limit, void* stream) {
    if (rows <= 0 || width <= 0) return;
    hipLaunchKernelGGL(swiglu_oai_kernel, dim3(row_groups(rows)), dim3(THREADS), 0, (hipStream_t)stream, gu, out, rows,
                       width, bounds, n_experts, gate_bias, up_bias, alpha, limit);
    (void)hipGetLastError();
}

static int launch_fold(const float* pairs, const float* weights, const int32_t* choices, int n_experts, const float* down_bias,
                       float* out, int64_t tokens, int topk, int cols, bool write, hipStream_t s) {
    if (tokens <= 0 || cols <= 0 || topk <= 0 || tokens > 65535 * (int64_t)65535) return LK_ERR_ARG;
    const bool vec = cols % 4 == 0 && (((uintptr_t)pairs | (uintptr_t)out | (uintptr_t)down_bias) & 15) == 0;
    // tokens ride the grid's second axis, 65535 at a time
    for (int64_t t0 = 0; t0 < tokens; t0 += 65535) {
        const unsigned ty = (unsigned)(tokens - t0 < 65535 ? tokens - t0 : 65535);
        const float* p = pairs + t0 * topk * cols;
        const float* w = weights + t0 * topk;
        const int32_t* ch = choices ? choices + t0 * topk : nullptr;
        float* o = out + t0 * cols;
        if (vec)
            hipLaunchKernelGGL(fold_kernel<true>, dim3((unsigned)((cols / 4 + THREADS - 1) / THREADS), ty), dim3(THREADS), 0, s, p, w,
                               ch, n_experts, down_bias, o, topk, cols, write ? 1 : 0);
        else
            hipLaunchKernelGGL(fold_kernel<false>, dim3((unsigned)((cols + THREADS - 1) / THREADS), ty), dim3(THREADS), 0, s, p, w,
                               ch, n_experts, down_bias, o, topk, cols, write ? 1 : 0);
    }
    return lk_launch_status();
}

extern "C" int lk_moe_fold(const float* pairs, const float* weights, const int32_t* choices, int n_experts, float* out, int64_t tokens,
                           int topk, int cols, int accumulate, void* stream) {
    if (tokens == 0) return LK_OK;
    if (!pairs || !weights || !out || (choices && n_experts <= 0)) return LK_ERR_ARG;
    return launch_fold(pairs, weights, choices, n_experts, nullptr, out, tokens, topk, cols, !accumulate, (hipStream_t)stream);
}

extern "C" void loken_moe_mmq_fold(const float* pairs, const float* weights, const int32_t* choices,
                                   const float* down_bias, float* out, int64_t tokens, int topk, int cols,
                                   void* stream) {
    // the count of experts is not among the arguments: a negative choice names none, nor does 0x7FFFFFFF (loken_topk_softmax)
    (void)launch_fold(pairs, weights, choices, 0x7FFFFFFF, down_bias, out, tokens, topk, cols, false, (hipStream_t)stream);
}
