// The router step in front of the expert block: softmax over a row of expert logits, the k largest
// probabilities in descending order (ties to the lower expert id), optionally renormalized to sum
// to one. Same name and arguments as the reference's launcher (loken_topk_softmax,
// cuda/moe/gate_topk.cu:405-451; semantics of topk_softmax, src/inference/moe_cuda_cpu/mod.rs:
// 2098-2113: softmax -> argsort descending -> take k -> optional renorm).
//
// One wave per row, lane l holding experts l, l + 64, ...: the maximum, the sum and each of the k
// arg-max rounds are wave reductions; rows are tiny (128 logits), so the launch is latency only.

#include "lk_common.h"
#include "stream_scratch.h"

namespace {

constexpr int MAX_PER_LANE = 8;   // up to 512 experts

static __device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, dpp_f32<0xB1>(v));
    v = fmaxf(v, dpp_f32<0x4E>(v));
    v = fmaxf(v, dpp_f32<0x141>(v));
    v = fmaxf(v, dpp_f32<0x140>(v));
    const int bits = __float_as_int(v);
    const float r0 = __int_as_float(__builtin_amdgcn_readlane(bits, 0));
    const float r1 = __int_as_float(__builtin_amdgcn_readlane(bits, 16));
    const float r2 = __int_as_float(__builtin_amdgcn_readlane(bits, 32));
    const float r3 = __int_as_float(__builtin_amdgcn_readlane(bits, 48));
    return fmaxf(fmaxf(r0, r1), fmaxf(r2, r3));
}

// Softmax over the logits a lane brings (p[i]: expert lane + 64 i, -INFINITY past n_experts) and the k largest, by
// the 64 lanes of one wave; PER = experts / 64 rounded up to a power of two. A round finds the largest
// probability through lane moves of the vector unit and scalar registers, and the lowest expert that has it by
// ballots (a permute through LDS per step of the reduction costs four times as much). Experts of a row are
// distinct; where nothing is left to choose the id is 0x7FFFFFFF and the weight not a number.
template <int PER>
static __device__ __forceinline__ void select_topk_softmax(float (&p)[PER], float* __restrict__ weights,
                                                           uint32_t* __restrict__ ids, int n_experts, int topk,
                                                           int with_norm, int lane) {
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < PER; ++i) mx = fmaxf(mx, p[i]);
    mx = wave_max(mx);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = lane + 64 * i;
        p[i] = e < n_experts ? expf(p[i] - mx) : -1.f;   // -1: never chosen, only probabilities >= 0 are
        sum += e < n_experts ? p[i] : 0.f;
    }
    sum = wave_sum(sum);
    float my_weight = 0.f;
    uint32_t my_id = 0;
    for (int j = 0; j < topk; ++j) {
        float best = p[0];
#pragma unroll
        for (int i = 1; i < PER; ++i) best = fmaxf(best, p[i]);
        best = wave_max(best);
        // Logits that are not numbers (and infinite ones, whose difference to the maximum is none) leave fewer
        // probabilities than choices: `best` is then -1 or not a number itself, and the choice names no expert.
        const float wanted = best >= 0.f ? best : NAN;   // equal to nothing
        int e = 0x7FFFFFFF;
#pragma unroll
        for (int i = PER - 1; i >= 0; --i) {
            const unsigned long long at = __ballot(p[i] == wanted);
            if (at) e = 64 * i + __ffsll((long long)at) - 1;
        }
        if (lane == j) { my_weight = best; my_id = (uint32_t)e; }
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (lane + 64 * i == e) p[i] = -1.f;
    }
    // the divisions of all choices at once, after the rounds that only depend on each other's maxima
    my_weight /= sum;
    float picked_sum = 0.f;
    if (with_norm)
        for (int j = 0; j < topk; ++j) picked_sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(my_weight), j));
    if (lane < topk) {
        weights[lane] = with_norm ? my_weight / picked_sum : my_weight;
        ids[lane] = my_id;
    }
}

static __device__ __forceinline__ void select_topk_softmax(const float* x, float* __restrict__ weights, uint32_t* __restrict__ ids,
                                                           int n_experts, int topk, int with_norm, int lane) {
    float p[MAX_PER_LANE];
#pragma unroll
    for (int i = 0; i < MAX_PER_LANE; ++i) p[i] = lane + 64 * i < n_experts ? x[lane + 64 * i] : -INFINITY;
    select_topk_softmax<MAX_PER_LANE>(p, weights, ids, n_experts, topk, with_norm, lane);
}

__global__ __launch_bounds__(64) void topk_softmax_kernel(const float* __restrict__ logits, float* __restrict__ weights,
                                                          uint32_t* __restrict__ ids, int n_experts, int topk,
                                                          int with_norm) {
    const size_t row = blockIdx.x;
    select_topk_softmax(logits + row * n_experts, weights + row * topk, ids + row * topk, n_experts, topk, with_norm,
                        threadIdx.x);
}

// ---------------------------------------------------------------------------------------------
// The gate product, softmax and top-k of every token (loken_gate_topk_softmax, cuda/moe/gate_topk.cu:253-295,
// 366-403), in two launches (a few tokens in one): the logits as an f32 product on the matrix unit, then a wave per token that adds
// the partial sums and selects. One workgroup per token (the kernel after these, still the one for rows that do
// not start on 16 bytes and for streams that record a graph before their scratch exists) reads the whole gate
// for each token through one CU: 28 us at one token of 2048 x 128, where the bytes take a microsecond, and 69 us
// at 1111.
//
// The logits: v_mfma_f32_{16x16x4,32x32x2}_f32 (f32 operands and sums), a tile of tokens x experts per
// workgroup. A lane takes four consecutive values of its token's row and of its expert's row at once, one component per
// instruction (any order of K serves as long as both operands agree). The four waves of a workgroup and the
// grid's z axis split K until the launch covers the chip; partial sums meet in LDS and in part[z].
// ---------------------------------------------------------------------------------------------
constexpr int LOGIT_WAVES = 4;
constexpr int LOGIT_SPREAD = 768;   // workgroups a launch aims at: loads wait a microsecond each, so three per CU

// A wave's share of the product of a 16 x 16 tile, rows straight from memory: lane (group, column), register v: token 4 grp + v,
// expert e0 + column.
static __device__ __forceinline__ v4f logits16_share(const float* __restrict__ x_in, const float* __restrict__ gate_w, int hidden, int n_rows,
                                                     int n_experts, int e0, int share, int shares) {
    constexpr int M = 16, UNIT = 16, AHEAD = 4;   // UNIT: values of K a load of the wave covers; AHEAD: loads per operand in flight
    const int lane = threadIdx.x & 63, at = lane % M, grp = lane / M;
    const int units = (hidden + UNIT - 1) / UNIT;
    const int u0 = (int)((int64_t)units * share / shares), u1 = (int)((int64_t)units * (share + 1) / shares);
    const float* xr = x_in + (size_t)min(at, n_rows - 1) * hidden;
    const float* wr = gate_w + (size_t)min(e0 + at, n_experts - 1) * hidden;
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    for (int u = u0; u < u1; u += AHEAD) {
        float4 a[AHEAD], b[AHEAD];
        bool live[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
            if (u + i < u1) {   // (the same for the whole wave: nothing is loaded past its share)
                const int k = (u + i) * UNIT + 4 * grp;
                live[i] = k < hidden;   // past the row's end, in its last unit: a repeat of the row's start, multiplied by zero
                a[i] = *(const float4*)(xr + (live[i] ? k : 0));
                b[i] = *(const float4*)(wr + (live[i] ? k : 0));
            }
        __builtin_amdgcn_sched_barrier(0);   // all of them out before the first is waited for
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
            if (u + i < u1) {
                if (!live[i]) a[i] = b[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].x, b[i].x, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].y, b[i].y, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].z, b[i].z, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i].w, b[i].w, acc, 0, 0, 0);
            }
    }
    return acc;
}

// Up to sixteen tokens.
__global__ __launch_bounds__(64 * LOGIT_WAVES) void gate_logits16_kernel(const float* __restrict__ x_in, const float* __restrict__ gate_w,
                                                                         float* __restrict__ part, int hidden, int n_rows,
                                                                         int n_experts) {
    constexpr int M = 16;
    __shared__ __align__(16) float meet[LOGIT_WAVES - 1][M * M];
    const int lane = threadIdx.x & 63, at = lane % M, grp = lane / M;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int e0 = blockIdx.y * M;
    v4f acc = logits16_share(x_in, gate_w, hidden, n_rows, n_experts, e0, blockIdx.z * LOGIT_WAVES + wave, gridDim.z * LOGIT_WAVES);
    if (wave > 0) *(v4f*)(meet[wave - 1] + lane * 4) = acc;
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 0; w < LOGIT_WAVES - 1; ++w) acc += *(const v4f*)(meet[w] + lane * 4);
#pragma unroll
    for (int v = 0; v < 4; ++v)
        if (4 * grp + v < n_rows && e0 + at < n_experts) part[((size_t)blockIdx.z * n_rows + 4 * grp + v) * n_experts + e0 + at] = acc[v];
}

// A few tokens: 16 x 16 tiles, rows straight from memory, the choice in the same launch. A workgroup is twice the four waves
// that share a partial sum; the last one of the launch to arrive (its stream's counter, which wraps to zero with it)
// reads all partial sums and gives a wave to each token. Its tail (the stores' way to memory, the counter, the partial sums, the choice:
// 3 us) takes what the second launch takes, so what it saves is the host's time for that launch, which bounds a call of so little work: one to four
// tokens called one by one 11.0 -> 8.6 us. Replayed in a graph, one launch against the two as they are now (128 experts of 2048, 1 / 4 / 8 / 16 tokens):
// 6.1 / 6.2 / 7.1 / 10.4 us against 5.4 / 5.7 / 5.9 / 6.0; 128 of 3072 6.4 / 6.6 / 7.6 / 10.9 against 5.6 / 5.9 / 6.2 / 6.3. So up to
// CHOICE_TOKENS tokens take it, outside a recording. Sums in the order of the two launches, hence the same bits.
__device__ uint32_t g_arrived[LK_SCRATCH_TICKETS];
constexpr int CHOICE_GROUPS = 2, CHOICE_THREADS = 64 * LOGIT_WAVES * CHOICE_GROUPS, CHOICE_TOKENS = 4;

// FRESH: partial sums of other XCDs' workgroups of this launch, read past this XCD's cache.
template <int PER, bool FRESH>
static __device__ __forceinline__ void sum_partials(float (&p)[PER], const float* part, int splits, int64_t row, int n_rows, int n_experts, int lane) {
    // partial sums in flight (one after the other they took 10 us of a one-token call, eight at a time a microsecond more than sixteen)
    constexpr int AHEAD = PER <= 2 ? 16 : 8;
    const int64_t step = (int64_t)n_rows * n_experts;
    const float* from = part + row * n_experts;   // uniform: a load is a scalar base and the lane's offset
    int at[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        at[i] = min(lane + 64 * i, n_experts - 1);
        p[i] = 0.f;
    }
    for (int z0 = 0; z0 < splits; z0 += AHEAD) {
        float v[AHEAD][PER];
#pragma unroll
        for (int z = 0; z < AHEAD; ++z) {
#pragma unroll
            for (int i = 0; i < PER; ++i) v[z][i] = FRESH ? __hip_atomic_load(from + at[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : from[at[i]];
            if (z0 + z + 1 < splits) from += step;
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int z = 0; z < AHEAD; ++z)
#pragma unroll
            for (int i = 0; i < PER; ++i) p[i] += z0 + z < splits ? v[z][i] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < PER; ++i)
        if (lane + 64 * i >= n_experts) p[i] = -INFINITY;
}

template <int PER>
__global__ __launch_bounds__(CHOICE_THREADS) void gate_topk16_kernel(const float* __restrict__ x_in, const float* __restrict__ gate_w,
                                                                     float* part, float* __restrict__ weights, uint32_t* __restrict__ ids,
                                                                     int hidden, int n_rows, int n_experts, int splits, int topk, int with_norm,
                                                                     int ticket) {
    constexpr int M = 16;
    __shared__ __align__(16) float meet[CHOICE_THREADS / 64][M * M];
    __shared__ int is_last;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int e0 = blockIdx.x * M, z0 = blockIdx.y * CHOICE_GROUPS, share = z0 * LOGIT_WAVES + wave;
    if (share < splits * LOGIT_WAVES)
        *(v4f*)(meet[wave] + lane * 4) = logits16_share(x_in, gate_w, hidden, n_rows, n_experts, e0, share, splits * LOGIT_WAVES);
    __syncthreads();
    {   // register v of lane (group, column): token 4 grp + v, expert `at` of the tile
        const int g = threadIdx.x / (M * M), i = threadIdx.x % (M * M), t = 4 * (i / 64) + i % 4, e = e0 + i / 4 % M, z = z0 + g;
        if (z < splits && t < n_rows && e < n_experts) {
            float sum = meet[LOGIT_WAVES * g][i];
#pragma unroll
            for (int w = 1; w < LOGIT_WAVES; ++w) sum += meet[LOGIT_WAVES * g + w][i];
            __hip_atomic_store(part + ((size_t)z * n_rows + t) * n_experts + e, sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    // Stores of agent scope go through the XCD's cache to where every XCD reads; once each wave has waited for its own, one thread
    // counts the workgroup in.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t last = gridDim.x * gridDim.y - 1;
        is_last = atomicInc(&g_arrived[ticket], last) == last;
    }
    __syncthreads();
    if (!is_last) return;
    if (wave >= n_rows) return;
    float p[PER];
    sum_partials<PER, true>(p, part, splits, wave, n_rows, n_experts, lane);
    select_topk_softmax<PER>(p, weights + (size_t)wave * topk, ids + (size_t)wave * topk, n_experts, topk, with_norm, lane);
}

// More tokens: 32 x 32 tiles. Taken from memory in operand order (a lane per row) a load touches 32 cache lines
// and the launch is bound by the address unit (1111 tokens: 22 us); here a wave copies 32 rows x 128 bytes of
// each operand into its own piece of LDS, eight lanes to a row, and reads the operands from there (row pitch 144 bytes:
// no bank conflicts). The next copy is in flight while this one is multiplied; waves share nothing until
// their sums meet.
__global__ __launch_bounds__(64 * LOGIT_WAVES) void gate_logits32_kernel(const float* __restrict__ x_in, const float* __restrict__ gate_w,
                                                                         float* __restrict__ part, int hidden, int n_rows,
                                                                         int n_experts) {
    constexpr int M = 32, UNIT = 32, PITCH = UNIT + 4, ROUNDS = M * UNIT / 4 / 64;
    __shared__ __align__(16) float stage[LOGIT_WAVES][2][M * PITCH];
    const int lane = threadIdx.x & 63, at = lane % M, grp = lane / M;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t0 = blockIdx.x * M, e0 = blockIdx.y * M;
    const int units = (hidden + UNIT - 1) / UNIT, shares = gridDim.z * LOGIT_WAVES, share = blockIdx.z * LOGIT_WAVES + wave;
    const int u0 = (int)((int64_t)units * share / shares), u1 = (int)((int64_t)units * (share + 1) / shares);
    const int row8 = lane >> 3, k4 = 4 * (lane & 7);
    float *sx = stage[wave][0], *sw = stage[wave][1];
    float4 xv[ROUNDS], wv[ROUNDS];
    auto fetch = [&](int u) {
        const int k = u * UNIT + k4;
        const bool live = k < hidden;   // in the row's last unit; past it: a repeat of the row's start, as zeros
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            xv[r] = *(const float4*)(x_in + (size_t)min(t0 + 8 * r + row8, n_rows - 1) * hidden + (live ? k : 0));
            wv[r] = *(const float4*)(gate_w + (size_t)min(e0 + 8 * r + row8, n_experts - 1) * hidden + (live ? k : 0));
            if (!live) xv[r] = wv[r] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    v16f acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
    if (u0 < u1) fetch(u0);
    for (int u = u0; u < u1; ++u) {
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            *(float4*)(sx + (8 * r + row8) * PITCH + k4) = xv[r];
            *(float4*)(sw + (8 * r + row8) * PITCH + k4) = wv[r];
        }
        __builtin_amdgcn_wave_barrier();   // a wave's LDS operations are served in order: the reads below see the writes
        if (u + 1 < u1) fetch(u + 1);
#pragma unroll
        for (int i = 0; i < UNIT / 8; ++i) {
            const float4 a = *(const float4*)(sx + at * PITCH + 8 * i + 4 * grp), b = *(const float4*)(sw + at * PITCH + 8 * i + 4 * grp);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b.z, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b.w, acc, 0, 0, 0);
        }
        __builtin_amdgcn_wave_barrier();
    }
    float* meet = &stage[0][0][0] + wave * M * M;
    __syncthreads();   // the pieces of LDS are read for the last time
    if (wave > 0) {
#pragma unroll
        for (int v = 0; v < 16; ++v) meet[v * 64 + lane] = acc[v];
    }
    __syncthreads();
    if (wave > 0) return;
    // lane (group, column), register v: token 8 (v / 4) + 4 grp + v % 4, expert `at` of the tile
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        float sum = acc[v];
#pragma unroll
        for (int w = 1; w < LOGIT_WAVES; ++w) sum += meet[w * M * M + v * 64 + lane];
        const int t = t0 + 8 * (v / 4) + 4 * grp + v % 4, e = e0 + at;
        if (t < n_rows && e < n_experts) part[((size_t)blockIdx.z * n_rows + t) * n_experts + e] = sum;
    }
}

template <int PER>
__global__ __launch_bounds__(256) void gate_select_kernel(const float* __restrict__ part, int splits, float* __restrict__ weights,
                                                          uint32_t* __restrict__ ids, int n_rows, int n_experts, int topk,
                                                          int with_norm) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= n_rows) return;
    float p[PER];
    sum_partials<PER, false>(p, part, splits, row, n_rows, n_experts, lane);
    select_topk_softmax<PER>(p, weights + row * topk, ids + row * topk, n_experts, topk, with_norm, lane);
}

// The same for one token per workgroup of 16 waves: a wave takes experts w, w + 16, ... and its lanes walk the
// row together (consecutive lanes read consecutive 16-byte pieces); the selection is run by wave 0 over the
// logits left in LDS.
constexpr int GATE_WAVES = 16;

__global__ __launch_bounds__(64 * GATE_WAVES) void gate_topk_softmax_kernel(const float* __restrict__ x_in,
                                                                            const float* __restrict__ gate_w,
                                                                            float* __restrict__ weights,
                                                                            uint32_t* __restrict__ ids, int hidden,
                                                                            int n_experts, int topk, int with_norm) {
    extern __shared__ __align__(16) float gate_lds[];   // [hidden] the token, then [n_experts] logits
    float* xs = gate_lds;
    float* logits = gate_lds + ((hidden + 3) & ~3);
    const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const float* x = x_in + (size_t)row * hidden;
    const bool vec = (hidden & 3) == 0 && (((uintptr_t)x_in | (uintptr_t)gate_w) & 15) == 0;
    if (vec) {
        for (int i = tid; i < hidden / 4; i += 64 * GATE_WAVES) ((float4*)xs)[i] = ((const float4*)x)[i];
    } else {
        for (int i = tid; i < hidden; i += 64 * GATE_WAVES) xs[i] = x[i];
    }
    __syncthreads();
    for (int e = wave; e < n_experts; e += GATE_WAVES) {
        const float* w = gate_w + (size_t)e * hidden;
        float acc = 0.f;
        if (vec) {
            for (int i = lane; i < hidden / 4; i += 64) {
                const float4 a = ((const float4*)w)[i], b = ((const float4*)xs)[i];
                acc += a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w;
            }
        } else {
            for (int i = lane; i < hidden; i += 64) acc += w[i] * xs[i];
        }
        acc = wave_sum(acc);
        if (lane == 0) logits[e] = acc;
    }
    __syncthreads();
    if (wave == 0) select_topk_softmax(logits, weights + (size_t)row * topk, ids + (size_t)row * topk, n_experts, topk, with_norm, lane);
}

// A sigmoid router (loken_topk_sigmoid_post, cuda/moe/gate_topk.cu:140-200, 329-364, 479-512):
// every expert's probability stands alone, 1 / (1 + exp(-logit)); the k experts are chosen on the
// probability plus a per-expert bias (ties to the lower id) while the weight handed back is the
// unbiased probability, divided by max(sum of the k, 2^-14) when with_norm, then times `scale`.
__global__ __launch_bounds__(64) void topk_sigmoid_post_kernel(const float* __restrict__ logits,
                                                               const float* __restrict__ bias, float* __restrict__ weights,
                                                               uint32_t* __restrict__ ids, int n_experts, int topk,
                                                               int with_norm, float scale) {
    const int row = blockIdx.x, lane = threadIdx.x;
    const float* x = logits + (size_t)row * n_experts;
    float prob[MAX_PER_LANE], sel[MAX_PER_LANE];
#pragma unroll
    for (int i = 0; i < MAX_PER_LANE; ++i) {
        const int e = lane + 64 * i;
        prob[i] = e < n_experts ? 1.0f / (1.0f + expf(-x[e])) : 0.f;
        sel[i] = e < n_experts ? prob[i] + (bias ? bias[e] : 0.f) : -INFINITY;
    }
    float picked_sum = 0.f, my_weight = 0.f;
    uint32_t my_id = 0;
    for (int j = 0; j < topk; ++j) {
        float best = -INFINITY, best_p = 0.f;
        int best_e = 0x7FFFFFFF;
#pragma unroll
        for (int i = 0; i < MAX_PER_LANE; ++i)
            if (sel[i] > best) { best = sel[i]; best_p = prob[i]; best_e = lane + 64 * i; }
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const float ob = __shfl_xor(best, o), op = __shfl_xor(best_p, o);
            const int oe = __shfl_xor(best_e, o);
            if (ob > best || (ob == best && oe < best_e)) { best = ob; best_p = op; best_e = oe; }
        }
        picked_sum += best_p;
        if (lane == j) { my_weight = best_p; my_id = (uint32_t)best_e; }
#pragma unroll
        for (int i = 0; i < MAX_PER_LANE; ++i)
            if (lane + 64 * i == best_e) sel[i] = -INFINITY;
    }
    if (lane < topk) {
        if (with_norm) my_weight *= 1.0f / fmaxf(picked_sum, 6.103515625e-5f);
        weights[(size_t)row * topk + lane] = my_weight * scale;
        ids[(size_t)row * topk + lane] = my_id;
    }
}

// Stable ascending rank sort of u32 keys (loken_argsort_small_u32 and loken_stable_sort_u32,
// cuda/moe/gate_topk.cu:453-477, 515-548): key i lands after every smaller key and every equal
// key before it; `sorted` receives the keys, `order` the index each came from. One lane per key;
// the keys pass through LDS a chunk at a time, every lane reading each once.
constexpr int SORT_WG = 256, SORT_CHUNK = 2048;

__global__ __launch_bounds__(SORT_WG) void stable_rank_sort_u32_kernel(const uint32_t* __restrict__ keys,
                                                                       uint32_t* __restrict__ sorted,
                                                                       uint32_t* __restrict__ order, int n) {
    __shared__ uint32_t chunk[SORT_CHUNK];
    const int i = blockIdx.x * SORT_WG + threadIdx.x;
    const uint32_t k = i < n ? keys[i] : 0u;
    int rank = 0;
    for (int base = 0; base < n; base += SORT_CHUNK) {
        const int len = min(SORT_CHUNK, n - base);
        __syncthreads();
        for (int j = threadIdx.x; j < len; j += SORT_WG) chunk[j] = keys[base + j];
        __syncthreads();
        for (int j = 0; j < len; ++j) {
            const uint32_t kj = chunk[j];
            rank += (kj < k) || (kj == k && base + j < i);
        }
    }
    if (i < n) {
        sorted[rank] = k;
        order[rank] = (uint32_t)i;
    }
}

}  // namespace

extern "C" void loken_topk_softmax(const float* logits, float* weights, uint32_t* ids, int n_rows, int n_experts,
                                   int n_expert_used, int with_norm, void* stream) {
    if (!logits || !weights || !ids || n_rows <= 0) return;
    if (n_experts <= 0 || n_experts > 64 * MAX_PER_LANE || n_expert_used <= 0 || n_expert_used > 64 ||
        n_expert_used > n_experts)
        return;   // the caller falls back, as with the reference's launcher
    hipLaunchKernelGGL(topk_softmax_kernel, dim3(n_rows), dim3(64), 0, (hipStream_t)stream, logits, weights, ids,
                       n_experts, n_expert_used, with_norm);
    (void)hipGetLastError();
}

static bool router_sizes_ok(int n_rows, int n_experts, int n_expert_used) {
    return n_rows > 0 && n_experts > 0 && n_experts <= 64 * MAX_PER_LANE && n_expert_used > 0 && n_expert_used <= 64 &&
           n_expert_used <= n_experts;
}

extern "C" void loken_gate_topk_softmax(const float* x_in, const float* gate_w, float* weights_out, uint32_t* ids_out,
                                        int hidden, int n_rows, int n_experts, int n_expert_used, int with_norm,
                                        void* stream) {
    if (!x_in || !gate_w || !weights_out || !ids_out || hidden <= 0 || hidden > 8192) return;   // the caller falls back
    if (!router_sizes_ok(n_rows, n_experts, n_expert_used)) return;
    hipStream_t s = (hipStream_t)stream;
    if (hidden % 4 == 0 && (((uintptr_t)x_in | (uintptr_t)gate_w) & 15) == 0) {
        LkScratch scratch(s);
        const int m = n_rows <= 16 ? 16 : 32;
        const int t_tiles = (n_rows + m - 1) / m, e_tiles = (n_experts + m - 1) / m;
        // K split until the launch has LOGIT_SPREAD workgroups, while a wave keeps at least two units of K
        const int units = hidden / m;
        int splits = LOGIT_SPREAD / (t_tiles < LOGIT_SPREAD ? t_tiles * e_tiles : LOGIT_SPREAD);
        if (splits > units / (2 * LOGIT_WAVES)) splits = units / (2 * LOGIT_WAVES);
        if (splits > 16) splits = 16;
        if (splits < 1) splits = 1;
        float* part = (float*)scratch.get(LK_SCRATCH_ROUTER, (size_t)splits * n_rows * n_experts * 4);
        if (part) {
            if (n_rows <= CHOICE_TOKENS && scratch.ticket() >= 0) {
                auto choice = n_experts <= 64 ? gate_topk16_kernel<1> : n_experts <= 128 ? gate_topk16_kernel<2> : n_experts <= 256 ? gate_topk16_kernel<4> : gate_topk16_kernel<8>;
                hipLaunchKernelGGL(choice, dim3(e_tiles, (splits + CHOICE_GROUPS - 1) / CHOICE_GROUPS), dim3(CHOICE_THREADS), 0, s, x_in, gate_w, part,
                                   weights_out, ids_out, hidden, n_rows, n_experts, splits, n_expert_used, with_norm, scratch.ticket());
                (void)hipGetLastError();
                return;
            }
            auto logits = m == 16 ? gate_logits16_kernel : gate_logits32_kernel;
            hipLaunchKernelGGL(logits, dim3(t_tiles, e_tiles, splits), dim3(64 * LOGIT_WAVES), 0, s, x_in, gate_w, part, hidden, n_rows,
                               n_experts);
            const dim3 waves((n_rows + 3) / 4);
            auto select = n_experts <= 64 ? gate_select_kernel<1> : n_experts <= 128 ? gate_select_kernel<2> : n_experts <= 256 ? gate_select_kernel<4> : gate_select_kernel<8>;
            hipLaunchKernelGGL(select, waves, dim3(256), 0, s, (const float*)part, splits, weights_out, ids_out, n_rows, n_experts,
                               n_expert_used, with_norm);
            (void)hipGetLastError();
            return;
        }
    }
    const int lds = (((hidden + 3) & ~3) + n_experts) * 4;
    hipLaunchKernelGGL(gate_topk_softmax_kernel, dim3(n_rows), dim3(64 * GATE_WAVES), lds, s, x_in,
                       gate_w, weights_out, ids_out, hidden, n_experts, n_expert_used, with_norm);
    (void)hipGetLastError();
}

extern "C" void loken_topk_sigmoid_post(const float* logits_in, const float* bias, float* weights_out, uint32_t* ids_out,
                                        int n_rows, int n_experts, int n_expert_used, int with_norm, float scale,
                                        void* stream) {
    if (!logits_in || !weights_out || !ids_out || !router_sizes_ok(n_rows, n_experts, n_expert_used)) return;
    hipLaunchKernelGGL(topk_sigmoid_post_kernel, dim3(n_rows), dim3(64), 0, (hipStream_t)stream, logits_in, bias,
                       weights_out, ids_out, n_experts, n_expert_used, with_norm, scale);
    (void)hipGetLastError();
}

extern "C" void loken_stable_sort_u32(const uint32_t* keys, uint32_t* sorted, uint32_t* order, int n, void* stream) {
    if (!keys || !sorted || !order || n <= 0) return;
    hipLaunchKernelGGL(stable_rank_sort_u32_kernel, dim3((n + SORT_WG - 1) / SORT_WG), dim3(SORT_WG), 0,
                       (hipStream_t)stream, keys, sorted, order, n);
    (void)hipGetLastError();
}

// The decode-size form of the same sort: the reference serves up to 32 keys with one warp and
// lets the caller fall back above; one workgroup here takes up to 256.
extern "C" void loken_argsort_small_u32(const uint32_t* in, uint32_t* sorted_out, uint32_t* index_out, int m,
                                        void* stream) {
    if (m <= 0 || m > SORT_WG) return;   // the caller falls back
    loken_stable_sort_u32(in, sorted_out, index_out, m, stream);
}
