"""GPU parity of the MoE expert block against the CPU oracle.

The oracle (lko_moe_forward) follows loken's host path: gate/up per routed pair, SiLU, down,
fold in expert-run order (src/inference/moe_cuda_cpu/mod.rs:459-605, 1478-1660). The GPU fold
runs in slot order (cuda/moe/moe_mmq.cu:155-176), so only the final [tokens, hidden] is
comparable and only to float summation order; the intermediate GLU rows are compared in sorted
order, which both sides share.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from loken_amd import lib, moe, ops, synth
from loken_amd.moe import MmqRouting
from moe_block_check import check_block, down_fold_from_rows

pytestmark = pytest.mark.gpu
RTOL, ATOL = 1e-3, 1e-4


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def assert_close(got, want, rtol=RTOL, atol=ATOL):
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    bad = np.abs(got - want) > rtol * np.abs(want) + atol
    assert not bad.any(), f"{bad.sum()} of {bad.size} outside tolerance; worst {np.abs(got - want).max()}"


def make_layer(tokens, hidden, ffn, n_experts, topk, seed, dt_down=lib.TYPE_Q4_K, x_scale=30.0, dt_gu=lib.TYPE_Q4_K):
    dt = dt_gu
    gate = synth.weight(dt, n_experts * ffn, hidden, seed=seed, stream=1)
    up = synth.weight(dt, n_experts * ffn, hidden, seed=seed, stream=2)
    down = synth.weight(dt_down, n_experts * hidden, ffn, seed=seed, stream=3)
    x = synth.activation(tokens, hidden, seed=seed) * np.float32(x_scale)
    logits = synth.activation(tokens, n_experts, seed=seed, stream=7)
    ids, w = oracle.topk_softmax(logits, topk)
    return gate, up, down, x, ids, w


def test_route_groups_pairs_stably_by_expert():
    rng = np.random.default_rng(50)
    tokens, topk, n_experts = 37, 4, 11
    choices = np.stack([rng.choice(n_experts, topk, replace=False) for _ in range(tokens)]).astype(np.int32)
    plan = MmqRouting.from_choices(dev(choices), n_experts)
    slots, experts = oracle.group_by_expert(choices)
    assert plan.slots.cpu().tolist() == slots.tolist()
    assert plan.src_rows.cpu().tolist() == (slots // topk).tolist()
    want_bounds = np.searchsorted(experts, np.arange(n_experts + 1))
    assert plan.bounds.cpu().tolist() == want_bounds.tolist()
    # the sorted-routing entry point builds the same plan
    plan2 = MmqRouting.new(dev(slots), dev(experts), topk, n_experts)
    assert torch.equal(plan2.bounds, plan.bounds) and torch.equal(plan2.slots, plan.slots)
    assert torch.equal(plan2.src_rows, plan.src_rows)


def test_route_with_experts_nobody_chose_and_one_token():
    choices = np.array([[5, 2]], np.int32)
    plan = MmqRouting.from_choices(dev(choices), 8)
    assert plan.bounds.cpu().tolist() == [0, 0, 0, 1, 1, 1, 2, 2, 2]
    assert plan.slots.cpu().tolist() == [1, 0]


@pytest.mark.parametrize("tokens,hidden,ffn,n_experts,topk", [(5, 512, 256, 6, 2), (40, 1024, 512, 8, 3),
                                                             (1, 256, 256, 4, 2), (70, 512, 768, 16, 4)])
@pytest.mark.parametrize("dt_down", [lib.TYPE_Q4_K, lib.TYPE_Q5_K, lib.TYPE_Q6_K])
@pytest.mark.parametrize("path", ["tiled", "rows"])
def test_expert_batched_block_matches_oracle(tokens, hidden, ffn, n_experts, topk, dt_down, path):
    """Both launch families of the expert-batched block: the tiled matmul, and (Q4_K stacks) the
    matrix-unit rows launch that serves short runs per expert."""
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=51, dt_down=dt_down)
    want, want_h = oracle.moe_forward(1, lib.TYPE_Q4_K, dt_down, x, gate, up, down, ids, w, n_experts, ffn, want_h=True)
    plan = MmqRouting.from_choices(dev(ids), n_experts).with_path(path)
    assert plan.takes_rows_launch(lib.TYPE_Q4_K, hidden) == (path == "rows")
    h = plan.gate_up_silu(lib.TYPE_Q4_K, dev(x), dev(gate), dev(up), ffn)
    # GLU rows in sorted order; expf differs from libm's in the last place, and silu(g)*u inherits
    # the relative error of g and u where they nearly cancel: compare against the scale of a row
    got_h = h.cpu().numpy()
    assert (np.abs(got_h - want_h) <= 1e-3 * np.abs(want_h) + 1e-4 * np.abs(want_h).max()).all()
    out = plan.down_fold(dt_down, h, dev(down), hidden, dev(w.reshape(-1)))
    # the strict bound with the oracle's second stage fed the card's own rows; end to end, whatever is
    # outside it belongs to a token with a flipped Q8_1 code of h (moe_block_check.py)
    slots = plan.slots.cpu().numpy()
    h_slot, want_h_slot = np.empty_like(got_h), np.empty_like(want_h)
    h_slot[slots], want_h_slot[slots] = got_h, want_h
    check_block(out.cpu().numpy(), h_slot, want, want_h_slot, dt_down, down, ids, w, n_experts, hidden)


NIBBLE_TILES = {"q4_0": lib.TYPE_Q4_0, "q4_1": lib.TYPE_Q4_1, "q5_0": lib.TYPE_Q5_0, "q5_1": lib.TYPE_Q5_1,
                "iq4_nl": lib.TYPE_IQ4_NL, "mxfp4": lib.TYPE_MXFP4, "iq4_xs": lib.TYPE_IQ4_XS, "q3_k": lib.TYPE_Q3_K,
                "q2_k": lib.TYPE_Q2_K,
                # the codebook formats only mixtures store (src/tensor/quantized/mmq.rs:335-343)
                "iq3_xxs": lib.TYPE_IQ3_XXS, "iq3_s": lib.TYPE_IQ3_S, "iq2_s": lib.TYPE_IQ2_S, "q2_0": lib.TYPE_Q2_0}


@pytest.mark.parametrize("tokens,hidden,ffn,n_experts,topk", [(40, 1024, 512, 8, 3), (70, 512, 768, 16, 4),
                                                             (1, 256, 256, 4, 2), (300, 512, 256, 3, 2)])
@pytest.mark.parametrize("name", sorted(NIBBLE_TILES))
def test_expert_batched_block_in_the_nibble_formats_matches_oracle(name, tokens, hidden, ffn, n_experts, topk):
    """The tiled launch for the 32-value formats, IQ4_XS and Q3_K; IQ4_NL, MXFP4 and IQ4_XS have no dense
    entry point. The last shape runs the 128-token tiles."""
    dt = NIBBLE_TILES[name]
    assert moe.moe_mmq_serves(dt, hidden)
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=53, dt_down=dt, dt_gu=dt, x_scale=4.0)
    want, want_h = oracle.moe_forward(1, dt, dt, x, gate, up, down, ids, w, n_experts, ffn, want_h=True)
    plan = MmqRouting.from_choices(dev(ids), n_experts).with_path("tiled")
    h = plan.gate_up_silu(dt, dev(x), dev(gate), dev(up), ffn)
    got_h = h.cpu().numpy()
    assert (np.abs(got_h - want_h) <= 1e-3 * np.abs(want_h) + 1e-4 * np.abs(want_h).max()).all()
    # down from the oracle's own rows, so that a code flipped by the last place of h does not enter
    out = plan.down_fold(dt, dev(want_h), dev(down), hidden, dev(w.reshape(-1)))
    scale = np.abs(want).max()
    assert (np.abs(out.cpu().numpy() - want) <= 1e-3 * np.abs(want) + 1e-4 * scale).all()


def test_down_fold_alone_is_tight_when_fed_the_oracle_rows():
    # feeding the oracle's own GLU rows removes the re-quantization ambiguity: 1e-3 rel + 1e-4 abs
    tokens, hidden, ffn, n_experts, topk = 24, 512, 512, 8, 2
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=52)
    want, want_h = oracle.moe_forward(1, lib.TYPE_Q4_K, lib.TYPE_Q4_K, x, gate, up, down, ids, w, n_experts, ffn, want_h=True)
    plan = MmqRouting.from_choices(dev(ids), n_experts)
    out = plan.down_fold(lib.TYPE_Q4_K, dev(want_h), dev(down), hidden, dev(w.reshape(-1)))
    assert_close(out.cpu().numpy(), want, atol=1e-4 * max(1.0, np.abs(want).max()))


def test_residual_is_the_starting_value_of_the_fold():
    tokens, hidden, ffn, n_experts, topk = 6, 256, 256, 4, 2
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=53)
    plan = MmqRouting.from_choices(dev(ids), n_experts)
    h = plan.gate_up_silu(lib.TYPE_Q4_K, dev(x), dev(gate), dev(up), ffn)
    base = plan.down_fold(lib.TYPE_Q4_K, h, dev(down), hidden, dev(w.reshape(-1)))
    res = torch.randn((tokens, hidden), device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    with_res = plan.down_fold(lib.TYPE_Q4_K, h, dev(down), hidden, dev(w.reshape(-1)), residual=res)
    # (res + a) + b against (0 + a + b) + res: float summation order only
    scale = base.abs().max().item() + res.abs().max().item()
    assert (with_res - (base + res)).abs().max().item() <= 1e-6 * scale


def test_result_does_not_depend_on_tile_width():
    tokens, hidden, ffn, n_experts, topk = 90, 512, 256, 4, 2
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=54)
    outs = []
    for width in (0, 32, 64, 128):
        plan = MmqRouting.from_choices(dev(ids), n_experts).with_tile_width(width)
        h = plan.gate_up_silu(lib.TYPE_Q4_K, dev(x), dev(gate), dev(up), ffn)
        outs.append(plan.down_fold(lib.TYPE_Q4_K, h, dev(down), hidden, dev(w.reshape(-1))))
    # The narrow tiles run the same int8 kernel, to the bit. The 128-token tile of Q4_K forms the
    # same integer dots on the f16 matrix unit and adds them up in another f32 order; the hidden
    # state is re-quantized between the two products, so a last-bit difference there can move a
    # code by one: a float tolerance, not equality.
    for o in outs[1:3]:
        assert torch.equal(o, outs[0])
    scale = outs[0].abs().max().item()
    assert (outs[3] - outs[0]).abs().max().item() <= 1e-4 * scale


@pytest.mark.parametrize("name", ["q4_k", "q5_k", "q6_k"])
@pytest.mark.parametrize("tokens,heavy", [(330, 40), (330, 150), (620, 260)])
def test_f16_tiles_of_uneven_runs_agree_with_the_int8_tiles(name, tokens, heavy, knobs):
    # expert 0 owns `heavy` rows more than its share, expert 1 none: full tiles, tiles of 32 tokens or fewer, and column
    # tiles past what the grid's first two dimensions cover. Same integers either way, so two f32 orders of the sums of
    # at most 16 sub-blocks of 512 values apart: 2e-5 of the largest result, as for the dense tiles.
    dt = getattr(lib, "TYPE_" + name.upper())
    hidden, ffn, n_experts, topk = 512, 512, 16, 2
    rng = np.random.default_rng(tokens)
    ids = np.stack([2 + rng.permutation(n_experts - 2)[:topk] for _ in range(tokens)]).astype(np.int32)
    ids[rng.permutation(tokens)[:heavy], 0] = 0
    gate, up, down = (dev(synth.weight(dt, n_experts * 512, 512, seed=58, stream=i)) for i in range(3))
    x = dev(synth.activation(tokens, hidden, seed=58))
    weights = torch.full((tokens * topk,), 0.5, device="cuda")
    plan = MmqRouting.from_choices(dev(ids), n_experts).with_path("tiled")
    assert plan.longest_run_expected() > 32
    h = plan.gate_up_silu(dt, x, gate, up, ffn)
    out = plan.down_fold(dt, h, down, hidden, weights)
    knobs.set("LK_MMQ_I8")
    h8 = plan.gate_up_silu(dt, x, gate, up, ffn)
    out8 = plan.down_fold(dt, h, down, hidden, weights)
    assert (h - h8).abs().max().item() <= 4e-5 * h8.abs().max().item()   # a product of two such results
    assert (out - out8).abs().max().item() <= 2e-5 * out8.abs().max().item()


def test_glu_kernels():
    rng = np.random.default_rng(55)
    rows, width, n_experts = 13, 40, 3
    gu = rng.standard_normal((rows, 2 * width)).astype(np.float32) * 3
    l = lib.load()
    s = torch.cuda.current_stream().cuda_stream
    gud = dev(gu)
    out = torch.empty((rows, width), device="cuda")
    l.loken_moe_mmq_silu_mul(gud.data_ptr(), out.data_ptr(), rows, width, s)
    g, u = gu[:, :width].astype(np.float64), gu[:, width:].astype(np.float64)
    np.testing.assert_allclose(out.cpu().numpy(), g / (1 + np.exp(-g)) * u, rtol=2e-6, atol=1e-7)
    bounds = np.array([0, 4, 4, 13], np.int32)
    gb = rng.standard_normal((n_experts, width)).astype(np.float32)
    ub = rng.standard_normal((n_experts, width)).astype(np.float32)
    alpha, limit = 1.702, 7.0
    bd, gbd, ubd = dev(bounds), dev(gb), dev(ub)   # named: a temporary would be freed before the launch
    l.loken_moe_mmq_swiglu_oai(gud.data_ptr(), out.data_ptr(), rows, width, bd.data_ptr(), n_experts,
                               gbd.data_ptr(), ubd.data_ptr(), alpha, limit, s)
    e_of = np.array([0] * 4 + [2] * 9)
    xx = np.minimum(g + gb[e_of], limit)
    uc = np.clip(u + ub[e_of], -limit, limit)
    np.testing.assert_allclose(out.cpu().numpy(), xx / (1 + np.exp(-alpha * xx)) * (1 + uc), rtol=3e-6, atol=1e-6)


def test_fold_is_in_slot_order_with_bias():
    rng = np.random.default_rng(56)
    tokens, topk, cols, n_experts = 5, 3, 33, 4
    pairs = rng.standard_normal((tokens * topk, cols)).astype(np.float32)
    wts = rng.random(tokens * topk).astype(np.float32)
    choices = rng.integers(0, n_experts, tokens * topk).astype(np.int32)
    bias = rng.standard_normal((n_experts, cols)).astype(np.float32)
    start = rng.standard_normal((tokens, cols)).astype(np.float32)
    out = dev(start.copy())
    pd, wd, cd, bd = dev(pairs), dev(wts), dev(choices), dev(bias)
    lib.load().loken_moe_mmq_fold(pd.data_ptr(), wd.data_ptr(), cd.data_ptr(), bd.data_ptr(), out.data_ptr(),
                                  tokens, topk, cols, torch.cuda.current_stream().cuda_stream)
    want = start.copy()
    for t in range(tokens):
        for k in range(topk):
            p = t * topk + k
            want[t] = want[t] + wts[p] * (pairs[p] + bias[choices[p]])   # same f32 steps, same order
    np.testing.assert_allclose(out.cpu().numpy(), want, rtol=1e-6, atol=1e-6)


def test_benchmark_shape_256_tokens_against_sampled_oracle():
    # Qwen3-30B-A3B-shaped layer: 128 experts, hidden 2048, ffn 768, top-8
    tokens, hidden, ffn, n_experts, topk = 256, 2048, 768, 128, 8
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=0)
    plan = MmqRouting.from_choices(dev(ids), n_experts)
    h = plan.gate_up_silu(lib.TYPE_Q4_K, dev(x), dev(gate), dev(up), ffn)
    out = plan.down_fold(lib.TYPE_Q4_K, h, dev(down), hidden, dev(w.reshape(-1))).cpu().numpy()
    # oracle on a sample of tokens (a token's output depends only on its own routed pairs)
    sample = [0, 17, 100, 255]
    want, want_h = oracle.moe_forward(1, lib.TYPE_Q4_K, lib.TYPE_Q4_K, x[sample], gate, up, down, ids[sample], w[sample],
                                      n_experts, ffn, want_h=True)
    slots = plan.slots.cpu().numpy()
    h_slot = np.empty((tokens * topk, ffn), np.float32)
    h_slot[slots] = h.cpu().numpy()
    rows = (np.array(sample)[:, None] * topk + np.arange(topk)[None, :]).reshape(-1)
    want_h_slot = np.empty_like(want_h)
    want_h_slot[oracle.group_by_expert(ids[sample])[0]] = want_h
    check_block(out[sample], h_slot[rows], want, want_h_slot, lib.TYPE_Q4_K, down, ids[sample], w[sample], n_experts, hidden)
    # every routed pair landed somewhere: the per-expert load adds up
    bounds = plan.bounds.cpu().numpy()
    assert bounds[-1] == tokens * topk and (np.diff(bounds) >= 0).all()


# ---------------------------------------------------------------- decode (per routed pair)
from loken_amd.moe import (ExpertRouting, moe_forward, moe_gemm_gguf, moe_gemm_gguf_down_reduce,
                           moe_gemm_gguf_gate_up_silu_mul)


def slot_order(h_sorted, ids):
    """oracle rows are in sorted order; the decode kernels write slot order"""
    slots, _ = oracle.group_by_expert(ids)
    out = np.empty_like(h_sorted)
    out[slots] = h_sorted
    return out


@pytest.mark.parametrize("tokens,hidden,ffn,n_experts,topk", [(1, 2048, 768, 128, 8), (3, 512, 256, 6, 2),
                                                             (16, 1024, 768, 32, 4)])
@pytest.mark.parametrize("dt_down", [lib.TYPE_Q4_K, lib.TYPE_Q5_K, lib.TYPE_Q6_K])
def test_per_pair_decode_block_matches_oracle(tokens, hidden, ffn, n_experts, topk, dt_down):
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=57, dt_down=dt_down)
    want, want_h = oracle.moe_forward(1, lib.TYPE_Q4_K, dt_down, x, gate, up, down, ids, w, n_experts, ffn, want_h=True)
    routing = ExpertRouting(dev(ids))
    slots, experts = oracle.group_by_expert(ids)
    assert routing.sorted_token_ids.cpu().tolist() == slots.tolist()
    assert routing.expert_ids.cpu().tolist() == experts.tolist()
    h = moe_gemm_gguf_gate_up_silu_mul(lib.TYPE_Q4_K, dev(x), dev(gate), dev(up), routing, n_experts, ffn)
    want_slot = slot_order(want_h, ids)
    assert (np.abs(h.cpu().numpy() - want_slot) <= 1e-3 * np.abs(want_slot) + 1e-4 * np.abs(want_slot).max()).all()
    out = moe_gemm_gguf_down_reduce(dt_down, h, dev(down), routing, dev(w.reshape(-1)), n_experts, hidden)
    check_block(out.cpu().numpy(), h.cpu().numpy(), want, want_slot, dt_down, down, ids, w, n_experts, hidden)


# the rows of the reference's expert table (src/inference/moe_cuda/gemm.rs:23-39) beyond the K-quant engines
TABLE_TAIL = {"q2_k": lib.TYPE_Q2_K, "q3_k": lib.TYPE_Q3_K, "q5_0": lib.TYPE_Q5_0, "mxfp4": lib.TYPE_MXFP4,
              "q5_1": lib.TYPE_Q5_1, "iq4_nl": lib.TYPE_IQ4_NL, "iq4_xs": lib.TYPE_IQ4_XS,
              "iq3_xxs": lib.TYPE_IQ3_XXS, "iq3_s": lib.TYPE_IQ3_S, "iq2_s": lib.TYPE_IQ2_S, "q2_0": lib.TYPE_Q2_0,
              "iq2_xxs": lib.TYPE_IQ2_XXS,   # wire ids 11..15
              "q5_k": lib.TYPE_Q5_K}   # and Q5_K on the K-quant engine, short rows and long


@pytest.mark.parametrize("hidden,ffn", [(256, 331), (1024, 129), (1024, 128), (2048, 331), (2048, 512), (2560, 331), (4096, 257)])
def test_gated_launch_of_many_tiles_a_wave(hidden, ffn):
    """1024 routed pairs leave a pair one workgroup, whose waves walk 4 to 42 tiles: one or several times the totals that wait in a
    wave's lanes at a time (4, 8 or 16 tiles of 4, 2 or 1 rows), a short last batch, and a last tile cut by the row count."""
    n_experts, topk, tokens = 3, 2, 512
    gate = synth.weight(lib.TYPE_Q4_K, n_experts * ffn, hidden, seed=61, stream=1)
    up = synth.weight(lib.TYPE_Q4_K, n_experts * ffn, hidden, seed=61, stream=2)
    x = synth.activation(tokens, hidden, seed=61) * np.float32(4.0)
    ids = np.stack([np.random.default_rng(t).choice(n_experts, topk, replace=False) for t in range(tokens)]).astype(np.int32)
    got = moe_gemm_gguf_gate_up_silu_mul(lib.TYPE_Q4_K, dev(x), dev(gate), dev(up), ExpertRouting(dev(ids)), n_experts, ffn).cpu().numpy()
    some = np.r_[0, 1, tokens // 2, tokens - 1]
    g = oracle.ob_matmul(lib.TYPE_Q4_K, x[some], gate, n_experts * ffn).reshape(len(some), n_experts, ffn).astype(np.float64)
    u = oracle.ob_matmul(lib.TYPE_Q4_K, x[some], up, n_experts * ffn).reshape(len(some), n_experts, ffn).astype(np.float64)
    h = g / (1.0 + np.exp(-g)) * u
    for i, t in enumerate(some):
        for j in range(topk):
            # 1e-3 of each factor, as the mat-vec's bound (1e-3 relative + 1e-4 absolute): both factors' errors add up, silu's slope is at most 1.1
            e = ids[t, j]
            bound = (1.1 * (1e-3 * np.abs(g[i, e]) + 1e-4)) * np.abs(u[i, e]) + np.abs(g[i, e]) * (1e-3 * np.abs(u[i, e]) + 1e-4) + 1e-6
            assert (np.abs(got[t * topk + j] - h[i, e]) <= bound).all()


@pytest.mark.parametrize("hidden,rows", [(256, 4), (1024, 4), (1280, 2), (2048, 2), (2560, 1), (4096, 1)])
@pytest.mark.parametrize("tiles", [1, 2, 3, 17])
def test_gated_register_launch_gives_the_bits_of_the_staged_one(hidden, rows, tiles, knobs):
    """1024 routed pairs leave a pair one workgroup of eight waves, so that a wave walks the given number of tiles of `rows` rows: one
    (a form of its own), fewer than the totals that wait in a wave's lanes at a time, and more; with the last wave cut and whole. The
    biases are read at rows that the lanes rebuild, so every activation goes through both."""
    from loken_amd.moe import (moe_gemm_gguf_gate_up_gelu_mul_concat, moe_gemm_gguf_gate_up_swiglu_limited,
                               moe_gemm_gguf_gate_up_swiglu_oai)
    n_experts, topk, tokens, dt = 3, 2, 512, lib.TYPE_Q4_K
    x = dev(synth.activation(tokens, hidden, seed=66) * np.float32(4.0))
    ids = np.stack([np.random.default_rng(t).choice(n_experts, topk, replace=False) for t in range(tokens)]).astype(np.int32)
    routing = ExpertRouting(dev(ids))
    for ffn in (8 * rows * tiles, 8 * rows * tiles - 1, 8 * rows * (tiles - 1) + 1):
        gate, up = (dev(synth.weight(dt, n_experts * ffn, hidden, seed=66, stream=i)) for i in (1, 2))
        both = dev(synth.weight(dt, n_experts * 2 * ffn, hidden, seed=66, stream=3))
        gb, ub = (dev(synth.normal(66, i, n_experts * ffn).reshape(n_experts, ffn)) for i in (11, 12))

        def run():
            return [moe_gemm_gguf_gate_up_silu_mul(dt, x, gate, up, routing, n_experts, ffn),
                    moe_gemm_gguf_gate_up_swiglu_oai(dt, x, gate, up, routing, n_experts, ffn, 1.702, 7.0, gb, ub),
                    moe_gemm_gguf_gate_up_swiglu_limited(dt, x, gate, up, routing, n_experts, ffn, 5.0),
                    moe_gemm_gguf_gate_up_gelu_mul_concat(dt, x, both, routing, n_experts, ffn)]

        one = run()
        knobs.set("LK_TUNE_NO_REG_MOE")
        two = run()
        knobs.clear("LK_TUNE_NO_REG_MOE")
        for a, b in zip(one, two):
            assert torch.equal(a, b), ffn


@pytest.mark.parametrize("gib", [2.5, 4.5])
def test_gated_launch_over_a_slab_of_more_than_31_and_than_32_bits(gib):
    # 2.5 GiB an expert is the register launch's (offsets of 32 bits), 4.5 GiB the staged one's. A period of rows over and over:
    # its outputs repeat.
    hidden, period, dt = 4096, 4093, lib.TYPE_Q4_K
    times = int(gib * 2**30) // (period * 16 * 144)
    one_gate, one_up = (dev(synth.weight(dt, period, hidden, seed=67, stream=i)) for i in (1, 2))
    x, routing = dev(synth.activation(1, hidden, seed=67) * np.float32(4.0)), ExpertRouting(dev(np.zeros((1, 1), np.int32)))
    want = moe_gemm_gguf_gate_up_silu_mul(dt, x, one_gate, one_up, routing, 1, period)
    gate, up = (w.reshape(-1).repeat(times) for w in (one_gate, one_up))
    got = moe_gemm_gguf_gate_up_silu_mul(dt, x, gate, up, routing, 1, period * times)
    assert torch.equal(got.reshape(times, period), want.expand(times, period))


@pytest.mark.parametrize("tokens,hidden,ffn,n_experts,topk", [(1, 1024, 768, 16, 4), (3, 512, 256, 6, 2), (2, 2560, 512, 4, 2)])
@pytest.mark.parametrize("name", sorted(TABLE_TAIL))
def test_per_pair_decode_block_in_the_tail_formats_matches_oracle(name, tokens, hidden, ffn, n_experts, topk):
    dt = TABLE_TAIL[name]
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=61, dt_down=dt, dt_gu=dt, x_scale=4.0)
    want, want_h = oracle.moe_forward(1, dt, dt, x, gate, up, down, ids, w, n_experts, ffn, want_h=True)
    routing = ExpertRouting(dev(ids))
    h = moe_gemm_gguf_gate_up_silu_mul(dt, dev(x), dev(gate), dev(up), routing, n_experts, ffn)
    want_slot = slot_order(want_h, ids)
    assert (np.abs(h.cpu().numpy() - want_slot) <= 1e-3 * np.abs(want_slot) + 1e-4 * np.abs(want_slot).max()).all()
    # down from the oracle's own intermediate rows, so the two stages are checked apart
    bias = torch.randn((n_experts, hidden), device="cuda", generator=torch.Generator(device="cuda").manual_seed(7))
    out = moe_gemm_gguf_down_reduce(dt, dev(want_slot), dev(down), routing, dev(w.reshape(-1)), n_experts, hidden)
    scale = np.abs(want).max()
    assert (np.abs(out.cpu().numpy() - want) <= 1e-3 * np.abs(want) + 1e-4 * scale).all()
    with_bias = moe_gemm_gguf_down_reduce(dt, dev(want_slot), dev(down), routing, dev(w.reshape(-1)), n_experts, hidden,
                                          down_bias=bias)
    add = (dev(w).unsqueeze(-1) * bias[dev(ids).long()]).sum(1)
    assert (with_bias - (out + add)).abs().max().item() <= 1e-5 * (scale + add.abs().max().item())
    # the plain launcher over the same pairs: the gate product alone
    plain = moe_gemm_gguf(dt, dev(x), dev(gate), routing, n_experts, ffn)
    slots, experts = oracle.group_by_expert(ids)
    gate_rows = gate.reshape(n_experts, ffn, -1)
    for j in range(len(slots)):
        want_row = oracle.ob_matmul(dt, x[slots[j] // topk][None, :], gate_rows[experts[j]].reshape(-1), ffn)[0]
        got_row = plain[slots[j]].cpu().numpy()
        assert (np.abs(got_row - want_row) <= 1e-3 * np.abs(want_row) + 1e-4 * np.abs(want_row).max()).all()


@pytest.mark.parametrize("name", ["q4_k", "q6_k", "q8_0", "mxfp4", "q5_0", "q3_k"])
def test_gated_decode_launch_with_the_other_activations(name):
    """The gate and up products are the same-codes oracle's; the activation on top of them is the
    closed form the reference's kernels state (cuda/moe/moe_gguf.cu:994-1003, 1178-1184, 1280-1289)."""
    from loken_amd.moe import (moe_gemm_gguf_gate_up_gelu_mul_concat, moe_gemm_gguf_gate_up_swiglu_limited,
                               moe_gemm_gguf_gate_up_swiglu_oai)
    dt = {"q4_k": lib.TYPE_Q4_K, "q6_k": lib.TYPE_Q6_K, "q8_0": lib.TYPE_Q8_0, **TABLE_TAIL}[name]
    tokens, hidden, ffn, n_experts, topk = 3, 512, 256, 5, 2
    gate, up, _, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=63, dt_gu=dt, x_scale=4.0)
    routing = ExpertRouting(dev(ids))
    slots, experts = oracle.group_by_expert(ids)
    gate_rows, up_rows = gate.reshape(n_experts, ffn, -1), up.reshape(n_experts, ffn, -1)
    g = np.empty((tokens * topk, ffn), np.float64)
    u = np.empty((tokens * topk, ffn), np.float64)
    for j in range(len(slots)):
        row = x[slots[j] // topk][None, :]
        g[slots[j]] = oracle.ob_matmul(dt, row, gate_rows[experts[j]].reshape(-1), ffn)[0]
        u[slots[j]] = oracle.ob_matmul(dt, row, up_rows[experts[j]].reshape(-1), ffn)[0]
    e_of_slot = ids.reshape(-1)

    def close(got, want):
        got = got.cpu().numpy()
        assert (np.abs(got - want) <= 1e-3 * np.abs(want) + 1e-4 * np.abs(want).max()).all()

    limit = float(np.quantile(np.abs(g), 0.7))   # so that both sides of every clamp occur
    alpha = 1.702
    gb = synth.normal(63, 11, n_experts * ffn).reshape(n_experts, ffn) * np.float32(0.1 * limit)
    ub = synth.normal(63, 12, n_experts * ffn).reshape(n_experts, ffn) * np.float32(0.1 * limit)
    for biased in (False, True):
        gg = g + (gb[e_of_slot] if biased else 0.0)
        uu = u + (ub[e_of_slot] if biased else 0.0)
        xx = np.minimum(gg, limit)
        want = xx / (1.0 + np.exp(-alpha * xx)) * (1.0 + np.clip(uu, -limit, limit))
        got = moe_gemm_gguf_gate_up_swiglu_oai(dt, dev(x), dev(gate), dev(up), routing, n_experts, ffn, alpha, limit,
                                               dev(gb) if biased else None, dev(ub) if biased else None)
        close(got, want)
    gl = np.minimum(g, limit)
    close(moe_gemm_gguf_gate_up_swiglu_limited(dt, dev(x), dev(gate), dev(up), routing, n_experts, ffn, limit),
          gl / (1.0 + np.exp(-gl)) * np.clip(u, -limit, limit))
    # one tensor per layer: every expert's gate rows, then its up rows
    both = np.concatenate([gate_rows, up_rows], axis=1)
    want = 0.5 * g * (1.0 + np.tanh(0.7978845608028654 * (g + 0.044715 * g ** 3))) * u
    close(moe_gemm_gguf_gate_up_gelu_mul_concat(dt, dev(x), dev(np.ascontiguousarray(both)), routing, n_experts, ffn), want)


@pytest.mark.parametrize("name", ["q4_k", "mxfp4"])
def test_live_count_variants_run_the_first_pairs_only(name):
    from loken_amd.moe import moe_gemm_gguf_down_pairs_live, moe_gemm_gguf_gate_up_silu_mul_live
    dt = {"q4_k": lib.TYPE_Q4_K, **TABLE_TAIL}[name]
    tokens, hidden, ffn, n_experts, topk = 4, 512, 256, 5, 2
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=64, dt_down=dt, dt_gu=dt, x_scale=4.0)
    routing = ExpertRouting(dev(ids))
    slots = routing.sorted_token_ids.cpu().numpy()
    pairs = tokens * topk
    full_h = moe_gemm_gguf_gate_up_silu_mul(dt, dev(x), dev(gate), dev(up), routing, n_experts, ffn)
    flat_w = dev(w.reshape(-1))
    for count in (5, pairs, 0):
        live = torch.tensor([count], dtype=torch.int32, device="cuda")   # the card reads it as a uint32
        marker = torch.full((pairs, ffn), -7.0, device="cuda")
        h = moe_gemm_gguf_gate_up_silu_mul_live(dt, dev(x), dev(gate), dev(up), routing, n_experts, ffn, live, out=marker)
        ran, idle = slots[:count], slots[count:]
        assert torch.equal(h[ran], full_h[ran])
        assert (h[idle] == -7.0).all()
        rows = moe_gemm_gguf_down_pairs_live(dt, full_h, dev(down), routing, flat_w, n_experts, hidden, live)
        assert (rows[idle] == 0).all()
        if count == pairs:
            want = moe_gemm_gguf_down_reduce(dt, full_h, dev(down), routing, flat_w, n_experts, hidden)
            got = rows.reshape(tokens, topk, hidden).sum(1)
            assert (got - want).abs().max().item() <= 1e-6 * want.abs().max().item()
            all_rows = rows
    live = torch.tensor([5], dtype=torch.int32, device="cuda")
    rows5 = moe_gemm_gguf_down_pairs_live(dt, full_h, dev(down), routing, flat_w, n_experts, hidden, live)
    assert torch.equal(rows5[slots[:5]], all_rows[slots[:5]])


@pytest.mark.parametrize("name", ["q4_k", "q6_k", "mxfp4"])
def test_experts_over_two_tensors_match_the_one_tensor_launch(name):
    from loken_amd.moe import (moe_gemm_gguf_down_pairs_over, moe_gemm_gguf_down_reduce_over,
                               moe_gemm_gguf_gate_up_silu_mul_over)
    dt = {"q4_k": lib.TYPE_Q4_K, "q6_k": lib.TYPE_Q6_K, **TABLE_TAIL}[name]
    tokens, hidden, ffn, n_experts, topk, cut = 5, 512, 256, 6, 3, 4
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=65, dt_down=dt, dt_gu=dt, x_scale=4.0)
    routing = ExpertRouting(dev(ids))
    flat_w = dev(w.reshape(-1))
    want_h = moe_gemm_gguf_gate_up_silu_mul(dt, dev(x), dev(gate), dev(up), routing, n_experts, ffn)
    want = moe_gemm_gguf_down_reduce(dt, want_h, dev(down), routing, flat_w, n_experts, hidden)

    def halves(stack):   # experts 0..cut-1 in one allocation, cut.. in another
        per = stack.reshape(n_experts, -1)
        return dev(np.ascontiguousarray(per[:cut])), dev(np.ascontiguousarray(per[cut:]))

    (g0, g1), (u0, u1), (d0, d1) = halves(gate), halves(up), halves(down)
    h = moe_gemm_gguf_gate_up_silu_mul_over(dt, dev(x), g0, u0, g1, u1, cut, routing, n_experts, ffn)
    assert torch.equal(h, want_h)
    # the second pair named by addresses on the card; the host-side ones are then ignored
    at = torch.tensor([g1.data_ptr(), u1.data_ptr()], dtype=torch.int64, device="cuda")
    h2 = moe_gemm_gguf_gate_up_silu_mul_over(dt, dev(x), g0, u0, g0, u0, cut, routing, n_experts, ffn, more_at=at)
    assert torch.equal(h2, want_h)
    bias = torch.randn((n_experts, hidden), device="cuda", generator=torch.Generator(device="cuda").manual_seed(8))
    assert torch.equal(moe_gemm_gguf_down_reduce_over(dt, want_h, d0, d1, cut, routing, flat_w, n_experts, hidden), want)
    assert torch.equal(moe_gemm_gguf_down_reduce_over(dt, want_h, d0, d1, cut, routing, flat_w, n_experts, hidden, down_bias=bias),
                       moe_gemm_gguf_down_reduce(dt, want_h, dev(down), routing, flat_w, n_experts, hidden, down_bias=bias))
    rows = moe_gemm_gguf_down_pairs_over(dt, want_h, d0, d1, cut, routing, flat_w, n_experts, hidden)
    assert (rows.reshape(tokens, topk, hidden).sum(1) - want).abs().max().item() <= 1e-6 * want.abs().max().item()
    at_d = torch.tensor([d1.data_ptr(), 0], dtype=torch.int64, device="cuda")
    assert torch.equal(moe_gemm_gguf_down_pairs_over(dt, want_h, d0, d0, cut, routing, flat_w, n_experts, hidden, more_at=at_d), rows)


def test_decode_launchers_refuse_wire_ids_outside_the_table():
    tokens, hidden, ffn, n_experts, topk = 2, 512, 256, 4, 2
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=62)
    routing = ExpertRouting(dev(ids))
    L = lib.load()
    out = torch.empty((tokens * topk, ffn), device="cuda")
    for wire in (16, 17, 99, -1):   # the table ends at 15 (src/inference/moe_cuda/gemm.rs:23-39)
        rc = L.loken_moe_gemm_gguf(dev(x).data_ptr(), dev(gate).data_ptr(), routing.sorted_token_ids.data_ptr(),
                                   routing.expert_ids.data_ptr(), None, out.data_ptr(), n_experts, topk,
                                   tokens * topk, ffn, hidden, wire, None)
        assert rc == lib.LK_ERR_TYPE


def test_decode_down_reduce_is_tight_on_oracle_rows_and_folds_in_slot_order():
    tokens, hidden, ffn, n_experts, topk = 4, 512, 512, 8, 3
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=58)
    want, want_h = oracle.moe_forward(1, lib.TYPE_Q4_K, lib.TYPE_Q4_K, x, gate, up, down, ids, w, n_experts, ffn, want_h=True)
    routing = ExpertRouting(dev(ids))
    h = dev(slot_order(want_h, ids))
    out = moe_gemm_gguf_down_reduce(lib.TYPE_Q4_K, h, dev(down), routing, dev(w.reshape(-1)), n_experts, hidden)
    assert_close(out.cpu().numpy(), want, atol=1e-4 * max(1.0, np.abs(want).max()))
    # residual as the starting value, add_after as a written sum, bias scaled by the router weight
    res = torch.randn((tokens, hidden), device="cuda", generator=torch.Generator(device="cuda").manual_seed(5))
    with_res = moe_gemm_gguf_down_reduce(lib.TYPE_Q4_K, h, dev(down), routing, dev(w.reshape(-1)), n_experts, hidden, residual=res)
    added = moe_gemm_gguf_down_reduce(lib.TYPE_Q4_K, h, dev(down), routing, dev(w.reshape(-1)), n_experts, hidden, add_after=res)
    scale = out.abs().max().item() + res.abs().max().item()
    assert (with_res - (out + res)).abs().max().item() <= 1e-6 * scale
    assert (added - (out + res)).abs().max().item() <= 1e-6 * scale
    bias = torch.randn((n_experts, hidden), device="cuda", generator=torch.Generator(device="cuda").manual_seed(6))
    biased = moe_gemm_gguf_down_reduce(lib.TYPE_Q4_K, h, dev(down), routing, dev(w.reshape(-1)), n_experts, hidden, down_bias=bias)
    wt = dev(w)
    extra = (wt.unsqueeze(-1) * bias[dev(ids).long()]).sum(dim=1)
    assert (biased - (out + extra)).abs().max().item() <= 1e-5 * (scale + extra.abs().max().item())


def test_generic_routed_product_with_and_without_weights():
    tokens, k, n, n_experts, topk = 5, 512, 96, 7, 2
    wq = synth.weight(lib.TYPE_Q8_0, n_experts * n, k, seed=59, stream=1)
    x = synth.activation(tokens, k, seed=59)
    ids, w = oracle.topk_softmax(synth.activation(tokens, n_experts, seed=59, stream=7), topk)
    routing = ExpertRouting(dev(ids))
    we = wq.reshape(n_experts, n, -1, 34)
    plain = moe_gemm_gguf(lib.TYPE_Q8_0, dev(x), dev(wq), routing, n_experts, n).cpu().numpy()
    for t in range(tokens):
        for j in range(topk):
            assert_close(plain[t * topk + j], oracle.ob_matmul(lib.TYPE_Q8_0, x[t:t + 1], we[ids[t, j]], n)[0])
    # with routing weights: one activation row per slot, output scaled
    xs = synth.activation(tokens * topk, k, seed=59, stream=8)
    scaled = moe_gemm_gguf(lib.TYPE_Q8_0, dev(xs), dev(wq), routing, n_experts, n, topk_weights=dev(w.reshape(-1))).cpu().numpy()
    for p in range(tokens * topk):
        e = ids.reshape(-1)[p]
        assert_close(scaled[p], w.reshape(-1)[p] * oracle.ob_matmul(lib.TYPE_Q8_0, xs[p:p + 1], we[e], n)[0])


@pytest.mark.parametrize("half", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("name", ["q4_k", "q6_k", "q8_0", "q5_1"])
def test_prefill_form_takes_half_precision_rows(name, half):
    # loken_moe_gemm_gguf_prefill: the rows arrive as f16 / bf16; the oracle is fed the values they hold
    from loken_amd.moe import moe_gemm_gguf_prefill
    wtype = {"q4_k": lib.TYPE_Q4_K, "q6_k": lib.TYPE_Q6_K, "q8_0": lib.TYPE_Q8_0, "q5_1": lib.TYPE_Q5_1}[name]
    tokens, k, n, n_experts, topk = 9, 512, 96, 6, 2
    wq = synth.weight(wtype, n_experts * n, k, seed=61, stream=1)
    ids, w = oracle.topk_softmax(synth.activation(tokens, n_experts, seed=61, stream=7), topk)
    routing = ExpertRouting(dev(ids))
    we = wq.reshape(n_experts, -1)   # an expert's n rows of blocks
    xh = dev(synth.activation(tokens, k, seed=61)).to(half)
    x_seen = xh.to(torch.float32).cpu().numpy()
    got = moe_gemm_gguf_prefill(wtype, xh, dev(wq), routing, n_experts, n).cpu().numpy()
    for t in range(tokens):
        for j in range(topk):
            assert_close(got[t * topk + j], oracle.ob_matmul(wtype, x_seen[t:t + 1], we[ids[t, j]], n)[0])
    # the same values as f32 rows through the decode-form launch: the same bits
    same = moe_gemm_gguf(wtype, xh.to(torch.float32), dev(wq), routing, n_experts, n).cpu().numpy()
    assert np.array_equal(got, same)
    # with routing weights: one activation row per slot, output scaled
    xs = dev(synth.activation(tokens * topk, k, seed=61, stream=8)).to(half)
    scaled = moe_gemm_gguf_prefill(wtype, xs, dev(wq), routing, n_experts, n, topk_weights=dev(w.reshape(-1))).cpu().numpy()
    xs_seen = xs.to(torch.float32).cpu().numpy()
    for p in range(tokens * topk):
        e = ids.reshape(-1)[p]
        assert_close(scaled[p], w.reshape(-1)[p] * oracle.ob_matmul(wtype, xs_seen[p:p + 1], we[e], n)[0])
    # an input width the launch does not know is a status, not a launch
    L = lib.load()
    assert L.loken_moe_gemm_gguf_prefill(xh.data_ptr(), dev(wq).data_ptr(), routing.sorted_token_ids.data_ptr(),
                                         routing.expert_ids.data_ptr(), None, dev(np.zeros(4, np.float32)).data_ptr(),
                                         n_experts, topk, tokens * topk, n, k, 2, 1, None) == lib.LK_ERR_TYPE


@pytest.mark.parametrize("tokens,hidden,ffn,n_experts,topk", [(1, 2048, 768, 128, 8), (16, 2048, 768, 128, 8),
                                                              (5, 100, 512, 9, 4), (7, 264, 1024, 12, 6),
                                                              (3, 77, 768, 5, 1), (40, 96, 512, 16, 8), (64, 64, 512, 16, 8)])
@pytest.mark.parametrize("name", ["q4_k", "q5_k", "q6_k"])
def test_down_and_fold_in_one_launch_gives_the_bits_of_the_two_launches(name, tokens, hidden, ffn, n_experts, topk, knobs):
    """Short K-quant rows at a handful of tokens take one launch (down + fold); with that launch switched
    off the same call takes the per-pair mat-vec and the fold kernel. Same bits, and both on the oracle."""
    dt, block_bytes = {"q4_k": (lib.TYPE_Q4_K, 144), "q5_k": (lib.TYPE_Q5_K, 176), "q6_k": (lib.TYPE_Q6_K, 210)}[name]
    down = synth.weight(dt, n_experts * hidden, ffn, seed=61, stream=3)
    ids, w = oracle.topk_softmax(synth.activation(tokens, n_experts, seed=61, stream=7), topk)
    h = synth.activation(tokens * topk, ffn, seed=61, stream=4) * np.float32(5.0)
    routing = ExpertRouting(dev(ids))
    bias = torch.randn((n_experts, hidden), device="cuda", generator=torch.Generator(device="cuda").manual_seed(9))
    res = torch.randn((tokens, hidden), device="cuda", generator=torch.Generator(device="cuda").manual_seed(10))
    down_d, h_d, w_d = dev(down), dev(h), dev(w.reshape(-1))

    def run(**kw):
        return moe_gemm_gguf_down_reduce(dt, h_d, down_d, routing, w_d, n_experts, hidden, **kw)

    cases = ({}, {"residual": res}, {"add_after": res}, {"down_bias": bias}, {"down_bias": bias, "add_after": res})
    one = [run(**kw) for kw in cases]
    # a pair whose expert is out of range, in the one launch
    keep = routing.expert_ids[0].item()
    routing.expert_ids[0] = -1
    one_dropped = run()
    knobs.set("LK_TUNE_DOWN_FOLD_OFF")
    two_dropped = run()
    routing.expert_ids[0] = keep
    two = [run(**kw) for kw in cases]
    for a, b in zip(one, two):
        assert torch.equal(a, b)
    assert torch.equal(one_dropped, two_dropped)
    we = down.reshape(n_experts, hidden, -1, block_bytes)
    want = np.zeros((tokens, hidden), np.float32)
    for t in range(tokens):
        for j in range(topk):
            p = t * topk + j
            want[t] += w[t, j] * oracle.ob_matmul(dt, h[p:p + 1], we[ids[t, j]], hidden)[0]
    assert_close(one[0].cpu().numpy(), want, atol=1e-4 * max(1.0, np.abs(want).max()))


@pytest.mark.parametrize("tokens,hidden,ffn,n_experts,topk", [(3, 331, 512, 6, 8), (2, 100, 768, 5, 4), (3, 331, 1024, 6, 4), (2, 203, 1024, 9, 8),
                                                              (2, 1031, 768, 4, 3)])
@pytest.mark.parametrize("name", ["q4_k", "q5_k", "q6_k"])
def test_down_and_fold_over_several_passes_and_a_cut_last_workgroup(name, tokens, hidden, ffn, n_experts, topk, knobs):
    """A workgroup takes 16 (up to four pairs a token) or 8 rows a pass and sums a row's pairs after its last one: one to sixteen
    passes, odd counts, and rows that end inside a workgroup's first, middle or last pass, against the mat-vec per pair and the sum."""
    dt = {"q4_k": lib.TYPE_Q4_K, "q5_k": lib.TYPE_Q5_K, "q6_k": lib.TYPE_Q6_K}[name]
    down = dev(synth.weight(dt, n_experts * hidden, ffn, seed=65, stream=3))
    ids = np.stack([np.arange(topk) % n_experts for _ in range(tokens)]).astype(np.int32)
    ids = np.stack([np.random.default_rng(t).permutation(row) for t, row in enumerate(ids)])
    w = synth.activation(tokens, topk, seed=65, stream=7)
    h = dev(synth.activation(tokens * topk, ffn, seed=65, stream=4) * np.float32(5.0))
    routing, w = ExpertRouting(dev(ids)), dev(w.reshape(-1))
    bias = torch.randn((n_experts, hidden), device="cuda", generator=torch.Generator(device="cuda").manual_seed(11))
    res = torch.randn((tokens, hidden), device="cuda", generator=torch.Generator(device="cuda").manual_seed(12))
    kinds = ({}, {"residual": res}, {"add_after": res}, {"down_bias": bias}, {"down_bias": bias, "add_after": res})

    def run():
        return [moe_gemm_gguf_down_reduce(dt, h, down, routing, w, n_experts, hidden, **kw) for kw in kinds]

    knobs.set("LK_TUNE_DOWN_FOLD_OFF")
    want = run()
    knobs.clear("LK_TUNE_DOWN_FOLD_OFF")
    for passes in (1, 2, 3, 4, 7, 16):
        knobs.set("LK_TUNE_DOWN_FOLD_PASSES", str(passes))
        for got, two in zip(run(), want):
            assert torch.equal(got, two), passes


def test_pairs_the_routing_leaves_out_add_nothing():
    tokens, hidden, ffn, n_experts, topk = 3, 256, 256, 4, 2
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=60)
    routing = ExpertRouting(dev(ids))
    h = moe_gemm_gguf_gate_up_silu_mul(lib.TYPE_Q4_K, dev(x), dev(gate), dev(up), routing, n_experts, ffn)
    full = moe_gemm_gguf_down_reduce(lib.TYPE_Q4_K, h, dev(down), routing, dev(w.reshape(-1)), n_experts, hidden)
    # mark the first sorted pair as belonging to no expert: the fold must see zeros for it
    dropped = routing.sorted_token_ids[0].item()
    routing.expert_ids[0] = n_experts + 3
    part = moe_gemm_gguf_down_reduce(lib.TYPE_Q4_K, h, dev(down), routing, dev(w.reshape(-1)), n_experts, hidden)
    t = dropped // topk
    others = [i for i in range(tokens) if i != t]
    assert torch.equal(part[others], full[others])
    assert not torch.equal(part[t], full[t])


def test_launchers_report_bad_arguments_and_formats():
    l = lib.load()
    buf = torch.zeros(4096, dtype=torch.uint8, device="cuda")
    p, s = buf.data_ptr(), torch.cuda.current_stream().cuda_stream
    assert l.loken_moe_gemm_gguf(p, p, p, p, None, p, 4, 2, 4, 8, 256, 16, s) == lib.LK_ERR_TYPE    # past the table's last row
    assert l.loken_moe_gemm_gguf(p, p, p, p, None, p, 4, 2, 4, 8, 250, 1, s) == lib.LK_ERR_ARG      # k not whole blocks
    assert l.loken_moe_gemm_gguf(p, p, p, p, None, p, 4, 2, 5, 8, 256, 1, s) == lib.LK_ERR_ARG      # pairs % topk
    assert l.loken_moe_gemm_gguf_down_reduce(p, p, p, p, None, p, 4, 2, 4, 8, 256, 1, None, None, s) == lib.LK_ERR_ARG
    assert l.loken_moe_gemm_gguf(p, p, p, p, None, p, 4, 2, 0, 8, 256, 1, s) == lib.LK_OK           # nothing routed
    l.loken_stream_scratch_release()


@pytest.mark.parametrize("tokens", [1, 16, 256])
def test_layer_entry_picks_a_path_and_both_agree(tokens):
    hidden, ffn, n_experts, topk = 512, 256, 16, 4
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=61)
    args = (lib.TYPE_Q4_K, lib.TYPE_Q4_K, dev(x), dev(gate), dev(up), dev(down), dev(ids), dev(w), n_experts, ffn)
    got, rows = moe_forward(*args, return_rows=True)
    want, want_h = oracle.moe_forward(1, lib.TYPE_Q4_K, lib.TYPE_Q4_K, x, gate, up, down, ids, w, n_experts, ffn, want_h=True)
    want_slot = slot_order(want_h, ids)
    sample = None if tokens <= 16 else np.arange(0, tokens, 16)
    check_block(got.cpu().numpy(), rows.cpu().numpy(), want, want_slot, lib.TYPE_Q4_K, down, ids, w, n_experts, hidden,
                tokens=sample)


@pytest.mark.parametrize("tokens,topk,n_experts,hidden,ffn,gu,dn", [
    (1, 2, 4, 512, 256, lib.TYPE_Q4_K, lib.TYPE_Q4_K), (7, 4, 60, 1024, 768, lib.TYPE_Q4_K, lib.TYPE_Q6_K),
    (3, 2, 8, 512, 1280, lib.TYPE_MXFP4, lib.TYPE_MXFP4), (70, 8, 512, 256, 512, lib.TYPE_Q4_K, lib.TYPE_Q4_K),
    (33, 4, 8, 512, 256, lib.TYPE_Q8_0, lib.TYPE_Q8_0), (129, 2, 8, 512, 768, lib.TYPE_Q4_K, lib.TYPE_Q4_K),
    (301, 8, 16, 256, 512, lib.TYPE_Q5_K, lib.TYPE_Q6_K)])
def test_block_in_one_call_is_the_block_launch_by_launch(tokens, topk, n_experts, hidden, ffn, gu, dn):
    """lk_moe_forward (pairs in slot order, sums written, the activation in the second quantizer) against the
    launches it is made of, sorted and summed into zeros: the same bits, two calls in a row."""
    gate, up = (dev(synth.weight(gu, n_experts * ffn, hidden, seed=62, stream=i)) for i in (1, 2))
    down = dev(synth.weight(dn, n_experts * hidden, ffn, seed=62, stream=3))
    for seed in (63, 64):
        x = dev(synth.activation(tokens, hidden, seed=seed))
        ids, w = oracle.topk_softmax(synth.activation(tokens, n_experts, seed=seed, stream=7), topk)
        args = (gu, dn, x, gate, up, down, dev(ids), dev(w), n_experts, ffn)
        assert torch.equal(moe_forward(*args), moe_forward(*args, return_rows=True)[0])


@pytest.mark.parametrize("gu,dn,tokens,topk,n_experts,hidden,ffn,grouped", [
    (lib.TYPE_Q4_K, lib.TYPE_Q4_K, 12, 2, 8, 2048, 512, False), (lib.TYPE_Q4_K, lib.TYPE_Q4_K, 24, 2, 8, 2048, 1024, True), (lib.TYPE_Q4_K, lib.TYPE_Q6_K, 11, 4, 8, 2048, 1024, True),
    (lib.TYPE_Q4_K, lib.TYPE_Q4_K, 25, 2, 8, 512, 256, True), (lib.TYPE_Q5_K, lib.TYPE_Q5_K, 10, 8, 64, 3072, 1536, True), (lib.TYPE_Q5_K, lib.TYPE_Q5_K, 10, 8, 64, 1024, 1024, False),
    (lib.TYPE_Q8_0, lib.TYPE_Q8_0, 20, 8, 64, 1536, 768, True), (lib.TYPE_Q8_0, lib.TYPE_Q8_0, 12, 4, 8, 2048, 768, False)])
def test_the_pairs_or_the_batch_by_the_weights_too(gu, dn, tokens, topk, n_experts, hidden, ffn, grouped):
    # both sides of the lines by the bytes of the pairs' matrices, against the same tokens one at a time
    # (rows small enough that the f16 scale of a Q8_1 block holds every product)
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, 84, dn, x_scale=3.0, dt_gu=gu)
    assert bool(lib.load().lk_moe_block_path(gu, dn, tokens, topk, n_experts, hidden, ffn) & lib.MOE_GROUPED) == grouped
    g, u, d, xd, idd, wd = (dev(a) for a in (gate, up, down, x, ids, w))
    got = moe.moe_forward(gu, dn, xd, g, u, d, idd, wd, n_experts, ffn)
    want = torch.cat([moe.moe_forward(gu, dn, xd[i:i + 1].contiguous(), g, u, d, idd[i:i + 1].contiguous(), wd[i:i + 1].contiguous(), n_experts, ffn)
                      for i in range(tokens)])
    assert ((got - want).abs() <= 1e-3 * want.abs() + 1e-3 * want.abs().max()).all()


@pytest.mark.parametrize("gu,dn", [(lib.TYPE_Q4_0, lib.TYPE_Q4_0), (lib.TYPE_Q4_1, lib.TYPE_Q4_1), (lib.TYPE_Q8_0, lib.TYPE_Q4_0), (lib.TYPE_Q4_1, lib.TYPE_Q4_K)])
@pytest.mark.parametrize("tokens,topk,n_experts,hidden,ffn", [(12, 2, 8, 512, 256), (23, 2, 8, 1024, 512), (25, 8, 60, 256, 256)])
def test_formats_without_a_mat_vec_per_pair_at_three_to_six_rows_an_expert(gu, dn, tokens, topk, n_experts, hidden, ffn):
    # small weights, where other formats take a mat-vec per routed pair
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, 85, dn, x_scale=4.0, dt_gu=gu)
    args = (gu, dn, dev(x), dev(gate), dev(up), dev(down), dev(ids), dev(w), n_experts, ffn)
    got, rows = moe_forward(*args, return_rows=True)
    want, want_h = oracle.moe_forward(1, gu, dn, x, gate, up, down, ids, w, n_experts, ffn, want_h=True)
    check_block(got.cpu().numpy(), rows.cpu().numpy(), want, slot_order(want_h, ids), dn, down, ids, w, n_experts, hidden)
    out = torch.empty(tokens, hidden, device="cuda")
    status = lib.load().lk_moe_forward(gu, dn, *(a.data_ptr() for a in args[2:8]), out.data_ptr(), tokens, topk, n_experts, hidden, ffn,
                                       torch.cuda.current_stream().cuda_stream)
    assert status == lib.LK_OK and torch.equal(out, got)


@pytest.mark.parametrize("tokens,topk,n_experts,hidden,ffn,tiles", [(24, 2, 8, 1280, 1536, True), (12, 2, 8, 1280, 1536, False), (40, 2, 8, 1792, 512, True),
                                                                    (24, 2, 8, 1792, 512, False), (40, 2, 8, 1280, 1024, False), (24, 2, 8, 2304, 1280, True),
                                                                    (40, 2, 8, 1024, 1280, False)])
def test_short_runs_of_rows_without_a_wave_a_tile_go_on_the_tiles(tokens, topk, n_experts, hidden, ffn, tiles):
    # Q4_K blocks on both sides of the line, against the same tokens one at a time (a mat-vec per routed pair)
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, 83, lib.TYPE_Q4_K, dt_gu=lib.TYPE_Q4_K)
    path = lib.load().lk_moe_block_path(lib.TYPE_Q4_K, lib.TYPE_Q4_K, tokens, topk, n_experts, hidden, ffn)
    assert bool(path & lib.MOE_TILES) == tiles
    g, u, d, xd, idd, wd = (dev(a) for a in (gate, up, down, x, ids, w))
    got = moe.moe_forward(lib.TYPE_Q4_K, lib.TYPE_Q4_K, xd, g, u, d, idd, wd, n_experts, ffn)
    want = torch.cat([moe.moe_forward(lib.TYPE_Q4_K, lib.TYPE_Q4_K, xd[i:i + 1].contiguous(), g, u, d, idd[i:i + 1].contiguous(),
                                      wd[i:i + 1].contiguous(), n_experts, ffn) for i in range(tokens)])
    assert ((got - want).abs() <= 1e-3 * want.abs() + 1e-3 * want.abs().max()).all()


@pytest.mark.parametrize("tokens,topk,n_experts,hidden,ffn,gu,rows_gu", [(41, 2, 8, 768, 256, lib.TYPE_Q4_K, True), (27, 4, 16, 256, 256, lib.TYPE_Q5_K, False),
                                                                        (67, 4, 32, 768, 256, lib.TYPE_Q5_K, False), (333, 1, 8, 1280, 512, lib.TYPE_Q6_K, False)])
def test_tokens_that_start_between_pieces_give_the_block_of_aligned_ones(tokens, topk, n_experts, hidden, ffn, gu, rows_gu):
    # the routing launch quantizes them too: rows of any number of 256-value blocks, from any float on
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, 77, gu, dt_gu=gu)
    path = lib.load().lk_moe_block_path(gu, gu, tokens, topk, n_experts, hidden, ffn)
    assert bool(path & lib.MOE_ROWS_GATE_UP) == rows_gu and bool(path & (lib.MOE_TILES | lib.MOE_ROWS_GATE_UP))
    args = [dev(a) for a in (gate, up, down, ids, w)]
    want = moe.moe_forward(gu, gu, dev(x), *args, n_experts, ffn)
    odd = torch.empty(x.size + 1, device="cuda")
    odd[1:].copy_(dev(x).reshape(-1))
    assert torch.equal(moe.moe_forward(gu, gu, odd[1:].view(tokens, hidden), *args, n_experts, ffn), want)


@pytest.mark.parametrize("tokens,topk,n_experts,hidden,ffn,dn,rows_gu", [
    (105, 2, 8, 512, 256, lib.TYPE_Q6_K, True), (115, 2, 8, 512, 256, lib.TYPE_Q6_K, False),   # longest run 36 / 39, down tiled
    (500, 4, 128, 2304, 256, lib.TYPE_Q4_K, False), (115, 2, 8, 2304, 256, lib.TYPE_Q4_K, True)])   # long rows: tiles fill the chip, or not
def test_block_launch_by_launch_makes_the_choices_of_the_one_call(tokens, topk, n_experts, hidden, ffn, dn, rows_gu):
    """Where a product's launch depends on the other one, or on how many tiles there are: the same bits both ways."""
    path = lib.load().lk_moe_block_path(lib.TYPE_Q4_K, dn, tokens, topk, n_experts, hidden, ffn)
    assert path & lib.MOE_GROUPED and bool(path & lib.MOE_ROWS_GATE_UP) == rows_gu
    assert MmqRouting(tokens, topk, n_experts, "cuda").takes_rows_launch(lib.TYPE_Q4_K, hidden)   # the stack's rule alone
    gate, up = (dev(synth.weight(lib.TYPE_Q4_K, 2 * ffn, hidden, seed=67, stream=i)).repeat(n_experts // 2, 1, 1) for i in (1, 2))
    down = dev(synth.weight(dn, 2 * hidden, ffn, seed=67, stream=3)).repeat(n_experts // 2, 1, 1)
    x = dev(synth.activation(tokens, hidden, seed=67))
    ids, w = oracle.topk_softmax(synth.activation(tokens, n_experts, seed=67, stream=7), topk)
    args = (lib.TYPE_Q4_K, dn, x, gate, up, down, dev(ids), dev(w), n_experts, ffn)
    assert torch.equal(moe_forward(*args), moe_forward(*args, return_rows=True)[0])


# runs around every edge of the token tiles (one to three of 32, then several tiles), none at all, and one far longer than expected
RUNS = [1, 32, 33, 64, 65, 96, 97, 128, 129, 0, 200, 31, 2, 95, 63, 34]


@pytest.mark.parametrize("gu,dn", [(lib.TYPE_Q4_K, lib.TYPE_Q4_K), (lib.TYPE_Q4_K, lib.TYPE_Q6_K), (lib.TYPE_Q6_K, lib.TYPE_Q6_K),
                                   (lib.TYPE_Q5_K, lib.TYPE_Q5_K), (lib.TYPE_Q6_K, lib.TYPE_Q5_K)])
@pytest.mark.parametrize("runs,hidden,ffn", [(RUNS, 256, 256), (RUNS, 768, 512), ([3] * 40 + [150] + [0, 1] * 11 + [12], 512, 256)])
def test_block_on_the_f16_tiles_at_every_run_length(runs, hidden, ffn, gu, dn):
    """Both products on the f16 tiles, operands gathered and handed on between them: the bits of the same launches through
    workspace records and f32 rows, and the oracle's block."""
    n_experts, tokens = len(runs), sum(runs)
    ids = np.random.default_rng(68).permutation(np.repeat(np.arange(n_experts, dtype=np.int32), runs)).reshape(tokens, 1)
    ids = np.concatenate([ids, np.roll(ids, 7, axis=0)], axis=1)
    w = np.abs(synth.activation(tokens, 2, seed=68)) + np.float32(0.1)
    # runs of a few rows over 64 experts: the rows launch of Q4_K and the int8 tiles of Q6_K, the same block
    tiles = n_experts < 60 or lib.TYPE_Q5_K in (gu, dn)
    assert bool(lib.load().lk_moe_block_path(gu, dn, tokens, 2, n_experts, hidden, ffn) & lib.MOE_TILES) == tiles
    gate, up = (synth.weight(gu, n_experts * ffn, hidden, seed=68, stream=i) for i in (1, 2))
    down = synth.weight(dn, n_experts * hidden, ffn, seed=68, stream=3)
    x = synth.activation(tokens, hidden, seed=69)
    args = (gu, dn, dev(x), dev(gate), dev(up), dev(down), dev(ids), dev(w), n_experts, ffn)
    got, rows = moe_forward(*args, return_rows=True)
    assert torch.equal(moe_forward(*args), got)
    sample = np.arange(0, tokens, 9)
    slabs = [np.ascontiguousarray(m).reshape(n_experts, -1) for m in (gate, up)]
    pairs = (sample[:, None] * 2 + np.arange(2)).reshape(-1)
    h = rows.cpu().numpy()[pairs]
    for p, hp in zip(pairs, h):
        e, row = ids[p // 2, p % 2], x[p // 2][None, :]
        g, u = (oracle.ob_matmul(gu, row, s[e], ffn)[0].astype(np.float64) for s in slabs)
        want = g / (1.0 + np.exp(-g)) * u
        assert (np.abs(hp - want) <= 1e-3 * np.abs(want) + 1e-4 * max(1.0, np.abs(want).max())).all()
    fed = down_fold_from_rows(dn, h, down, ids[sample], w[sample], n_experts, hidden)
    bound = 1e-3 * np.abs(fed) + 1e-4 * max(1.0, np.abs(fed).max())
    assert (np.abs(got.cpu().numpy()[sample] - fed) <= bound).all()


@pytest.mark.parametrize("gu,dn", [(lib.TYPE_Q4_K, lib.TYPE_Q6_K), (lib.TYPE_Q5_K, lib.TYPE_Q5_K), (lib.TYPE_Q6_K, lib.TYPE_Q6_K),
                                   (lib.TYPE_Q8_0, lib.TYPE_Q4_0), (lib.TYPE_MXFP4, lib.TYPE_IQ4_NL)])
def test_block_on_the_f16_tiles_keeps_odd_tokens_and_missing_choices_to_themselves(gu, dn):
    """Zeros, tiny and large values, infinities and NaN among the tokens, choices outside the expert range among the pairs: the
    launches' own bits, every other token as without them, a missing pair as one of weight zero."""
    hidden, ffn, n_experts, tokens, topk = 512, 256, 16, 300, 4
    assert lib.load().lk_moe_block_path(gu, dn, tokens, topk, n_experts, hidden, ffn) & lib.MOE_TILES
    gate, up = (dev(synth.weight(gu, n_experts * ffn, hidden, seed=71, stream=i)) for i in (1, 2))
    down = dev(synth.weight(dn, n_experts * hidden, ffn, seed=71, stream=3))
    x = dev(synth.activation(tokens, hidden, seed=71))
    ids, w = (dev(a) for a in oracle.topk_softmax(synth.activation(tokens, n_experts, seed=71, stream=7), topk))
    run = lambda x, ids, w, **how: moe_forward(gu, dn, x, gate, up, down, ids, w, n_experts, ffn, **how)
    clean = run(x, ids, w)
    odd = x.clone()
    odd[3] = 0
    odd[50] *= 1e-7
    odd[51, ::32] = 30.0   # (a Q8_1 scale holds 65504 x 127: the gated products of larger values are infinite)
    odd[77, 5], odd[130, 511], odd[299] = float("inf"), float("nan"), float("-inf")
    got = run(odd, ids, w)
    changed = torch.tensor([3, 50, 51, 77, 130, 299], device="cuda")
    kept = torch.ones(tokens, dtype=torch.bool, device="cuda")
    kept[changed] = False
    assert torch.equal(got[kept], clean[kept]) and not got[3].any() and torch.isfinite(got[[50, 51]]).all()
    assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(run(odd, ids, w, return_rows=True)[0]))
    missing, weights = ids.clone(), w.clone()
    for token, slot, to in ((0, 0, -1), (9, 3, n_experts), (64, 1, 2 ** 31 - 1), (64, 2, -2 ** 31), (298, 0, 1 << 20)):
        missing[token, slot], weights[token, slot] = to, 0.0
    missing[200], weights[200] = -1, 0.0   # a token without any expert
    got = run(x, missing, w)
    assert torch.equal(got, run(x, ids, weights)) and not got[200].any()
    assert torch.equal(got, run(x, missing, w, return_rows=True)[0])


@pytest.mark.parametrize("gu,dn", [(lib.TYPE_Q8_0, lib.TYPE_Q8_0), (lib.TYPE_Q4_0, lib.TYPE_Q8_0), (lib.TYPE_Q4_K, lib.TYPE_Q4_0),
                                   (lib.TYPE_MXFP4, lib.TYPE_MXFP4), (lib.TYPE_IQ4_NL, lib.TYPE_MXFP4), (lib.TYPE_Q5_K, lib.TYPE_IQ4_NL)])
@pytest.mark.parametrize("runs,hidden,ffn", [(RUNS, 256, 256), (RUNS, 768, 512)])
def test_block_of_plain_blocks_on_the_f16_tiles(runs, hidden, ffn, gu, dn):
    test_block_on_the_f16_tiles_at_every_run_length(runs, hidden, ffn, gu, dn)


@pytest.mark.parametrize("wtype,second,mapped", [(lib.TYPE_Q4_K, True, False), (lib.TYPE_Q6_K, False, True)])
def test_expert_product_of_more_rows_than_its_operands_buffer_holds(wtype, second, mapped):
    """17000 rows of 14336 values: 564 MB of token operands, which the launch makes and multiplies in passes of 256 MB at most,
    runs cut at their ends: the bits of calls over less than a pass each."""
    l, k, n, stacks = lib.load(), 14336, 128, 2 if second else 1
    runs, info, s = [5000, 0, 11963, 37], ops.MMQ_DEVICE_INFO, torch.cuda.current_stream().cuda_stream
    w = dev(synth.weight(wtype, stacks * len(runs) * n, k, seed=70, stream=1))
    half = w.numel() // stacks
    base = dev(synth.activation(500, k, seed=70))
    bounds = np.concatenate([[0], np.cumsum(runs)]).astype(np.int32)

    def launch(y, rows, cut, dst, ids):
        w2 = w.reshape(-1)[half:].data_ptr() if second else None
        assert getattr(l, moe.MMQ_MOE_LAUNCHER[wtype])(
            w.data_ptr(), w2, n, y.data_ptr(), dst.data_ptr(), cut.data_ptr(), ids.data_ptr() if ids is not None else None, half // len(runs), k, n, rows,
            k // synth.BLOCK_LEN[wtype], stacks * n, len(runs), 12000, 12000, 0, info["cc"], info["smpbo"], info["warp_size"], s) != 0

    total = int(bounds[-1])
    x = base.repeat(total // 500 + 1, 1)[:total].contiguous()
    y = ops.mmq_quantize(wtype, x)
    ids = dev(np.random.default_rng(70).permutation(total).astype(np.int32)) if mapped else None
    out = torch.full((total, stacks * n), float("nan"), device="cuda")
    launch(ops.mmq_quantize(wtype, base), 500, dev(np.array([0, 500, 500, 500, 500], np.int32)), torch.empty_like(out[:500]), None)   # kernels loaded
    l.loken_stream_scratch_release()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    launch(y, total, dev(bounds), out, ids)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] <= 336 << 20   # 256 MB and the quarter more that a buffer grows by
    if mapped:
        out = out[ids.long()]
    for m0 in range(0, total, 500):
        m1 = min(m0 + 500, total)
        part = torch.empty((m1 - m0, stacks * n), device="cuda")
        y = ops.mmq_quantize(wtype, x[m0:m1])
        launch(y, m1 - m0, dev(np.clip(bounds, m0, m1) - np.int32(m0)), part, None)
        assert torch.equal(out[m0:m1], part), m0
    l.loken_stream_scratch_release()


@pytest.mark.parametrize("n,n_experts,topk", [(1, 3, 1), (63, 5, 3), (64, 1, 1), (1025, 130, 5), (4097, 512, 1), (8888, 128, 8)])
def test_routing_is_a_stable_grouping(n, n_experts, topk):
    choices = synth.rand_ints(23, n, n, n_experts).astype(np.int32).reshape(-1, topk)
    plan = MmqRouting.from_choices(dev(choices), n_experts)
    order = np.argsort(choices.reshape(-1), kind="stable")
    assert np.array_equal(plan.slots.cpu().numpy(), order)
    assert np.array_equal(plan.src_rows.cpu().numpy(), order // topk)
    assert np.array_equal(plan.bounds.cpu().numpy(), np.searchsorted(np.sort(choices.reshape(-1)), np.arange(n_experts + 1)))


@pytest.mark.parametrize("n,n_experts,topk", [(1, 3, 1), (65, 5, 5), (1025, 130, 5), (4100, 64, 4)])
@pytest.mark.parametrize("share", [0.2, 1.0])
def test_pairs_without_an_expert_come_behind_all_others(n, n_experts, topk, share):
    """Every entry of slots and src_rows is written whatever the choices hold: the quantizer gathers all of them."""
    choices = synth.rand_ints(24, n, n, n_experts).astype(np.int32)
    out = synth.rand_ints(25, n, n, 1000) < 1000 * share
    choices[out] = np.array([-1, n_experts, 0x7FFFFFFF, -2 ** 31], np.int32)[synth.rand_ints(26, n, n, 4)[out]]
    expert = np.where((choices < 0) | (choices >= n_experts), n_experts, choices)
    order = np.argsort(expert, kind="stable")
    cd = dev(choices)
    counts, bounds, slots, src = (torch.full((m,), -9, dtype=torch.int32, device="cuda") for m in (n_experts, n_experts + 1, n, n))
    lib.load().loken_moe_mmq_route(cd.data_ptr(), n, topk, n_experts, counts.data_ptr(), bounds.data_ptr(), slots.data_ptr(),
                                   src.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert np.array_equal(slots.cpu().numpy(), order)
    assert np.array_equal(src.cpu().numpy(), order // topk)
    assert np.array_equal(bounds.cpu().numpy(), np.searchsorted(np.sort(expert), np.arange(n_experts + 1)))
    assert np.array_equal(counts.cpu().numpy(), np.bincount(expert, minlength=n_experts + 1)[:n_experts])


@pytest.mark.parametrize("tokens,topk,n_experts,hidden,ffn,gu,dn", [
    (1, 2, 4, 512, 256, lib.TYPE_Q4_K, lib.TYPE_Q4_K),          # a mat-vec per pair
    (3, 2, 8, 512, 1280, lib.TYPE_MXFP4, lib.TYPE_MXFP4),
    (24, 4, 16, 512, 256, lib.TYPE_Q4_K, lib.TYPE_Q4_K),        # rows launches
    (33, 4, 8, 512, 256, lib.TYPE_Q8_0, lib.TYPE_Q8_0),         # int8 tiles
    (7, 4, 4, 1024, 768, lib.TYPE_Q4_K, lib.TYPE_Q6_K),         # rows, then tiles
    (129, 2, 8, 512, 768, lib.TYPE_Q4_K, lib.TYPE_Q4_K),        # f16 tiles
    (301, 8, 16, 256, 512, lib.TYPE_Q5_K, lib.TYPE_Q6_K)])
def test_choices_that_name_no_expert_add_nothing(tokens, topk, n_experts, hidden, ffn, gu, dn):
    """Left-out pairs (-1, the count itself, what the router leaves for a token that is not a number): the block's
    output is that of the same choices with a weight of zero, bit for bit (a sum gains 0 x a finite row)."""
    gate, up = (dev(synth.weight(gu, n_experts * ffn, hidden, seed=65, stream=i)) for i in (1, 2))
    down = dev(synth.weight(dn, n_experts * hidden, ffn, seed=65, stream=3))
    x = synth.activation(tokens, hidden, seed=65)
    ids, w = oracle.topk_softmax(synth.activation(tokens, n_experts, seed=65, stream=7), topk)
    left_out = synth.rand_ints(66, tokens, tokens * topk, 4).reshape(tokens, topk) == 0
    left_out[-1] = True                                         # a token without any expert: the NaN row below
    ids_out, w_zero = ids.copy(), w.copy()
    ids_out[left_out] = np.resize(np.array([-1, n_experts, 0x7FFFFFFF], np.int32), left_out.sum())
    w_zero[left_out] = 0.0
    want = moe_forward(gu, dn, dev(x), gate, up, down, dev(ids), dev(w_zero), n_experts, ffn)
    x_nan, w_nan = x.copy(), w.copy()
    x_nan[-1] = np.nan
    w_nan[-1] = np.nan
    args = (gu, dn, dev(x_nan), gate, up, down, dev(ids_out), dev(w_nan), n_experts, ffn)
    # the scratch the block works in, left full of values that are no indices and no numbers
    junk = moe_forward(gu, dn, torch.full((2 * tokens, hidden), float("nan"), device="cuda"), gate, up, down,
                       dev(np.concatenate([ids, ids])), dev(np.concatenate([w, w])), n_experts, ffn)
    assert junk.shape == (2 * tokens, hidden)
    got = moe_forward(*args)
    assert torch.equal(got, want) and (got[-1] == 0).all()
    by_launch, rows = moe_forward(*args, return_rows=True)
    assert torch.equal(by_launch, got)
    assert (rows[dev(left_out.reshape(-1))] == 0).all() and torch.isfinite(rows).all()


# ---------------------------------------------------------------- router
@pytest.mark.parametrize("tokens,experts,topk,renorm", [(1, 128, 8, True), (16, 128, 8, True), (256, 128, 8, False),
                                                        (7, 60, 4, True), (5, 512, 64, True), (3, 8, 8, False)])
def test_router_topk_softmax_matches_oracle(tokens, experts, topk, renorm):
    logits = synth.normal(90, tokens * 1000 + experts, tokens * experts).astype(np.float32).reshape(tokens, experts)
    want_ids, want_w = oracle.topk_softmax(logits, topk, renorm)
    w, ids = moe.topk_softmax(dev(logits), topk, renorm)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.allclose(w.cpu().numpy(), want_w, rtol=1e-5, atol=1e-7)


def test_router_ties_go_to_the_lower_expert_and_weights_descend():
    logits = np.zeros((2, 128), np.float32)
    logits[1, [5, 40, 41, 100]] = [2.0, 3.0, 3.0, 2.0]
    w, ids = moe.topk_softmax(dev(logits), 8, True)
    ids, w = ids.cpu().numpy(), w.cpu().numpy()
    assert ids[0].tolist() == list(range(8)) and np.allclose(w[0], 1.0 / 8)
    assert ids[1, :4].tolist() == [40, 41, 5, 100] and ids[1, 4:].tolist() == [0, 1, 2, 3]
    assert (np.diff(w[1]) <= 0).all() and abs(w[1].sum() - 1.0) < 1e-6


@pytest.mark.parametrize("tokens,topk,n_experts", [(3, 2, 5), (8, 4, 16), (1, 8, 128)])
def test_q4k_pair_rows_over_caller_quantized_rows_with_one_expert_per_pair(tokens, topk, n_experts):
    """loken_moe_q4k_imma_m8_gate_up and loken_moe_q4k_imma_m8_down: Q8_1 rows from the caller,
    expert ids per pair (one of them out of range), GELU on the gate. The products are the
    same-codes oracle's (cuda/moe/moe_q4k_imma_m8.cu:273-296, moe_q4k_imma_m8_down.cu:196-230)."""
    from loken_amd.moe import moe_q4k_imma_m8_down_reduce, moe_q4k_imma_m8_gate_up
    hidden, ffn = 512, 256
    gate, up, down, x, ids, w = make_layer(tokens, hidden, ffn, n_experts, topk, seed=66, x_scale=4.0)
    slots, experts = oracle.group_by_expert(ids)
    experts = experts.copy()
    dropped = len(slots) // 2
    experts[dropped] = n_experts + 3          # a pair the routing leaves out
    gate_rows, up_rows = gate.reshape(n_experts, ffn, -1), up.reshape(n_experts, ffn, -1)
    both = np.ascontiguousarray(np.concatenate([gate_rows, up_rows], axis=1))
    pairs = tokens * topk
    want_h = np.zeros((pairs, ffn), np.float64)
    for j in range(pairs):
        if experts[j] >= n_experts:
            continue
        row = x[slots[j] // topk][None, :]
        g = oracle.ob_matmul(lib.TYPE_Q4_K, row, gate_rows[experts[j]].reshape(-1), ffn)[0].astype(np.float64)
        u = oracle.ob_matmul(lib.TYPE_Q4_K, row, up_rows[experts[j]].reshape(-1), ffn)[0].astype(np.float64)
        want_h[slots[j]] = 0.5 * g * (1.0 + np.tanh(0.7978845608028654 * (g + 0.044715 * g ** 3))) * u
    sd, ed = dev(slots.astype(np.int32)), dev(experts.astype(np.int32))
    h = moe_q4k_imma_m8_gate_up(dev(x), dev(both), sd, ed, n_experts, topk, ffn)
    got_h = h.cpu().numpy()
    assert (got_h[slots[dropped]] == 0).all()
    assert (np.abs(got_h - want_h) <= 1e-3 * np.abs(want_h) + 1e-4 * np.abs(want_h).max()).all()

    # down from the device's own h, so that the two sides quantize the same rows
    down_rows = down.reshape(n_experts, hidden, -1)
    flat_w = w.reshape(-1).astype(np.float32)
    want = np.zeros((tokens, hidden), np.float64)
    for slot in range(pairs):                 # slot order: the fold's order
        j = int(np.nonzero(slots == slot)[0][0])
        if experts[j] >= n_experts:
            continue
        y = oracle.ob_matmul(lib.TYPE_Q4_K, got_h[slot][None, :], down_rows[experts[j]].reshape(-1), hidden)[0]
        want[slot // topk] += (y * flat_w[slot]).astype(np.float64)
    got = moe_q4k_imma_m8_down_reduce(h, dev(down), sd, ed, dev(flat_w), n_experts, topk, hidden).cpu().numpy()
    assert (np.abs(got - want) <= 1e-3 * np.abs(want) + 1e-4 * np.abs(want).max()).all()


@pytest.mark.parametrize("hint", [1, 9, 40])
# a wave per 16-row tile (2, 3, 4, 8 super-blocks: every load depth), a wave per 32-row tile (1, 5, 6), or four
# waves splitting a tile's super-blocks (10)
@pytest.mark.parametrize("k", [256, 512, 768, 1024, 1280, 1536, 2048, 2560])
def test_rows_launch_serves_any_run_length_whatever_the_hint(hint, k):
    """lk_moe_q4k_rows_grouped: the hint only picks the pass width (8, 16 or 32 rows); an expert with
    more rows takes more passes, one without rows none, and gather / scatter follow the routing."""
    rng = np.random.default_rng(67)
    n_experts, n, tokens = 5, 100, 30
    counts = [37, 0, 1, 9, 13]                              # sorted rows per expert
    rows = sum(counts)
    bounds = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    src = rng.integers(0, tokens, rows).astype(np.int32)    # sorted row -> token
    dst_map = rng.permutation(rows).astype(np.int32)        # sorted row -> output row
    w = synth.weight(lib.TYPE_Q4_K, n_experts * n, k, seed=67, stream=1)
    w2 = synth.weight(lib.TYPE_Q4_K, n_experts * n, k, seed=67, stream=2)
    x = synth.activation(tokens, k, seed=67) * np.float32(4.0)
    q = ops.quantize_q8_1_rows(dev(x), k_padded=k)
    expert_of = np.repeat(np.arange(n_experts), counts)
    per = w.reshape(n_experts, n, -1), w2.reshape(n_experts, n, -1)
    prod = [np.stack([oracle.ob_matmul(lib.TYPE_Q4_K, x[src[i]][None, :], m[expert_of[i]].reshape(-1), n)[0]
                      for i in range(rows)]).astype(np.float64) for m in per]
    L = lib.load()
    s = torch.cuda.current_stream().cuda_stream
    wd, w2d, bd, sd, dd = dev(w), dev(w2), dev(bounds), dev(src), dev(dst_map)
    # plain product, scattered
    out = torch.full((rows, n), -9.0, device="cuda")
    lib.check("lk_moe_q4k_rows_grouped", L.lk_moe_q4k_rows_grouped(
        wd.data_ptr(), None, 0, q.data_ptr(), k // 32, bd.data_ptr(), sd.data_ptr(), dd.data_ptr(), out.data_ptr(), n,
        n_experts, n * (k // 256) * 144, n, k, hint, s))
    got = out.cpu().numpy()
    want = np.empty_like(prod[0])
    want[dst_map] = prod[0]
    assert (np.abs(got - want) <= 1e-3 * np.abs(want) + 1e-4).all()
    # gate and up with SiLU, rows left in sorted order
    out2 = torch.full((rows, n), -9.0, device="cuda")
    lib.check("lk_moe_q4k_rows_grouped", L.lk_moe_q4k_rows_grouped(
        wd.data_ptr(), w2d.data_ptr(), 0, q.data_ptr(), k // 32, bd.data_ptr(), sd.data_ptr(), None, out2.data_ptr(), n,
        n_experts, n * (k // 256) * 144, n, k, hint, s))
    g, u = prod
    want2 = g / (1.0 + np.exp(-g)) * u
    got2 = out2.cpu().numpy()
    assert (np.abs(got2 - want2) <= 1e-3 * np.abs(want2) + 1e-4 * np.abs(want2).max()).all()
