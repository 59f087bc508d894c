"""Calls that work in the library's scratch memory, recorded into graphs: replays beside calls and other graphs on
streams that nothing orders against them, every one the eager bits."""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from loken_amd import lib, moe, synth
from test_gpu_host_mirror import Linear

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def record(fn, stream):
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            out = fn()
    return graph, out


def check_replays(calls, stream):
    """`calls`: functions of one operation over inputs of their own. The first two are recorded, both on `stream`, and
    replayed on two more while the last runs eagerly where all were warmed up and where they were recorded."""
    want = [fn() for fn in calls]
    torch.cuda.synchronize()
    graphs = [record(fn, stream) for fn in calls[:2]]
    c, d = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    for _ in range(4):
        for _, out in graphs:
            out.zero_()
        torch.cuda.synchronize()
        for _ in range(5):
            for (graph, _), s in zip(graphs, (c, d)):
                with torch.cuda.stream(s):
                    graph.replay()
            here = calls[2]()
            with torch.cuda.stream(stream):
                there = calls[2]()
        torch.cuda.synchronize()
        for got, w in zip([out for _, out in graphs] + [here, there], [want[0], want[1], want[2], want[2]]):
            assert torch.equal(got, w)


@pytest.mark.parametrize("tokens,topk,n_experts,hidden,ffn,gu,dn", [
    (2, 2, 16, 1024, 512, lib.TYPE_Q8_0, lib.TYPE_Q8_0),         # mat-vec per pair
    (64, 4, 16, 1024, 512, lib.TYPE_Q4_K, lib.TYPE_Q4_K),        # rows launches
    (200, 4, 8, 1024, 768, lib.TYPE_Q4_K, lib.TYPE_Q6_K)])       # tiles
def test_mixture_layer(tokens, topk, n_experts, hidden, ffn, gu, dn):
    gate, up = (dev(synth.weight(gu, n_experts * ffn, hidden, seed=70, stream=i)) for i in (1, 2))
    down = dev(synth.weight(dn, n_experts * hidden, ffn, seed=70, stream=3))
    router = dev((synth.normal(70, 4, n_experts * hidden) * 0.05).reshape(n_experts, hidden).astype(np.float32))
    L = lib.load()

    def layer(seed):
        x = dev(synth.activation(tokens, hidden, seed=seed))

        def call():
            w, ids = moe.gate_topk_softmax(x, router, topk)
            out = torch.empty((tokens, hidden), device="cuda")
            lib.check("lk_moe_forward", L.lk_moe_forward(
                gu, dn, x.data_ptr(), gate.data_ptr(), up.data_ptr(), down.data_ptr(), ids.data_ptr(), w.data_ptr(), out.data_ptr(),
                tokens, topk, n_experts, hidden, ffn, torch.cuda.current_stream().cuda_stream))
            return out
        return call

    check_replays([layer(seed) for seed in (71, 72, 73)], torch.cuda.Stream())


@pytest.mark.parametrize("wtype,n,k,rows,half", [(lib.TYPE_Q8_0, 300, 1024, 5, False), (lib.TYPE_Q4_K, 4096, 1024, 12, True),
                                                  (lib.TYPE_Q5_K, 600, 4096, 77, True), (lib.TYPE_Q4_K, 4096, 1024, 200, False)])
def test_linear(wtype, n, k, rows, half):
    lin = Linear(wtype, dev(synth.weight(wtype, n, k, seed=74, stream=1)), n, k)

    def call(seed):
        x = dev(synth.activation(rows, k, seed=seed)).to(torch.float16 if half else torch.float32)
        return lambda: lin(x)

    try:
        check_replays([call(seed) for seed in (75, 76, 77)], torch.cuda.Stream())
    finally:
        lin.close()


def test_every_capture_has_an_id_of_its_own():
    """What the library tells one recording from the next by, on one stream and on another."""
    hip = C.CDLL("libamdhip64.so")
    x, sides, ids = torch.zeros(8, device="cuda"), [torch.cuda.Stream(), torch.cuda.Stream()], []

    def body(stream):
        x.add_(1.0)
        for s in (stream, torch.cuda.default_stream()):
            status, at = C.c_int(-1), C.c_ulonglong(0)
            assert hip.hipStreamGetCaptureInfo(C.c_void_p(s.cuda_stream), C.byref(status), C.byref(at)) == 0
            assert status.value == (1 if s is stream else 0)
            if s is stream:
                ids.append(at.value)

    keep = [record(lambda: body(side), side) for side in sides + sides]
    assert len(keep) == len(set(ids)) == 4


def test_scratch_that_grows_after_a_recording():
    """A graph keeps what it was recorded with, whatever the streams' buffers become."""
    wtype, n, k = lib.TYPE_Q4_K, 640, 2048
    lin = Linear(wtype, dev(synth.weight(wtype, n, k, seed=78, stream=1)), n, k)
    x = dev(synth.activation(20, k, seed=78))
    side = torch.cuda.Stream()
    want = lin(x)
    graph, out = record(lambda: lin(x), side)
    for rows in (100, 300, 900):
        big = dev(synth.activation(rows, k, seed=79))
        with torch.cuda.stream(side):
            there = lin(big)
        here = lin(big)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(here, there)
    lin.close()


@pytest.mark.parametrize("wtype,n,k,rows", [(lib.TYPE_Q4_K, 2986, 6144, 26), (lib.TYPE_Q6_K, 2048, 6912, 48), (lib.TYPE_Q5_K, 1152, 4864, 40)])
def test_a_linear_recorded_after_larger_calls_alone_runs_in_their_buffers(wtype, n, k, rows):
    """Rows kernels and tiles work in different buffers: where only calls on the tiles ran before, the tiles serve the recorded one."""
    w = synth.weight(wtype, 64, k, seed=82, stream=1).reshape(64, -1).repeat((n + 63) // 64, axis=0)[:n]
    x = synth.activation(rows, k, seed=82)
    lin, xd = Linear(wtype, dev(w), n, k), dev(x)
    lib.load().lkh_release_workspaces()
    lib.load().loken_stream_scratch_release()
    lin(dev(synth.activation(700, k, seed=83)))
    assert lin.path == "tiled"
    graph, out = record(lambda: lin(xd), torch.cuda.Stream())
    assert lin.path == "tiled"
    eager = lin(xd)
    assert lin.path == "rows-on-matrix-unit"
    ends = np.r_[:20, n - 20:n]
    want = oracle.ob_matmul(wtype, x, w[ends], len(ends))
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert (np.abs(out.cpu().numpy()[:, ends] - want) <= 1e-3 * np.abs(want) + 1e-4).all()
        assert (out - eager).abs().max() <= 2e-5 * eager.abs().max()
    lin.close()


@pytest.mark.parametrize("gu,dn,tokens,n_experts,hidden,ffn", [(lib.TYPE_Q4_K, lib.TYPE_Q4_K, 15, 8, 512, 256), (lib.TYPE_Q8_0, lib.TYPE_Q8_0, 24, 8, 512, 256),
                                                               (lib.TYPE_MXFP4, lib.TYPE_MXFP4, 9, 6, 256, 512), (lib.TYPE_Q5_K, lib.TYPE_Q5_K, 1, 8, 512, 512)])
def test_a_block_recorded_after_larger_calls_alone_runs_in_their_buffers(gu, dn, tokens, n_experts, hidden, ffn):
    """A block of few pairs works in another buffer than a batched one, unless down and fold are one launch: where only batched
    blocks ran before, the batched launches serve the recorded one."""
    topk = 2
    gate, up = (dev(synth.weight(gu, n_experts * ffn, hidden, seed=84, stream=i)) for i in (1, 2))
    down = dev(synth.weight(dn, n_experts * hidden, ffn, seed=84, stream=3))
    L = lib.load()

    def call(tokens, seed):
        ids, w = oracle.topk_softmax(synth.activation(tokens, n_experts, seed=seed, stream=7), topk)
        x, ids, w = dev(synth.activation(tokens, hidden, seed=seed)), dev(ids), dev(w)

        def run():
            out = torch.empty((tokens, hidden), device="cuda")
            lib.check("lk_moe_forward", L.lk_moe_forward(gu, dn, x.data_ptr(), gate.data_ptr(), up.data_ptr(), down.data_ptr(), ids.data_ptr(), w.data_ptr(),
                                                         out.data_ptr(), tokens, topk, n_experts, hidden, ffn, torch.cuda.current_stream().cuda_stream))
            return out
        return run

    assert not L.lk_moe_block_path(gu, dn, tokens, topk, n_experts, hidden, ffn) & lib.MOE_GROUPED
    assert L.lk_moe_block_path(gu, dn, 300, topk, n_experts, hidden, ffn) & lib.MOE_GROUPED
    L.loken_stream_scratch_release()
    call(300, 85)()
    small = call(tokens, 86)
    graph, out = record(small, torch.cuda.Stream())
    eager = small()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert ((out - eager).abs() <= 1e-3 * eager.abs() + 1e-3 * eager.abs().max()).all()


@pytest.mark.parametrize("wtype,n,k,rows,most", [(lib.TYPE_Q4_K, 4096, 4096, 200, 16), (lib.TYPE_Q6_K, 1186, 10240, 1661, 32)])
def test_a_recorded_tiled_linear_holds_what_its_partial_products_need(wtype, n, k, rows, most):
    """16 MiB beside the operands, 32 where the plan cuts K of a product of many rows and columns: the eager call's plan, and its bits."""
    L = lib.load()
    blob = dev(synth.weight(wtype, 2, k, seed=87, stream=1)).reshape(2, -1).repeat(n // 2, 1)
    lin, x = Linear(wtype, blob, n, k), dev(synth.activation(200, k, seed=87)).repeat(9, 1)[:rows].contiguous()
    want, out = lin(x), torch.empty((rows, n), device="cuda")
    assert lin.path == "tiled"

    def call():
        lib.check("forward", L.lkh_qkernel_matmul_forward(lin.h, x.data_ptr(), lib.TYPE_F32, rows, out.data_ptr(), torch.cuda.current_stream().cuda_stream, 0))

    side, graphs = torch.cuda.Stream(), []
    graphs.append(record(call, side)[0])
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    for _ in range(4):
        graphs.append(record(call, side)[0])
    torch.cuda.synchronize()
    operands = (rows + 128) * (k // 256) * 592 * 5 / 4
    assert free - torch.cuda.mem_get_info()[0] <= 4 * (operands + (most + 6 << 20))
    for graph in graphs:
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    lin.close()
    L.lkh_release_workspaces()
    L.loken_stream_scratch_release()


def test_dropping_the_linears_workspaces_leaves_the_mixtures_graph():
    tokens, topk, n_experts, hidden, ffn = 64, 4, 8, 512, 256
    gate, up = (dev(synth.weight(lib.TYPE_Q6_K, n_experts * ffn, hidden, seed=81, stream=i)) for i in (1, 2))
    down = dev(synth.weight(lib.TYPE_Q6_K, n_experts * hidden, ffn, seed=81, stream=3))
    ids, w = oracle.topk_softmax(synth.activation(tokens, n_experts, seed=81, stream=7), topk)
    args = (lib.TYPE_Q6_K, lib.TYPE_Q6_K, dev(synth.activation(tokens, hidden, seed=81)), gate, up, down, dev(ids), dev(w), n_experts, ffn)
    want = moe.moe_forward(*args)
    graph, out = record(lambda: moe.moe_forward(*args), torch.cuda.Stream())
    for _ in range(3):
        lib.load().lkh_release_workspaces()
        filler = torch.full((64 << 20,), 7.0, device="cuda")   # over what a release of too much would have given back
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and (filler == 7.0).all()
        del filler
        torch.cuda.empty_cache()


def test_router_recorded_before_any_call_takes_its_form_without_scratch():
    lib.load().loken_stream_scratch_release()
    x = dev(synth.activation(9, 512, seed=80))
    gate = dev((synth.normal(80, 2, 64 * 512) * 0.05).reshape(64, 512).astype(np.float32))
    graph, (w, ids) = record(lambda: moe.gate_topk_softmax(x, gate, 4), torch.cuda.Stream())
    want_ids, want_w = oracle.topk_softmax((x.double() @ gate.double().T).float().cpu().numpy(), 4)
    for _ in range(3):
        ids.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(ids.cpu().numpy(), want_ids) and np.abs(w.cpu().numpy() - want_w).max() < 2e-5
