"""Calls through the library's scratch memory from many streams and several host threads: more streams than hold
buffers of their own, threads that share a stream, threads with one each. Every result the bits of a call alone."""
import ctypes as C
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from loken_amd import lib, moe, synth
from test_gpu_host_mirror import Linear

pytestmark = pytest.mark.gpu
OWN_STREAMS = 32   # LK_SCRATCH_STREAMS


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.fixture
def streams():
    """Non-blocking streams of the default priority, past what torch's pool hands out; the scratch they used goes with them."""
    hip = C.CDLL("libamdhip64.so")
    made = []

    def make(count):
        for _ in range(count):
            h = C.c_void_p()
            assert hip.hipStreamCreateWithFlags(C.byref(h), 1) == 0
            made.append(h.value)
        return list(made)

    yield make
    torch.cuda.synchronize()
    lib.load().loken_stream_scratch_release()
    lib.load().lkh_release_workspaces()
    for h in made:
        assert hip.hipStreamDestroy(C.c_void_p(h)) == 0


def linear_work(count, seed):
    """(call on a stream handle -> output, expected) per index, over inputs of their own; two kernels' worth of scratch."""
    lins = [Linear(lib.TYPE_Q8_0, dev(synth.weight(lib.TYPE_Q8_0, 300, 1024, seed=seed, stream=1)), 300, 1024),
            Linear(lib.TYPE_Q6_K, dev(synth.weight(lib.TYPE_Q6_K, 640, 2048, seed=seed, stream=2)), 640, 2048)]
    work = []
    for i in range(count):
        lin = lins[i % 2]
        x = dev(synth.activation((5, 70)[i % 2], lin.k, seed=seed + i))
        work.append((lin, x, lin(x), torch.empty((x.shape[0], lin.n), device="cuda")))
    torch.cuda.synchronize()

    def call(i, stream):
        lin, x, _, out = work[i]
        lib.check("forward", lib.load().lkh_qkernel_matmul_forward(lin.h, x.data_ptr(), lib.TYPE_F32, x.shape[0], out.data_ptr(), stream, 0))

    def check():
        torch.cuda.synchronize()
        for lin, x, want, out in work:
            assert torch.equal(out, want)
            out.zero_()
        torch.cuda.synchronize()

    return call, check, lambda: [lin.close() for lin in lins]


def test_more_streams_than_hold_buffers(streams):
    lib.load().lkh_release_workspaces()
    lib.load().loken_stream_scratch_release()
    handles = streams(OWN_STREAMS + 5)
    call, check, close = linear_work(len(handles), 90)
    for _ in range(4):
        for _ in range(3):
            for i, s in enumerate(handles):
                call(i, s)
        check()
    close()


@pytest.mark.parametrize("shared", [True, False])
def test_threads(streams, shared):
    threads = 6
    handles = streams(threads)
    call, check, close = linear_work(threads, 91)
    failed = []

    def body(i):
        try:
            for _ in range(60):
                call(i, handles[0 if shared else i])
        except Exception as e:   # noqa: BLE001 -- reported by the test's own thread
            failed.append(e)

    for _ in range(2):
        running = [threading.Thread(target=body, args=(i,)) for i in range(threads)]
        for t in running:
            t.start()
        for t in running:
            t.join()
        assert not failed, failed
        check()
    close()


def test_mixture_layers_of_two_threads_on_one_stream(streams):
    tokens, topk, n_experts, hidden, ffn, wt = 40, 4, 8, 512, 256, lib.TYPE_Q6_K
    gate, up = (dev(synth.weight(wt, n_experts * ffn, hidden, seed=92, stream=i)) for i in (1, 2))
    down = dev(synth.weight(wt, n_experts * hidden, ffn, seed=92, stream=3))
    L, handle = lib.load(), streams(1)[0]
    work = []
    for i in range(2):
        ids, w = oracle.topk_softmax(synth.activation(tokens, n_experts, seed=93 + i, stream=7), topk)
        a = (dev(synth.activation(tokens, hidden, seed=93 + i)), dev(ids), dev(w))
        want = moe.moe_forward(wt, wt, a[0], gate, up, down, a[1], a[2], n_experts, ffn)
        work.append((a, want, torch.zeros_like(want)))
    torch.cuda.synchronize()
    codes = []

    def body(i):
        (x, ids, w), _, out = work[i]
        for _ in range(60):
            codes.append(L.lk_moe_forward(wt, wt, x.data_ptr(), gate.data_ptr(), up.data_ptr(), down.data_ptr(), ids.data_ptr(),
                                          w.data_ptr(), out.data_ptr(), tokens, topk, n_experts, hidden, ffn, handle))

    running = [threading.Thread(target=body, args=(i,)) for i in range(2)]
    for t in running:
        t.start()
    for t in running:
        t.join()
    torch.cuda.synchronize()
    assert set(codes) == {lib.LK_OK}
    for _, want, out in work:
        assert torch.equal(out, want)


def test_a_call_that_grows_beside_a_recording_thread(streams):
    """Another stream's call may allocate, and free what it outgrew, while this thread records: the recording stands."""
    wtype, n, k = lib.TYPE_Q6_K, 640, 2048
    lin = Linear(wtype, dev(synth.weight(wtype, n, k, seed=95, stream=1)), n, k)
    handle = streams(1)[0]
    lib.load().lkh_release_workspaces()
    sizes = (20, 60, 200, 700)
    xs = [dev(synth.activation(rows, k, seed=95)) for rows in sizes]
    want = [lin(x) for x in xs]
    outs = [torch.empty_like(w) for w in want]
    x0 = xs[0].clone()
    graph, out, codes = torch.cuda.CUDAGraph(), torch.empty_like(want[0]), []
    side = torch.cuda.Stream()
    torch.cuda.synchronize()

    def grow():
        for x, o in zip(xs, outs):
            codes.append(lib.load().lkh_qkernel_matmul_forward(lin.h, x.data_ptr(), lib.TYPE_F32, x.shape[0], o.data_ptr(), handle, 0))

    other = Linear(wtype, lin.w, n, k)
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            for at in range(2):
                lib.check("forward", lib.load().lkh_qkernel_matmul_forward(other.h, x0.data_ptr(), lib.TYPE_F32, sizes[0], out.data_ptr(),
                                                                           side.cuda_stream, 0))
                if at == 0:
                    t = threading.Thread(target=grow)
                    t.start()
                    t.join()
    torch.cuda.synchronize()
    assert codes == [lib.LK_OK] * len(sizes)
    for o, w in zip(outs, want):
        assert torch.equal(o, w)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want[0])
    lin.close()
    other.close()
