"""Router-side launchers on the card: the fused gate mat-vec + softmax + top-k, the sigmoid
router and the stable sorts, against the oracle and numpy."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from loken_amd import moe, synth

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("tokens,hidden,experts,k,renorm", [(1, 2048, 128, 8, True), (16, 2048, 128, 8, True),
                                                            (256, 2048, 128, 8, False), (3, 4096, 64, 4, True),
                                                            (2, 1030, 32, 2, True), (5, 8192, 256, 8, True),
                                                            (2, 514, 40, 3, False), (17, 1028, 33, 4, True), (16, 36, 65, 5, True),
                                                            (97, 2048, 129, 8, True), (1111, 768, 512, 8, True)])
def test_gate_topk_softmax_matches_the_two_step_path(tokens, hidden, experts, k, renorm):
    x = synth.normal(20, 1, tokens * hidden).reshape(tokens, hidden)
    gate = (synth.normal(20, 2, experts * hidden) * (1.5 / np.sqrt(hidden))).reshape(experts, hidden).astype(np.float32)
    logits = x.astype(np.float64) @ gate.astype(np.float64).T
    want_ids, want_w = oracle.topk_softmax(logits.astype(np.float32), k, renorm)
    w, ids = moe.gate_topk_softmax(dev(x), dev(gate), k, renorm)
    w, ids = w.cpu().numpy(), ids.cpu().numpy()
    # a logit here is a 64-lane f32 sum: where two probabilities at the cut lie closer than that
    # rounding, either order is right; everywhere else the experts must be the oracle's
    p = np.exp(logits - logits.max(axis=1, keepdims=True))
    p /= p.sum(axis=1, keepdims=True)
    ranked = -np.sort(-p, axis=1)
    clear = (ranked[:, :k] - ranked[:, 1:k + 1]).min(axis=1) > 1e-5 * ranked[:, :1].ravel()
    assert clear.mean() > 0.9
    assert np.array_equal(ids[clear], want_ids[clear])
    assert np.abs(w[clear] - want_w[clear]).max() < 2e-5
    # the launch agrees with itself split in two: logits through the unfused router
    w2, ids2 = moe.topk_softmax(dev(logits.astype(np.float32)), k, renorm)
    assert np.array_equal(ids2.cpu().numpy()[clear], ids[clear])


NONE = 0x7FFFFFFF


def chosen_of(logits, k):
    """The selection's rule in numpy: probabilities that are numbers, largest first, ties to the lower id."""
    with np.errstate(invalid="ignore"):
        p = np.exp(logits - np.fmax.reduce(logits), dtype=np.float32)
    ids = [e for e in np.argsort(-p, kind="stable") if not np.isnan(p[e])][:k]
    return np.array(ids + [NONE] * (k - len(ids)), np.int32), bool(np.isnan(p).any())


@pytest.mark.parametrize("experts,k", [(5, 5), (40, 3), (64, 8), (100, 64), (128, 8), (200, 16), (512, 64)])
def test_logits_that_are_not_numbers_are_never_chosen_and_no_expert_twice(experts, k):
    base = synth.normal(28, experts, 8 * experts).reshape(8, experts).astype(np.float32)
    base[1, experts // 2] = np.nan
    base[2] = np.nan
    base[3, k // 2:] = np.nan                    # fewer numbers than choices
    base[4, 0] = np.inf                          # inf - inf: not a probability
    base[5] = -np.inf
    base[6, 1:] = -np.inf                        # one expert and zeros
    w, ids = moe.topk_softmax(dev(base), k, True)
    w, ids = w.cpu().numpy(), ids.cpu().numpy()
    for row in range(8):
        want, not_a_number = chosen_of(base[row], k)
        assert np.array_equal(ids[row], want), row
        assert np.isnan(w[row]).all() if not_a_number else np.isfinite(w[row]).all(), row


@pytest.mark.parametrize("tokens,experts,k", [(1, 40, 8), (16, 128, 8), (17, 33, 4), (40, 300, 8)])
@pytest.mark.parametrize("aligned", [True, False])   # in two launches, or one (rows that do not start on 16 bytes)
def test_gate_of_weights_and_tokens_that_are_not_numbers(tokens, experts, k, aligned):
    hidden = 128
    x = synth.normal(29, 1, tokens * hidden).reshape(tokens, hidden)
    gate = (0.1 * synth.normal(29, 2, experts * hidden)).reshape(experts, hidden).astype(np.float32)
    gate[k - 2:] = np.nan                        # fewer experts with a logit than choices
    if tokens > 1:
        x[3] = np.nan
    xd = torch.empty(tokens * hidden + 1, device="cuda")[0 if aligned else 1:][:tokens * hidden].view(tokens, hidden)
    xd.copy_(dev(x))
    w, ids = moe.gate_topk_softmax(xd, dev(gate), k, True)
    w, ids = w.cpu().numpy(), ids.cpu().numpy()
    assert np.isnan(w).all() and (ids[:, k - 2:] == NONE).all()
    for t in range(tokens):
        if t == 3:
            assert (ids[t] == NONE).all()
        else:
            assert sorted(ids[t, :k - 2].tolist()) == list(range(k - 2))


@pytest.mark.parametrize("tokens,experts,k,renorm,scale,with_bias", [(1, 256, 8, True, 2.5, True), (33, 128, 8, True, 1.0, False),
                                                                     (7, 64, 6, False, 1.0, True), (4, 40, 3, True, 0.5, True),
                                                                     (2, 512, 10, True, 1.0, True)])
def test_topk_sigmoid_post(tokens, experts, k, renorm, scale, with_bias):
    logits = synth.normal(21, 1, tokens * experts).reshape(tokens, experts) * 2.0
    bias = (0.2 * synth.normal(21, 2, experts)).astype(np.float32) if with_bias else None
    want_ids, want_w = oracle.topk_sigmoid(logits, k, bias=bias, renorm=renorm, scale=scale)
    w, ids = moe.topk_sigmoid_post(dev(logits), k, dev(bias) if with_bias else None, renorm, scale)
    assert np.array_equal(ids.cpu().numpy(), want_ids)
    assert np.abs(w.cpu().numpy() - want_w).max() <= 1e-6 * scale


def test_sigmoid_ties_and_floor():
    w, ids = moe.topk_sigmoid_post(dev(np.zeros((2, 64), np.float32)), 5)
    assert ids.cpu().numpy().tolist() == [[0, 1, 2, 3, 4]] * 2 and np.allclose(w.cpu().numpy(), 0.2)
    deep = np.full((1, 64), -30.0, np.float32)
    w, _ = moe.topk_sigmoid_post(dev(deep), 4)
    want_ids, want_w = oracle.topk_sigmoid(deep, 4)
    assert np.allclose(w.cpu().numpy(), want_w, rtol=1e-5)


@pytest.mark.parametrize("n,experts,small", [(1, 128, True), (8, 128, True), (32, 128, True), (200, 8, True), (257, 128, False),
                                              (2048, 128, False), (5000, 3, False), (4096, 100000, False)])
def test_stable_sorts_match_numpy(n, experts, small):
    keys = synth.rand_ints(22, n, n, experts).astype(np.uint32)
    got, order = moe.stable_sort_u32(dev(keys.view(np.int32)), small=small)
    want_order = np.argsort(keys, kind="stable")
    assert np.array_equal(order.cpu().numpy().view(np.uint32), want_order.astype(np.uint32))
    assert np.array_equal(got.cpu().numpy().view(np.uint32), keys[want_order])


@pytest.mark.parametrize("tokens,hidden,experts,k", [(1, 2048, 128, 8), (4, 2048, 128, 8), (5, 512, 17, 2), (4, 132, 512, 64), (2, 8192, 60, 4), (3, 64, 200, 1)])
def test_a_few_tokens_choose_alike_on_every_stream_and_in_graphs(tokens, hidden, experts, k):
    # up to four tokens one launch, whose workgroups count themselves in a counter of the stream: whatever ran before, it is at zero;
    # more tokens, and recorded calls, two launches with the same bits
    x, gate = dev(synth.normal(31, 1, tokens * hidden).reshape(tokens, hidden)), dev(synth.normal(31, 2, experts * hidden).reshape(experts, hidden) * 0.05)
    logits = x.double() @ gate.double().T
    want_w, want_ids = moe.topk_softmax(logits.float(), k)
    ranked = logits.softmax(1).sort(dim=1, descending=True).values
    gap = (ranked[:, :k] - ranked[:, 1:k + 1]).min() if k < experts else (ranked[:, :-1] - ranked[:, 1:]).min()
    first = moe.gate_topk_softmax(x, gate, k)
    if gap > 1e-5 * ranked.max():
        assert torch.equal(first[1], want_ids)
    assert (first[0].sort(dim=1).values - want_w.sort(dim=1).values).abs().max() < 2e-5
    streams = [torch.cuda.Stream() for _ in range(3)]
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side), torch.cuda.graph(graph, stream=side):
        recorded = moe.gate_topk_softmax(x, gate, k)
    torch.cuda.synchronize()
    for _ in range(4):
        graph.replay()
        results = []
        for s in streams:
            with torch.cuda.stream(s):
                results += [moe.gate_topk_softmax(x, gate, k), moe.gate_topk_softmax(x[:1], gate, k)]
        torch.cuda.synchronize()
        for w, ids in results:
            assert torch.equal(w, first[0][:w.shape[0]]) and torch.equal(ids, first[1][:w.shape[0]])
        assert torch.equal(recorded[0], first[0]) and torch.equal(recorded[1], first[1])
