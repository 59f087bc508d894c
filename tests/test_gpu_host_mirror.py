"""The C++ host mirror of QKernelMatMul (include/loken_host.hpp) through its C symbols: path chosen
by row count, results equal to the launchers called one by one, workspace rules."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from loken_amd import lib, ops, synth

pytestmark = pytest.mark.gpu

DT = {"q4_k": lib.TYPE_Q4_K, "q5_k": lib.TYPE_Q5_K, "q6_k": lib.TYPE_Q6_K, "q8_0": lib.TYPE_Q8_0,
      "q4_0": lib.TYPE_Q4_0, "q4_1": lib.TYPE_Q4_1, "q5_0": lib.TYPE_Q5_0, "q5_1": lib.TYPE_Q5_1, "iq4_nl": lib.TYPE_IQ4_NL, "mxfp4": lib.TYPE_MXFP4, "q2_k": lib.TYPE_Q2_K, "q3_k": lib.TYPE_Q3_K}
PATH = {1: "matvec-fused", 2: "matvec", 3: "rows-on-matrix-unit", 4: "tiled"}
X_TYPES = {torch.float32: lib.TYPE_F32, torch.float16: lib.TYPE_F16, torch.bfloat16: lib.TYPE_BF16}


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


class Linear:
    def __init__(self, wtype, w, n, k):
        self.l = lib.load()
        self.w = w   # keeps the blob alive
        self.n, self.k = n, k
        self.h = self.l.lkh_qkernel_matmul_new(wtype, n, k, w.data_ptr(), torch.cuda.current_device())

    def __call__(self, x, decode_order=False, stream=None):
        out = torch.empty((x.shape[0], self.n), dtype=x.dtype, device=x.device)
        s = stream if stream is not None else torch.cuda.current_stream().cuda_stream
        rc = self.l.lkh_qkernel_matmul_forward(self.h, x.data_ptr(), X_TYPES[x.dtype], x.shape[0], out.data_ptr(), s,
                                               int(decode_order))
        if rc:
            raise lib.LokenError("lkh_qkernel_matmul_forward", rc)
        return out

    @property
    def path(self):
        return PATH.get(self.l.lkh_qkernel_matmul_last_path(self.h), "none")

    def close(self):
        self.l.lkh_qkernel_matmul_free(self.h)


def close(got, want, rtol=1e-3, atol=1e-4):
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    return bool((np.abs(got - want) <= rtol * np.abs(want) + atol).all())


@pytest.mark.parametrize("name,rows,n,expect", [
    ("q4_k", 1, 200, "matvec-fused"), ("q4_k", 2, 200, "matvec-fused"), ("q4_k", 5, 200, "matvec"),
    ("q4_k", 8, 200, "matvec"), ("q4_k", 9, 200, "rows-on-matrix-unit"), ("q4_k", 40, 200, "rows-on-matrix-unit"),
    # a handful of rows over a matrix large enough to pay for staging them in every workgroup
    ("q4_k", 2, 4000, "matvec-fused"), ("q4_k", 3, 4000, "rows-on-matrix-unit"), ("q4_k", 8, 1100, "rows-on-matrix-unit"),
    ("q5_k", 4, 2100, "rows-on-matrix-unit"), ("q5_k", 4, 2000, "rows-on-matrix-unit"), ("q4_k", 3, 300, "rows-on-matrix-unit"), ("q6_k", 5, 256, "rows-on-matrix-unit"),
    # above 16 rows the rows kernel keeps a matrix too small to fill the chip with tiles (n x rows up to 450 thousand)
    ("q4_k", 80, 200, "rows-on-matrix-unit"), ("q4_k", 80, 24000, "tiled"),
    ("q6_k", 1, 200, "matvec-fused"), ("q6_k", 8, 200, "matvec"), ("q6_k", 20, 200, "rows-on-matrix-unit"),
    ("q6_k", 40, 200, "rows-on-matrix-unit"), ("q6_k", 200, 24000, "tiled"),
    ("q8_0", 3, 200, "matvec"), ("q8_0", 16, 200, "matvec"), ("q8_0", 17, 200, "tiled"), ("q5_k", 1, 200, "matvec-fused"), ("q5_k", 8, 200, "matvec"),
    ("q5_k", 20, 200, "rows-on-matrix-unit"), ("q5_k", 200, 200, "rows-on-matrix-unit"), ("q5_k", 80, 24000, "tiled"), ("q5_k", 18, 24000, "rows-on-matrix-unit"),
    ("q4_0", 1, 200, "matvec"), ("q4_0", 12, 200, "matvec"), ("q5_1", 9, 200, "matvec"), ("iq4_nl", 3, 200, "matvec"),
    # four of the 32-value formats have tiles: from 16 rows, or from 9 over 48 M weights
    ("q4_0", 50, 200, "tiled"), ("q5_0", 16, 200, "tiled"), ("q5_1", 30, 12000, "tiled"), ("q4_1", 12, 12000, "matvec"),
    ("q4_0", 9, 49152, "tiled"),
    ("q4_1", 130, 300, "tiled"), ("iq4_nl", 60, 200, "matvec"), ("q3_k", 41, 200, "tiled"), ("q3_k", 17, 12000, "tiled"),
    ("q2_k", 50, 200, "tiled"),
    ("mxfp4", 17, 200, "matvec"), ("q2_k", 12, 200, "matvec"), ("q3_k", 1, 200, "matvec")])
def test_forward_takes_the_path_of_its_row_count_and_matches_the_oracle(name, rows, n, expect):
    wtype, k = DT[name], 1024
    w = synth.weight(wtype, n, k, seed=80, stream=1)
    x = synth.activation(rows, k, seed=80)
    lin = Linear(wtype, dev(w), n, k)
    try:
        got = lin(dev(x))
        assert lin.path == expect
        pick = np.arange(n) if n <= 400 else np.sort(np.random.default_rng(80).choice(n, 300, replace=False))
        assert close(got.cpu().numpy()[:, pick], oracle.ob_matmul(wtype, x, w[pick], len(pick)))
    finally:
        lin.close()


def test_decode_order_keeps_every_row_on_the_matvec_family_and_rows_independent():
    wtype, n, k = lib.TYPE_Q4_K, 300, 2048
    w = dev(synth.weight(wtype, n, k, seed=81, stream=1))
    x = dev(synth.activation(20, k, seed=81))
    lin = Linear(wtype, w, n, k)
    try:
        batch = lin(x, decode_order=True)
        assert lin.path == "matvec"
        q = ops.quantize_q8_1_rows(x)
        for r in (0, 7, 8, 19):
            assert torch.equal(batch[r:r + 1], ops.mmvq(wtype, w, q[r:r + 1], k, n))
    finally:
        lin.close()


def test_half_inputs_stay_in_their_type_on_the_matvec_family():
    wtype, n, k = lib.TYPE_Q6_K, 64, 512
    w = dev(synth.weight(wtype, n, k, seed=82, stream=1))
    lin = Linear(wtype, w, n, k)
    try:
        x = dev(synth.activation(3, k, seed=82)).to(torch.bfloat16)
        y = lin(x)
        assert y.dtype == torch.bfloat16 and lin.path == "matvec"
        want = ops.mmvq(wtype, w, ops.quantize_q8_1_rows(x), k, n, out_dtype=torch.bfloat16)
        assert torch.equal(y, want)
    finally:
        lin.close()


# every kernel that stores in the rows' type itself, at ragged row counts: 16- and 32-row tiles, int8 tiles whole and
# with K cut, f16 tiles, the wide ones
@pytest.mark.parametrize("half", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("name,rows,n,k", [
    ("q4_k", 12, 2050, 1024), ("q4_k", 12, 70, 1280), ("q5_k", 24, 2051, 1024), ("q6_k", 12, 1030, 2048), ("q6_k", 40, 601, 2048),
    ("q6_k", 24, 601, 1280), ("q6_k", 9, 601, 1280), ("q8_0", 70, 1027, 512), ("q8_0", 70, 1028, 1024), ("q8_0", 200, 12289, 256),
    ("q4_k", 150, 4099, 1024), ("q6_k", 200, 4099, 512), ("q5_k", 130, 16387, 256), ("q4_k", 512, 9001, 256), ("q4_1", 33, 201, 512)])
def test_half_rows_are_the_f32_rows_rounded_once(name, rows, n, k, half):
    w = dev(synth.weight(DT[name], n, k, seed=84, stream=rows))
    lin = Linear(DT[name], w, n, k)
    x = dev(synth.activation(rows, k, seed=84)).to(half)
    want = lin(x.float())
    path = lin.path
    got = lin(x)
    assert lin.path == path and torch.equal(got, want.to(half))
    lin.close()


@pytest.mark.parametrize("half", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("name,rows,n,expect", [
    ("q6_k", 50, 64, "rows-on-matrix-unit"), ("q4_k", 20, 200, "rows-on-matrix-unit"), ("q4_k", 4, 4000, "rows-on-matrix-unit"),
    ("q4_k", 130, 24000, "tiled"), ("q4_k", 300, 6000, "tiled"), ("q6_k", 200, 24000, "tiled"), ("q8_0", 40, 200, "tiled"),
    ("q5_1", 60, 200, "tiled"), ("q5_k", 90, 24000, "tiled")])
def test_half_rows_above_the_matvec_family_follow_the_oracle_and_leave_in_their_type(name, rows, n, expect, half):
    # the reference's forward serves f16 / bf16 rows at every row count and returns their type
    # (src/tensor/quantized/kernel_matmul.rs:1086-1714): the oracle is fed the values the rows hold, and
    # the result is the f32 call's result rounded once to the narrow type
    wtype, k = DT[name], 1024
    w = synth.weight(wtype, n, k, seed=83, stream=1)
    xh = dev(synth.activation(rows, k, seed=83)).to(half)
    x_seen = xh.to(torch.float32)
    lin = Linear(wtype, dev(w), n, k)
    try:
        got = lin(xh)
        assert got.dtype == half and lin.path == expect
        wide = lin(x_seen)
        assert lin.path == expect
        assert torch.equal(got, wide.to(half))
        pick = np.arange(n) if n <= 400 else np.sort(np.random.default_rng(83).choice(n, 300, replace=False))
        want = oracle.ob_matmul(wtype, x_seen.cpu().numpy(), w[pick], len(pick))
        eps = 2.0 ** -8 if half == torch.bfloat16 else 2.0 ** -11   # one rounding to the narrow type
        gotf = got.to(torch.float32).cpu().numpy()[:, pick].astype(np.float64)
        assert (np.abs(gotf - want) <= (1e-3 + eps) * np.abs(want) + 1e-4).all()
    finally:
        lin.close()


def test_workspace_grows_outside_a_capture_only_and_replays_then():
    # twenty rows: up to sixteen over a matrix like this are quantized in the launch and need no workspace
    wtype, n, k = lib.TYPE_Q4_K, 128, 1024
    w = dev(synth.weight(wtype, n, k, seed=83, stream=1))
    lin = Linear(wtype, w, n, k)
    lib.load().lkh_release_workspaces()
    try:
        x = dev(synth.activation(20, k, seed=83))
        side = torch.cuda.Stream()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(side):
            with pytest.raises(lib.LokenError) as err:      # nothing reserved yet: refused while recording
                with torch.cuda.graph(graph, stream=side):
                    lin(x, stream=side.cuda_stream)
            assert "LK_ERR_NOMEM" in str(err.value)
        torch.cuda.synchronize()
        eager = lin(x)                                       # reserves the workspace
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        out = torch.empty((20, n), device="cuda")
        with torch.cuda.stream(side):
            with torch.cuda.graph(graph, stream=side):
                rc = lib.load().lkh_qkernel_matmul_forward(lin.h, x.data_ptr(), lib.TYPE_F32, 20, out.data_ptr(),
                                                           side.cuda_stream, 0)
                assert rc == 0
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, eager)
    finally:
        lin.close()


def test_argument_errors_are_status_codes():
    l = lib.load()
    assert l.lkh_matvec_rows(lib.TYPE_Q4_K, 4096) == 8 and l.lkh_matvec_rows(lib.TYPE_Q6_K, 4096) == 8
    assert l.lkh_matvec_rows(lib.TYPE_Q8_0, 4096) == 16
    h = l.lkh_qkernel_matmul_new(99, 8, 256, 16, 0)
    assert l.lkh_qkernel_matmul_forward(h, 16, lib.TYPE_F32, 1, 16, None, 0) == lib.LK_ERR_TYPE
    l.lkh_qkernel_matmul_free(h)
    h = l.lkh_qkernel_matmul_new(lib.TYPE_Q4_K, 8, 250, 16, 0)
    assert l.lkh_qkernel_matmul_forward(h, 16, lib.TYPE_F32, 1, 16, None, 0) == lib.LK_ERR_ARG
    assert l.lkh_qkernel_matmul_forward(h, 16, lib.TYPE_F32, 0, 16, None, 0) == lib.LK_OK
    l.lkh_qkernel_matmul_free(h)


def test_rows_too_long_for_the_matrix_unit_rows_kernel_go_to_the_tiles():
    # 12 rows of 40960 values: the rows kernel's scale tables do not fit LDS; the call must end on the
    # tiled matmul with a written buffer, and the direct wrapper must raise instead of returning
    wtype, n, k, rows = lib.TYPE_Q4_K, 64, 40960, 12
    w = synth.weight(wtype, n, k, seed=84, stream=1)
    x = synth.activation(rows, k, seed=84)
    lin = Linear(wtype, dev(w), n, k)
    try:
        out = torch.full((rows, n), float("nan"), device="cuda")
        rc = lib.load().lkh_qkernel_matmul_forward(lin.h, dev(x).data_ptr(), lib.TYPE_F32, rows, out.data_ptr(),
                                                   torch.cuda.current_stream().cuda_stream, 0)
        assert rc == 0 and lin.path == "tiled"
        # 160 blocks per row summed one after the other in f32: held to the row scale, not element by
        # element (the test is about which kernel ran and that it wrote the buffer)
        want = oracle.ob_matmul(wtype, x, w, n)
        assert np.abs(out.cpu().numpy() - want).max() <= 1e-5 * np.abs(want).max() + 1e-4
    finally:
        lin.close()
    with pytest.raises(lib.LokenError):
        ops.dense_q4k_rows(dev(w), dev(x), n)


@pytest.mark.parametrize("name,rows,n", [("q4_k", 1, 300), ("q4_k", 2, 300), ("q4_k", 7, 300), ("q6_k", 5, 260), ("q8_0", 12, 200),
                                        ("q5_k", 1, 130), ("q4_0", 6, 200), ("q3_k", 3, 200)])
@pytest.mark.parametrize("xt", [torch.float32, torch.float16])
def test_an_activation_quantized_once_serves_several_weights_with_the_bits_of_forward(name, rows, n, xt):
    # quantize_for_matvec / forward_quantized of the reference (src/tensor/quantized/kernel_matmul.rs:695-812):
    # the Q8_1 rows are made once and every weight over them returns what its own forward returns
    l = lib.load()
    wtype, k = DT[name], 1024
    lins = [Linear(wtype, dev(synth.weight(wtype, n + 8 * i, k, seed=90 + i, stream=1)), n + 8 * i, k) for i in range(2)]
    x = dev(synth.activation(rows, k, seed=90)).to(xt)
    q81 = torch.empty(l.lkh_quantized_activation_bytes(k, rows), dtype=torch.uint8, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    try:
        assert l.lkh_qkernel_matmul_quantize_for_matvec(lins[0].h, x.data_ptr(), X_TYPES[xt], rows, q81.data_ptr(), s, 0) == 0
        for lin in lins:
            out = torch.empty((rows, lin.n), dtype=xt, device="cuda")
            assert l.lkh_qkernel_matmul_forward_quantized(lin.h, q81.data_ptr(), X_TYPES[xt], rows, out.data_ptr(), s, 0) == 0
            path = lin.path
            assert torch.equal(out, lin(x))
            assert path == ("matvec" if rows <= 2 else lin.path)   # (one or two rows: forward quantizes them in the mat-vec launch)
    finally:
        for lin in lins:
            lin.close()


def test_a_pair_of_weights_over_one_quantized_row_in_one_launch():
    # forward_quantized_pair (kernel_matmul.rs:814-876): one f32-born row, two weights of one format and k
    l = lib.load()
    k = 2048
    a = Linear(lib.TYPE_Q4_K, dev(synth.weight(lib.TYPE_Q4_K, 520, k, seed=91, stream=1)), 520, k)
    b = Linear(lib.TYPE_Q4_K, dev(synth.weight(lib.TYPE_Q4_K, 136, k, seed=92, stream=1)), 136, k)
    c = Linear(lib.TYPE_Q6_K, dev(synth.weight(lib.TYPE_Q6_K, 136, k, seed=93, stream=1)), 136, k)
    x = dev(synth.activation(1, k, seed=91))
    q81 = torch.empty(l.lkh_quantized_activation_bytes(k, 1), dtype=torch.uint8, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    try:
        assert l.lkh_qkernel_matmul_quantize_for_matvec(a.h, x.data_ptr(), lib.TYPE_F32, 1, q81.data_ptr(), s, 0) == 0
        oa, ob = torch.empty((1, 520), device="cuda"), torch.empty((1, 136), device="cuda")
        assert l.lkh_qkernel_matmul_forward_quantized_pair(a.h, b.h, q81.data_ptr(), oa.data_ptr(), ob.data_ptr(), s) == 0
        assert torch.equal(oa, a(x)) and torch.equal(ob, b(x))
        # two formats do not pair: the reference's None
        assert l.lkh_qkernel_matmul_forward_quantized_pair(a.h, c.h, q81.data_ptr(), oa.data_ptr(), ob.data_ptr(), s) == lib.LK_NOT_TAKEN
    finally:
        for lin in (a, b, c):
            lin.close()


def test_rows_that_forward_serves_another_way_are_not_quantized_for_the_matvec():
    l = lib.load()
    s = torch.cuda.current_stream().cuda_stream
    k = 1024
    x = dev(synth.activation(40, k, seed=94))
    q81 = torch.empty(l.lkh_quantized_activation_bytes(k, 40), dtype=torch.uint8, device="cuda")
    out = torch.empty((40, 4000), device="cuda")
    big = Linear(lib.TYPE_Q4_K, dev(synth.weight(lib.TYPE_Q4_K, 4000, k, seed=94, stream=1)), 4000, k)
    try:
        # 40 rows go to the matrix-unit kernels, 4 rows over this matrix to the 16-row tiles
        for rows in (40, 4):
            assert l.lkh_qkernel_matmul_quantize_for_matvec(big.h, x.data_ptr(), lib.TYPE_F32, rows, q81.data_ptr(), s, 0) == lib.LK_NOT_TAKEN
            assert l.lkh_qkernel_matmul_forward_quantized(big.h, q81.data_ptr(), lib.TYPE_F32, rows, out.data_ptr(), s, 0) == lib.LK_NOT_TAKEN
        # in decode order every row count stays on the mat-vec kernels
        assert l.lkh_qkernel_matmul_quantize_for_matvec(big.h, x.data_ptr(), lib.TYPE_F32, 40, q81.data_ptr(), s, 1) == 0
        assert l.lkh_qkernel_matmul_forward_quantized(big.h, q81.data_ptr(), lib.TYPE_F32, 40, out.data_ptr(), s, 1) == 0
        assert torch.equal(out, big(x, decode_order=True))
        assert l.lkh_qkernel_matmul_quantize_for_matvec(big.h, x.data_ptr(), 77, 2, q81.data_ptr(), s, 0) == lib.LK_ERR_TYPE
        assert l.lkh_qkernel_matmul_quantize_for_matvec(big.h, None, lib.TYPE_F32, 2, q81.data_ptr(), s, 0) == lib.LK_ERR_ARG
    finally:
        big.close()


@pytest.mark.parametrize("name,rows,n,k,expect", [
    ("q4_k", 12, 2048, 8192, "rows-on-matrix-unit"), ("q5_k", 16, 2048, 8192, "rows-on-matrix-unit"), ("q6_k", 12, 2048, 8192, "rows-on-matrix-unit"),
    ("q4_k", 8, 2048, 8192, "matvec"), ("q5_k", 9, 2288, 7680, "rows-on-matrix-unit"), ("q4_k", 16, 8200, 8192, "tiled")])
def test_long_rows_at_nine_to_sixteen_activation_rows(name, rows, n, k, expect):
    # Q4_K / Q5_K: the 16-row tiles up to 8192 matrix rows (2048 x 8192 at 12 rows 9.2 us, the tiled matmul with K cut 17.0), the tiled
    # matmul past them
    wtype = DT[name]
    w = synth.weight(wtype, n, k, seed=96, stream=1)
    x = synth.activation(rows, k, seed=96)
    lin = Linear(wtype, dev(w), n, k)
    try:
        got = lin(dev(x))
        assert lin.path == expect
        pick = np.sort(np.random.default_rng(96).choice(n, 200, replace=False))
        assert close(got.cpu().numpy()[:, pick], oracle.ob_matmul(wtype, x, w[pick], len(pick)))
    finally:
        lin.close()


@pytest.mark.parametrize("name,k,rows,expect", [("q4_k", 8192, 17, "tiled"), ("q5_k", 8192, 32, "tiled"), ("q4_k", 8192, 33, "tiled"),
                                                 ("q4_k", 12288, 33, "tiled"), ("q6_k", 8192, 32, "rows-on-matrix-unit"),
                                                 ("q6_k", 8192, 33, "tiled")])
def test_long_rows_above_sixteen_activation_rows(name, k, rows, expect):
    wtype, n = DT[name], 1100
    w = synth.weight(wtype, n, k, seed=97, stream=1)
    x = synth.activation(rows, k, seed=97)
    lin = Linear(wtype, dev(w), n, k)
    got = lin(dev(x))
    assert lin.path == expect
    lin.close()
    pick = np.sort(np.random.default_rng(97).choice(n, 100, replace=False))
    assert close(got.cpu().numpy()[:, pick], oracle.ob_matmul(wtype, x, w[pick], len(pick)))


@pytest.mark.parametrize("half", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("name,n,k,rows", [
    ("q4_k", 260, 1280, 3), ("q5_k", 256, 4096, 8), ("q4_k", 4100, 2048, 7), ("q5_k", 8200, 2304, 5), ("q4_k", 16384, 2048, 8), ("q6_k", 270, 1280, 4),
    ("q6_k", 300, 4096, 8), ("q6_k", 2050, 3072, 3), ("q6_k", 6144, 2048, 6), ("q4_k", 2048, 4096, 16), ("q5_k", 2050, 2048, 9),
    ("q6_k", 2030, 2816, 15), ("q4_k", 1, 256, 9), ("q5_k", 200, 4096, 16), ("q6_k", 40, 1280, 12)])
def test_a_few_rows_straight_into_the_launch_carry_the_quantizers_codes(name, n, k, rows, half):
    # the same products from Q8_1 rows of the stand-alone quantizer: bit for bit, with zeros, a row's largest code everywhere, halves between two codes,
    # tiny values and infinities among the rows; rows that start off a 16-byte piece too
    w = dev(synth.weight(DT[name], n, k, seed=86, stream=3))
    x = dev(synth.activation(rows, k, seed=86))
    x[0, :64] = 0
    x[1] = torch.arange(k, device="cuda").remainder(255) - 127.0
    x[1, ::3] *= 0.5
    x[2] *= 1e-6
    x = x.to(half)
    lin = Linear(DT[name], w, n, k)
    fn = ops.dense_q6k_rows if name == "q6_k" else (lambda *a: ops.dense_q4k_rows(*a, q5=name == "q5_k"))
    got = lin(x)
    assert lin.path == "rows-on-matrix-unit" and torch.equal(got, fn(w, x.float(), n).to(half))
    flat = torch.zeros(rows * k + 1, device="cuda", dtype=half)
    flat[1:] = x.reshape(-1)
    assert torch.equal(lin(flat[1:].view(rows, k)), got)
    x[0, 5], x[rows - 1, k - 1] = float("inf"), float("nan")
    assert torch.equal(torch.nan_to_num(lin(x)), torch.nan_to_num(fn(w, x.float(), n).to(half)))
    lin.close()


# a workgroup to the CU, two, three and one more than that; last sets of one row and of eight
@pytest.mark.parametrize("half", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name,n,k,rows", [("q4_k", 512, 4096, 64), ("q4_k", 511, 4096, 64), ("q5_k", 1030, 2304, 25), ("q4_k", 2040, 2048, 31), ("q5_k", 512, 1792, 97), ("q4_k", 768, 1024, 128),
                                           ("q5_k", 2050, 768, 41), ("q4_k", 4090, 512, 17), ("q6_k", 640, 4096, 44), ("q6_k", 1360, 1024, 24), ("q6_k", 520, 768, 65)])
def test_sets_of_eight_rows_straight_into_the_launch_carry_the_quantizers_codes(name, n, k, rows, half):
    test_a_few_rows_straight_into_the_launch_carry_the_quantizers_codes(name, n, k, rows, half)


@pytest.mark.parametrize("half", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("name,n,k,rows", [("q4_k", 260, 4096, 3), ("q5_k", 2030, 2048, 9), ("q6_k", 2050, 3072, 8), ("q6_k", 1030, 1024, 16),
                                           ("q4_k", 128, 1024, 12), ("q5_k", 17, 256, 9), ("q6_k", 255, 4096, 16)])
def test_a_few_rows_off_a_vector_boundary_are_one_launch_without_a_workspace(name, n, k, rows, half):
    # a recorded call with nothing reserved is refused where it needs a workspace; rows on any element need none
    lin = Linear(DT[name], dev(synth.weight(DT[name], n, k, seed=88, stream=1)), n, k)
    x = dev(synth.activation(rows, k, seed=88)).to(half)
    want = lin(x)
    flat = torch.zeros(rows * k + 1, device="cuda", dtype=half)
    flat[1:] = x.reshape(-1)
    lib.load().lkh_release_workspaces()
    side, graph, out = torch.cuda.Stream(), torch.cuda.CUDAGraph(), torch.zeros_like(want)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=side):
        rc = lib.load().lkh_qkernel_matmul_forward(lin.h, flat[1:].data_ptr(), X_TYPES[half], rows, out.data_ptr(), side.cuda_stream, 0)
    assert rc == 0 and lin.path == "rows-on-matrix-unit"
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    # half an element off: no such rows
    assert lib.load().lkh_qkernel_matmul_forward(lin.h, flat.data_ptr() + 1, X_TYPES[half], rows, out.data_ptr(), None, 0) == lib.LK_ERR_ARG
    lin.close()


@pytest.mark.parametrize("name", ["q4_k", "q5_k", "q6_k"])
@pytest.mark.parametrize("knob,rows,off", [("LK_TUNE_ROWS16_OFF", 5, True), ("LK_TUNE_ROWS16_OFF", 12, True), ("LK_TUNE_ROWS16_MAX8", 8, False),
                                           ("LK_TUNE_ROWS16_MAX8", 12, True)])
def test_the_overrides_turn_the_short_launches_off_too(name, knob, rows, off, knobs):
    # without them the rows go by way of the quantizer and its workspace, without which a recorded call is refused
    l, n, k = lib.load(), 520, 1024
    w, x = synth.weight(DT[name], n, k, seed=87, stream=1), synth.activation(rows, k, seed=87)
    lin, xd = Linear(DT[name], dev(w), n, k), dev(x)
    knobs.set(knob)
    l.lkh_release_workspaces()
    side, graph, out = torch.cuda.Stream(), torch.cuda.CUDAGraph(), torch.empty((rows, n), device="cuda")
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=side):
        rc = l.lkh_qkernel_matmul_forward(lin.h, xd.data_ptr(), lib.TYPE_F32, rows, out.data_ptr(), side.cuda_stream, 0)
    assert rc == (lib.LK_ERR_NOMEM if off else 0)
    got = lin(xd)
    assert lin.path == "rows-on-matrix-unit" and close(got.cpu().numpy(), oracle.ob_matmul(DT[name], x, w, n))
    lin.close()


@pytest.mark.parametrize("name,n,k,rows,expect", [
    ("q4_k", 8193, 7168, 9, "tiled"), ("q4_k", 8192, 7168, 9, "rows-on-matrix-unit"), ("q5_k", 512, 8448, 16, "rows-on-matrix-unit"),
    ("q5_k", 520, 4608, 17, "tiled"), ("q5_k", 520, 4352, 32, "rows-on-matrix-unit"), ("q4_k", 700, 5120, 200, "rows-on-matrix-unit"),
    ("q4_k", 700, 5120, 33, "tiled"), ("q4_k", 600, 1024, 600, "rows-on-matrix-unit"), ("q5_k", 600, 2304, 600, "tiled"),
    ("q6_k", 12289, 4864, 9, "tiled"), ("q6_k", 520, 4864, 9, "rows-on-matrix-unit"), ("q6_k", 4100, 4096, 20, "rows-on-matrix-unit"),
    ("q6_k", 2049, 12544, 17, "tiled"), ("q6_k", 2048, 12544, 32, "rows-on-matrix-unit"), ("q6_k", 1025, 6400, 64, "tiled"),
    ("q6_k", 520, 5120, 200, "rows-on-matrix-unit"), ("q6_k", 520, 5888, 65, "tiled"), ("q6_k", 2800, 3072, 33, "rows-on-matrix-unit"),
    ("q6_k", 1023, 3072, 300, "rows-on-matrix-unit"), ("q6_k", 520, 768, 7, "rows-on-matrix-unit"), ("q4_k", 4096, 8192, 4, "matvec"),
    ("q4_k", 4112, 8192, 4, "rows-on-matrix-unit"), ("q4_k", 255, 2048, 3, "matvec"), ("q6_k", 256, 1280, 3, "rows-on-matrix-unit")])
def test_both_sides_of_the_lines_around_the_rows_kernels(name, n, k, rows, expect):
    wtype = DT[name]
    w = synth.weight(wtype, n, k, seed=98, stream=1)
    x = synth.activation(rows, k, seed=98)
    lin = Linear(wtype, dev(w), n, k)
    got = lin(dev(x))
    assert lin.path == expect
    lin.close()
    pick, some = np.r_[:40, n - 40:n], np.unique(np.r_[:min(4, rows), max(0, rows - 4):rows])
    assert close(got.cpu().numpy()[some][:, pick], oracle.ob_matmul(wtype, x[some], w[pick], len(pick)))


@pytest.mark.parametrize("name,n,k,rows,expect", [
    ("q8_0", 12289, 4096, 9, "tiled"), ("q8_0", 12287, 4096, 11, "matvec"), ("q8_0", 8193, 4096, 12, "tiled"), ("q8_0", 513, 4096, 14, "tiled"), ("q8_0", 513, 4096, 13, "matvec"),
    ("q8_0", 513, 8192, 12, "tiled"),
    ("q8_0", 513, 3840, 16, "matvec"), ("q8_0", 511, 4096, 16, "matvec"), ("q8_0", 12289, 4096, 8, "matvec"), ("q4_0", 512, 256, 9, "tiled"),
    ("q4_0", 511, 768, 15, "matvec"), ("q4_0", 645, 2304, 12, "tiled"), ("q4_0", 645, 2304, 8, "matvec")])
def test_nine_to_sixteen_rows_of_plain_blocks(name, n, k, rows, expect):
    test_both_sides_of_the_lines_around_the_rows_kernels(name, n, k, rows, expect)
    q81 = torch.empty(lib.load().lkh_quantized_activation_bytes(k, rows), dtype=torch.uint8, device="cuda")
    lin = Linear(DT[name], dev(synth.weight(DT[name], 8, k, seed=98).reshape(8, -1).repeat((n + 7) // 8, axis=0)[:n]), n, k)
    x = dev(synth.activation(rows, k, seed=98))
    s = torch.cuda.current_stream().cuda_stream
    # rows quantized beforehand are served whichever launch forward takes, with its bits
    assert lib.load().lkh_qkernel_matmul_quantize_for_matvec(lin.h, x.data_ptr(), X_TYPES[x.dtype], rows, q81.data_ptr(), s, 0) == 0
    out = torch.empty((rows, n), device="cuda")
    assert lib.load().lkh_qkernel_matmul_forward_quantized(lin.h, q81.data_ptr(), X_TYPES[x.dtype], rows, out.data_ptr(), s, 0) == 0
    assert lin.path == expect and torch.equal(out, lin(x))
    lin.close()


# three to eight rows of the K-quants on the rows kernels (rows whose padded length is more than their own among them), nine to
# sixteen of Q8_0 and Q4_0 on the tiles
@pytest.mark.parametrize("xt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name,rows,n,k,expect", [
    ("q4_k", 3, 2100, 1280, "rows-on-matrix-unit"), ("q4_k", 8, 520, 2048, "rows-on-matrix-unit"), ("q5_k", 7, 1100, 4096, "rows-on-matrix-unit"),
    ("q6_k", 5, 2050, 2048, "rows-on-matrix-unit"), ("q6_k", 8, 601, 1280, "rows-on-matrix-unit"), ("q6_k", 3, 4099, 2816, "rows-on-matrix-unit"),
    ("q8_0", 14, 513, 4352, "tiled"), ("q8_0", 16, 1030, 8192, "tiled"), ("q4_0", 9, 512, 256, "tiled"), ("q4_0", 15, 645, 1280, "tiled")])
def test_rows_quantized_beforehand_are_served_by_the_launches_of_forward(name, rows, n, k, expect, xt):
    l, s = lib.load(), torch.cuda.current_stream().cuda_stream
    w = synth.weight(DT[name], n, k, seed=95, stream=1)
    lin = Linear(DT[name], dev(w), n, k)
    q81 = torch.empty(l.lkh_quantized_activation_bytes(k, rows), dtype=torch.uint8, device="cuda")
    x = dev(synth.activation(rows, k, seed=95)).to(xt)
    x[0, :64] = 0
    x[1] *= 1e-6
    for bad in (False, True):
        if bad:
            x[0, 5], x[rows - 1, k - 1] = float("inf"), float("nan")
        want = lin(x)
        assert lin.path == expect
        out = torch.empty((rows, n), dtype=xt, device="cuda")
        assert l.lkh_qkernel_matmul_quantize_for_matvec(lin.h, x.data_ptr(), X_TYPES[xt], rows, q81.data_ptr(), s, 0) == 0
        assert l.lkh_qkernel_matmul_forward_quantized(lin.h, q81.data_ptr(), X_TYPES[xt], rows, out.data_ptr(), s, 0) == 0
        assert lin.path == expect and torch.equal(torch.nan_to_num(out), torch.nan_to_num(want))
        assert l.lkh_qkernel_matmul_forward_quantized(lin.h, q81.data_ptr() + 2, X_TYPES[xt], rows, out.data_ptr(), s, 0) == lib.LK_ERR_ARG
        if not bad:
            pick = np.arange(0, n, 7)
            eps = 0.0 if xt == torch.float32 else 2.0 ** -8   # one rounding to the narrow type
            assert close(out.float().cpu().numpy()[:, pick], oracle.ob_matmul(DT[name], x.float().cpu().numpy(), w[pick], len(pick)), rtol=1e-3 + eps)
    lin.close()


@pytest.mark.parametrize("rows,n,k,expect", [(3, 1030, 2816, "matvec"), (8, 1030, 2816, "matvec"), (5, 2050, 4096, "matvec"),
                                             (9, 1030, 2816, "rows-on-matrix-unit"), (20, 300, 1280, "rows-on-matrix-unit")])
def test_q6k_weights_off_a_16_byte_boundary(rows, n, k, expect):
    w = synth.weight(lib.TYPE_Q6_K, n, k, seed=89, stream=1)
    flat = torch.zeros(w.size + 16, dtype=torch.uint8, device="cuda")
    flat[2:2 + w.size] = dev(w).reshape(-1)
    x = synth.activation(rows, k, seed=89)
    lin = Linear(lib.TYPE_Q6_K, flat[2:], n, k)
    got = lin(dev(x))
    assert lin.path == expect
    lin.close()
    pick = np.arange(0, n, 5)
    assert close(got.cpu().numpy()[:, pick], oracle.ob_matmul(lib.TYPE_Q6_K, x, w[pick], len(pick)))


@pytest.mark.parametrize("name,rows,n,k", [("q4_k", 3, 4096, 2048), ("q5_k", 4, 14336, 4096), ("q6_k", 7, 1024, 2048), ("q6_k", 3, 4096, 14336),
                                           ("q8_0", 17, 513, 4096), ("q4_0", 16, 645, 1024)])
def test_large_matrices_and_tiled_row_counts_refuse_rows_quantized_beforehand(name, rows, n, k):
    l, s = lib.load(), torch.cuda.current_stream().cuda_stream
    lin = Linear(DT[name], torch.zeros(1 << 26, dtype=torch.uint8, device="cuda"), n, k)
    q81 = torch.zeros(l.lkh_quantized_activation_bytes(k, rows), dtype=torch.uint8, device="cuda")
    x, out = torch.zeros((rows, k), device="cuda"), torch.zeros((rows, n), device="cuda")
    assert l.lkh_qkernel_matmul_quantize_for_matvec(lin.h, x.data_ptr(), lib.TYPE_F32, rows, q81.data_ptr(), s, 0) == lib.LK_NOT_TAKEN
    assert l.lkh_qkernel_matmul_forward_quantized(lin.h, q81.data_ptr(), lib.TYPE_F32, rows, out.data_ptr(), s, 0) == lib.LK_NOT_TAKEN
    lin.close()


@pytest.mark.parametrize("name", ["q4_k", "q5_k", "q6_k", "q8_0"])
@pytest.mark.parametrize("half", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,n,k,shift,expect", [(1, 1, 256, 0, "matvec-fused"), (2, 7, 1024, 4, "matvec-fused"), (1, 301, 2048, 0, "matvec-fused"),
                                                   (2, 4099, 4096, 8, "matvec-fused"), (1, 9001, 3840, 0, "matvec-fused"), (2, 2050, 2048, 0, "matvec-fused"),
                                                   (1, 64, 1024, 2, "matvec"), (2, 70, 8192, 0, "matvec-fused"),
                                                   (1, 70, 4352, 4, "matvec-fused"), (2, 64, 8448, 0, "matvec"),
                                                   (2, 4096, 4352, 0, "matvec"), (1, 9637, 4352, 0, "matvec-fused"), (2, 2890, 4352, 0, "matvec-fused")])
def test_half_rows_quantized_in_the_launch_carry_the_quantizers_codes(name, rows, n, k, shift, expect, half):
    # One launch over one or two half rows: the bits of quantizer and mat-vec, rows from any 8-byte boundary; rows off it,
    # and longer ones, go on as two launches. Zeros, the largest codes, tiny values, infinities and NaN among them.
    w = dev(synth.weight(DT[name], n, k, seed=99, stream=1))
    x = dev(synth.activation(rows, k, seed=99))
    x[0, :32] = 0
    x[0, 32:64] *= 1e-6
    x[rows - 1, 64] = 127
    flat = torch.zeros(rows * k + shift, device="cuda", dtype=half)
    flat[shift:] = x.reshape(-1).to(half)
    x = flat[shift:].view(rows, k)
    lin = Linear(DT[name], w, n, k)
    for _ in range(2):
        got = lin(x)
        assert lin.path == expect and got.dtype == half
        want = ops.mmvq(DT[name], w, ops.quantize_q8_1_rows(x.contiguous()), k, n, out_dtype=half)
        assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(want))
        x[0, 5], x[rows - 1, k - 1] = float("inf"), float("nan")
    lin.close()


@pytest.mark.parametrize("name", ["q4_k", "q5_k", "q6_k"])
@pytest.mark.parametrize("rows,n,k,shift", [(450, 2048, 256, 0), (180, 2561, 1280, 0), (33, 14336, 512, 1)])
def test_operands_straight_from_the_rows_are_those_of_the_records(name, rows, n, k, shift):
    # The tiled products' token operands written by the quantizer itself, or from the workspace records: one rule, so the same
    # bits; rows that start off a 16-byte piece too. Zeros, the type's largest codes and tiny values among them.
    w = dev(synth.weight(DT[name], n, k, seed=85, stream=2))
    x = dev(synth.activation(rows, k, seed=85))
    x[0] = 0
    x[1, ::32] = 127
    x[2] *= 1e-7
    flat = torch.zeros(rows * k + shift, device="cuda")
    flat[shift:] = x.reshape(-1)
    x = flat[shift:].view(rows, k)
    lin = Linear(DT[name], w, n, k)
    got = lin(x)
    assert lin.path == "tiled" and torch.equal(got, ops.mmq_forward(DT[name], w, x.clone(), n))
    lin.close()


@pytest.mark.parametrize("name,n,k,rows,expect", [
    ("q6_k", 4112, 4608, 17, "tiled"), ("q6_k", 2056, 4352, 32, "rows-on-matrix-unit"), ("q6_k", 8200, 2560, 17, "tiled"),
    ("q6_k", 5200, 4096, 17, "rows-on-matrix-unit"), ("q6_k", 9700, 768, 33, "tiled"), ("q6_k", 9696, 768, 33, "rows-on-matrix-unit"),
    ("q5_k", 4096, 3328, 17, "rows-on-matrix-unit"), ("q5_k", 520, 3328, 161, "tiled"), ("q4_k", 2080, 3328, 65, "rows-on-matrix-unit")])
def test_the_lines_that_moved_to_the_tiles_dealt_evenly(name, n, k, rows, expect):
    test_both_sides_of_the_lines_around_the_rows_kernels(name, n, k, rows, expect)


@pytest.mark.parametrize("name,n,k,rows,expect", [
    ("q4_k", 2986, 6144, 26, "rows-on-matrix-unit"), ("q4_k", 2064, 14336, 40, "rows-on-matrix-unit"), ("q4_k", 1030, 4096, 128, "rows-on-matrix-unit"),
    ("q4_k", 1030, 5632, 128, "tiled"), ("q4_k", 14336, 5120, 64, "tiled"), ("q5_k", 3456, 5632, 19, "rows-on-matrix-unit"),
    ("q5_k", 8208, 5632, 19, "tiled"), ("q6_k", 4096, 6144, 17, "rows-on-matrix-unit"), ("q6_k", 4097, 6144, 17, "tiled"),
    ("q6_k", 2048, 6912, 48, "rows-on-matrix-unit"), ("q6_k", 2049, 6912, 48, "tiled"), ("q6_k", 1360, 4096, 96, "rows-on-matrix-unit"),
    ("q6_k", 1361, 5632, 96, "tiled"), ("q6_k", 1024, 5632, 128, "rows-on-matrix-unit"), ("q6_k", 2056, 34816, 18, "tiled"), ("q5_k", 1152, 4864, 40, "rows-on-matrix-unit")])
def test_the_lines_that_moved_to_sets_of_rows(name, n, k, rows, expect):
    test_both_sides_of_the_lines_around_the_rows_kernels(name, n, k, rows, expect)



@pytest.mark.parametrize("name,n,k,rows,expect", [
    ("q6_k", 8192, 1024, 64, "rows-on-matrix-unit"), ("q6_k", 8196, 1024, 64, "tiled"), ("q6_k", 7000, 2048, 49, "rows-on-matrix-unit"),
    ("q6_k", 6000, 2304, 60, "tiled"), ("q6_k", 6145, 4608, 30, "rows-on-matrix-unit"), ("q6_k", 6144, 4608, 30, "tiled"),
    ("q6_k", 8192, 6144, 17, "rows-on-matrix-unit"), ("q6_k", 8196, 4352, 17, "tiled"), ("q6_k", 11264, 3072, 25, "rows-on-matrix-unit"),
    ("q6_k", 13660, 3072, 25, "tiled"), ("q6_k", 9216, 2560, 20, "rows-on-matrix-unit"), ("q6_k", 9215, 2560, 20, "tiled"),
    ("q4_k", 7930, 11264, 64, "tiled"), ("q4_k", 6102, 512, 125, "tiled"), ("q4_k", 2986, 6144, 26, "rows-on-matrix-unit")])
def test_the_lines_where_the_tiles_or_the_sets_had_been_slower(name, n, k, rows, expect):
    test_both_sides_of_the_lines_around_the_rows_kernels(name, n, k, rows, expect)


def test_q6k_weights_off_a_piece_keep_the_tiles_where_sets_of_rows_would_pay():
    n, k, rows = 4000, 6144, 24
    w, x = synth.weight(DT["q6_k"], 50, k, seed=98, stream=3).reshape(50, -1), synth.activation(rows, k, seed=98)
    want = np.tile(oracle.ob_matmul(DT["q6_k"], x, w, 50), (1, n // 50))
    flat = torch.zeros(n * w.shape[1] + 32, dtype=torch.uint8, device="cuda")
    for shift, expect in ((0, "rows-on-matrix-unit"), (2, "tiled")):
        blob = flat[shift:shift + n * w.shape[1]]
        blob.view(n // 50, -1)[:] = dev(w).reshape(1, -1)
        lin = Linear(DT["q6_k"], blob, n, k)
        got, path = lin(dev(x)), lin.path
        lin.close()
        assert path == expect and close(got.cpu().numpy(), want)


@pytest.mark.parametrize("name,n,k,rows", [("q6_k", 4000, 6144, 24), ("q6_k", 1360, 5632, 96), ("q4_k", 2986, 6144, 26)])
def test_without_the_short_launches_their_rows_keep_the_tiles(name, n, k, rows, knobs):
    w, x = np.tile(synth.weight(DT[name], 50, k, seed=99, stream=3).reshape(50, -1), ((n + 49) // 50, 1))[:n], synth.activation(rows, k, seed=99)
    lin, xd = Linear(DT[name], dev(w), n, k), dev(x)
    want = np.tile(oracle.ob_matmul(DT[name], x, w[:50], 50), (1, (n + 49) // 50))[:, :n]
    got = lin(xd)
    assert lin.path == "rows-on-matrix-unit" and close(got.cpu().numpy(), want)
    knobs.set("LK_TUNE_ROWS16_OFF")
    got = lin(xd)
    assert lin.path == "tiled" and close(got.cpu().numpy(), want)
    lin.close()
