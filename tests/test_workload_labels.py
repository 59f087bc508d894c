"""What the measured workloads call the kernels they time (no GPU needed)."""
import pytest

pytest.importorskip("torch")

from loken_amd import lib, workloads


@pytest.mark.parametrize("wtype,n,m,f16", [
    (lib.TYPE_Q4_K, 14336, 512, True), (lib.TYPE_Q8_0, 14336, 512, True), (lib.TYPE_Q4_0, 4096, 64, True), (lib.TYPE_Q6_K, 512, 9, True),
    (lib.TYPE_Q5_K, 511, 512, False), (lib.TYPE_Q4_K, 4096, 8, False), (lib.TYPE_Q4_1, 4096, 512, False), (lib.TYPE_Q3_K, 4096, 512, False)])
def test_tiled_calls_are_priced_by_the_unit_they_run_on(wtype, n, m, f16, knobs):
    knobs.clear("LK_MMQ_I8")
    kernel, peak, dtype = workloads.tile_kernel(wtype, n, m)
    assert kernel.startswith("tile_dense_kernel" if f16 else "mmq_dense_kernel")
    assert peak == (workloads.F16_PEAK_TFLOPS if f16 else workloads.INT8_PEAK_TOPS) and dtype.startswith("f16" if f16 else "int8")
    knobs.set("LK_MMQ_I8")
    assert workloads.tile_kernel(wtype, n, m)[0].startswith("mmq_dense_kernel")
