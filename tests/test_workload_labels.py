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


@pytest.mark.parametrize("wtype", [lib.TYPE_Q4_K, lib.TYPE_Q5_K, lib.TYPE_Q8_0, lib.TYPE_MXFP4])
def test_the_expert_workload_times_the_launches_of_the_block(wtype):
    # 128 experts of 2048 -> 768, top-8: Q5_K at 24 to 31 tokens and Q8_0 at 36 to 47 are batched for the bytes of their weights
    for tokens in (1, 16, 24, 31, 40, 64, 256, 1111):
        path = lib.load().lk_moe_block_path(wtype, wtype, tokens, 8, 128, 2048, 768)
        assert workloads.moe_launches("auto", wtype, tokens, 8, 128, 2048, 768) == path
    assert workloads.moe_launches("pairs", wtype, 256, 8, 128, 2048, 768) == 0
    assert workloads.moe_launches("tiled", wtype, 1, 8, 128, 2048, 768) == lib.MOE_GROUPED
    assert workloads.moe_launches("rows", lib.TYPE_Q4_K, 1, 8, 128, 2048, 768) == lib.MOE_GROUPED | lib.MOE_ROWS_GATE_UP | lib.MOE_ROWS_DOWN
    assert workloads.moe_launches("tiled", lib.TYPE_IQ2_XXS, 256, 8, 128, 2048, 768) == 0   # no batched launch
