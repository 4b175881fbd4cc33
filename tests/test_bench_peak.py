"""bench.py prices a launch's products at the rate of the instructions that they run on."""
import os
import sys

import pytest

import product_programs as PP

from anvil.backend import hip

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench                                                       # noqa: E402


@pytest.mark.parametrize("low,split", [
    (PP.product("NT", 4096, 2944, 72), True),                      # shared tiles
    (PP.product("TN", 1030, 520, 2065), True),                     # the bf16 K split
    (PP.product("NN", 64, 96, 64), False),                         # the float32 K split
    (PP.attention(4, 700, 700, 128), True)])
def test_peak_is_that_of_the_kernels_products(low, split):
    src = hip.generate(low.prog, library=True)
    names = [line.split(") ", 1)[1].split("(")[0] for line in src.splitlines() if line.startswith("__global__ void __launch_bounds__(")]
    peaks = {bench.matrix_peak(src, f"{name} gemm: y") for name in names if name.startswith(("k", "fk"))}
    assert (bench.PEAK_SPLIT_MFMA in peaks) == split


def test_peak_of_a_side_by_side_launch_is_that_of_its_parts():
    part = "__device__ __forceinline__ void fk{0}_k{0}(const float *a) {{\n    anvil_mm_tile_{1}<4, 2, 2>(a);\n}}\n"
    launch = "__global__ void __launch_bounds__(256) fk{0}(const float *a) {{\n    fk{0}_k{0}(a);\n}}\n"
    source = "".join(text.format(k, tile) for k, tile in ((1, "kpipe"), (2, "split"), (21, "kpipe")) for text in (part, launch))
    assert [bench.matrix_peak(source, f"fk{k} fused: k{k} gemm: y") == bench.PEAK_SPLIT_MFMA for k in (1, 2, 21)] == [False, True, False]
