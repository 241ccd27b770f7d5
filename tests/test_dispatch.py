"""Which kernel a GEMM runs (on the CPU: the rules take a shape and a CU count)."""
import importlib

import pytest

# Test modules whose shapes are there for one kernel each.
PLANNED = ["test_gpu_kranges", "test_gpu_packed_out", "test_gpu_parity", "test_gpu_producers", "test_gpu_tiles16"]


@pytest.mark.parametrize("module", PLANNED)
def test_shapes_reach_their_kernels(gemm_plan, module):
    for m, k, n, epilogue, split, name in importlib.import_module(f"tests.{module}").PLANS:
        assert gemm_plan(m, k, n, epilogue, split) == name, (m, k, n, epilogue, split)


def test_k_ranges(gemm_plan):
    from tests import test_gpu_kranges as kranges
    for ranges, shapes in kranges.RANGES.items():
        for shape in shapes:
            assert gemm_plan(*shape).startswith(f"k{ranges} "), shape


def test_row_counts_and_fused_tiles_reach_their_kernels(exact_plan, fused_plan):
    from tests import test_gpu_exact_rows as exact
    from tests import test_gpu_fused_tiles as fused
    for m, _, n, rows in exact.SHAPES + exact.NONFINITE:
        assert exact_plan(m, n) == rows, (m, n)
    assert {rows for *_, rows in exact.NONFINITE} == {1, 2, 4, 8, 16}
    for m, k, n, tile in fused.SHAPES:
        assert fused_plan(m, k, n) == tile, (m, k, n)


# (m, k, n, epilogue, split): us on an MI355X with the persistent kernel and
# with the faster of the one-range tiles of 64 x 192 and 128 x 192
MEASURED = [
    (4592, 3072, 12288, "plain", 0, 319.8, 303.5), (4000, 3072, 9216, "plain", 0, 219.6, 203.6),
    (2200, 3072, 3072, "plain", 0, 60.2, 51.5), (1024, 3072, 18432, "plain", 0, 123.7, 110.7),
    (4096, 3072, 12288, "plain", 0, 260.9, 269.9), (4240, 3072, 9216, "plain", 0, 221.8, 225.0),
    (4608, 15360, 3072, "plain", 0, 326.2, 421.0), (3840, 3072, 3072, "plain", 0, 63.0, 68.4),
    (2200, 3072, 3072, "gate_residual", 0, 65.6, 55.0), (1500, 9216, 3072, "gate_residual", 0, 201.5, 107.9),
    (2836, 1152, 24640, "gate_residual", 0, 233.9, 242.8), (3968, 1536, 26304, "gate_residual", 0, 391.4, 408.1),
    (3000, 3072, 18432, "swiglu", 0, 309.3, 300.9), (2200, 3072, 18432, "swiglu", 0, 227.0, 233.0),
    (4592, 3072, 12288, "packed_swiglu", 0, 310.2, 318.5), (3744, 768, 19456, "packed_swiglu", 6464, 126.3, 146.6),
    (4498, 768, 8896, "packed_swiglu", 0, 77.9, 87.4), (3808, 2688, 22528, "packed_swiglu", 7488, 411.4, 447.0),
    (1600, 768, 7104, "packed_swiglu", 0, 25.1, 31.5), (594, 1152, 15488, "packed_swiglu", 5120, 30.5, 36.4),
    (3300, 3072, 21504, "packed_gelu", 9216, 385.7, 394.8), (3773, 768, 15040, "packed_gelu", 0, 107.1, 108.8),
    (1024, 3072, 18432, "packed_swiglu", 0, 125.7, 118.2),
]


@pytest.mark.parametrize("m,k,n,epilogue,split,persistent,tiles", MEASURED)
def test_picks_the_faster_kernel(gemm_plan, m, k, n, epilogue, split, persistent, tiles):
    name = gemm_plan(m, k, n, epilogue, split)
    us = tiles if name.startswith("k1 ") else persistent
    assert us <= 1.03 * min(persistent, tiles), name


# (m, k, n): us with the fused-conversion GEMM's tiles of 128 x 512, 64 x 256,
# 64 x 128 and 32 x 64
FUSED = [
    (599, 3968, 14704, 114.9, 117.7, 135.3, 190.2),
    (4484, 3648, 2176, 107.8, 103.2, 123.2, 181.6),
    (2884, 4544, 4096, 130.8, 142.1, 167.9, 269.3),
    (3531, 4160, 2816, 120.4, 117.6, 140.5, 207.6),
    (2269, 7488, 9472, 420.9, 438.9, 505.7, 838.4),
    (2752, 256, 3968, 21.7, 17.8, 19.6, 20.6),
    (738, 576, 15488, 31.3, 27.7, 31.1, 38.5),
    (3753, 3968, 1792, 109.6, 74.2, 99.4, 135.6),
    (572, 1856, 10240, 58.8, 38.5, 39.4, 64.1),
    (1582, 1344, 1928, 42.4, 22.7, 20.3, 27.7),
    (1756, 192, 3840, 18.6, 12.9, 12.4, 12.9),
    (273, 1024, 3336, 34.1, 16.9, 13.0, 11.5),
    (29, 192, 10208, 10.8, 7.5, 6.3, 6.2),
]


@pytest.mark.parametrize("m,k,n,t512,t256,t128,t64", FUSED)
def test_picks_the_faster_tile(fused_plan, m, k, n, t512, t256, t128, t64):
    us = dict(zip(("128x512", "64x256", "64x128", "32x64"), (t512, t256, t128, t64)))
    name = fused_plan(m, k, n)
    assert us[name] <= 1.05 * min(us.values()), name
