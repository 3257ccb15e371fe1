"""CPU: which loop a launch takes, by its sizes (256 workgroups, the library's count without a GPU)."""
import math
import time

import pytest

from momoe_amd import _hip

ROWS, TRANSPOSED, KBLOCKED = 0, 1, 2


# Times in us at 32 and 64 rows a stage, on one MI355X: rows spread as by a router without preferences | skewed
@pytest.mark.parametrize("rows_per_expert,N,X,Y,b_layout,stage", [
    (192, 64, 512, 1024, ROWS, 32),        # 39, 42
    (256, 64, 512, 1024, ROWS, 32),        # 44, 46
    (280, 64, 1024, 1024, KBLOCKED, 32),   # 68, 72 | 77, 73
    (236, 96, 256, 128, ROWS, 64),         # 166, 104 with a load falling as rank^-1.8
    (200, 96, 256, 512, ROWS, 64),         # 24, 26 | 64, 59: no more tiles than workgroups
    (448, 64, 512, 1024, ROWS, 64),        # 69, 67
    (192, 32, 768, 2048, ROWS, 32),        # 48, 52
    (512, 16, 4096, 2048, KBLOCKED, 64),   # 182, 167
    (192, 64, 512, 512, KBLOCKED, 64),     # 18.9, 20.9: no more tiles than workgroups
    (192, 64, 2048, 4096, KBLOCKED, 32),   # 361, 381: ten tiles a workgroup and more
    (200, 128, 2048, 2048, KBLOCKED, 64),  # 402, 378 | 396, 403
    (256, 128, 2048, 2048, KBLOCKED, 64),  # 454, 435
    (192, 128, 1024, 2048, ROWS, 64),      # 215, 205
    (200, 64, 1024, 2048, ROWS, 64),       # 111, 104 | 110, 109: eight tiles a workgroup
    (192, 64, 2048, 2048, ROWS, 64),       # 214, 199
    (128, 128, 2048, 2048, ROWS, 32),
])
def test_rows_of_a_weight_gradient_stage(rows_per_expert, N, X, Y, b_layout, stage):
    msum = rows_per_expert * N
    assert _hip._lib.momoe_wgrad_stage_rows(N, X, Y, msum, b_layout) == stage
    if b_layout == ROWS:  # (hs, the other operand of the Wl2 gradient, does not matter)
        assert _hip._lib.momoe_wgrad_stage_rows(N, X, Y, msum, TRANSPOSED) == stage


def test_no_weight_gradient_launch():
    assert _hip._lib.momoe_wgrad_stage_rows(8, 64, 64, 0, ROWS) == 0


def _row_tiles(mean, height, first=0):
    """Row tiles per expert as the choice of loop for the row-tile GEMMs estimates them, the first terms taken as 1."""
    spread, t, k = math.sqrt(mean), 1.0 + first, 1 + first
    while k * height < mean + 6 * spread:
        t += 1 / (1 + math.exp(1.7 * (k * height - mean) / spread))
        k += 1
    return t


@pytest.mark.parametrize("mean", [1, 90, 300, 515, 4096, 8000, 131072])
def test_terms_left_out_of_the_sum_of_row_tiles_are_ones(mean):
    for height in (256, 320):
        first, spread = math.floor((mean - 24 * math.sqrt(mean)) / height), math.sqrt(mean)
        assert _row_tiles(mean, height) == _row_tiles(mean, height, max(0, first))
        if first > 0:
            assert 1 / (1 + math.exp(1.7 * (first * height - mean) / spread)) == 1


def test_choice_for_many_rows_per_expert_is_quick():
    """Host time of a choice does not grow with the rows per expert (120 ms for these with every term added)."""
    lib = _hip._lib
    lib.momoe_gemm_tile_rows(1 << 10, 1, 4096, 4096)
    best = 1.0
    for _ in range(5):
        t0 = time.perf_counter()
        lib.momoe_gemm_tile_rows(1 << 30, 1, 4096, 4096)
        best = min(best, time.perf_counter() - t0)
    assert best < 1e-3


# Times in us of the loops with 32 and 64 k-values a stage, rows spread as by a router without preferences
@pytest.mark.parametrize("rows_per_expert,N,cols,contraction,span", [
    (130, 96, 512, 512, False),      # x.Wl1, 18.2, 20.8: one round, a short contraction
    (176, 96, 512, 512, False),      # dL/dx, 20.4, 21.6
    (300, 96, 512, 512, False),      # x.Wl1, 27, 31
    (224, 48, 3072, 512, True),      # h.Wl2, 66, 57: three rounds
    (512, 128, 2048, 2048, True),
    (62, 128, 2048, 2048, False),    # few rows per expert
    (300, 64, 2048, 2048, True),     # x.Wl1, 218, 178 (163, 178 with 300 rows in every expert)
])
def test_loop_of_the_row_tile_gemms(rows_per_expert, N, cols, contraction, span):
    rows = _hip._lib.momoe_gemm_tile_rows(rows_per_expert * N, N, cols, contraction)
    assert rows == (_hip.RECOMPUTE_TILE_ROWS if span else 0)


@pytest.mark.parametrize("rows_per_expert,N,D,H,stage", [
    (176, 64, 1024, 512, 32),   # 43, 49
    (200, 64, 1024, 512, 32),   # 44, 48
    (130, 64, 1024, 512, 32),   # 35, 40
    (512, 32, 1024, 512, 64),   # 71, 54
    (152, 32, 2048, 768, 64),   # 65, 58
    (269, 8, 1152, 64, 64),     # 27, 20: 16 tiles, cut into pieces
    (512, 128, 2048, 1024, 64),
    (62, 128, 2048, 768, 32),
])
def test_loop_of_the_recomputing_gemm(rows_per_expert, N, D, H, stage):
    assert _hip._lib.momoe_recompute_stage_k(rows_per_expert * N, N, D, H) == stage


def test_no_recomputing_launch():
    assert _hip._lib.momoe_recompute_stage_k(0, 8, 64, 64) == 0


# (times of either side beside the constants, csrc/router.hip)
@pytest.mark.parametrize("M,D,N,own", [
    (1024, 2048, 128, True), (1025, 2048, 128, False), (2048, 1024, 128, True), (2049, 128, 8, False),  # rows of partial sums, tokens
    (1024, 1024, 256, True), (1025, 1024, 256, False), (1000, 2048, 256, False), (2048, 128, 256, True),  # partial sums
    (512, 1024, 512, True), (513, 1024, 512, False), (2000, 1024, 512, False), (1, 8192, 512, True),
])
def test_tokens_of_the_router_with_its_product(M, D, N, own):
    parts = -(-D // 128)
    assert _hip._lib.momoe_gate_router_workspace_bytes(M, D, N) == (parts * M * N * 4 if own else -1)
