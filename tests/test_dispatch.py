"""CPU: which loop a launch takes, by its sizes (256 workgroups, the library's count without a GPU)."""
import pytest

from momoe_amd import _hip

ROWS, TRANSPOSED, KBLOCKED = 0, 1, 2


# Times in us at 32 and 64 rows a stage, on one MI355X, rows spread as by a router without preferences
@pytest.mark.parametrize("rows_per_expert,N,X,Y,b_layout,stage", [
    (192, 64, 512, 1024, ROWS, 32),        # 39, 42
    (256, 64, 512, 1024, ROWS, 32),        # 44, 46
    (400, 64, 512, 1024, ROWS, 32),        # 64, 69
    (448, 64, 512, 1024, ROWS, 64),        # 69, 67
    (192, 32, 768, 2048, ROWS, 32),        # 48, 52
    (304, 16, 4096, 2048, KBLOCKED, 32),   # 124, 133
    (512, 16, 4096, 2048, KBLOCKED, 64),   # 182, 167
    (192, 64, 512, 512, KBLOCKED, 32),     # 18.9, 20.9
    (192, 64, 2048, 4096, KBLOCKED, 32),   # 361, 381: ten tiles a workgroup and more
    (256, 128, 2048, 2048, KBLOCKED, 64),  # 454, 435
    (192, 128, 1024, 2048, ROWS, 64),      # 215, 205
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
