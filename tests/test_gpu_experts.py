"""GPU: MoMoE forward + backward through the C ABI against the CPU oracle on the same
seeded inputs.  Tolerance: rtol 2e-2 / atol 2e-2 (bf16 results vs fp32-accumulated
oracle) plus a norm-wise bound; tokens-per-expert bit-exact."""
import pytest
import torch

import oracle
from gpu_util import (assert_close, device_layer_inputs, oracle_forward_for_tokens, rel_err,
                      run_device_layer, run_oracle_layer,
                      sampled_parity_on_device_inputs as _sampled_parity_on_device_inputs)
from helpers import make_layer_inputs, make_routing

pytestmark = pytest.mark.gpu


def _check_all(dev, ref, rel=1e-2):
    assert torch.equal(dev["sizes"], ref["sizes"])
    for k in ("y", "G_x", "G_W1", "G_W2", "G_s"):
        assert_close(dev[k], ref[k], k, rel=rel)


@pytest.mark.parametrize("save_percent", [0, 50, 100])
def test_tiny_reference_config(save_percent):
    # B=2, S=64, D=128, H=64, N=8, K=2
    M, D, H, N, K = 128, 128, 64, 8, 2
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, seed=0)
    dev = run_device_layer(x, W1, W2, mask, s, dy, K, save_percent, B=2)
    ref = run_oracle_layer(x, W1, W2, mask, s, dy)
    _check_all(dev, ref)
    assert dev["y"].dtype == torch.bfloat16 and dev["G_s"].dtype == torch.float32
    assert dev["G_W1"].dtype == torch.bfloat16 and dev["G_x"].dtype == torch.bfloat16
    assert torch.all(dev["G_s"][mask == 0] == 0)


@pytest.mark.parametrize("M,D,H,N,K,Ks,skew,sp", [
    (1024, 512, 256, 16, 4, 0, None, 0),
    (1024, 512, 256, 16, 4, 0, None, 37),    # save boundary in the middle of a tile
    (999, 256, 320, 12, 3, 0, None, 100),    # ragged token count, H not a multiple of the column tile
    (2048, 512, 384, 20, 6, 2, 1.8, 0),      # skew + shared experts, H = 1.5 column tiles
    (2048, 512, 384, 20, 6, 2, 1.8, 100),
    (16, 256, 128, 32, 4, 0, None, 0),       # decode-sized: most experts empty
    (64, 64, 32, 1, 1, 0, None, 0),          # one expert, smallest supported D and H
    (33, 96, 160, 5, 5, 0, None, 50),        # every token on every expert, odd token count
    (700, 160, 96, 3, 2, 1, None, 0),        # experts taller than one tile, one shared expert
    (9000, 64, 96, 3, 2, 1, None, 0),        # a shared expert with enough rows that its weight
                                             # gradient is contracted in several pieces
    (12000, 96, 64, 6, 1, 0, 1.8, 50),       # one routed expert holds most rows
])
def test_layer_parity(M, D, H, N, K, Ks, skew, sp):
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, Ks=Ks, seed=5, skew=skew)
    dev = run_device_layer(x, W1, W2, mask, s, dy, K, sp)
    ref = run_oracle_layer(x, W1, W2, mask, s, dy)
    _check_all(dev, ref)


@pytest.mark.parametrize("seed", range(16))
def test_random_small_shapes(seed):
    # shapes drawn from a seeded generator: odd token counts, D and H any multiple of 32,
    # few or many experts, shared experts, every save_percent regime
    import random
    rng = random.Random(1000 + seed)
    D, H = 32 * rng.randint(1, 10), 32 * rng.randint(1, 10)
    N = rng.randint(1, 40)
    K = rng.randint(1, min(N, 6))
    Ks = rng.randint(0, K - 1) if rng.random() < 0.4 else 0
    M = rng.choice([1, 7, 64, 255, 256, 257, 600, 901])
    sp = rng.choice([0, 0, 25, 50, 100])
    skew = rng.choice([None, None, 1.5])
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, Ks=Ks, seed=seed, skew=skew)
    dev = run_device_layer(x, W1, W2, mask, s, dy, K, sp)
    ref = run_oracle_layer(x, W1, W2, mask, s, dy)
    _check_all(dev, ref)
    # the same through the 320-row code path of the forward and data-gradient GEMMs, which small
    # routings never choose by themselves: bit-identical to the run above
    from momoe_amd import _hip, experts
    try:
        experts.TILE_ROWS = _hip.TILE_ROWS
        tall = run_device_layer(x, W1, W2, mask, s, dy, K, sp)
    finally:
        experts.TILE_ROWS = _hip.AUTO_TILE_ROWS
    for k in dev:
        assert torch.equal(tall[k], dev[k]), k


@pytest.mark.parametrize("M,D,H,N,K,sp", [
    (2000, 352, 288, 72, 3, 0),     # too many tiles for narrow ones: every GEMM takes the wide ones
    (1100, 800, 416, 16, 4, 40),    # 275 rows per expert: narrow tiles of halved 320-row ones
    (1, 2048, 768, 128, 8, 0),      # one token
    (640, 1056, 544, 20, 2, 0),     # narrow, column counts one fragment past a tile, 64 rows
    (1300, 160, 1056, 24, 4, 100),  # x.Wl1 wide, the products over D columns narrow
])
def test_wide_and_narrow_tiles(M, D, H, N, K, sp):
    from momoe_amd import _hip, experts
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, seed=3)
    dev = run_device_layer(x, W1, W2, mask, s, dy, K, sp)
    _check_all(dev, run_oracle_layer(x, W1, W2, mask, s, dy))
    # any tile height gives the same sums: halved 320-row tiles, tiles of one fragment row
    for rows in (_hip.TILE_ROWS, 32):
        try:
            experts.TILE_ROWS = rows
            other = run_device_layer(x, W1, W2, mask, s, dy, K, sp)
        finally:
            experts.TILE_ROWS = _hip.AUTO_TILE_ROWS
        for k in dev:
            assert torch.equal(other[k], dev[k]), (rows, k)


@pytest.mark.parametrize("M,D,H,N,K,Ks,skew,sp,span", [
    (8000, 352, 544, 8, 2, 0, None, 0, (1, 1, 1, 1)),  # a full round of x.Wl1 and 6 to 9 tiles per XCD in 2 or 4 pieces each;
                                             # contractions of 5.5, 8.5 and 17 stages, columns past a tile
    (3000, 480, 608, 30, 4, 0, None, 60, (1, 0, 1, 0)),  # 2 to 6 tiles per XCD in 4 or 8 pieces
    (4100, 544, 352, 10, 4, 1, 1.0, 100, (1, 1, 1, 1)),  # skew: tiles of 1 to 8 fragment rows
    (2900, 352, 544, 20, 6, 2, 0.3, 30, (1, 1, 1, 1)),
])
def test_tiles_of_64_k_values(M, D, H, N, K, Ks, skew, sp, span):
    """span: which of x.Wl1, h.Wl2, dL/dh and dL/dx run in the loop of 64 k-values a stage."""
    from momoe_amd import _hip, experts
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, Ks=Ks, seed=6, skew=skew)
    gemms = ((2 * H, D), (D, H), (H, D), (D, 2 * H))
    assert tuple(_hip._lib.momoe_gemm_tile_rows(M * K, N, *g) // _hip.RECOMPUTE_TILE_ROWS for g in gemms) == span
    dev = run_device_layer(x, W1, W2, mask, s, dy, K, sp)
    _check_all(dev, run_oracle_layer(x, W1, W2, mask, s, dy))
    # halved tiles of 320 rows, tiles of three fragment rows: the same sums
    for rows in (_hip.TILE_ROWS, 96):
        try:
            experts.TILE_ROWS = rows
            other = run_device_layer(x, W1, W2, mask, s, dy, K, sp)
        finally:
            experts.TILE_ROWS = _hip.AUTO_TILE_ROWS
        for k in ("y", "G_x"):
            assert torch.equal(other[k], dev[k]), (rows, k)


@pytest.mark.parametrize("M,D,H,N,K,Ks,skew,rows", [
    (1024, 992, 480, 32, 4, 1, 0.5, 256),    # a partial dL/ds per 64 of 480 hidden columns: 8
    (1000, 1024, 416, 32, 4, 2, 0.3, 256),   # 7: the last 128-column tile has no second one
    (1020, 992, 480, 32, 4, 1, 1.0, 320),    # the library chooses 320-row tiles
])
def test_more_tiles_than_a_narrow_launch_was_chosen_for(M, D, H, N, K, Ks, skew, rows):
    """The kernels of few tiles go by the table: experts of several row tiles make them take wide ones."""
    from momoe_amd import _hip
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, Ks=Ks, seed=3, skew=skew)
    table = _hip.index_build(mask.to("cuda:0"), K)["tile_table"][:2].tolist()
    # (256 CUs; chosen as if each of the N experts were one tile)
    assert table[1] == rows and N * -(-H // 64) <= 256 < table[0] * -(-H // 64)
    ref = run_oracle_layer(x, W1, W2, mask, s, dy)
    dev = run_device_layer(x, W1, W2, mask, s, dy, K, 0)
    _check_all(dev, ref)
    # rows of saved pre-activations leave their partial sums among the others'; their bf16 rounding
    # is held to the bound of test_save_percent_only_changes_rounding
    saved = run_device_layer(x, W1, W2, mask, s, dy, K, 40)
    assert torch.equal(saved["y"], dev["y"])
    for k in ("G_x", "G_W1", "G_W2", "G_s"):
        assert rel_err(saved[k], dev[k]) < 1e-2, k


@pytest.mark.parametrize("M,D,H,N,K,skew", [
    (300, 2080, 544, 120, 2, None),   # both matrices above 256 MiB, no dimension a multiple of the tile
    (1300, 2080, 544, 120, 2, 1.8),   # experts of one row tile and of several in one launch
])
def test_weights_read_once(M, D, H, N, K, skew):
    """The forward only: no kernel of the backward reads weights this way."""
    import momoe_amd
    from momoe_amd import _hip, experts
    x, _, W1, W2, mask, s = device_layer_inputs(M, D, H, N, K, skew=skew)
    layer = momoe_amd.MoMoE(D, H, N, K, Wl1_ND2H=W1, Wl2_NHD=W2)
    args = x.reshape(1, M, D), mask.to("cuda:0"), s.T.contiguous().to("cuda:0").T
    with torch.no_grad():
        y, sizes = layer(*args)
        try:
            given = []
            for experts.TILE_ROWS in (_hip.RECOMPUTE_TILE_ROWS, _hip.TILE_ROWS, 64):
                given.append(layer(*args)[0])
        finally:
            experts.TILE_ROWS = _hip.AUTO_TILE_ROWS
    assert torch.equal(sizes.cpu(), (mask != 0).sum(1)) and all(torch.equal(g, y) for g in given)
    tok = torch.arange(0, M, M // 16)[:16]
    want, _ = oracle_forward_for_tokens(x, W1, W2, mask, s, tok)
    assert_close(y.reshape(M, D)[tok.to("cuda:0")], want, "y (sampled tokens)")


@pytest.mark.parametrize("M,D,H,N,K,Ks,sp", [
    (1, 2048, 768, 128, 8, 0, 0),    # one token
    (32, 96, 160, 8, 3, 1, 100),     # the most rows a tile takes, last stages of 96 and 32 k-values
    (31, 64, 32, 5, 5, 0, 50),       # last stages of 64 and 32
    (17, 640, 544, 4, 2, 0, 0),      # five stages: one more than are in flight, columns past a tile
    (33, 448, 320, 4, 2, 0, 0),      # one token too many for it
])
def test_tiles_of_few_rows(M, D, H, N, K, Ks, sp):
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, Ks=Ks, seed=4)
    dev = run_device_layer(x, W1, W2, mask, s, dy, K, sp)
    _check_all(dev, run_oracle_layer(x, W1, W2, mask, s, dy))


@pytest.mark.parametrize("M", [7, 8, 9, 16, 17, 25, 32])
def test_gate_weights_of_few_rows(M):
    """Every expert holds every token: h.Wl2 takes the gate weights eight rows at a time, in either layout of s."""
    D, H, N = 160, 96, 3
    x, W1, W2, mask, s, _ = make_layer_inputs(M, D, H, N, N, seed=M, wstd=0.2)  # (outputs of some units)
    b = lambda t: t.to("cuda:0", torch.bfloat16)
    import momoe_amd
    layer = momoe_amd.MoMoE(D, H, N, N, Wl1_ND2H=b(W1), Wl2_NHD=b(W2))
    f = lambda t: t.to(torch.bfloat16).float()
    want = torch.zeros(M, D)
    for i in range(N):
        ab = f(x) @ f(W1)[i]
        want += s[i][:, None] * (f(ab[:, :H] * torch.nn.functional.silu(ab[:, H:])) @ f(W2)[i])
    for s_dev in (s.contiguous().to("cuda:0"), s.T.contiguous().to("cuda:0").T):
        with torch.no_grad():
            y, _ = layer(b(x).reshape(1, M, D), mask.to("cuda:0"), s_dev)
        assert_close(y.reshape(M, D), want, "y")


@pytest.mark.parametrize("rows", [32, 256, 320])
@pytest.mark.parametrize("sizes", [[33, 0, 1, 64, 2, 0, 0, 0], [0, 0, 250, 0, 0, 0, 0, 0], [0, 700, 5, 0, 0, 31, 0, 0]])
def test_index_that_repeats_tokens(sizes, rows):
    """The entry points take any list of tokens per expert, also of few tokens an expert holds many times."""
    from momoe_amd import _hip
    M, D, H, N, dev = 32, 160, 96, len(sizes), "cuda:0"
    x, W1, W2, _, s, _ = make_layer_inputs(M, D, H, N, 2, seed=13)
    msum = sum(sizes)
    cumsums = torch.zeros(N + 1, dtype=torch.int32)
    cumsums[1:] = torch.cumsum(torch.tensor(sizes), 0)
    idx = torch.randint(0, M, (msum,), generator=torch.Generator().manual_seed(2), dtype=torch.int32)
    s = torch.rand(N, M, generator=torch.Generator().manual_seed(3))
    b = lambda t: t.to(dev, torch.bfloat16)
    table = _hip.tile_table_build(cumsums.to(dev), 1, msum, rows)
    h = torch.full((H // 32, msum, 32), 7.0, device=dev, dtype=torch.bfloat16)
    ys = torch.full((msum, D), 7.0, device=dev, dtype=torch.bfloat16)
    _hip.lin1_swiglu_fwd(b(x), b(W1), idx.to(dev), table, h, None, 0, 0)
    _hip.lin2_scale_fwd(h, b(W2), s.to(dev), idx.to(dev), table, ys, M)
    f = lambda t: t.to(torch.bfloat16).float()
    got_h = h.permute(1, 0, 2).reshape(msum, H).float().cpu()
    for i in range(N):
        r = slice(int(cumsums[i]), int(cumsums[i + 1]))
        if sizes[i] == 0:
            continue
        tok = idx[r].long()
        ab = f(x)[tok] @ f(W1)[i]
        assert_close(got_h[r], ab[:, :H] * torch.nn.functional.silu(ab[:, H:]), f"h of expert {i}")
        assert_close(ys[r], (got_h[r] @ f(W2)[i]) * s[i, tok][:, None], f"rows of expert {i}")


@pytest.mark.parametrize("sizes,rows,H", [
    ([100] + [1] * 7, 32, 96),      # 11 entries, three column blocks in either GEMM
    ([250, 1] + [0] * 6, 32, 96),   # the one entry too many is another expert's than the one before it
    ([33] * 7 + [1], 32, 768),      # 15 entries in 24 column blocks: more tiles than workgroups
    ([257] + [1] * 15, 256, 256),   # 17 entries
    ([700] + [1] * 31, 256, 96), ([700] + [1] * 31, 320, 96),
])
def test_more_tiles_than_experts_of_few_rows(sizes, rows, H):
    """At most 32 tokens and an index that repeats them: a table of more entries than experts.  Nothing is written behind the results."""
    from momoe_amd import _hip
    M, D, N, msum, dev = 32, 160, len(sizes), sum(sizes), "cuda:0"
    assert msum <= M * N and sum(-(-n // rows) for n in sizes) > min(N, msum) and N * -(-2 * H // 64) <= 256  # what such launches take
    x, W1, W2, _, s, _ = make_layer_inputs(M, D, H, N, 2, seed=17)
    cumsums = torch.zeros(N + 1, dtype=torch.int32)
    cumsums[1:] = torch.cumsum(torch.tensor(sizes), 0)
    idx = torch.randint(0, M, (msum,), generator=torch.Generator().manual_seed(2), dtype=torch.int32)
    s = torch.rand(N, M, generator=torch.Generator().manual_seed(3))
    b = lambda t: t.to(dev, torch.bfloat16)
    table = _hip.tile_table_build(cumsums.to(dev), 1, msum, rows)
    owned = []

    def guarded(*size):  # as many elements again behind the result
        n = torch.Size(size).numel()
        owned.append((torch.full((2 * n,), 7.0, device=dev, dtype=torch.bfloat16), n))
        return owned[-1][0][:n].view(size)

    h, ys, ab = guarded(H // 32, msum, 32), guarded(msum, D), guarded(msum, 2 * H)
    lo = sizes[0]  # rows of the first expert are not saved, and its tiles left out
    _hip.lin1_swiglu_fwd(b(x), b(W1), idx.to(dev), table, h, None, 0, 0)
    _hip.lin1_swiglu_fwd(b(x), b(W1), idx.to(dev), table, None, ab, lo, msum)
    _hip.lin2_scale_fwd(h, b(W2), s.to(dev), idx.to(dev), table, ys, M)
    assert all(bool((t[n:] == 7.0).all()) for t, n in owned) and bool((ab[:lo] == 7.0).all())
    f = lambda t: t.to(torch.bfloat16).float()
    got_h = h.permute(1, 0, 2).reshape(msum, H).float().cpu()
    for i in range(N):
        r = slice(int(cumsums[i]), int(cumsums[i + 1]))
        if sizes[i] == 0:
            continue
        tok = idx[r].long()
        want = f(x)[tok] @ f(W1)[i]
        assert_close(got_h[r], want[:, :H] * torch.nn.functional.silu(want[:, H:]), f"h of expert {i}")
        assert_close(ys[r], (got_h[r] @ f(W2)[i]) * s[i, tok][:, None], f"rows of expert {i}")
        if i > 0:
            assert_close(ab[r], want, f"a|b of expert {i}")


@pytest.mark.parametrize("gather_a", [True, False])
def test_weight_gradient_of_cut_experts(gather_a):
    # experts of 20000 / 3 / 0 / 5000 rows: the first is contracted in pieces that meet in the
    # fp32 workspace.  Checked against a plain fp32 matmul per expert and against the same
    # launch without a workspace (no expert is cut then).
    from momoe_amd import _hip
    dev = "cuda:0"
    sizes = [20000, 3, 0, 5000]
    N, X, Y, M = len(sizes), 320, 512, 20000
    msum = sum(sizes)
    g = torch.Generator(device=dev).manual_seed(11)
    cumsums = torch.tensor([0] + list(torch.tensor(sizes).cumsum(0)), dtype=torch.int32, device=dev)
    A = torch.randn(M if gather_a else msum, X, generator=g, device=dev).to(torch.bfloat16)
    B = torch.randn(msum if gather_a else M, Y, generator=g, device=dev).to(torch.bfloat16)
    ids = torch.cat([torch.randperm(M, generator=g, device=dev)[:n].sort().values for n in sizes]).to(torch.int32)
    ga, gb = (ids, None) if gather_a else (None, ids)
    need = _hip._lib.momoe_wgrad_workspace_bytes(N, X, Y, msum)
    assert need >= 3 * 4 * 262144
    out = {}
    for ws in (need, 262144 * 16, 0):
        GW = torch.full((N, X, Y), float("nan"), device=dev, dtype=torch.bfloat16)
        _hip.wgrad(A, ga, B, gb, cumsums, GW, M, msum, workspace_bytes=ws)
        out[ws] = GW.float()
    torch.cuda.synchronize()
    for e, n in enumerate(sizes):
        r0 = int(cumsums[e])
        Ae = A[ids[r0:r0 + n].long()] if gather_a else A[r0:r0 + n]
        Be = B[r0:r0 + n] if gather_a else B[ids[r0:r0 + n].long()]
        want = Ae.float().T @ Be.float()
        for ws, got in out.items():
            assert_close(got[e].cpu(), want.cpu(), f"GW[{e}] ws={ws}", rel=5e-3)
    assert torch.equal(out[0][2], torch.zeros(X, Y, device=dev))
    assert torch.equal(out[need][1:3], out[0][1:3])  # uncut experts: bit-identical


@pytest.mark.parametrize("sizes,M", [([300, 0, 17, 1000, 64], 1000), ([20000, 3, 0, 5000], 20000)])
def test_weight_gradient_from_a_transposed_operand(sizes, M):
    # either operand handed over as [padded sorted row / 32, feature, 32] (the layout the SwiGLU
    # backward writes s*h in): same result as from the row layout, against a plain fp32 matmul
    from momoe_amd import _hip
    dev = "cuda:0"
    N, X, Y = len(sizes), 320, 512
    msum = sum(sizes)
    g = torch.Generator(device=dev).manual_seed(5)
    c = [0] + list(torch.tensor(sizes).cumsum(0).tolist())
    cumsums = torch.tensor(c, dtype=torch.int32, device=dev)
    A = torch.randn(msum, X, generator=g, device=dev).to(torch.bfloat16)
    B = torch.randn(msum, Y, generator=g, device=dev).to(torch.bfloat16)

    def grouped(rows):
        F = rows.shape[1]
        mpad = _hip.padded_rows(msum, N)
        assert mpad == (msum + 31) // 32 * 32 + 32 * N
        # garbage outside the experts' own 32-row groups must not matter; zeros inside them do
        T = torch.full((F, mpad), float("nan"), device=dev, dtype=rows.dtype)
        for e in range(N):
            p0 = (c[e] + 31) // 32 * 32 + 32 * e
            n = c[e + 1] - c[e]
            T[:, p0:p0 + (n + 31) // 32 * 32] = 0
            T[:, p0:p0 + n] = rows[c[e]:c[e + 1]].T
        return T.reshape(F, mpad // 32, 32).permute(1, 0, 2).contiguous()

    # k-blocked B: [feature / 32, row, 32]
    blocked_B = B.reshape(msum, Y // 32, 32).permute(1, 0, 2).contiguous()
    want = torch.stack([A[c[e]:c[e + 1]].float().T @ B[c[e]:c[e + 1]].float() for e in range(N)])
    for kw, a, b in ((dict(a_transposed=True), grouped(A), B), (dict(b_transposed=True), A, grouped(B)),
                     (dict(b_kblocked=True), A, blocked_B)):
        for ws in (None, 0):
            GW = torch.full((N, X, Y), float("nan"), device=dev, dtype=torch.bfloat16)
            _hip.wgrad(a, None, b, None, cumsums, GW, M, msum, workspace_bytes=ws, **kw)
            torch.cuda.synchronize()
            for e in range(N):
                assert_close(GW[e], want[e], f"GW[{e}] {kw} ws={ws}", rel=5e-3)
    with pytest.raises(RuntimeError):  # both transposed: refused
        _hip.wgrad(grouped(A), None, grouped(B), None, cumsums, GW, M, msum, a_transposed=True, b_transposed=True)


def _pieces(lib, sizes, X, Y, M):
    """Pieces that momoe_wgrad cuts the experts' rows into, given all the workspace it can use: at least kc
    stages of 32 rows each, so that the partial tiles fit, and none where no expert can hold two such pieces."""
    N, msum, tiles = len(sizes), sum(sizes), -(-X // 256) * -(-Y // 256)
    room = min(lib.momoe_wgrad_workspace_bytes(N, X, Y, msum) // 262144, 8 * 256)
    kc = max(64, -(-tiles * (msum // 32 + N) // room)) if room else 1 << 30
    if -(-min(M, msum) // 32) < 2 * kc:
        return [1] * N
    return [max(1, -(-n // 32) // kc) for n in sizes]


@pytest.mark.parametrize("sizes,X,Y,stage,pieces", [
    ([0, 1, 33, 64, 65, 130, 1100, 257], 264, 328, 64, 1),  # 206 rows per expert on average, edges in X and Y
    ([0, 1, 33, 64, 65, 130, 900, 257], 264, 328, 32, 1),   # 181: the same in the short loop
    ([2000, 0, 31, 1500], 512, 256, 64, 1),                  # whole tiles
    ([129, 1, 0, 300, 128, 127, 95, 5], 520, 72, 32, 1),     # 98 rows per expert: the short loop
    ([9031, 31, 0, 6000], 264, 328, 64, 4),                  # cut by rows, into pieces of 71 groups of 32
    ([31, 9031, 0, 6] + [2] * 50, 264, 328, 32, 4),          # cut in the short loop
])
@pytest.mark.parametrize("form", ["gather_a", "gather_b", "a_transposed", "b_transposed", "b_kblocked"])
def test_weight_gradient_loops_at_the_edges(sizes, X, Y, stage, pieces, form):
    # Bound: products of bf16 pairs are exact in fp32, so n of them sum to within n 2^-24 of their
    # absolute sum, and the result is rounded to bf16 once (2^-8 relative).
    from momoe_amd import _hip
    dev = "cuda:0"
    if form == "b_kblocked":
        Y = Y // 32 * 32
    N, msum, M = len(sizes), sum(sizes), 1500
    M = max(M, max(sizes))
    layout = {"a_transposed": 1, "b_transposed": 1, "b_kblocked": 2}.get(form, 0)
    assert _hip._lib.momoe_wgrad_stage_rows(N, X, Y, msum, layout) == stage
    assert max(_pieces(_hip._lib, sizes, X, Y, M)) == pieces
    c = [0] + list(torch.tensor(sizes).cumsum(0).tolist())
    cumsums = torch.tensor(c, dtype=torch.int32, device=dev)
    g = torch.Generator(device=dev).manual_seed(21)
    A = torch.randn(M if form == "gather_a" else msum, X, generator=g, device=dev).to(torch.bfloat16)
    B = torch.randn(M if form == "gather_b" else msum, Y, generator=g, device=dev).to(torch.bfloat16)
    ids = torch.randint(0, M, (msum,), generator=g, device=dev, dtype=torch.int32)

    def grouped(rows):
        mpad = _hip.padded_rows(msum, N)
        T = torch.full((mpad, rows.shape[1]), float("nan"), device=dev, dtype=rows.dtype)
        for e in range(N):
            p0, n = (c[e] + 31) // 32 * 32 + 32 * e, sizes[e]
            T[p0:p0 + (n + 31) // 32 * 32] = 0
            T[p0:p0 + n] = rows[c[e]:c[e + 1]]
        return T.reshape(mpad // 32, 32, -1).permute(0, 2, 1).contiguous()

    a, b, kw, ga, gb = A, B, {}, None, None
    rows_a, rows_b = A, B
    if form == "gather_a":
        ga, rows_a = ids, A[ids.long()]
    elif form == "gather_b":
        gb, rows_b = ids, B[ids.long()]
    elif form == "a_transposed":
        a, kw = grouped(A), dict(a_transposed=True)
    elif form == "b_transposed":
        b, kw = grouped(B), dict(b_transposed=True)
    else:
        b, kw = B.reshape(msum, Y // 32, 32).permute(1, 0, 2).contiguous(), dict(b_kblocked=True)
    for ws in (None, 0):
        GW = torch.full((N, X, Y), float("nan"), device=dev, dtype=torch.bfloat16)
        _hip.wgrad(a, ga, b, gb, cumsums, GW, M, msum, workspace_bytes=ws, **kw)
        for e in range(N):
            pa, pb = (t[c[e]:c[e + 1]].double().cpu() for t in (rows_a, rows_b))
            want, size = pa.T @ pb, pa.abs().T @ pb.abs()
            bound = want.abs() * 2.0**-8 + size * (sizes[e] * 2.0**-24 * (1 + 2.0**-8))
            assert torch.all((GW[e].double().cpu() - want).abs() <= bound), f"expert {e} ws={ws}"


@pytest.mark.parametrize("sizes,X,Y,pieces", [
    ([3000, 2600, 64, 0, 3100], 2048, 2304, 1),   # 72 tiles each, 360 items
    ([9000, 2600, 64, 0, 3100], 2048, 2304, 4),   # one cut by rows
    ([70, 0, 4000, 0, 4000, 4000], 2304, 2048, 1),  # short items in front, items without rows between
])
@pytest.mark.parametrize("form", ["a_transposed", "b_kblocked"])
def test_weight_gradients_in_whole_rounds(sizes, X, Y, pieces, form):
    """Few experts with thousands of rows and more tiles than workgroups: the XCDs take whole rounds.  Every tile of
    every expert is written, bounds as above.  (The conditions of WorkItems::whole_rounds, in its units of cost:
    32 rows, and 4 for an item's stores.)"""
    from momoe_amd import _hip
    dev, N, msum, M = "cuda:0", len(sizes), sum(sizes), max(sizes)
    tiles = -(-X // 256) * -(-Y // 256)
    assert _hip._lib.momoe_wgrad_stage_rows(N, X, Y, msum, 2) == 64
    assert max(_pieces(_hip._lib, sizes, X, Y, M)) == pieces
    items = lambda cut: [(tiles * p, -(-(-(-n // 32)) // p) + 4) for n, p in zip(sizes, cut)]
    for cut in ([1] * N, _pieces(_hip._lib, sizes, X, Y, M)):
        share = sum(n * cost for n, cost in items(cut)) // 256
        assert sum(n for n, _ in items(cut)) > 256 and share >= 8 * N and 8 * max(cost for _, cost in items(cut)) > share
    c = [0] + list(torch.tensor(sizes).cumsum(0).tolist())
    cumsums = torch.tensor(c, dtype=torch.int32, device=dev)
    g = torch.Generator(device=dev).manual_seed(24)
    A = torch.randn(M if form == "b_kblocked" else msum, X, generator=g, device=dev).to(torch.bfloat16)
    B = torch.randn(msum if form == "b_kblocked" else M, Y, generator=g, device=dev).to(torch.bfloat16)
    ids = torch.randint(0, M, (msum,), generator=g, device=dev, dtype=torch.int32)
    if form == "b_kblocked":
        blocked = B.reshape(msum, Y // 32, 32).permute(1, 0, 2).contiguous()
        args, kw, rows_a, rows_b = (A, ids, blocked, None), dict(b_kblocked=True), A[ids.long()], B
    else:
        T = torch.zeros(_hip.padded_rows(msum, N), X, device=dev, dtype=torch.bfloat16)
        for e in range(N):
            p0 = (c[e] + 31) // 32 * 32 + 32 * e
            T[p0:p0 + sizes[e]] = A[c[e]:c[e + 1]]
        grouped = T.reshape(-1, 32, X).permute(0, 2, 1).contiguous()
        args, kw, rows_a, rows_b = (grouped, None, B, ids), dict(a_transposed=True), A, B[ids.long()]
    for ws in (None, 0):
        GW = torch.full((N, X, Y), float("nan"), device=dev, dtype=torch.bfloat16)
        _hip.wgrad(*args, cumsums, GW, M, msum, workspace_bytes=ws, **kw)
        for e in range(N):
            pa, pb = (t[c[e]:c[e + 1]].double() for t in (rows_a, rows_b))
            want, size = pa.T.contiguous() @ pb, pa.abs().T.contiguous() @ pb.abs()
            bound = want.abs() * 2.0**-8 + size * (sizes[e] * 2.0**-24 * (1 + 2.0**-8))
            assert torch.all((GW[e].double() - want).abs() <= bound), f"expert {e} ws={ws}"


def _microseconds(launch, launches=20, rounds=5):
    """Shortest time of a launch over `rounds` runs of `launches`."""
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    times = []
    for _ in range(rounds + 1):
        a.record()
        for _ in range(launches):
            launch()
        b.record()
        torch.cuda.synchronize()
        times.append(a.elapsed_time(b) * 1e3 / launches)
    return min(times[1:])


@pytest.mark.parametrize("N,held,rows,X,Y", [(64, 8, 3584, 1024, 1024), (32, 4, 4096, 2048, 1536)])
def test_weight_gradient_of_experts_without_rows_costs_their_zeros(N, held, rows, X, Y):
    """A launch in which most experts are empty takes as long as that of the others and a fill of the rest (95 us
    against 83 + 18, 148 against 140 + 27; 117 and 181 with two stages of the loop for each empty tile)."""
    from momoe_amd import _hip
    dev, msum = "cuda:0", held * rows
    assert _hip._lib.momoe_wgrad_stage_rows(N, X, Y, msum, 2) == 64
    cumsums = torch.tensor([min(e, held) * rows for e in range(N + 1)], dtype=torch.int32, device=dev)
    g = torch.Generator(device=dev).manual_seed(22)
    A = torch.randn(rows, X, generator=g, device=dev).to(torch.bfloat16)
    B = torch.randn(Y // 32, msum, 32, generator=g, device=dev).to(torch.bfloat16)
    ids = torch.arange(rows, dtype=torch.int32, device=dev).repeat(held)
    buffers = [torch.full((N, X, Y), float("nan"), device=dev, dtype=torch.bfloat16) for _ in range(4)]
    turn = iter(range(1 << 30))
    GW = lambda: buffers[next(turn) % 4]  # (in turn: one alone would stay in the last-level cache)
    some = cumsums[:held + 1].contiguous()
    for attempt in range(3):
        all_of_it = _microseconds(lambda: _hip.wgrad(A, ids, B, None, cumsums, GW(), rows, msum, b_kblocked=True))
        if attempt == 0:
            assert all(torch.all(b[held:] == 0) and torch.isfinite(b[:held]).all() for b in buffers)
        of_held = _microseconds(lambda: _hip.wgrad(A, ids, B, None, some, GW()[:held], rows, msum, b_kblocked=True))
        fill = _microseconds(lambda: GW()[held:].zero_())
        if all_of_it <= of_held + 1.25 * fill:
            return
    raise AssertionError(f"{all_of_it:.0f} us, {of_held:.0f} without the empty experts, {fill:.0f} to fill theirs")


def test_ids_of_gathered_rows_are_not_waited_for():
    """Loop of 32 rows a stage: the ids are asked for a stage ahead, so gathering costs next to nothing (74 us
    gathered and 66 not when every stage waited for its ids)."""
    from momoe_amd import _hip
    dev, N, X, Y = "cuda:0", 32, 1024, 1024
    sizes = torch.tensor([2000] + [225] * (N - 1))
    msum = int(sizes.sum())
    assert _hip._lib.momoe_wgrad_stage_rows(N, X, Y, msum, 2) == 32
    cumsums = torch.cat([torch.zeros(1, dtype=torch.int64), sizes.cumsum(0)]).to(torch.int32).to(dev)
    ids = torch.arange(msum, dtype=torch.int32, device=dev)
    A = torch.ones(msum, X, device=dev, dtype=torch.bfloat16)
    B = torch.ones(Y // 32, msum, 32, device=dev, dtype=torch.bfloat16)
    GW = torch.empty(N, X, Y, device=dev, dtype=torch.bfloat16)
    launch = lambda gather: _hip.wgrad(A, gather, B, None, cumsums, GW, msum, msum, b_kblocked=True, workspace_bytes=0)
    for attempt in range(3):
        gathered, plain = (_microseconds(lambda: launch(g)) for g in (ids, None))
        if gathered <= 1.06 * plain:
            return
    raise AssertionError(f"{gathered:.1f} us gathered, {plain:.1f} not")


def test_experts_without_tokens_get_zero_weight_grads():
    M, D, H, N, K = 256, 128, 64, 8, 2
    x, W1, W2, _, _, dy = make_layer_inputs(M, D, H, N, K, seed=9)
    mask = torch.zeros(N, M, dtype=torch.int32)
    mask[1] = 1
    mask[6] = 1
    s = torch.rand(N, M) * mask
    dev = run_device_layer(x, W1, W2, mask, s, dy, K, 0)
    ref = run_oracle_layer(x, W1, W2, mask, s, dy)
    _check_all(dev, ref)
    for i in (0, 2, 3, 4, 5, 7):
        assert torch.all(dev["G_W1"][i] == 0) and torch.all(dev["G_W2"][i] == 0)


def test_save_percent_only_changes_rounding():
    M, D, H, N, K = 2048, 512, 256, 16, 4
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, seed=12)
    r0 = run_device_layer(x, W1, W2, mask, s, dy, K, 0)
    r100 = run_device_layer(x, W1, W2, mask, s, dy, K, 100)
    assert torch.equal(r0["y"], r100["y"])  # forward does not depend on what is saved
    for k in ("G_x", "G_W1", "G_W2", "G_s"):
        assert rel_err(r0[k], r100[k]) < 1e-2, k


def test_headline_shape_properties_and_sampled_parity():
    # Full headline layer: D=2048, H=1024, N=128, K=8, 8192 tokens.  The oracle is evaluated
    # on a sample of tokens / experts; size-independent properties cover the rest.
    import momoe_amd
    M, D, H, N, K = 8192, 2048, 1024, 128, 8
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, seed=21)
    dev = "cuda:0"
    layer = momoe_amd.MoMoE(D, H, N, K, 0, Wl1_ND2H=W1.to(dev), Wl2_NHD=W2.to(dev))
    xd = x.to(dev, torch.bfloat16).reshape(4, 2048, D).requires_grad_()
    sd = s.T.contiguous().to(dev).T.requires_grad_()
    y, sizes = layer(xd, mask.to(dev), sd)
    y.backward(dy.to(dev, torch.bfloat16).reshape(4, 2048, D))
    torch.cuda.synchronize()
    assert sizes.sum().item() == M * K and torch.equal(sizes.cpu(), (mask != 0).sum(1))
    assert torch.isfinite(y).all() and torch.isfinite(layer.Wl1_ND2H.grad).all()
    # linearity in the gate weights: y(2s) == 2*y(s) up to bf16 rounding
    with torch.no_grad():
        y2, _ = layer(xd, mask.to(dev), 2 * sd)
    assert rel_err(y2, 2 * y) < 5e-3
    # sampled forward parity: 48 tokens, all of their experts
    r = lambda t: t.to(torch.bfloat16).float()
    tok = torch.arange(0, M, M // 48)[:48]
    yo = oracle.experts_forward(r(x[tok]), r(W1), r(W2), mask[:, tok], s[:, tok])
    assert_close(y.reshape(M, D)[tok], yo, "y (sampled tokens)")
    # sampled weight-gradient / dL/ds parity: experts 0, 77 and 127 from the closed form
    for i in (0, 77, 127):
        sel = torch.nonzero(mask[i]).flatten()
        one = torch.zeros(1, sel.numel(), dtype=torch.int32) + 1
        _, gW1, gW2, gs = oracle.experts_backward_closed_form(
            r(x[sel]), r(W1[i:i + 1]), r(W2[i:i + 1]), one, s[i:i + 1, sel], r(dy[sel]), dtype=torch.float32)
        assert_close(layer.Wl1_ND2H.grad[i], gW1[0], f"G_W1[{i}]")
        assert_close(layer.Wl2_NHD.grad[i], gW2[0], f"G_W2[{i}]")
        assert_close(sd.grad[i, sel], gs[0], f"G_s[{i}]")
    # sampled dL/dx parity for the same tokens
    xs = r(x[tok]).requires_grad_()
    oracle.experts_forward(xs, r(W1), r(W2), mask[:, tok], s[:, tok]).backward(r(dy[tok]))
    assert_close(xd.grad.reshape(M, D)[tok], xs.grad, "G_x (sampled tokens)")


def test_skewed_routing_with_shared_experts_full_size():
    # D=2048, H=1408, 60 routed + 4 shared experts, 4 routed + 4 shared per token, 16384 tokens,
    # Zipf-like load: a few experts hold ~10x the mean, the shared ones hold every token
    _sampled_parity_on_device_inputs(16384, 2048, 1408, 64, 8, 4, 1.8, 0, 8, experts=(0, 59))


def test_headline_layer_full_size_with_everything_saved():
    # the headline layer at save_percent=100: every row takes the saved-pre-activation branch
    # of the SwiGLU backward (momoe/momoe.py:486-491)
    _sampled_parity_on_device_inputs(8192, 2048, 1024, 128, 8, 0, None, 100, 4, experts=(0, 77, 127))


@pytest.mark.parametrize("sp", [0, 50, 100])
def test_memory_stress_layer_full_size(sp):
    # D=4096, H=2048, N=64, K=8, 65536 tokens: 524288 sorted rows, 4 GiB intermediates
    _sampled_parity_on_device_inputs(65536, 4096, 2048, 64, 8, 0, None, sp, 16, experts=(63,), n_tok=8)


def test_input_formats_and_partial_gradients():
    # what a caller may hand over besides the router's own outputs: fp32 x (cast to bf16 like
    # the reference, momoe/momoe.py:863), non-contiguous x and G_y, a contiguous s_NM, a strided
    # mask; and backward with only some inputs requiring gradients.
    import momoe_amd
    M, D, H, N, K = 384, 128, 96, 10, 3
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, seed=21)
    ref = run_oracle_layer(x, W1, W2, mask, s, dy)
    dev = "cuda:0"
    layer = momoe_amd.MoMoE(D, H, N, K, 0, Wl1_ND2H=W1.to(dev), Wl2_NHD=W2.to(dev))
    # the oracle sees bf16-rounded x: hand the device the same values as fp32, in a strided view
    x32 = x.to(torch.bfloat16).float()
    wide = torch.zeros(M, 2 * D, device=dev)
    wide[:, ::2] = x32.to(dev)
    xd = wide[:, ::2].reshape(2, M // 2, D).requires_grad_()
    assert not xd.is_contiguous() or xd.dtype == torch.float32
    sd = s.contiguous().to(dev).requires_grad_()                      # plain [N, M]
    maskd = mask.T.contiguous().to(dev).T                             # strides (1, N)
    y, sizes = layer(xd, maskd, sd)
    assert y.dtype == torch.bfloat16 and y.shape == (2, M // 2, D) and sizes.dtype == torch.int64
    dy_wide = torch.zeros(2, M // 2, 2 * D, device=dev, dtype=torch.bfloat16)
    dy_wide[..., ::2] = dy.to(dev, torch.bfloat16).reshape(2, M // 2, D)
    y.backward(dy_wide[..., ::2])
    torch.cuda.synchronize()
    assert torch.equal(sizes.cpu(), ref["sizes"])
    assert_close(y.reshape(M, D), ref["y"], "y")
    assert_close(xd.grad.reshape(M, D), ref["G_x"], "G_x")
    assert_close(sd.grad, ref["G_s"], "G_s")
    assert_close(layer.Wl1_ND2H.grad, ref["G_W1"], "G_W1")
    assert_close(layer.Wl2_NHD.grad, ref["G_W2"], "G_W2")

    # frozen experts: only x and s get gradients; then only the weights
    frozen = momoe_amd.MoMoE(D, H, N, K, 50, Wl1_ND2H=W1.to(dev), Wl2_NHD=W2.to(dev))
    for p in frozen.parameters():
        p.requires_grad_(False)
    xb = x.to(dev, torch.bfloat16).reshape(1, M, D).requires_grad_()
    sb = s.contiguous().to(dev).requires_grad_()
    yb, _ = frozen(xb, mask.to(dev), sb)
    yb.backward(dy.to(dev, torch.bfloat16).reshape(1, M, D))
    assert frozen.Wl1_ND2H.grad is None and frozen.Wl2_NHD.grad is None
    assert_close(xb.grad.reshape(M, D), ref["G_x"], "G_x (frozen experts)")
    assert_close(sb.grad, ref["G_s"], "G_s (frozen experts)")
    xc = x.to(dev, torch.bfloat16).reshape(1, M, D)
    yc, _ = layer(xc, mask.to(dev), s.contiguous().to(dev))
    layer.zero_grad(set_to_none=True)
    yc.backward(dy.to(dev, torch.bfloat16).reshape(1, M, D))
    assert_close(layer.Wl1_ND2H.grad, ref["G_W1"], "G_W1 (weights only)")
    assert_close(layer.Wl2_NHD.grad, ref["G_W2"], "G_W2 (weights only)")
    # no_grad forward keeps nothing for a backward
    with torch.no_grad():
        yn, _ = layer(xc, mask.to(dev), s.contiguous().to(dev))
    assert not yn.requires_grad and torch.equal(yn, yc.detach())


@pytest.mark.parametrize("grad", [True, False])
def test_traced_modules_run_the_layer(grad):
    """A graph of torch.jit.trace does on other inputs, of other sizes too, what the module does:
    results, gradients and the selection bias's update."""
    import momoe_amd
    dev = "cuda:0"
    D, H, N, K, Ks = 64, 32, 8, 3, 1
    torch.manual_seed(4)
    eager = momoe_amd.MoE(D, H, N, K, Ks, save_percent=50, bias_update_rate=0.5)
    module = momoe_amd.MoE(D, H, N, K, Ks, save_percent=50, bias_update_rate=0.5)
    module.load_state_dict(eager.state_dict())

    def inputs(M, seed):
        x, _, _, mask, s, dy = make_layer_inputs(M, D, H, N, K, Ks, seed=seed)
        return (x.to(dev, torch.bfloat16).reshape(1, M, D), mask.to(dev), s.to(dev),
                dy.to(dev, torch.bfloat16).reshape(1, M, D))

    x, mask, s, _ = inputs(40, 1)
    with torch.set_grad_enabled(grad):
        traced_experts = torch.jit.trace(module.momoe, (x, mask, s))
        traced_router = torch.jit.trace(module.router, (x, module.biases_N))
        traced = torch.jit.trace(module, x, check_trace=False)  # a call moves the bias
    module.load_state_dict(eager.state_dict())
    for M, seed in ((40, 2), (40, 3), (40, 4), (75, 5)):
        x, mask, s, dy = inputs(M, seed)
        results = []
        for moe, router, experts_of in ((eager, eager.router, eager.momoe), (traced, traced_router, traced_experts)):
            params = eager if moe is eager else module
            params.zero_grad(set_to_none=True)
            xd, sd = x.clone().requires_grad_(grad), s.clone().requires_grad_(grad)
            with torch.set_grad_enabled(grad):
                y, sizes = experts_of(xd, mask, sd)
                xr, chosen, gates = router(xd, params.biases_N)
                out = [y, sizes, xr, chosen, gates, moe(xd)]
            if grad:
                torch.autograd.backward([y, gates, out[5]], [dy, torch.ones_like(gates), dy])
                out += [xd.grad, sd.grad, params.router.Wg_DN.grad, params.momoe.Wl1_ND2H.grad,
                        params.momoe.Wl2_NHD.grad]
            results.append([t.detach() for t in out] + [params.biases_N.detach().clone()])
        for i, (a, b) in enumerate(zip(*results)):
            assert a.dtype == b.dtype and torch.equal(a, b), (M, i)


def test_saved_tensor_hooks():
    """A hook may hand every saved tensor back as a copy; one that hands back something else than was
    saved (host memory, another type, fewer elements) is refused before any kernel reads it."""
    import momoe_amd
    dev = "cuda:0"
    D, H, N, K, M = 64, 32, 4, 2, 48
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, seed=6)
    moe = momoe_amd.MoE(D, H, N, K, 0, save_percent=50, bias_update_rate=0.0, Wg_DN=torch.randn(D, N).to(dev),
                        Wl1_ND2H=W1.to(dev), Wl2_NHD=W2.to(dev))
    xd = x.to(dev, torch.bfloat16).reshape(1, M, D).requires_grad_()
    sd, dyd, maskd = s.to(dev).requires_grad_(), dy.to(dev, torch.bfloat16).reshape(1, M, D), mask.to(dev)

    def experts():
        y, _ = moe.momoe(xd, maskd, sd)
        return [y], [dyd]

    def router():
        _, _, gates = moe.router(xd, moe.biases_N)
        return [gates], [torch.ones_like(gates) * 0.5 + gates.detach()]

    def gradients(call, unpack):
        saved = []

        def pack(t):
            saved.append(t.clone())
            return len(saved) - 1

        for t in (xd, sd, *moe.parameters()):
            t.grad = None
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda i: unpack(i, saved[i])):
            out, grads = call()
        torch.autograd.backward(out, grads)
        return [t.grad for t in (xd, sd, *moe.parameters()) if t.grad is not None], len(saved)

    def at(i, change):  # the i-th saved tensor changed, the others as they were
        return lambda j, t: change(t) if i == j else t

    for call, count in ((experts, 6), (router, 6)):
        want, n = gradients(call, lambda i, t: t)
        got, _ = gradients(call, lambda i, t: t.cpu().to(dev))
        assert n == count and len(want) >= 2 and all(torch.equal(a, b) for a, b in zip(got, want))
        for i in range(count):
            for change in (torch.Tensor.cpu, lambda t: t.to(torch.float16), lambda t: t[..., :-1].contiguous()):
                with pytest.raises(RuntimeError, match="saved tensor"):
                    gradients(call, at(i, change))


@pytest.mark.parametrize("grad", [True, False])
def test_forward_mode_is_refused(grad):
    """Neither function has a forward-mode rule: a tangent on an input is an error, also where no
    input wants a gradient, never a result without it."""
    import momoe_amd
    import torch.autograd.forward_ad as fwAD
    x, W1, W2, mask, s, _ = make_layer_inputs(32, 64, 32, 4, 2, seed=1)
    layer = momoe_amd.MoMoE(64, 32, 4, 2, Wl1_ND2H=W1.to("cuda:0"), Wl2_NHD=W2.to("cuda:0"))
    moe = momoe_amd.MoE(64, 32, 4, 2, 0, Wg_DN=torch.randn(64, 4).to("cuda:0"), Wl1_ND2H=W1.to("cuda:0"),
                        Wl2_NHD=W2.to("cuda:0"))
    xd = x.to("cuda:0", torch.bfloat16).reshape(1, 32, 64)
    with fwAD.dual_level(), torch.set_grad_enabled(grad):
        dual = fwAD.make_dual(xd, torch.ones_like(xd))
        with pytest.raises(RuntimeError):
            layer(dual, mask.to("cuda:0"), s.to("cuda:0"))
        with pytest.raises(RuntimeError):
            moe(dual)


@pytest.mark.parametrize("M,D,H,N,K,skew", [
    (1, 32, 32, 1, 1, None), (128, 64, 96, 8, 2, None), (300, 96, 160, 9, 3, 1.8),  # one to three stages, a half column block
    (257, 416, 64, 3, 3, None), (1024, 1024, 512, 32, 4, None),  # a second tile of one row; one tile per CU
    (800, 160, 2048, 8, 2, 1.8),                                 # more tiles than CUs: u goes through memory
])
@pytest.mark.parametrize("overflow", [False, True])
def test_dgrad_h_on_the_way_to_the_swiglu_backward(M, D, H, N, K, skew, overflow):
    """The two products in one launch are those of the two launches, bit for bit."""
    from momoe_amd import _hip
    dev, msum = "cuda:0", M * K
    assert _hip._lib.momoe_dgrad_h_lin1_bwd_fits(M, D, H, N, msum) == 1
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, seed=3, skew=skew)
    if overflow:
        if N == K:
            pytest.skip("a token cannot have more than all experts")
        mask = torch.ones_like(mask)  # more pairs than rows: nothing is written
    x, Gy, W1, W2 = (t.to(dev, torch.bfloat16) for t in (x, dy, W1, W2))
    s = s.to(dev)
    ib = _hip.index_build(mask.to(dev), K, tile_rows=_hip.RECOMPUTE_TILE_ROWS)
    idx, table = ib["idx_Msum"], ib["tile_table"]
    nparts = _hip._lib.momoe_gs_parts(H, N, msum)
    new = lambda *size: torch.full(size, 7, device=dev, dtype=torch.bfloat16)
    outs = lambda: (new(2 * H // 32, msum, 32), new(_hip.padded_rows(msum, N) // 32, H, 32), torch.full((nparts, msum), 7.0, device=dev))
    u, want, got = new(msum, H), outs(), outs()
    _hip.dgrad_h(Gy, W2, idx, table, u)
    p = lambda t: t.data_ptr()
    _hip._call("momoe_lin1_swiglu_bwd_parts", p(x), p(W1), p(idx), p(table), p(u), p(s), s.stride(0), s.stride(1), 0, p(want[0]),
               p(want[1]), H, p(want[2]), nparts, M, D, H, N, msum, _hip._stream())
    _hip.dgrad_h_lin1_bwd(Gy, W2, x, W1, idx, table, s, new(msum, H), *got)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("M,D,H,N,K,skew", [(300, 96, 160, 9, 3, 1.8), (800, 160, 2048, 8, 2, 1.8)])  # u in registers, through memory
def test_tables_that_the_joined_launch_does_not_take(M, D, H, N, K, skew):
    from momoe_amd import _hip
    dev, msum = "cuda:0", M * K
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, seed=3, skew=skew)
    x, Gy, W1, W2 = (t.to(dev, torch.bfloat16) for t in (x, dy, W1, W2))
    ib = _hip.index_build(mask.to(dev), K, tile_rows=_hip.TILE_ROWS)
    full = lambda *size, dt=torch.bfloat16: torch.full(size, 7.0, device=dev, dtype=dt)
    outs = (full(msum, H), full(2 * H // 32, msum, 32), full(_hip.padded_rows(msum, N) // 32, H, 32),
            full(_hip._lib.momoe_gs_parts(H, N, msum), msum, dt=torch.float32))
    _hip.dgrad_h_lin1_bwd(Gy, W2, x, W1, ib["idx_Msum"], ib["tile_table"], s.to(dev), *outs)
    assert all(bool((t == 7.0).all()) for t in outs)  # tiles too tall: nothing is written


@pytest.mark.parametrize("M,D,H,N,K,skew", [
    (1, 32, 32, 1, 1, None), (128, 128, 64, 8, 2, None), (300, 352, 288, 9, 3, 1.8),  # a tile each, tiles cut off, few rows
    (4095, 64, 32, 70, 3, 1.8), (1000, 1056, 544, 16, 1, None),   # the most tokens; more tiles than workgroups
    (64, 1056, 544, 80, 3, None),  # weights past the last-level cache: dL/dx behind both weight gradients
])
@pytest.mark.parametrize("overflow", [False, True])
def test_tail_of_a_small_backward(M, D, H, N, K, skew, overflow):
    """The three products in one launch are those of the three launches, bit for bit."""
    from momoe_amd import _hip
    dev, msum = "cuda:0", M * K
    assert _hip._lib.momoe_backward_tail_fits(M, D, H, N, msum) == 1
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, seed=2, skew=skew)
    if overflow:
        if N == K:
            pytest.skip("a token cannot have more than all experts")
        mask = torch.ones_like(mask)  # more pairs than rows: no rows for anyone, the gradients are zeros
    elif N > 2:
        mask[N // 2] = 0  # an expert without tokens
    rnd = lambda *size: torch.randn(*size, generator=torch.Generator(device=dev).manual_seed(5), device=dev).to(torch.bfloat16)
    new = lambda *size: torch.full(size, 7, device=dev, dtype=torch.bfloat16)
    x, Gy, W1 = (t.to(dev, torch.bfloat16) for t in (x, dy, W1))
    ib = _hip.index_build(mask.to(dev), K)
    idx, cumsums, table = (ib[k] for k in ("idx_Msum", "cumsums_N", "tile_table"))
    gz, hsT = rnd(2 * H // 32, msum, 32), rnd(_hip.padded_rows(msum, N) // 32, H, 32)
    GW1, GW2, gxs = new(N, D, 2 * H), new(N, H, D), new(msum, D)
    part = torch.randn(3, msum, device=dev)
    Gs, wantGs = torch.full((M, N), 7.0, device=dev), torch.full((M, N), 7.0, device=dev)
    _hip.backward_tail(hsT, Gy, x, gz, W1, idx, cumsums, table, GW2, GW1, gxs, part, Gs)
    _hip.gs_scatter_tokens(part, idx, cumsums, wantGs)
    want1, want2, wantx = new(N, D, 2 * H), new(N, H, D), new(msum, D)
    _hip.wgrad(hsT, None, Gy, idx, cumsums, want2, M, msum, workspace_bytes=0, a_transposed=True)
    _hip.wgrad(x, idx, gz, None, cumsums, want1, M, msum, workspace_bytes=0, b_kblocked=True)
    _hip.dgrad_x(gz, W1, table, wantx, M)
    results = ((GW1, want1), (GW2, want2), (gxs, wantx), (Gs, wantGs))
    assert all(torch.equal(a, b) for a, b in results)
    for a, _ in results:
        a.fill_(7)  # (what there are no rows for stays as it was)
    _hip.backward_tail(hsT, Gy, x, gz, W1, idx, cumsums, table, GW2, GW1, gxs)  # without dL/ds
    assert (Gs == 7).all() and all(torch.equal(a, b) for a, b in results[:3])


def test_calls_that_are_too_large_for_the_tail():
    from momoe_amd import _hip
    fits = _hip._lib.momoe_backward_tail_fits
    assert fits(4096, 64, 32, 70, 4096 * 3) == 0         # an expert may be cut
    assert fits(1024, 1024, 512, 32, 4096) == 1 and fits(1024, 8192, 4096, 32, 4096) == 0  # 64 MiB of rows
    assert fits(2048, 512, 256, 16, 8192) == 0           # the loop of 64 rows a stage
    assert fits(128, 100, 64, 8, 256) == 0
    assert fits(4000, 1 << 20, 32, 1, 1) == 0            # gathered rows are addressed with 32 bits
    z = torch.zeros(16, device="cuda:0", dtype=torch.bfloat16)
    with pytest.raises(RuntimeError):
        _hip._call("momoe_backward_tail", *[z.data_ptr() if i != 1 else 64 for i in range(12)], None, 0, None, 128, 100, 64, 8, 256, _hip._stream())


@pytest.mark.parametrize("M,N,K,nparts,skew", [
    (1, 1, 1, 1, None), (63, 15, 4, 2, None), (64, 16, 4, 1, None), (65, 17, 17, 3, None),  # tiles of 64 x 16
    (256, 1, 1, 1, None), (257, 2, 2, 1, None),    # 256 rows are read without probing
    (2049, 8, 1, 2, 1.8), (70001, 20, 6, 8, 1.8),  # experts of up to all rows and of none, several probes
])
def test_gate_gradient_in_the_layout_of_the_router(M, N, K, nparts, skew):
    """The same sums as momoe_gs_scatter, element for element, with the experts of a token next to each other."""
    from momoe_amd import _hip
    mask, _ = make_routing(M, N, K, seed=M, skew=skew)
    if M > 2:
        mask[:, 1] = 0  # a token without experts: the last rows are nobody's
    ib = _hip.index_build(mask.to("cuda:0"), K)
    part = torch.randn(nparts, M * K, device="cuda:0")
    want = torch.full((N, M), 7.0, device="cuda:0")
    got = torch.full((M, N), 7.0, device="cuda:0")
    _hip.gs_scatter(part, ib["idx_Msum"], ib["cumsums_N"], want)
    _hip.gs_scatter_tokens(part, ib["idx_Msum"], ib["cumsums_N"], got)
    assert torch.equal(got.T, want)
    # more pairs than rows: nothing but zeros
    ib = _hip.index_build(torch.ones(N + 1, M, dtype=torch.int32, device="cuda:0"), N)
    got = torch.full((M, N + 1), 7.0, device="cuda:0")
    _hip.gs_scatter_tokens(torch.randn(1, M * N, device="cuda:0"), ib["idx_Msum"], ib["cumsums_N"], got)
    assert not got.any()


@pytest.mark.parametrize("transposed", [False, True])
def test_gate_gradient_has_the_layout_of_the_gate_weights(transposed):
    x, W1, W2, mask, s, dy = make_layer_inputs(70, 64, 32, 9, 3, seed=4)
    want = run_device_layer(x, W1, W2, mask, s, dy, 3, 0)["G_s"]
    import momoe_amd
    layer = momoe_amd.MoMoE(64, 32, 9, 3, save_percent=0, Wl1_ND2H=W1.to("cuda:0"), Wl2_NHD=W2.to("cuda:0"))
    s_dev = (s.T.contiguous().to("cuda:0").T if transposed else s.contiguous().to("cuda:0")).requires_grad_()
    y, _ = layer(x.to("cuda:0", torch.bfloat16)[None], mask.to("cuda:0"), s_dev)
    y.backward(dy.to("cuda:0", torch.bfloat16)[None])
    assert s_dev.grad.stride() == s_dev.stride() and torch.equal(s_dev.grad.cpu(), want)


@pytest.mark.parametrize("M,D,H,N,K,sp", [
    (300, 128, 96, 8, 3, 40),      # few tiles: the module has a partial dL/ds per 64 hidden columns
    (2000, 352, 288, 72, 3, 100),
    (2000, 352, 288, 72, 3, 0),
])
def test_entry_points_one_by_one(M, D, H, N, K, sp):
    """The launch sequence of a forward and backward through the C entry points, in buffers of the
    caller's own, gives what the module gives."""
    from momoe_amd import _hip
    dev = "cuda:0"
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, seed=9)
    want = run_device_layer(x, W1, W2, mask, s, dy, K, sp)
    b = lambda t: t.to(dev, torch.bfloat16)
    new = lambda *size, dtype=torch.bfloat16: torch.full(size, 7, device=dev, dtype=dtype)
    x, W1, W2, Gy, sd = b(x), b(W1), b(W2), b(dy), s.T.contiguous().to(dev).T
    msum, msave = M * K, M * K * sp // 100
    ib = _hip.index_build(mask.to(dev), K, recompute_table=True)
    idx, cumsums, inv, table = (ib[k] for k in ("idx_Msum", "cumsums_N", "inv_MK", "tile_table"))

    h, ab, ys, y = new(H // 32, msum, 32), new(msave, 2 * H) if msave else None, new(msum, D), new(M, D)
    _hip.lin1_swiglu_fwd(x, W1, idx, table, h, ab, 0, msave)
    _hip.lin2_scale_fwd(h, W2, sd, idx, table, ys, M)
    _hip.combine(ys, inv, y)

    u, gz, hsT = new(msum, H), new(2 * H // 32, msum, 32), new(_hip.padded_rows(msum, N) // 32, H, 32)
    gs_part, Gs = new(-(-H // _hip.GS_BLOCK), msum, dtype=torch.float32), new(N, M, dtype=torch.float32)
    GW1, GW2, gxs, Gx = new(N, D, 2 * H), new(N, H, D), new(msum, D), new(M, D)
    ws = lambda X, Y: min(msum * H * 2, _hip.wgrad_workspace_bytes(N, X, Y, msum))
    _hip.dgrad_h(Gy, W2, idx, table, u)
    if msave:
        _hip.swiglu_bwd_saved(ab, u, sd, idx, cumsums, msave, gz, hsT, gs_part)
    _hip.lin1_swiglu_bwd(x, W1, idx, ib["recompute_table"], u, sd, msave, gz, hsT, gs_part)
    _hip.gs_scatter(gs_part, idx, cumsums, Gs)
    _hip.wgrad(hsT, None, Gy, idx, cumsums, GW2, M, msum, workspace_bytes=ws(H, D), a_transposed=True)
    _hip.wgrad(x, idx, gz, None, cumsums, GW1, M, msum, workspace_bytes=ws(D, 2 * H), b_kblocked=True)
    _hip.dgrad_x(gz, W1, table, gxs, M)
    _hip.combine(gxs, inv, Gx)
    torch.cuda.synchronize()
    for k, got in (("sizes", ib["sizes_N"]), ("y", y), ("G_x", Gx), ("G_W1", GW1), ("G_W2", GW2)):
        assert torch.equal(got.cpu(), want[k]), k
    # fp32 sums of at most ceil(H/64) partial sums in another grouping
    torch.testing.assert_close(Gs.cpu(), want["G_s"], rtol=1e-5, atol=1e-5 * want["G_s"].abs().max().item())


def test_recomputing_gemm_ignores_a_table_of_taller_tiles():
    """momoe_lin1_swiglu_bwd takes row tiles of at most 256 rows: given the 320-row table of the other
    GEMMs it must leave its outputs alone instead of computing on tiles it cannot hold."""
    from momoe_amd import _hip
    M, D, H, N, K = 2048, 128, 64, 2, 1
    x, W1, _, mask, s, _ = make_layer_inputs(M, D, H, N, K, seed=5)
    dev = "cuda:0"
    ib = _hip.index_build(mask.to(dev), K, tile_rows=_hip.TILE_ROWS)
    msum = M * K
    assert _hip.TILE_ROWS > _hip.RECOMPUTE_TILE_ROWS and int(ib["sizes_N"].max()) > _hip.RECOMPUTE_TILE_ROWS
    u = torch.randn(msum, H, device=dev).to(torch.bfloat16)
    xb, W1b, sd = x.to(dev).to(torch.bfloat16), W1.to(dev), s.to(dev)

    def run(table):
        gz = torch.full((2 * H // 32, msum, 32), 7.0, device=dev, dtype=torch.bfloat16)
        hsT = torch.full((_hip.padded_rows(msum, N) // 32, H, 32), 7.0, device=dev, dtype=torch.bfloat16)
        gs_part = torch.full(((H + _hip.GS_BLOCK - 1) // _hip.GS_BLOCK, msum), 7.0, device=dev)
        _hip.lin1_swiglu_bwd(xb, W1b, ib["idx_Msum"], table, u, sd, 0, gz, hsT, gs_part)
        torch.cuda.synchronize()
        return gz, hsT, gs_part

    for t in run(ib["tile_table"]):
        assert bool((t == 7.0).all())
    own = _hip.tile_table_build(ib["cumsums_N"], M, K, _hip.RECOMPUTE_TILE_ROWS)
    assert not bool((run(own)[0] == 7.0).all())


@pytest.mark.parametrize("M,D,H,N,K,Ks,skew,row_lo", [
    (3000, 1056, 416, 12, 4, 0, None, 0),     # 16.5 stages; a column block whose second half is past H
    (2500, 2080, 352, 14, 4, 1, 1.0, 4001),   # tiles of 1 to 8 fragment rows, a boundary inside an expert
    (2600, 2048, 288, 24, 3, 0, 0.5, 2048),   # one 32-column block in the last tile
])
def test_recomputing_gemm_in_the_span_loop(M, D, H, N, K, Ks, skew, row_lo):
    """G_z, hs^T and the partial dL/ds against 64-bit arithmetic.  Bounds: a and b are fp32 sums of D exact
    products, D 2^-24 of their absolute sum off; that error times the derivatives (|silu'| <= 1.1, |silu''| <=
    0.5); fp32 arithmetic and the fast exp and reciprocal, 2^-19 of the factors; bf16 results, 2^-8."""
    from momoe_amd import _hip
    dev = "cuda:0"
    x, W1, _, mask, s, _ = make_layer_inputs(M, D, H, N, K, Ks=Ks, seed=8, skew=skew)
    msum = M * K
    assert _hip._lib.momoe_recompute_stage_k(msum, N, D, H) == 64
    ib = _hip.index_build(mask.to(dev), K, recompute_table=True)
    idx, c = ib["idx_Msum"], [0] + mask.sum(1).cumsum(0).tolist()
    xb, W1b, sd = x.to(dev).to(torch.bfloat16), W1.to(dev).to(torch.bfloat16), s.to(dev)
    u = torch.randn(msum, H, generator=torch.Generator(device=dev).manual_seed(3), device=dev).to(torch.bfloat16)

    def run(table):
        full = lambda *shape, dt=torch.bfloat16: torch.full(shape, 7.0, device=dev, dtype=dt)
        out = (full(2 * H // 32, msum, 32), full(_hip.padded_rows(msum, N) // 32, H, 32),
               full(-(-H // _hip.GS_BLOCK), msum, dt=torch.float32))
        _hip.lin1_swiglu_bwd(xb, W1b, idx, table, u, sd, row_lo, *out)
        return out

    tall = _hip.tile_table_build(ib["cumsums_N"], M, K, _hip.TILE_ROWS)
    assert all(bool((t == 7.0).all()) for t in run(tall))  # tiles too tall: nothing is written
    gz, hsT, gs = run(ib["recompute_table"])
    gz = gz.permute(1, 0, 2).reshape(msum, 2 * H)
    hs = hsT.permute(0, 2, 1).reshape(-1, H)
    assert torch.isfinite(gs).all()
    for e in range(N):
        r0, r1 = c[e], c[e + 1]
        lo = r0 + max(0, row_lo - r0) // 32 * 32  # groups of 32 rows from the expert's first
        if row_lo >= r1:  # its rows are all below
            assert bool((gz[r0:r1] == 7.0).all()) and bool((gs[:, r0:r1] == 7.0).all())
            continue
        assert bool((gz[r0:lo] == 7.0).all()) and bool((gs[:, r0:lo] == 7.0).all())
        tok, x64, w64 = idx[lo:r1].long(), xb[idx[lo:r1].long()].double().cpu(), W1b[e].double().cpu()
        ab, size = x64 @ w64, x64.abs() @ w64.abs() * (D * 2.0**-24)
        (va, vb), (ea, eb) = ab.split(H, 1), size.split(H, 1)
        sv, u64 = sd[e, tok].double().cpu()[:, None], u[lo:r1].double().cpu()
        sg = torch.sigmoid(vb)
        silu, d = vb * sg, sg * (1 + vb * (1 - sg))
        su, near = (sv * u64).abs(), 2.0**-19 * (1 + va.abs()) * (1 + vb.abs())

        def check(got, want, err, what):
            bound = want.abs() * 2.0**-8 + 1.01 * err
            assert bool(((got.double().cpu() - want).abs() <= bound).all()), f"{what} of expert {e}"

        eh = 1.1 * va.abs() * eb + silu.abs() * ea + near  # of a silu(b)
        check(gz[lo:r1, :H], sv * u64 * silu, su * (1.1 * eb + near), "G_a")
        check(gz[lo:r1, H:], sv * u64 * va * d, su * (1.1 * ea + 0.5 * va.abs() * eb + near), "G_b")
        p0 = (r0 + 31) // 32 * 32 + 32 * e + lo - r0
        n = r1 - lo
        check(hs[p0:p0 + n], sv * va * silu, sv.abs() * eh, "hs")
        assert bool((hs[p0 + n:p0 + (n + 31) // 32 * 32] == 0).all())
        for b in range(gs.shape[0]):
            cols = slice(128 * b, min(H, 128 * b + 128))
            t = u64[:, cols] * (va * silu)[:, cols]
            err = (u64.abs() * eh)[:, cols].sum(1) + 128 * 2.0**-24 * t.abs().sum(1)
            assert bool(((gs[b, lo:r1].double().cpu() - t.sum(1)).abs() <= err).all()), f"dL/ds {b} of expert {e}"


@pytest.mark.parametrize("sp", [0, 40])
def test_both_row_tile_geometries_give_the_same_layer(sp):
    """Experts of 1..700 rows on 256-row and on 320-row tiles (and on the library's own choice): the
    contraction order does not depend on the tile height, so every result is bit-identical, and
    the 320-row path is checked against the oracle like any other."""
    from momoe_amd import _hip, experts
    M, D, H, N, K = 1500, 160, 96, 12, 3
    x, W1, W2, mask, s, dy = make_layer_inputs(M, D, H, N, K, seed=21, skew=1.2)
    assert int(mask.sum(1).max()) > 2 * _hip.RECOMPUTE_TILE_ROWS  # several tiles, ragged
    outs = {}
    try:
        for rows in (_hip.RECOMPUTE_TILE_ROWS, _hip.TILE_ROWS, _hip.AUTO_TILE_ROWS, 288):
            experts.TILE_ROWS = rows
            outs[rows] = run_device_layer(x, W1, W2, mask, s, dy, K, sp)
    finally:
        experts.TILE_ROWS = _hip.AUTO_TILE_ROWS
    ref = run_oracle_layer(x, W1, W2, mask, s, dy)
    _check_all(outs[_hip.TILE_ROWS], ref)
    base = outs[_hip.RECOMPUTE_TILE_ROWS]
    for rows, got in outs.items():
        for k in base:
            assert torch.equal(got[k], base[k]), (rows, k)
