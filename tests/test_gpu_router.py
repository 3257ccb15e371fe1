"""GPU: TopKRouter kernels and the MoE wrapper against the oracle."""
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


def _logits(M, N, seed):
    return torch.randn(M, N, generator=torch.Generator().manual_seed(seed))


@pytest.mark.parametrize("M,N,K,Ks,f32", [
    (128, 8, 2, 0, True), (8192, 128, 8, 0, True), (1000, 64, 8, 4, True),
    (513, 200, 6, 1, True), (2048, 128, 8, 0, False),
    (77, 300, 8, 3, True),      # more than 256 experts: 8 columns per lane
    (33, 64, 3, 0, True),       # one column per lane, a partial block of tokens
    (4096, 96, 6, 2, True),     # the most tokens with one per wavefront
    (4097, 130, 6, 2, True),    # one more: two per wavefront, a last block of one token
    (17, 512, 8, 1, True),      # the most experts, a last block of one token
    (64, 8, 8, 0, True),        # every expert is chosen
    (1, 1, 1, 0, True), (3, 65, 4, 1, True), (5, 129, 4, 0, True), (7, 257, 5, 2, True),  # blocks of four tokens, a part of one
    (3072, 64, 4, 0, True), (3073, 64, 4, 0, True),  # the most tokens in blocks of four, one more
])
def test_router_forward(M, N, K, Ks, f32):
    from momoe_amd import _hip
    lg = _logits(M, N, 1)
    if not f32:
        lg = lg.to(torch.bfloat16)
    g = torch.Generator().manual_seed(2)
    bias = torch.cat([torch.randn(N - Ks, generator=g) * 1e-3, torch.full((Ks,), float("-inf"))])
    ref = oracle.router_forward(None, None, bias, N, K, Ks, logits=lg.float())
    mask, s_MN, p_sel, Ng_M, Ks_M = _hip.router_fwd(lg.to("cuda:0"), bias.to("cuda:0"), K, Ks)
    torch.cuda.synchronize()
    if f32:
        assert torch.equal(mask.cpu(), ref["mask_NM"])  # routing bit-exact on tie-free fp32 logits
    else:
        # bf16 logits contain exact ties, whose order torch.topk leaves unspecified:
        # compare only tokens whose K-th and (K+1)-th scores differ
        sc = torch.softmax(lg.float()[:, :N - Ks], -1) + bias[:N - Ks]
        top = torch.topk(sc, K - Ks + 1, dim=-1).values
        clear = (top[:, -2] - top[:, -1]) > 1e-6
        assert clear.float().mean() > 0.9
        assert torch.equal(mask.cpu()[:, clear], ref["mask_NM"][:, clear])
        return
    assert mask.dtype == torch.int32 and mask.is_contiguous()
    torch.testing.assert_close(s_MN.cpu(), ref["s_NM"].T, rtol=1e-5, atol=1e-7)
    torch.testing.assert_close(p_sel.cpu(), ref["p_sel_MN"], rtol=1e-5, atol=1e-7)
    torch.testing.assert_close(Ng_M.cpu(), ref["Ng_M"], rtol=1e-5, atol=1e-7)
    if Ks:
        torch.testing.assert_close(Ks_M.cpu(), ref["Ks_M"], rtol=1e-5, atol=1e-7)


def test_router_forward_takes_equal_scores_in_column_order():
    """Whole numbers as logits (few distinct scores, the two lowest -inf through the bias) and every
    column: of equal scores the lowest columns are taken, as a stable sort gives them."""
    from momoe_amd import _hip
    M, N, K = 300, 130, 8
    lg = torch.randint(0, 3, (M, N), generator=torch.Generator().manual_seed(5)).float()
    lg[0] = 1.0
    bias = torch.zeros(N)
    bias[3:] = torch.where(torch.arange(3, N) % 5 == 0, torch.tensor(0.0), torch.tensor(float("-inf")))
    bias[40:] = float("-inf")
    mask = _hip.router_fwd(lg.to("cuda:0"), bias.to("cuda:0"), K, 0)[0].cpu()
    # every column's exponential is one of three values, so equal logits have equal probabilities
    key = torch.where(torch.isinf(bias), torch.tensor(-1.0), lg)
    want = torch.zeros(M, N, dtype=torch.int32)
    want.scatter_(1, torch.sort(key, dim=1, descending=True, stable=True).indices[:, :K], 1)
    assert torch.equal(mask.T, want)


@pytest.mark.parametrize("M,N,K,Ks", [(256, 16, 4, 0), (1000, 64, 8, 4), (300, 130, 5, 2),
                                      (90, 300, 8, 3),     # more than 256 experts: blocks of 16 tokens
                                      (8192, 128, 8, 0)])  # the headline routing
def test_router_backward(M, N, K, Ks):
    from momoe_amd import _hip
    lg = _logits(M, N, 3)
    bias = torch.cat([torch.zeros(N - Ks), torch.full((Ks,), float("-inf"))])
    ref = oracle.router_forward(None, None, bias, N, K, Ks, logits=lg)
    G_s = torch.randn(N, M, generator=torch.Generator().manual_seed(4)) * (ref["mask_NM"] != 0)
    want = oracle.router_backward_closed_form(G_s, ref["p_sel_MN"], ref["s_NM"], ref["Ng_M"], ref["Ks_M"],
                                              ref["mask_NM"], Ks, round_bf16=True)
    d = lambda t: t.contiguous().to("cuda:0")
    got = _hip.router_bwd(d(G_s), d(ref["p_sel_MN"]), d(ref["s_NM"].T), d(ref["Ng_M"]), d(ref["Ks_M"]),
                          d(ref["mask_NM"]), Ks)
    torch.cuda.synchronize()
    assert got.dtype == torch.bfloat16
    torch.testing.assert_close(got.float().cpu(), want, rtol=1e-2, atol=1e-6)
    # strided G_s (transposed view) gives the same answer
    got2 = _hip.router_bwd(d(G_s.T).T, d(ref["p_sel_MN"]), d(ref["s_NM"].T), d(ref["Ng_M"]),
                           d(ref["Ks_M"]), d(ref["mask_NM"]), Ks)
    assert torch.equal(got, got2)


def test_moe_wrapper_against_oracle_and_state_dict():
    import momoe_amd
    torch.manual_seed(0)
    B, S, D, H, N, K, Ks = 2, 256, 256, 128, 16, 4, 1
    Wg = torch.randn(D, N) * 0.1
    W1 = torch.randn(N, D, 2 * H) * 0.02
    W2 = torch.randn(N, H, D) * 0.02
    x = torch.randn(B, S, D)
    dy = torch.randn(B, S, D)
    moe = momoe_amd.MoE(D, H, N, K, Ks, save_percent=0, bias_update_rate=1e-2,
                        Wg_DN=Wg.cuda(), Wl1_ND2H=W1.cuda(), Wl2_NHD=W2.cuda())
    assert set(moe.state_dict().keys()) == {"biases_N", "router.Wg_DN", "momoe.Wl1_ND2H", "momoe.Wl2_NHD"}
    ref = oracle.OracleMoE(D, H, N, K, Ks, bias_update_rate=1e-2, Wg_DN=Wg, Wl1_ND2H=W1.bfloat16(),
                           Wl2_NHD=W2.bfloat16())
    ref.load_state_dict({k: v.cpu().float() if "Wl" in k else v.cpu() for k, v in moe.state_dict().items()})
    xd = x.cuda().bfloat16().requires_grad_()
    xo = x.bfloat16().float().requires_grad_()
    # The gate logits are bf16 (momoe/topk_router.py:95) and contain exact ties, whose order
    # torch.topk leaves unspecified while the device kernel picks the lower index.  So the
    # device's selection is first checked to be A valid top-k under the oracle's own scores
    # (no unselected expert scores higher than a selected one, up to one rounding step of the
    # logits), then handed to the oracle, and everything after it is compared element by element.
    with torch.no_grad():
        _, mask_dev, _ = moe.router(xd, moe.biases_N)
    mask_dev = mask_dev.cpu()
    own = oracle.router_forward(xo.reshape(B * S, D), Wg, ref.biases_N, N, K, Ks)
    sc = own["sel_scores_MNg"]
    chosen = mask_dev[:N - Ks].T != 0
    assert torch.all(chosen.sum(1) == K - Ks) and torch.all(mask_dev[N - Ks:] == 1)
    worst_in = torch.where(chosen, sc, torch.full_like(sc, float("inf"))).min(1).values
    best_out = torch.where(chosen, torch.full_like(sc, float("-inf")), sc).max(1).values
    assert torch.all(worst_in >= best_out - 1e-2 * sc.max(1).values)
    print(f"[routing] {int((mask_dev != own['mask_NM']).any(0).sum())} of {B * S} tokens are routed "
          "differently by torch.topk on the CPU (ties / last-bit logit differences)")
    ref.router.forced_mask_NM = mask_dev

    y = moe(xd)
    yo = ref(xo)
    y.backward(dy.cuda().bfloat16())
    yo.backward(dy.bfloat16().float())
    torch.cuda.synchronize()
    from gpu_util import assert_close, rel_err
    assert torch.equal(moe.biases_N.cpu(), ref.biases_N)
    assert_close(y, yo, "y")
    assert_close(xd.grad, xo.grad, "G_x", rel=2e-2)
    assert_close(moe.momoe.Wl1_ND2H.grad, ref.momoe.Wl1_ND2H.grad, "G_Wl1", rel=2e-2)
    assert_close(moe.momoe.Wl2_NHD.grad, ref.momoe.Wl2_NHD.grad, "G_Wl2", rel=2e-2)
    # dL/dWg = x^T . G_logit sums over all tokens, and G_logit = p*(o - <o,p>) cancels heavily,
    # so the bf16-level differences of dL/ds are amplified: the element-wise bound is relative
    # to the tensor's RMS (a misplaced row or column would be off by the RMS itself)
    gw, gwo = moe.router.Wg_DN.grad.float().cpu(), ref.router.Wg_DN.grad.float()
    rms = gwo.pow(2).mean().sqrt()
    assert torch.all((gw - gwo).abs() <= 0.15 * rms + 2e-2 * gwo.abs())
    assert rel_err(gw, gwo) < 5e-2
    assert moe.biases_N[-1].item() == float("-inf")


@pytest.mark.parametrize("grad", [True, False])
def test_router_under_autocast(grad):
    """autocast decides the type of the gate product: bfloat16 changes nothing, float16 (its default)
    is refused, since the kernel reads bfloat16 and float32 logits only."""
    import momoe_amd
    torch.manual_seed(3)
    D, H, N, K, Ks = 64, 32, 8, 3, 1
    moe = momoe_amd.MoE(D, H, N, K, Ks, bias_update_rate=0.0)
    x = torch.randn(2, 24, D, device="cuda", dtype=torch.bfloat16)
    with torch.set_grad_enabled(grad):
        want = [*moe.router(x, moe.biases_N), moe(x)]
        with torch.autocast("cuda", dtype=torch.bfloat16):
            got = [*moe.router(x, moe.biases_N), moe(x)]
        with torch.autocast("cuda", dtype=torch.float16):
            with pytest.raises(AssertionError, match="logits"):
                moe.router(x, moe.biases_N)
            with pytest.raises(AssertionError, match="logits"):
                moe(x)
    for g, w in zip(got, want):
        assert g.dtype == w.dtype and torch.equal(g, w)


def test_training_smoke_loss_decreases():
    # scaled-down version of the reference's only test (momoe/test.py): AdamW on
    # mean((y - x)^2); the loss starts near 1 and must go down.
    import momoe_amd
    torch.manual_seed(0)
    B, S, D, H, N, K, Ks = 4, 1024, 256, 128, 32, 6, 1
    x = torch.randn(B, S, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    moe = momoe_amd.MoE(D, H, N, K, Ks, save_percent=0, bias_update_rate=1e-4)
    opt = torch.optim.AdamW(moe.parameters(), lr=1e-3)
    losses = []
    for _ in range(40):
        y = moe(x)
        loss = torch.mean(torch.square(y.float() - x.float()))
        loss.backward()
        opt.step()
        opt.zero_grad()
        losses.append(loss.item())
    assert 0.5 < losses[0] < 1.5
    assert losses[-1] < 0.9 * losses[0]


def test_training_smoke_at_the_reference_size():
    # momoe/test.py as written: B,S,D,H = 4,8192,1024,512; N,K,Ks = 32,6,1; 10 warm-up forwards,
    # then 200 AdamW steps (lr 1e-3) on mean((y - x)^2).  Its docstring is the only expected
    # result the reference states: the loss starts around 1 and goes down towards 0.
    import momoe_amd
    torch.manual_seed(0)
    B, S, D, H, N, K, Ks = 4, 8192, 1024, 512, 32, 6, 1
    x = torch.randn(B, S, D, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    moe = momoe_amd.MoE(D, H, N, K, Ks, save_percent=0, bias_update_rate=1e-4)
    for _ in range(10):
        moe(x)
    opt = torch.optim.AdamW(moe.parameters(), lr=1e-3)
    losses = []
    for _ in range(200):
        x.grad = torch.zeros_like(x)
        y = moe(x)
        loss = torch.mean(torch.square(y.float() - x.float()))
        loss.backward()
        opt.step()
        opt.zero_grad()
        losses.append(loss.item())
    assert all(l == l for l in losses), "loss became NaN"
    assert 0.8 < losses[0] < 1.2
    assert losses[-1] < 0.5 * losses[0]
    assert losses[-1] == min(losses[-20:]) or losses[-1] < 1.05 * min(losses[-20:])
    # the routed experts' selection bias moved by at most 210 steps of the update rate
    b = moe.biases_N[:N - Ks]
    assert torch.all(b.abs() <= 210 * 1e-4 + 1e-6) and torch.all(torch.isinf(moe.biases_N[N - Ks:]))


@pytest.mark.parametrize("M,D,N", [
    (1, 8, 8), (64, 128, 128), (65, 136, 136), (255, 120, 16),   # tiles of 128 x 128, stages of 64 tokens
    (256, 128, 8), (257, 256, 64), (1537, 40, 24), (8200, 2048, 128),  # one range of tokens and several, the last a part
])
def test_gate_weight_gradient(M, D, N):
    from momoe_amd import _hip
    g = torch.Generator(device="cuda:0").manual_seed(M)
    wide = torch.randn(M, D + 8, generator=g, device="cuda:0").to(torch.bfloat16)
    gl = torch.randn(M, N, generator=g, device="cuda:0").to(torch.bfloat16)
    for x in (wide[:, :D].contiguous(), wide[:, :D]):
        got = torch.full((D, N), 7.0, device="cuda:0", dtype=torch.bfloat16)
        _hip.gate_wgrad(x, gl, got)
        xd, gd = x.double(), gl.double()
        ref, size = xd.T.contiguous() @ gd, xd.abs().T.contiguous() @ gd.abs()
        # bf16 rounding of the result, and M fp32 additions of products of that size
        assert ((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + M * 2.0 ** -24 * size).all()
    # an infinite token stays in its own column of x
    x = wide[:, :D].contiguous()
    x[M - 1, 3] = float("inf")
    _hip.gate_wgrad(x, gl.abs() + 1, got)
    assert torch.isinf(got[3]).all() and torch.isfinite(torch.cat([got[:3], got[4:]])).all()


def test_gate_weight_gradient_in_many_tiles():
    """130 tiles: one range, though of more tokens than a range has elsewhere."""
    from momoe_amd import _hip
    M, D, N = 600, 16520, 8
    ranges = lambda D: _hip._lib.momoe_gate_wgrad_workspace_bytes(M, D, N) // (D * N * 4)
    assert ranges(D) == 1 and ranges(8256) == 3
    test_gate_weight_gradient(M, D, N)


@pytest.mark.parametrize("M,D,N", [
    (1, 8, 8), (64, 64, 32), (127, 128, 40), (129, 136, 136), (300, 264, 512), (8192, 64, 64),  # tiles of 128 x 128, 32 k-values
])
@pytest.mark.parametrize("add", [False, True])
def test_gate_input_gradient(M, D, N, add):
    from momoe_amd import _hip
    g = torch.Generator(device="cuda:0").manual_seed(M)
    rnd = lambda *size: torch.randn(*size, generator=g, device="cuda:0").to(torch.bfloat16)
    gl, Wg, gx = rnd(M, N), rnd(D, N), rnd(M, D)
    out = torch.full((M, D), 7.0, device="cuda:0", dtype=torch.bfloat16)
    kept = gx.clone()
    _hip.gate_dgrad(gl, Wg, gx if add else None, out)
    assert torch.equal(gx, kept)
    ref, size = gl.double() @ Wg.double().T.contiguous(), gl.double().abs() @ Wg.double().abs().T.contiguous()
    if add:
        ref, size = ref + gx.double(), size + gx.double().abs()
    # bf16 rounding of the result, and N + 1 fp32 additions of that size
    assert ((out.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + (N + 1) * 2.0 ** -24 * size).all()
    gl[M // 2, N - 1] = float("inf")  # a token that is not finite is alone in that
    want, rest = out.clone(), torch.arange(M, device="cuda:0") != M // 2
    _hip.gate_dgrad(gl, Wg, gx if add else None, out)
    assert torch.equal(out[rest], want[rest]) and not torch.isfinite(out[M // 2]).any()


@pytest.mark.parametrize("M,D,N", [(1, 64, 16), (300, 64, 16), (2000, 72, 20), (1600, 96, 24)])
@pytest.mark.parametrize("pitch", [0, 4, 8])
def test_gate_gradients_of_the_module(M, D, N, pitch):
    """Whichever product the module takes, by the widths and the layout of x, the gradients are those of
    the library's, which a backward that is itself recorded takes."""
    import momoe_amd
    g = torch.Generator(device="cuda:0").manual_seed(D)
    r = momoe_amd.TopKRouter(D, N, 4, 0, Wg_DN=torch.randn(D, N, generator=g, device="cuda:0").to(torch.bfloat16) / 8)
    x = torch.randn(1, M, D + pitch, generator=g, device="cuda:0").to(torch.bfloat16)[..., :D]
    w = torch.randn(N, M, generator=g, device="cuda:0")
    x.requires_grad_()
    for through in (False, True):  # a gradient of x from elsewhere is added
        grads = []
        for recorded in (False, True):
            out = r(x, torch.zeros(N, device="cuda:0"))
            loss = (out[2] * w).sum() + (out[0].float().square().sum() if through else 0.0)
            grads.append([t.detach().double() for t in torch.autograd.grad(loss, (r.Wg_DN, x), create_graph=recorded)])
        for got, want in zip(*grads):
            assert got.shape == want.shape and (got - want).abs().max() <= 2.0 ** -7 * want.abs().max()


def _gate_backward(M, D, N):
    """The entry points that a backward of the router calls, and its gradients next to the library's."""
    import momoe_amd
    from momoe_amd import _hip
    g = torch.Generator(device="cuda:0").manual_seed(D)
    r = momoe_amd.TopKRouter(D, N, 4, 0, Wg_DN=torch.randn(D, N, generator=g, device="cuda:0").to(torch.bfloat16) / D ** 0.5)
    x = torch.randn(1, M, D, generator=g, device="cuda:0").to(torch.bfloat16).requires_grad_()
    w = torch.randn(M, N, generator=g, device="cuda:0").T

    def grads(recorded):
        out = r(x, torch.zeros(N, device="cuda:0"))
        return torch.autograd.grad((out[2], out[0]), (r.Wg_DN, x), (w, x.detach()), create_graph=recorded)

    want = grads(True)  # (a backward that is itself recorded takes the library's products)
    with _hip.kernel_timer() as kt:
        got = grads(False)
    for a, b in zip(got, want):
        assert a.shape == b.shape and (a.double() - b.double()).abs().max() <= 2.0 ** -7 * b.double().abs().max()
    return [n for n, _ in kt.durations_ms()]


@pytest.mark.parametrize("M,D,N,own", [
    (5000, 8192, 128, True), (64, 512, 256, True), (4096, 1024, 512, True), (2048, 4096, 256, True),
    (2049, 4096, 256, False), (4097, 1024, 512, False),  # more than 128 experts and 2^31 terms
])
def test_which_product_takes_the_gradient_of_the_tokens(M, D, N, own):
    assert ("momoe_gate_dgrad" in _gate_backward(M, D, N)) == own


@pytest.mark.parametrize("M,D,N,own", [
    (1, 2048, 128, True), (1, 2056, 128, False),                              # up to 2^18 results: any number of tokens
    (512, 2048, 256, True), (511, 2048, 256, False), (1024, 2048, 512, True),  # more: by tokens
    (4200, 4096, 264, False),                                                # more than 2^20
])
def test_which_product_takes_the_gradient_of_the_gate_weights(M, D, N, own):
    assert ("momoe_gate_wgrad" in _gate_backward(M, D, N)) == own


def _whole_numbers(M, D, N, pitch=0):
    """x, Wg whose products have the same sum in any order: small whole numbers."""
    g = torch.Generator().manual_seed(M + D + N)
    x = torch.randint(-3, 4, (M, D + pitch), generator=g).to("cuda:0", torch.bfloat16)[:, :D]
    return x, torch.randint(-2, 3, (D, N), generator=g).to("cuda:0", torch.bfloat16)


@pytest.mark.parametrize("M,D,N,K,Ks", [
    (1, 8, 8, 1, 0), (3, 40, 24, 5, 1), (63, 128, 128, 8, 0), (64, 136, 136, 4, 0),  # parts of 128 k-values, blocks of
    (65, 192, 64, 4, 2), (16, 2048, 128, 8, 0), (130, 1000, 512, 8, 0),              # 128 experts and 64 tokens
    (2048, 256, 16, 2, 0), (2, 2184, 32, 4, 0),  # the most tokens; 18 parts, two rounds of them
])
@pytest.mark.parametrize("pitch", [0, 8])
def test_router_with_its_product(M, D, N, K, Ks, pitch):
    from momoe_amd import _hip
    x, Wg = _whole_numbers(M, D, N, pitch)
    bias = torch.cat([torch.randn(N - Ks, generator=torch.Generator().manual_seed(1)) * 1e-3, torch.full((Ks,), float("-inf"))]).to("cuda:0")
    logits = (x.double().cpu() @ Wg.double().cpu()).to("cuda:0", torch.float32).to(torch.bfloat16)
    want = _hip.router_fwd(logits, bias, K, Ks)
    for a, b in zip(_hip.gate_router_fwd(x, Wg, bias, K, Ks), want):
        assert torch.equal(a, b)
    # a token that is not finite is alone in that
    x[M // 2, D - 1] = float("inf")
    got = _hip.gate_router_fwd(x, Wg, bias, K, Ks)
    rest = torch.arange(M, device="cuda:0") != M // 2
    assert torch.equal(got[0][:, rest], want[0][:, rest]) and torch.equal(got[1][rest], want[1][rest])


def test_sizes_the_router_with_its_product_refuses():
    from momoe_amd import _hip
    for M, D, N in [(2049, 64, 8), (1025, 2048, 8), (4, 20, 8), (4, 64, 12), (4, 64, 520)]:
        assert _hip._lib.momoe_gate_router_workspace_bytes(M, D, N) == -1
        with pytest.raises(RuntimeError):
            _hip.gate_router_fwd(*_whole_numbers(M, D, N), torch.zeros(N, device="cuda:0"), 2, 0)


@pytest.mark.parametrize("M,D,N,pitch", [(2048, 64, 8, 0), (2049, 64, 8, 0), (5, 20, 8, 0), (5, 64, 12, 0), (5, 64, 8, 4), (5, 64, 8, 8)])
def test_module_routes_alike_by_either_product(M, D, N, pitch):
    import momoe_amd
    from momoe_amd import _hip
    x, Wg = _whole_numbers(M, D, N, pitch)
    bias = torch.zeros(N, device="cuda:0")
    want = _hip.router_fwd((x.double().cpu() @ Wg.double().cpu()).to("cuda:0", torch.bfloat16), bias, 2, 0)
    for weight in (Wg, Wg.T.contiguous().T):
        r = momoe_amd.TopKRouter(D, N, 2, 0, Wg_DN=Wg)
        r.Wg_DN.data = weight
        for grad in (False, True):
            with torch.set_grad_enabled(grad):
                out = r(x[None], bias)
            assert torch.equal(out[1], want[0]) and torch.equal(out[2], want[1].T)


def test_the_product_of_many_tokens_comes_before_what_the_host_allocates():
    """The GPU has the product to work on while the host goes on with the call."""
    import momoe_amd
    from torch.utils._python_dispatch import TorchDispatchMode

    class Recorded(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            names.append(func.overloadpacket.__name__)
            return func(*args, **(kwargs or {}))

    names = []
    x, Wg = _whole_numbers(3000, 64, 8)
    r, bias = momoe_amd.TopKRouter(64, 8, 2, 0, Wg_DN=Wg), torch.zeros(8, device="cuda:0")
    with torch.no_grad(), Recorded():
        r(x[None], bias)
    assert "mm" in names and "empty" in names and names.index("mm") < names.index("empty")
    r.Wg_DN.data = Wg.flatten()  # what is no matrix is refused as the product refuses it
    with pytest.raises(RuntimeError):
        r(x[None, :5], bias)


def test_gate_gradients_of_widths_that_the_kernels_refuse():
    import momoe_amd
    from momoe_amd import _hip
    M, D, N, K = 3, (1 << 20) + 8, 8, 2
    x, Wg = _whole_numbers(M, D, N)
    r = momoe_amd.TopKRouter(D, N, K, 0, Wg_DN=Wg)
    w = torch.randn(M, N, generator=torch.Generator(device="cuda:0").manual_seed(3), device="cuda:0").T
    xg = x[None].clone().requires_grad_()
    out = r(xg, torch.zeros(N, device="cuda:0"))
    GW, Gx = torch.autograd.grad((out[2], out[0]), (r.Wg_DN, xg), (w, x[None]))
    mask, s, p_sel, Ng, Ks = _hip.router_fwd(torch.mm(x, Wg), torch.zeros(N, device="cuda:0"), K, 0)
    assert torch.equal(out[1], mask) and torch.equal(out[2], s.T)
    G, xd, Wd = _hip.router_bwd(w, p_sel, s, Ng, Ks, mask, 0).double(), x.double(), Wg.double()
    # one rounding to bf16 (2^-8), and of the sums in fp32
    for got, want, terms in ((GW, xd.T @ G, xd.T.abs() @ G.abs()), (Gx[0], xd + G @ Wd.T, xd.abs() + G.abs() @ Wd.T.abs())):
        assert got.shape == want.shape and ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -20 * terms).all()

