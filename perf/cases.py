"""The workloads this framework is timed on: what its users run, through `MoMoE` and `MoE`.

A case is one call of a mixture-of-experts layer: a forward under `no_grad` (decode, prefill) or a
forward and backward (a training step without the optimizer).  `draw` gives further cases of the
same ranges.  Sizes: D = model width, H = hidden width of an expert, N = experts (the shared ones
included), K = experts per token (shared included), Ks = shared experts, tokens = rows of x.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("momoe-impl_amd"))
import momoe_amd  # noqa: E402

DEV = "cuda:0"


def _case(name, tokens, D, H, N, K, train, Ks=0, skew=0.0, save_percent=0, router=False):
    return {"name": name, "tokens": tokens, "D": D, "H": H, "N": N, "K": K, "Ks": Ks, "skew": skew,
            "save_percent": save_percent, "train": train, "router": router}


def listed():
    return [
        # one sequence being decoded: eight experts' weights stream, launches and host work show
        _case("decode 1 token", 1, 2048, 768, 128, 8, False),
        # a decode batch through the whole layer, gate included, as a serving loop calls it
        _case("decode 16 tokens, router", 16, 2048, 768, 128, 8, False, router=True),
        # a large decode batch or a short prompt, no multiple of anything: every expert's weights stream
        _case("decode 131 tokens", 131, 2048, 768, 128, 8, False),
        # a prompt of ordinary length through the whole layer: between streaming and multiplying
        _case("prefill 1000 tokens, router", 1000, 2048, 768, 128, 8, False, router=True),
        # batched prefill: bound by the matrix products
        _case("prefill 8192 tokens", 8192, 2048, 768, 128, 8, False),
        # a unit-test or debugging sized training step: launches and host work only
        _case("train tiny", 128, 128, 64, 8, 2, True),
        # the smallest model that is trained in earnest: 2 x 512 tokens
        _case("train small", 1024, 1024, 512, 32, 4, True),
        # the headline training layer, least memory: pre-activations are recomputed
        _case("train headline", 8192, 2048, 1024, 128, 8, True),
        # the same layer as a model holds it, with its router, when memory is plentiful
        _case("train headline, router, all saved", 8192, 2048, 1024, 128, 8, True, save_percent=100, router=True),
        # widths that are no power of two, K that does not divide N, half of the rows saved
        _case("train ragged, half saved", 7680, 2176, 1152, 64, 6, True, save_percent=50),
        # few experts receive ten times the mean load and four see every token
        _case("train skewed, shared experts", 16384, 2048, 1408, 64, 8, True, Ks=4, skew=1.8),
        # the largest layer, 8 x 8192 tokens
        _case("train large", 65536, 4096, 2048, 64, 8, True),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    limit = _flops(listed()[-1])
    while True:
        train = rng.random() < 0.5
        step = rng.choice((32, 64, 128))  # D and H are multiples of 32
        case = {
            "tokens": int(_log_uniform(rng, 64 if train else 1, 32768)),
            "D": max(step, int(_log_uniform(rng, 128, 4096)) // step * step),
            "H": max(step, int(_log_uniform(rng, 64, 2048)) // step * step),
            "N": rng.choice((8, 16, 32, 48, 64, 96, 128)),
            "K": rng.choice((1, 2, 4, 6, 8)),
            "Ks": rng.choice((0, 0, 0, 1, 2)),
            "skew": rng.choice((0.0, 0.0, 0.5, 1.8)),
            "save_percent": rng.choice((0, 0, 50, 100)) if train else 0,
            "train": train,
            "router": rng.random() < 0.5,
        }
        if case["K"] > case["Ks"] and case["K"] <= case["N"] // 2 and _flops(case) < limit and _weights(case) < 2 << 30:
            return case


def _routing(case, gen):
    """What a router hands to `MoMoE`: the 0/1 mask [N, tokens] and the gate weights (the transposed
    view of a [tokens, N] matrix).  Top-k of softmax(N(0,1) logits), renormalised; with `skew` the
    logits fall with the logarithm of an expert's rank; the last Ks experts hold every token."""
    M, N, K, Ks = case["tokens"], case["N"], case["K"], case["Ks"]
    Ng = N - Ks
    logits = torch.randn(M, N, generator=gen, device=DEV)
    logits[:, :Ng] -= case["skew"] * torch.log(torch.arange(1, Ng + 1, device=DEV, dtype=torch.float32))
    p = torch.softmax(logits[:, :Ng], -1)
    chosen = torch.zeros(M, Ng, dtype=torch.bool, device=DEV)
    chosen.scatter_(1, torch.topk(p, K - Ks, dim=-1).indices, True)
    w = p * chosen
    s_MN = torch.cat([w / w.sum(-1, keepdim=True), torch.softmax(logits[:, Ng:], -1)], -1)
    mask = torch.ones(N, M, dtype=torch.int32, device=DEV)
    mask[:Ng] = chosen.T.to(torch.int32)
    return mask, s_MN.contiguous().T


def prepare(case, seed):
    M, D, H, N, K, Ks, train = (case[k] for k in ("tokens", "D", "H", "N", "K", "Ks", "train"))
    gen = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(1, M, D, generator=gen, device=DEV).to(torch.bfloat16)
    W1 = torch.empty(N, D, 2 * H, device=DEV, dtype=torch.bfloat16).normal_(0, 0.02, generator=gen)
    W2 = torch.empty(N, H, D, device=DEV, dtype=torch.bfloat16).normal_(0, 0.02, generator=gen)
    state = {"train": train, "router": case["router"], "x": x}
    if case["router"]:
        # gate logits of about N(0,1), the skew as a common component of the tokens
        Wg = torch.randn(D, N, generator=gen, device=DEV) / math.sqrt(D)
        if case["skew"]:
            x[..., 0] = 1.0
            Wg[0, :N - Ks] = -case["skew"] * torch.log(torch.arange(1, N - Ks + 1, device=DEV, dtype=torch.float32))
        # a model that serves keeps the selection bias it was trained to
        state["layer"] = momoe_amd.MoE(D, H, N, K, Ks, save_percent=case["save_percent"],
                                       bias_update_rate=1e-4 if train else 0.0,
                                       Wg_DN=Wg.to(torch.bfloat16), Wl1_ND2H=W1, Wl2_NHD=W2)
    else:
        state["layer"] = momoe_amd.MoMoE(D, H, N, K, case["save_percent"], Wl1_ND2H=W1, Wl2_NHD=W2)
        state["mask"], state["s"] = _routing(case, gen)
    if train:
        state["dy"] = torch.randn(1, M, D, generator=gen, device=DEV).to(torch.bfloat16)
        x.requires_grad_()
        if not case["router"]:
            state["s"].requires_grad_()
    return state


def run(state):
    layer, x = state["layer"], state["x"]
    if not state["train"]:
        with torch.no_grad():
            return layer(x) if state["router"] else layer(x, state["mask"], state["s"])
    layer.zero_grad(set_to_none=True)
    x.grad = None
    if state["router"]:
        y = layer(x)
        y.backward(state["dy"])
        experts = layer.momoe
        return [y.detach(), x.grad, layer.router.Wg_DN.grad, experts.Wl1_ND2H.grad, experts.Wl2_NHD.grad,
                layer.biases_N.detach()]
    s = state["s"]
    s.grad = None
    y, sizes = layer(x, state["mask"], s)
    y.backward(state["dy"])
    return [y.detach(), sizes, x.grad, layer.Wl1_ND2H.grad, layer.Wl2_NHD.grad, s.grad]


def _weights(case):
    return 3 * case["D"] * case["H"] * case["N"]


def _flops(case):
    # 6 D H per (token, expert) pair forward, twice that backward; what is recomputed does not count
    passes = 3 if case["train"] else 1
    experts = 6 * case["D"] * case["H"] * case["tokens"] * case["K"]
    gate = 2 * case["D"] * case["N"] * case["tokens"] if case["router"] else 0
    return passes * (experts + gate)


def work(case):
    M, D, N, K, Ks = (case[k] for k in ("tokens", "D", "N", "K", "Ks"))
    # experts that hold a token, had every routed expert the same chance
    held = Ks + (N - Ks) * (1 - (1 - (K - Ks) / (N - Ks)) ** M)
    weights = 2 * _weights(case) * held / N
    rows = 2 * M * D
    gate = 2 * D * N if case["router"] else 8 * N * M  # gate weights, or mask and gate weights given
    if not case["train"]:
        return {"bytes": weights + 2 * rows + gate, "flops": _flops(case)}
    # every weight gradient is written, also of an expert without tokens; dL/ds is [N, tokens] fp32
    grads = 2 * _weights(case) + (2 * D * N if case["router"] else 4 * N * M)
    return {"bytes": weights + 4 * rows + gate + grads, "flops": _flops(case)}


def tolerance(case):
    # bf16 operands and results with fp32 sums: an intermediate rounded at another place moves a
    # result by a few 2^-9 of its size; tokens per expert are whole numbers and stay the same
    return {"rel": 1e-2}
