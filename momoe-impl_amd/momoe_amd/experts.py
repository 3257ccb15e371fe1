"""`MoMoE`: the experts of a SwiGLU mixture-of-experts layer, forward and backward,
on the gfx950 kernels of libmomoe_hip.so.

Mirrors the module and autograd contract of the reference (momoe/momoe.py:847-972):
`MoMoE(embedding_dim, intermediate_dim, num_experts, num_chosen_experts, save_percent,
Wl1_ND2H, Wl2_NHD)`, `forward(x_BSD, mask_NM, s_NM) -> (y_BSD bf16, sizes_N int64)`;
gradients for x (bf16), Wl1/Wl2 (bf16) and s_NM (fp32 [N,M], zero off-mask).

The host path (allocations, launches, autograd) is native: csrc/layer_binding.cpp.
"""
import torch
import torch.nn as nn

from . import _hip, _layer


# The layer requires every token to be routed to exactly K experts (momoe/momoe.py:831, the
# reference's README) and, like the reference, does not verify it: the index build counts the
# offending tokens on the device and reading that counter would stall the host.  With too few
# pairs the missing contributions are simply absent from y and the gradients; with too many (more
# pairs than the M*K sorted rows) the routing is refused on the device: no GEMM runs, y and all
# gradients are zero.  Set CHECK_ROUTING = True to read the counter after
# every forward (one device synchronisation per call) and raise on a violation.
CHECK_ROUTING = False

# Row-tile height of the grouped GEMMs: _hip.AUTO_TILE_ROWS leaves it to the library, 256 rows for the
# launches that take no taller tiles whole and for the others 256 or 320, chosen by the index build on the
# device from the routing.  A fixed height (a multiple of 32 from 32 to _hip.TILE_ROWS) is for
# experiments and for tests that must cover every code path.
TILE_ROWS = _hip.AUTO_TILE_ROWS


class MoEFunction:
    """(x_BSD, Wl1_ND2H, Wl2_NHD, mask_NM, s_NM, K, save_percent) -> (y_BSD, sizes_N): the autograd
    function of the layer, native (csrc/layer_binding.cpp).

    Forward (momoe/momoe.py:856-874): routing index, x.Wl1 with fused SwiGLU,
    h.Wl2 scaled by the gate weight, K-way combine.  With save_percent > 0 the
    pre-activation halves a|b of the first int(M*K*save_percent/100) sorted rows are kept for the
    backward; everything else is recomputed there.

    Backward (momoe/momoe.py:881-903).  Differences from the reference that do not
    change results beyond rounding: x and G_y are gathered inside the GEMM loads
    instead of being materialised in sorted order; dL/ds is obtained from
    (G_y.Wl2^T).h, which equals G_y.(h.Wl2), so the down projection is never
    recomputed and y_pre is never saved; dL/ds is reduced without atomics.
    """

    @staticmethod
    def apply(x_BSD, Wl1_ND2H, Wl2_NHD, mask_NM, s_NM, K, save_percent):
        return _layer.experts(x_BSD, Wl1_ND2H, Wl2_NHD, mask_NM, s_NM, K, save_percent, TILE_ROWS, CHECK_ROUTING)


class MoMoE(nn.Module):
    """Memory-optimised mixture of SwiGLU experts (momoe/momoe.py:914-972).

    Args:
        embedding_dim: D.  intermediate_dim: H.  num_experts: N (shared experts included,
        as the last rows of mask_NM/s_NM).  num_chosen_experts: K per token (shared included).
        save_percent: share of the (token, expert) rows whose pre-activations are kept
        for the backward, 0..100.
        Wl1_ND2H / Wl2_NHD: optional initial weights, [N, D, 2H] and [N, H, D]; the first
        H columns of Wl1 are the linear half, the last H go through SiLU.
    D and H must be multiples of 32 (the k-depth of one GEMM stage).
    """

    def __init__(self, embedding_dim, intermediate_dim, num_experts, num_chosen_experts,
                 save_percent=0, Wl1_ND2H=None, Wl2_NHD=None):
        assert save_percent >= 0 and save_percent <= 100, (
            "save_percent must be between 0 and 100 inclusive, got {}".format(save_percent))
        super().__init__()
        self.D = embedding_dim
        self.H = intermediate_dim
        self.N = num_experts
        self.K = num_chosen_experts
        self.save_percent = save_percent

        if Wl1_ND2H is None:
            Wl1_ND2H = torch.randn((self.N, self.D, 2 * self.H), device="cuda", dtype=torch.bfloat16) / self.D
        if Wl2_NHD is None:
            Wl2_NHD = torch.randn((self.N, self.H, self.D), device="cuda", dtype=torch.bfloat16) / self.D
        self.Wl1_ND2H = nn.Parameter(Wl1_ND2H.clone().detach().to(torch.bfloat16), requires_grad=True)
        self.Wl2_NHD = nn.Parameter(Wl2_NHD.clone().detach().to(torch.bfloat16), requires_grad=True)

    def forward(self, x_BSD, mask_NM, s_NM):
        """x_BSD [B,S,D]; mask_NM int32 0/1 [N,M] with exactly K ones per token; s_NM [N,M]
        gate weights (zero off-mask).  Returns (y_BSD bf16, tokens per expert int64 [N])."""
        return MoEFunction.apply(x_BSD, self.Wl1_ND2H, self.Wl2_NHD, mask_NM, s_NM, self.K, self.save_percent)
