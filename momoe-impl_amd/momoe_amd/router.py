"""`TopKRouter`: top-k + softmax gate with a selection bias (auxiliary-loss-free load
balancing) and shared experts, mirroring momoe/topk_router.py:83-173.

The gate product of many tokens is a plain library GEMM (torch); that of few tokens, its gradients and the
softmax / top-k / renormalise pass with its backward are HIP kernels.
"""
import torch
import torch.nn as nn

from . import _layer


class TopKRouterFunction:
    """(x_BSD, Wg_DN, biases_N, N, K, Ks) -> (x_BSD, mask_NM int32 [N,M], s_NM fp32 [N,M]): the
    autograd function of the router, native (csrc/layer_binding.cpp).

    s_NM is the transposed view of an [M,N] matrix, as in the reference
    (momoe/topk_router.py:120); x_BSD is passed through so its gradient picks up
    the gate's contribution (:124, :139).
    """

    @staticmethod
    def apply(x_BSD, Wg_DN, biases_N, N, K, Ks):
        return _layer.router(x_BSD, Wg_DN, biases_N, N, K, Ks)


class TopKRouter(nn.Module):
    """momoe/topk_router.py:151-173."""

    def __init__(self, embedding_dim, num_experts, num_chosen_experts, num_shared_experts,
                 Wg_DN=None):
        super().__init__()
        self.D = embedding_dim
        self.N = num_experts
        self.K = num_chosen_experts
        self.Ks = num_shared_experts
        if Wg_DN is None:
            Wg_DN = torch.randn((self.D, self.N), device="cuda", dtype=torch.bfloat16) / self.D
        self.Wg_DN = nn.Parameter(Wg_DN.clone().detach().to(torch.bfloat16), requires_grad=True)

    def forward(self, x_BSD, biases_N):
        return TopKRouterFunction.apply(x_BSD, self.Wg_DN, biases_N, self.N, self.K, self.Ks)
