"""Linears with few weights in training: the stream mappings' projection
(mhc.py:283-318) and the MoE router (moe.py:383-416)."""
import torch
import torch.nn.functional as F

from . import kernels
from ._common import first_order, plain_eager

# Where the weight gradient runs on the HIP kernel: the library gives a product
# with a small output few workgroups.  Kernel against library in us at 64 / 1,024
# / 2,048 / 8,192 tokens: 24 x 2,048 6.6 / 7.8 / 8.9 / 14 against 6.9 / 14 / 18 / 55;
# 128 x 512 6.8 / 8.1 / 9.4 / 14 against 7.3 / 15 / 22 / 65; 256 x 1,024 7.3 / 12.7 / 14
# / 20 against 6.9 / 13.6 / 18 / 55.  Past 2^18 weights its partial sums count: 24 x
# 16,384 7.4 / 13.2 / 18 / 47 against 6.9 / 15 / 20 / 62 (at 512 tokens 11.5 against
# 10.8), 320 x 1,280 7.5 / 16.4 / 20 / 39 against 7.1 / 13.5 / 18 / 56 (at 3,072 21
# against 25); past the line 1,024 x 4,096 25 / 47 / 61 / 191 against 15 / 27 / 34 / 93.
MAX_WEIGHTS = 400 * 1024
ANY_ROWS_WEIGHTS = 2 ** 18


def _few_rows(M, N, K) -> bool:
    return N <= 1024 and (N * K <= ANY_ROWS_WEIGHTS
                          or (N <= 512 and N * K <= MAX_WEIGHTS and M >= (1024 if N <= 32 else 3072)))


class _FewRowsLinearFunction(torch.autograd.Function):
    """F.linear(x, wb) for wb = w.to(bf16) of a float32 weight w: the plain
    backward gives w its gradient in float32, one that is itself differentiated
    or batched gives wb its own, as F.linear's.  Of the weights only wb is
    saved, so w may change between the forward and its backward."""

    @staticmethod
    def forward(ctx, x, w, wb):
        ctx.save_for_backward(x, wb)
        return F.linear(x, wb)

    @staticmethod
    def backward(ctx, gy):
        x, wb = ctx.saved_tensors
        nx, nw, _ = ctx.needs_input_grad
        g2, x2 = gy.reshape(-1, gy.shape[-1]), x.reshape(-1, x.shape[-1])
        gx = (g2 @ wb).view(x.shape) if nx else None
        if not first_order(gy):
            return gx, None, g2.t() @ x2 if nw else None
        return gx, kernels.linear_wgrad(g2, x2) if nw else None, None


class FewRowsLinear:
    """F.linear(x, w.to(bf16)) of bf16 rows with a float32 weight w; dw on the
    HIP kernel (float32, not rounded to bf16 on the way)."""

    @staticmethod
    def takes(x, w) -> bool:
        N, K = w.shape
        return (x.is_cuda and x.dtype == torch.bfloat16 and w.dtype == torch.float32 and w.device == x.device
                and type(x) is torch.Tensor and type(w) in (torch.Tensor, torch.nn.Parameter) and x.numel() > 0
                and x.shape[-1] == K and x.is_contiguous() and x.data_ptr() % 16 == 0
                and _few_rows(x.numel() // K, N, K) and K % 8 == 0 and x.numel() // K * max(N, K) * 2 < 2 ** 31
                and (not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") == torch.bfloat16)
                and plain_eager())

    @staticmethod
    def apply(x, w):
        return _FewRowsLinearFunction.apply(x, w, w.to(x.dtype))
