"""Linears with few weights in training: the stream mappings' projection
(mhc.py:283-318) and the MoE router (moe.py:383-416)."""
import torch
import torch.nn.functional as F

from . import kernels
from ._common import first_order, plain_eager

# N * K up to which the weight gradient runs on the HIP kernel: the library
# gives a product with a small output few workgroups.  Kernel against library
# in us at 64 / 2,048 / 8,192 tokens: 24 x 2,048 6.8 / 9.1 / 14 against 7.5 /
# 18 / 56; 128 x 512 6.9 / 9.6 / 15 against 7.4 / 22 / 65; 24 x 16,384 7.8 / 18
# / 47 against 7.5 / 21 / 62; past the line 384 x 1,536 8.5 / 23.5 / 52 against
# 7.7 / 19 / 56 and 1,024 x 4,096 25 / 61 / 191 against 15 / 34 / 93.
MAX_WEIGHTS = 400 * 1024


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
                and x.shape[-1] == K and x.is_contiguous() and x.data_ptr() % 16 == 0 and N <= 1024
                and N * K <= MAX_WEIGHTS and K % 8 == 0 and x.numel() // K * max(N, K) * 2 < 2 ** 31
                and (not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") == torch.bfloat16)
                and plain_eager())

    @staticmethod
    def apply(x, w):
        return _FewRowsLinearFunction.apply(x, w, w.to(x.dtype))
