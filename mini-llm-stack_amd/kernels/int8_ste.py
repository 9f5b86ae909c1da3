"""INT8 straight-through-estimator linear on the gfx950 kernels: the INT8 part of
the reference's kernels/autograd_ops.py:95-134, under a module name of its own.

The reference's autograd_ops also holds the attention and MoE autograd functions
(autograd_ops.py:22-92), which this build does not replace. With the reference
checkout on sys.path after this package, the reference's autograd_ops imports
unchanged and its Int8MatmulSTE binds this package's int8_matmul / int8_dgrad;
this module serves callers without the checkout.

Forward: y = int8_matmul(x, W_q, s). Backward: dx = int8_dgrad(dy, W_q, s) on the
device, and the fp32 master weight receives dy^T @ x (nothing quantized in it), for fp32
on the matrix cores at the sizes where that is faster than the library's fp32 product.
"""

from __future__ import annotations

import torch

import kernels
from kernels._hip import ld, plain, rows, stream
from kernels.dequant_matmul import int8_dgrad, int8_matmul


def _weight_grad(dy: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """dy [M, N]^T @ x [M, K]. The kernel takes ordinary fp32 tensors; what torch has to see (a
    gradient of the gradient, tracing, autocast) and other dtypes are torch's."""
    if dy.dtype != torch.float32 or x.dtype != torch.float32 or dy.dim() != 2 or x.dim() != 2:
        return dy.t() @ x
    # the sizes first: a small step is bound by its host work (100 tokens, 512 x 512: all checks
    # in front of the library's product 23.1 us, the product's own call 19.7)
    M, N = dy.shape
    K = x.shape[1]
    lib = kernels.lib()
    if (not lib.mlsx_dw_fp32_pays(M, N, K) or x.shape[0] != M or not plain(dy) or not plain(x)
            or dy.device != x.device or torch.is_autocast_enabled("cuda")):
        return dy.t() @ x
    dy, x = rows(dy), rows(x)
    need = lib.mlsx_dw_fp32_workspace(M, N, K)
    ws = torch.empty(need, dtype=torch.uint8, device=dy.device)
    dw = torch.empty(N, K, dtype=torch.float32, device=dy.device)
    kernels.check(lib.mlsx_dw_fp32(dy.data_ptr(), ld(dy), x.data_ptr(), ld(x), dw.data_ptr(), ld(dw), M, N, K,
                                   ws.data_ptr(), need, stream(dy.device)), "weight gradient")
    return dw


class Int8MatmulSTE(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w_q, scale, master_weight):
        ctx.save_for_backward(x, w_q, scale)
        return int8_matmul(x, w_q, scale)

    @staticmethod
    def backward(ctx, dy):
        x, w_q, scale = ctx.saved_tensors
        dy = dy.contiguous()
        dx = int8_dgrad(dy, w_q, scale)
        dw = _weight_grad(dy, x)
        return dx, None, None, dw


class QuantLinearSTE(torch.nn.Module):
    """Linear layer for quantization-aware training: the parameter stays fp32 and is
    re-quantized to INT8 (per-row scales) at every forward; its gradient passes straight
    through the quantizer."""

    def __init__(self, in_features: int, out_features: int):
        super().__init__()
        self.weight = torch.nn.Parameter(torch.randn(out_features, in_features) * 0.02)

    def forward(self, x):
        from serve.quantize import quantize_int8
        w_q, scale = quantize_int8(self.weight.detach())
        shape = x.shape
        flat = x.reshape(-1, shape[-1])
        y = Int8MatmulSTE.apply(flat, w_q, scale, self.weight)
        return y.reshape(*shape[:-1], -1)
