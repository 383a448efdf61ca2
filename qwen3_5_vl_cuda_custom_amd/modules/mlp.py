"""CudaSwiGLUMLP / CudaVisionMLP (reference modules/mlp.py:10-34)."""
from __future__ import annotations

import torch
from torch import nn

from ..kernels import gelu_tanh, matmul_gelu, matmul_swiglu, rmsnorm_matmul_swiglu, swiglu
from ..kernels.backward import needs_grad
from ..kernels.matmul import line_padded_rows
from .linear import CudaLinear
from .norms import CudaRMSNorm, fused_norm_ok


# Rows from which CudaVisionMLP pads its hidden rows to whole 128-byte lines (line_padded_rows). It makes fc2 about
# 5 us faster from 256 rows on and costs about 5 us of host time, and a tower of fewer rows is bound by the host: the
# 27 blocks with padding against without, 784 rows 5236 / 5098 us, 1520 rows 5367 / 5306, 1764 rows 5446 / 5551,
# 3528 rows 6616 / 6711.
PAD_ROWS = 1536


class CudaSwiGLUMLP(nn.Module):
    """down_proj(silu(gate_proj(x)) · up_proj(x)); gate/up (I, h), down (h, I)."""

    def __init__(self, hidden_size: int, intermediate_size: int, bias: bool = False) -> None:
        super().__init__()
        self.gate_proj = CudaLinear(hidden_size, intermediate_size, bias=bias)
        self.up_proj = CudaLinear(hidden_size, intermediate_size, bias=bias)
        self.down_proj = CudaLinear(intermediate_size, hidden_size, bias=bias)

    def forward(self, x: torch.Tensor, residual: torch.Tensor | None = None, *,
                input_norm: CudaRMSNorm | None = None) -> torch.Tensor:
        """`input_norm`: x is taken before this RMSNorm; for decode shapes (at
        most 32 bf16 tokens) it runs inside the gate/up GEMM, else first."""
        if needs_grad(x, residual, *self.parameters()):  # training: modules/mlp.py:19-22 on differentiable ops
            if input_norm is not None:
                x = input_norm(x)
            return self.down_proj(swiglu(self.gate_proj(x), self.up_proj(x)), residual=residual)
        no_bias = self.gate_proj.bias is None and self.up_proj.bias is None
        if input_norm is not None and no_bias and fused_norm_ok(x, input_norm):
            act = rmsnorm_matmul_swiglu(x, input_norm.weight, input_norm.eps, self.gate_proj.weight,
                                        self.up_proj.weight)
            return self.down_proj(act, residual=residual)
        if input_norm is not None:
            x = input_norm(x)
        if no_bias:
            act = matmul_swiglu(x, self.gate_proj.weight, self.up_proj.weight)  # gate, up and swiglu in one GEMM
        else:
            act = swiglu(self.gate_proj(x), self.up_proj(x))
        return self.down_proj(act, residual=residual)


class CudaVisionMLP(nn.Module):
    """linear_fc2(gelu_tanh(linear_fc1(x))), both with bias; the gelu runs in fc1's GEMM epilogue."""

    def __init__(self, hidden_size: int, intermediate_size: int) -> None:
        super().__init__()
        self.linear_fc1 = CudaLinear(hidden_size, intermediate_size, bias=True)
        self.linear_fc2 = CudaLinear(intermediate_size, hidden_size, bias=True)

    def forward(self, x: torch.Tensor, residual: torch.Tensor | None = None) -> torch.Tensor:
        if needs_grad(x, residual, *self.parameters()):  # training: modules/mlp.py:33-34 on differentiable ops
            return self.linear_fc2(gelu_tanh(self.linear_fc1(x)), residual=residual)
        w1 = self.linear_fc1.weight
        padded = line_padded_rows(x, w1.shape[0]) if x.numel() >= PAD_ROWS * x.shape[-1] else None
        h = matmul_gelu(x, w1, self.linear_fc1.bias, out=padded)
        return self.linear_fc2(h, residual=residual)
