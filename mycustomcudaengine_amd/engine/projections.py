"""The engine's projections of more tokens than the decode-sized GEMMs take:
this package's prompt GEMM (csrc/prompt_gemm.hip) for the sizes at which it is
the faster one, torch.matmul and the separate ops otherwise (the reference
runs all of them through torch.matmul, engine/models/llama.py:94-174,
benchmarks/benchmark_engine.py:40-122).
"""
from __future__ import annotations

import torch

import my_cuda_engine_cpp as ops

from .. import _lib
from ..ops import _native

_STORE, _ADD, _SWIGLU = 0, 1, 2  # MCE_EPI_*


def _prompt_gemm(x, weight, out, epilogue, norm_weight, eps):
    if x.is_cuda:
        _lib.load()  # binds the native call, also where this is a process's first op
    return _native.prompt_gemm(x, weight, out, epilogue, norm_weight, eps)


def linear(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """x [M, K] . weight [N, K]^T"""
    y = _prompt_gemm(x, weight, None, _STORE, None, None)
    return torch.matmul(x, weight.T) if y is NotImplemented else y


def linear_swiglu(x: torch.Tensor, gate_up: torch.Tensor) -> torch.Tensor:
    """silu(x W_gate^T) * (x W_up^T), gate_up [2 N, K] with the gate rows first"""
    y = _prompt_gemm(x, gate_up, None, _SWIGLU, None, None)
    return ops.swiglu(torch.matmul(x, gate_up.T)) if y is NotImplemented else y


def linear_add(x: torch.Tensor, weight: torch.Tensor, residual: torch.Tensor) -> None:
    """residual += x . weight^T, in place"""
    if _prompt_gemm(x, weight, residual, _ADD, None, None) is NotImplemented:
        residual.addmm_(x, weight.T)


def linear_add_norm(x: torch.Tensor, weight: torch.Tensor, residual: torch.Tensor,
                    norm_weight: torch.Tensor, eps: float) -> torch.Tensor:
    """residual += x . weight^T in place; returns RMSNorm(residual)"""
    y = _prompt_gemm(x, weight, residual, _ADD, norm_weight, eps)
    if y is NotImplemented:
        residual.addmm_(x, weight.T)
        y = ops.rmsnorm(residual, norm_weight, eps)
    return y
