"""TriangleMultiplication with the reference's constructor, parameter names and call
signature (``xfold/nn/triangle_multiplication.py:21-46``), running on the HIP backend.

:func:`triangle_multiplication_hip` takes any module that carries the reference's
parameters (this class or the reference's own), so the reference can call it from a
``'hip'`` branch of its ``forward`` without changing checkpoints.
"""

from __future__ import annotations

from typing import Optional

import torch
import torch.nn as nn

from ..fastnn import LayerNorm
from ..fastnn import config as fastnn_config
from ..fastnn import native_hip as nh


_WEIGHTS = ("projection", "gate", "output_projection", "gating_linear")
_NORMS = ("left_norm_input", "center_norm")


def triangle_multiplication_hip(module: nn.Module, pair: torch.Tensor, mask: Optional[torch.Tensor],
                                accumulate_into: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Update of ``xfold/nn/triangle_multiplication.py:71-105`` (or ``pair += update`` in
    place when ``accumulate_into`` is the contiguous pair tensor itself)."""
    nh.check_gpu_inference(pair, mask)
    nh.check_module(module)
    dtype, (w_proj, w_gate, w_out, w_gating, lw, lb, cw, cb) = nh.gather(
        module, "triangle_multiplication", nh.params(module, _WEIGHTS, _NORMS), 4, pair,
        lambda dt: (*nh.linear_weights(module, _WEIGHTS, dt),
                    *nh.norm_params(module, _NORMS[0]), *nh.norm_params(module, _NORMS[1])))
    if pair.dim() != 3 or pair.shape[0] != pair.shape[1] or pair.shape[2] != module.c_pair:
        raise ValueError("TriangleMultiplication expects pair [N, N, c_pair].")
    n, c = pair.shape[0], pair.shape[2]
    outgoing = module.equation == "cik,cjk->cij"
    pair_c = pair.contiguous()
    mask_t, mask_code = nh.mask_arg(mask, (n, n))
    if accumulate_into is not None:
        out, accumulate = accumulate_into, 1
        if not out.is_contiguous() or out.shape != pair.shape:
            raise ValueError("accumulate_into must be a contiguous tensor shaped like pair")
    else:
        out, accumulate = torch.empty((n, n, c), dtype=dtype, device=pair.device), 0
    lib = nh.load_library()
    ws = nh.workspace(lib.xfh_triangle_multiplication_workspace_size(n, c, nh.dtype_code(dtype)),
                      pair.device)
    nh.call("xfh_triangle_multiplication", nh.ptr(pair_c), nh.dtype_code(pair.dtype), nh.ptr(mask_t),
            mask_code, n, c, int(outgoing), nh.ptr(lw), nh.ptr(lb), float(module.left_norm_input.eps),
            nh.ptr(w_proj), nh.ptr(w_gate), nh.ptr(cw), nh.ptr(cb), float(module.center_norm.eps),
            nh.ptr(w_out), nh.ptr(w_gating), nh.dtype_code(dtype),
            nh.ptr(out), nh.dtype_code(out.dtype), accumulate, nh.ptr(ws), ws.numel(),
            nh.stream_of(pair.device))
    return out


class TriangleMultiplication(nn.Module):
    def __init__(self, c_pair: int = 128, _outgoing: bool = True) -> None:
        super().__init__()
        self.c_pair = c_pair
        self.left_norm_input = LayerNorm(c_pair)
        self.projection = nn.Linear(c_pair, 2 * c_pair, bias=False)
        self.gate = nn.Linear(c_pair, 2 * c_pair, bias=False)
        self.center_norm = LayerNorm(c_pair)
        self.output_projection = nn.Linear(c_pair, c_pair, bias=False)
        self.gating_linear = nn.Linear(c_pair, c_pair, bias=False)
        self.equation = "cik,cjk->cij" if _outgoing else "ckj,cki->cij"

    def forward(self, pair: torch.Tensor, mask: torch.Tensor) -> torch.Tensor:
        if fastnn_config.triangle_multiplication_implementation == fastnn_config.HIP:
            return triangle_multiplication_hip(self, pair, mask)
        raise ValueError("Unknown triangle_multiplication_implementation for xfold_cpu_amd: "
                         f"{fastnn_config.triangle_multiplication_implementation!r} (only 'hip')")
