"""PairformerBlock and EvoformerBlock with the reference's constructors, submodule names and
call signatures (``xfold/nn/pairformer.py:26-156``), running on the HIP backend.

The block applies its five pair updates in place, each op's final kernel adding its
result straight into ``pair`` (the residual ``pair += op(pair)`` of ``pairformer.py:96-100``
without a separate update tensor), then the single track (``pairformer.py:102-113``).
"""

from __future__ import annotations

import ctypes
from typing import Optional

import torch
import torch.nn as nn

from ..fastnn import LayerNorm
from ..fastnn import config as fastnn_config
from ..fastnn import native_hip as nh
from ..fastnn import ops
from .attention import _GRID_WEIGHTS, GridSelfAttention, MSAAttention, grid_self_attention_hip, msa_attention_hip
from .diffusion_transformer import _QKV, SelfAttention, qkvg_weights, self_attention_hip
from .primitives import OuterProductMean, Transition, outer_product_mean_hip, transition_hip
from .triangle_multiplication import _NORMS as _TRIANGLE_NORMS, _WEIGHTS as _TRIANGLE_WEIGHTS
from .triangle_multiplication import TriangleMultiplication, triangle_multiplication_hip

_ATTENTION = _QKV + ("gating_query",)


def pair_logits_hip(block: nn.Module, pair: torch.Tensor, dtype: torch.dtype):
    """``Linear(LN(pair)).permute(2, 0, 1)`` (``pairformer.py:103-106``): with bf16 compute,
    128 pair channels and at most ``attention_max_keys()`` tokens one kernel writes it as the
    attention's packed bias (:class:`ops.PackedBias`), else a [H, N, N] view."""
    norm = block.single_pair_logits_norm
    proj = block.single_pair_logits_projection
    if dtype == torch.bfloat16 and pair.shape[-1] == 128 and proj.weight.shape[0] <= 384 \
            and tuple(norm.normalized_shape) == (128,) and pair.shape[0] <= nh.attention_max_keys():
        w = nh.linear_weight(block, "single_pair_logits_projection", dtype)
        return ops.PackedBias(ops.pair_attention_bias(pair, norm.weight, norm.bias, norm.eps, w, owner=norm))
    normed = ops.layer_norm(pair, norm.normalized_shape, norm.weight, norm.bias, norm.eps,
                            out_dtype=dtype, owner=norm)
    logits = ops.linear(normed, nh.linear_weight(block, "single_pair_logits_projection", dtype), None, dtype)
    return logits.permute(2, 0, 1)


# The single-track block's pair transition and pair logits in one kernel (when the shapes
# allow it); False runs them as two kernels, with the same results bit for bit.
FUSE_TRANSITION_AND_LOGITS = True


def _transition_with_logits_hip(block: nn.Module, pair: torch.Tensor) -> Optional[ops.PackedBias]:
    """``pair += pair_transition(pair)`` and then the pair logits of the updated pair
    (``pairformer.py:100``, ``:103-106``) in one kernel, whose epilogue computes the logits
    from the values it stores: bf16 pair [N, N, 128], hidden 512, at most 16 heads. None
    (nothing done) for other shapes."""
    tr, norm, proj = block.pair_transition, block.single_pair_logits_norm, nh.param(block, "single_pair_logits_projection")
    names = ("transition1", "transition2")
    w1_src, w2_src, *tr_norm = nh.params(tr, names, ("input_layer_norm",))
    n, c = pair.shape[0], pair.shape[-1]
    if (pair.dtype != torch.bfloat16 or pair.dim() != 3 or pair.shape[1] != n or c != 128
            or w2_src.shape != (c, 512) or w1_src.shape != (1024, c)
            or tuple(norm.normalized_shape) != (c,) or tuple(tr.input_layer_norm.normalized_shape) != (c,)
            or proj.shape[0] > 16 or n > nh.attention_max_keys()):
        return None
    sources = [w1_src, w2_src, proj, *tr_norm, norm.weight, norm.bias]
    # Not this dtype: None, and the general path builds its own copies.
    dtype, values = nh.gather(
        block, "transition_pair_bias", sources, 3, pair,
        lambda dt: None if dt != torch.bfloat16 else (
            nh.linear_weight(tr, "transition1", dt, "glu"), nh.linear_weight(tr, "transition2", dt),
            nh.linear_weight(block, "single_pair_logits_projection", dt), *nh.norm_params(tr, "input_layer_norm"),
            *nh.norm_params(block, "single_pair_logits_norm")))
    if values is None:
        return None
    nh.check_gpu_inference(pair)
    nh.check_module(tr)
    w1, w2, wb, nw, nb, bw, bb = values
    heads = wb.shape[0]
    packed = torch.empty((heads, n, (n + 63) // 64 * 64), dtype=torch.float32, device=pair.device)
    nh.call("xfh_transition_pair_bias", nh.ptr(pair), n, c, 512, nh.ptr(nw), nh.ptr(nb),
            float(tr.input_layer_norm.eps), nh.ptr(w1), nh.ptr(w2), nh.ptr(bw), nh.ptr(bb), float(norm.eps),
            nh.ptr(wb), heads, nh.ptr(packed), nh.stream_of(pair.device))
    return ops.PackedBias(packed)


def pairformer_block_hip(block: nn.Module, pair: torch.Tensor, pair_mask: torch.Tensor,
                         single: Optional[torch.Tensor] = None,
                         seq_mask: Optional[torch.Tensor] = None):
    """``PairformerBlock.forward`` (``pairformer.py:77-114``); ``pair`` (and ``single``)
    must be contiguous and are updated in place, as the reference's ``+=`` does."""
    if not pair.is_contiguous() or (single is not None and not single.is_contiguous()):
        raise ValueError("PairformerBlock (hip) updates pair/single in place; pass contiguous tensors")
    if not block.with_single:
        _pair_updates_hip(block, pair, pair_mask)
        return pair
    _pair_updates_hip(block, pair, pair_mask, transition=False)
    if FUSE_TRANSITION_AND_LOGITS and _single_track_hip(block, pair, single, seq_mask):
        return pair, single
    logits = _transition_with_logits_hip(block, pair) if FUSE_TRANSITION_AND_LOGITS else None
    if logits is None:
        transition_hip(block.pair_transition, pair, accumulate_into=pair)
        dtype = nh.compute_dtype(pair, block.single_pair_logits_projection.weight)
        logits = pair_logits_hip(block, pair, dtype)
    self_attention_hip(block.single_attention_, single, seq_mask, logits, None, accumulate_into=single)
    transition_hip(block.single_transition, single, accumulate_into=single)
    return pair, single


def _single_track_hip(block: nn.Module, pair: torch.Tensor, single: torch.Tensor,
                      seq_mask: Optional[torch.Tensor]) -> bool:
    """The pair transition with its logits and the whole single track in one library call
    (``xfh_pairformer_single``), where the operators' own bf16 paths take those shapes; False
    (nothing done) otherwise."""
    if nh.first_pass(block, "single_track"):
        return False
    m = block._modules
    tr, norm, att, str_ = (m[name] for name in ("pair_transition", "single_pair_logits_norm", "single_attention_",
                                                "single_transition"))
    proj = nh.param(block, "single_pair_logits_projection")
    aln, zero = att._modules["adaptive_layernorm"], att._modules["adaptive_zero_init"]
    n, heads, c = pair.shape[0], att.num_head, single.shape[-1]
    if (pair.dtype != torch.bfloat16 or pair.dim() != 3 or tuple(pair.shape) != (n, n, 128) or heads > 16
            or tuple(single.shape) != (n, c) or single.dtype not in (torch.float32, torch.bfloat16)
            or c % 32 or c % heads or not ops.AttentionOperands.supported(n, heads, c // heads)
            or aln.use_single_cond or zero.use_single_cond
            or (seq_mask is not None and tuple(seq_mask.shape) != (n,))):
        return False
    names = ("transition1", "transition2")
    tr_w, str_w, att_w = nh.params(tr, names), nh.params(str_, names), nh.params(att, _ATTENTION)
    out_w = nh.param(zero, "transition2")
    f = str_w[1].shape[1]
    if (tr_w[0].shape != (1024, 128) or tr_w[1].shape != (128, 512) or proj.shape != (heads, 128)
            or str_w[0].shape != (2 * f, c) or str_w[1].shape != (c, f) or out_w.shape != (c, c)
            or any(w.shape != (c, c) for w in att_w)):
        return False
    norms = ((tr, "input_layer_norm", 128), (block, "single_pair_logits_norm", 128), (aln, "layer_norm", c),
             (str_, "input_layer_norm", c))
    if any(tuple(owner._modules[name].normalized_shape) != (size,) for owner, name, size in norms):
        return False
    nh.check_gpu_inference(pair, single, seq_mask)
    nh.check_module(block)
    norm_sources = []
    for owner, name, _ in norms:
        norm_sources += (nh.param(owner, name), nh.param(owner, name, "bias"))

    def build(dt):
        if dt != torch.bfloat16:
            return None
        n0, n1, n2, n3 = (nh.norm_params(owner, name) for owner, name, _ in norms)
        return [*n0, nh.linear_weight(tr, "transition1", dt, "glu"), nh.linear_weight(tr, "transition2", dt),
                *n1, nh.linear_weight(block, "single_pair_logits_projection", dt),
                *n2, *qkvg_weights(att, dt), nh.linear_weight(zero, "transition2", dt),
                *n3, nh.linear_weight(str_, "transition1", dt, "glu"), nh.linear_weight(str_, "transition2", dt)]
    # The operators resolve the compute dtype from the pair or the single track and their own
    # weights: one group when both have one dtype, else the general path.
    if single.dtype != pair.dtype and not torch.is_autocast_enabled("cuda"):
        return False
    _, values = nh.gather(block, "single_track", [*tr_w, proj, *att_w, *str_w, out_w, nh.param(att, "q_projection", "bias"),
                                                  *norm_sources], 9, pair, build, again=True)
    if values is None:
        return False
    operands = ops.shared_attention_operands(1, n, heads, c // heads, single.device)
    operands.set_mask(seq_mask)
    eps = (ctypes.c_float * 4)(*(owner._modules[name].eps for owner, name, _ in norms))
    lib = nh.load_library()
    ws = nh.workspace(lib.xfh_pairformer_single_workspace_size(n, c, heads, f), pair.device)
    nh.call("xfh_pairformer_single", nh.ptr(pair), nh.ptr(single), nh.dtype_code(single.dtype), n, c, heads, f,
            nh.ptrs(values), eps, (c // heads) ** -0.5 * 1.4426950408889634, nh.ptr(operands.q), nh.ptr(operands.k),
            nh.ptr(operands.vt), nh.ptr(operands.gate), nh.ptr(operands.words), nh.ptr(ws), ws.numel(),
            nh.stream_of(pair.device))
    return True


_TRIANGLES = ("triangle_multiplication_outgoing", "triangle_multiplication_incoming")
_GRIDS = ("pair_attention1", "pair_attention2")


def _pair_updates_hip(block: nn.Module, pair: torch.Tensor, pair_mask: torch.Tensor,
                      transition: bool = True) -> None:
    """The pair updates (``pairformer.py:96-100``), as one library call (``xfh_pair_updates``) when
    the five modules agree in their widths."""
    m = block._modules
    triangles, grids = [m[name] for name in _TRIANGLES], [m[name] for name in _GRIDS]
    tr = m["pair_transition"]

    def one_by_one():
        triangle_multiplication_hip(triangles[0], pair, pair_mask, accumulate_into=pair)
        triangle_multiplication_hip(triangles[1], pair, pair_mask, accumulate_into=pair)
        grid_self_attention_hip(grids[0], pair, pair_mask, accumulate_into=pair)
        grid_self_attention_hip(grids[1], pair, pair_mask, accumulate_into=pair)
        if transition:
            transition_hip(tr, pair, accumulate_into=pair)
    if nh.first_pass(block, "pair_updates"):
        return one_by_one()
    tr_w = nh.params(tr, ("transition1", "transition2"))
    c, heads, f = pair.shape[-1], grids[0].num_head, tr_w[1].shape[1]
    if (pair.dim() != 3 or pair.shape[0] != pair.shape[1] or pair_mask is None or heads != grids[1].num_head
            or any(t.c_pair != c for t in triangles + grids) or tr_w[0].shape != (2 * f, c)):
        return one_by_one()
    nh.check_gpu_inference(pair, pair_mask)
    nh.check_module(block)
    n = pair.shape[0]
    weights, norms = [], []
    for t in triangles:
        weights += nh.params(t, _TRIANGLE_WEIGHTS)
        norms += nh.params(t, (), _TRIANGLE_NORMS)
    for g in grids:
        weights += nh.params(g, _GRID_WEIGHTS)
        norms += nh.params(g, (), ("act_norm",))
    norms += nh.params(tr, (), ("input_layer_norm",))

    def build(dt):
        out = []
        for t in triangles:
            out += (*nh.norm_params(t, _TRIANGLE_NORMS[0]), *nh.norm_params(t, _TRIANGLE_NORMS[1]))
            out += nh.linear_weights(t, _TRIANGLE_WEIGHTS, dt)
        for g in grids:
            out += nh.norm_params(g, "act_norm")
            out += nh.linear_weights(g, _GRID_WEIGHTS, dt)
        out += nh.norm_params(tr, "input_layer_norm")
        out += (nh.linear_weight(tr, "transition1", dt, "glu"), nh.linear_weight(tr, "transition2", dt))
        return out
    dtype, values = nh.gather(block, "pair_updates", weights + tr_w + norms, len(weights) + 2, pair, build, again=True)
    if values is None:
        return one_by_one()
    mask_t, mask_code = nh.mask_arg(pair_mask, (n, n))
    outgoing = (ctypes.c_int * 2)(*(t.equation == "cik,cjk->cij" for t in triangles))
    transpose = (ctypes.c_int * 2)(*(bool(g.transpose) for g in grids))
    eps = (ctypes.c_float * 7)(*(t._modules[name].eps for t in triangles for name in _TRIANGLE_NORMS),
                               *(g.act_norm.eps for g in grids), tr.input_layer_norm.eps)
    f_now = f if transition else 0
    lib, code = nh.load_library(), nh.dtype_code(dtype)
    ws = nh.workspace(lib.xfh_pair_updates_workspace_size(n, c, heads, f_now, code), pair.device)
    nh.call("xfh_pair_updates", nh.ptr(pair), nh.dtype_code(pair.dtype), nh.ptr(mask_t), mask_code, n, c, heads, f_now,
            outgoing, transpose, nh.ptrs(values), eps, code, nh.ptr(ws), ws.numel(), nh.stream_of(pair.device))


def _require_hip_backends() -> None:
    for name in ("layer_norm_implementation", "dot_product_attention_implementation",
                 "gated_linear_unit_implementation", "triangle_multiplication_implementation"):
        if getattr(fastnn_config, name) != fastnn_config.HIP:
            raise ValueError(f"Unknown {name} for xfold_cpu_amd: "
                             f"{getattr(fastnn_config, name)!r} (only 'hip')")


class PairformerBlock(nn.Module):
    def __init__(self, n_heads: int = 16, c_pair: int = 128, c_single: int = 384,
                 c_hidden_mul: int = 128, n_heads_pair: int = 4, num_intermediate_factor: int = 4,
                 with_single: bool = True) -> None:
        super().__init__()
        self.n_heads = n_heads
        self.with_single = with_single
        self.num_intermediate_factor = num_intermediate_factor
        self.triangle_multiplication_outgoing = TriangleMultiplication(c_pair=c_pair, _outgoing=True)
        self.triangle_multiplication_incoming = TriangleMultiplication(c_pair=c_pair, _outgoing=False)
        self.pair_attention1 = GridSelfAttention(c_pair=c_pair, num_head=n_heads_pair, transpose=False)
        self.pair_attention2 = GridSelfAttention(c_pair=c_pair, num_head=n_heads_pair, transpose=True)
        self.pair_transition = Transition(c_x=c_pair, num_intermediate_factor=num_intermediate_factor)
        self.c_single = c_single
        if with_single:
            self.single_pair_logits_norm = LayerNorm(c_pair)
            self.single_pair_logits_projection = nn.Linear(c_pair, n_heads, bias=False)
            self.single_attention_ = SelfAttention(c_x=c_single, num_head=n_heads, use_single_cond=False)
            self.single_transition = Transition(c_x=c_single)

    def forward(self, pair, pair_mask, single=None, seq_mask=None):
        _require_hip_backends()
        return pairformer_block_hip(self, pair, pair_mask, single, seq_mask)


def evoformer_block_hip(block: nn.Module, msa: torch.Tensor, pair: torch.Tensor, msa_mask: torch.Tensor,
                        pair_mask: torch.Tensor):
    """``EvoformerBlock.forward`` (``pairformer.py:139-156``): OuterProductMean into the pair,
    MSA attention (over the updated pair) and transition into the MSA, then the five pair
    updates. ``msa`` and ``pair`` must be contiguous and are updated in place."""
    if not pair.is_contiguous() or not msa.is_contiguous():
        raise ValueError("EvoformerBlock (hip) updates msa/pair in place; pass contiguous tensors")
    outer_product_mean_hip(block.outer_product_mean, msa, msa_mask, accumulate_into=pair)
    msa_attention_hip(block.msa_attention1, msa, msa_mask, pair, accumulate_into=msa)
    transition_hip(block.msa_transition, msa, accumulate_into=msa)
    _pair_updates_hip(block, pair, pair_mask)
    return msa, pair


class EvoformerBlock(nn.Module):
    def __init__(self, c_msa: int = 64, c_pair: int = 128, n_heads_pair: int = 4) -> None:
        super().__init__()
        self.outer_product_mean = OuterProductMean(c_msa=c_msa, num_output_channel=c_pair)
        self.msa_attention1 = MSAAttention(c_msa=c_msa, c_pair=c_pair)
        self.msa_transition = Transition(c_x=c_msa)
        self.triangle_multiplication_outgoing = TriangleMultiplication(c_pair=c_pair, _outgoing=True)
        self.triangle_multiplication_incoming = TriangleMultiplication(c_pair=c_pair, _outgoing=False)
        self.pair_attention1 = GridSelfAttention(c_pair=c_pair, num_head=n_heads_pair, transpose=False)
        self.pair_attention2 = GridSelfAttention(c_pair=c_pair, num_head=n_heads_pair, transpose=True)
        self.pair_transition = Transition(c_x=c_pair)

    def forward(self, msa, pair, msa_mask, pair_mask):
        _require_hip_backends()
        return evoformer_block_hip(self, msa, pair, msa_mask, pair_mask)
