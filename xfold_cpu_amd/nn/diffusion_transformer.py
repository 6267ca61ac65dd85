"""Diffusion-transformer modules with the reference's constructors, parameter names and
call signatures (``xfold/nn/diffusion_transformer.py:27-272``), running on the HIP backend:
AdaptiveLayerNorm, AdaLNZero, DiffusionTransition, SelfAttention (also the Pairformer's
single-track attention), DiffusionTransformer and the atom CrossAttention (:275-350).

The ``*_hip`` functions take any module carrying the reference's parameters. Activations
may carry a leading sample dim ([S, N, c]); conditioning tensors ([N, c_cond]) and pair
logits ([H, N, N]) are shared by all samples, which is what the reference computes one
sample at a time.
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
from .cache import InputCache


def _adaptive_layer_norm(aln: nn.Module, x: torch.Tensor, single_cond: Optional[torch.Tensor],
                         dtype: torch.dtype, out_dtype: Optional[torch.dtype] = None,
                         cond: Optional[tuple] = None, stacked: Optional[tuple] = None) -> torch.Tensor:
    """``AdaptiveLayerNorm.forward`` (``diffusion_transformer.py:51-64``); Linears in
    ``dtype``, result in ``out_dtype`` (default ``dtype``). ``cond`` = (scale, shift) already
    computed from single_cond (see :func:`_block_conditioning`); ``stacked`` = the weights of
    :func:`_scale_shift_weights` that the caller has at hand."""
    if (single_cond is None) != (not aln.use_single_cond):
        raise ValueError("single_cond must be given exactly when use_single_cond is set")
    out_dtype = out_dtype or dtype
    if cond is not None:
        return ops.adaptive_layer_norm(x, cond[0], cond[1], aln.layer_norm.eps, out_dtype=out_dtype)
    if not aln.use_single_cond:
        ln = aln.layer_norm
        return ops.layer_norm(x, ln.normalized_shape, ln.weight, ln.bias, ln.eps, out_dtype=out_dtype,
                              owner=ln)
    cln = aln.single_cond_layer_norm
    cond = ops.layer_norm(single_cond, cln.normalized_shape, nh.param(aln, "single_cond_layer_norm"),
                          nh.param(aln, "single_cond_layer_norm", "bias"), cln.eps, out_dtype=dtype, owner=cln)
    # scale and shift stay fp32 (one rounding fewer before the sigmoid and the add); one launch over the
    # stacked weights, made on the first pass (the next one may be a graph capture). Weights of which
    # nothing is kept are not worth stacking on every call (fp32 CrossAttention 300 us, 279 in two launches).
    if stacked is None:
        sources = _scale_shift_sources(aln)
        if sources[0].is_inference():
            scale, shift = (ops.linear(cond, nh.linear_weight(aln, name, dtype), b, dtype, out_dtype=torch.float32)
                            for name, b in (("single_cond_scale", sources[2]), ("single_cond_bias", None)))
            return ops.adaptive_layer_norm(x, scale, shift, aln.layer_norm.eps, out_dtype=out_dtype)
        stacked = nh.derived_weight(aln, f"scale_shift:{dtype}", [t for t in sources if t is not None],
                                    lambda *ts: _scale_shift_weights(dtype, *ts))
    scale, shift = ops.linear_batched(cond.reshape(-1, cond.shape[-1]), *stacked[:2], dtype, out_dtype=torch.float32)
    return ops.adaptive_layer_norm(x, scale, shift, aln.layer_norm.eps, out_dtype=out_dtype)


def _scale_shift_sources(aln: nn.Module) -> tuple:
    return (*nh.params(aln, ("single_cond_scale", "single_cond_bias")), nh.param(aln, "single_cond_scale", "bias"))


def _scale_shift_weights(dtype: torch.dtype, scale: torch.Tensor, shift: torch.Tensor,
                         bias: Optional[torch.Tensor] = None, others=()):
    """single_cond_scale and single_cond_bias as one [2, c, c_cond] weight in ``dtype`` and their
    [2, c] fp32 bias (zeros for single_cond_bias, which has none; None without a bias); then copies
    of ``others``, made by the same call."""
    nh.check_one_device([scale, shift, *others])
    c, k = scale.shape
    w = torch.empty((2, c, k), dtype=dtype, device=scale.device)
    copies = [torch.empty(t.shape, dtype=dtype, device=t.device) for t in others]
    torch._foreach_copy_([*w.unbind(0), *copies], [scale, shift, *others])
    if bias is None:
        return (w, None, *copies)
    b = torch.zeros((2, c), dtype=torch.float32, device=scale.device)
    b[0].copy_(bias)
    return (w, b, *copies)


def _ada_ln_zero(zero: nn.Module, hidden: torch.Tensor, single_cond: Optional[torch.Tensor],
                 dtype: torch.dtype, accumulate_into: Optional[torch.Tensor],
                 cond: Optional[torch.Tensor] = None, weights: Optional[tuple] = None) -> torch.Tensor:
    """``AdaLNZero.forward`` (``diffusion_transformer.py:85-95``), optionally added in place;
    ``cond`` = adaptive_zero_cond(single_cond) already computed, in the output dtype; ``weights`` =
    the prepared transition2 and adaptive_zero_cond that the caller has at hand."""
    w = weights[0] if weights is not None else nh.linear_weight(zero, "transition2", dtype)
    out = accumulate_into
    out_dtype = out.dtype if out is not None else dtype
    acc = out is not None
    if zero.use_single_cond:
        if cond is None:
            w_cond = weights[1] if weights is not None else nh.linear_weight(zero, "adaptive_zero_cond", dtype)
            cond = ops.linear(single_cond, w_cond, nh.param(zero, "adaptive_zero_cond", "bias"), dtype,
                              out_dtype=out_dtype)
        epi = nh.EPI_MUL_SIGMOID_AUX_ACCUMULATE if acc else nh.EPI_MUL_SIGMOID_AUX
        return ops.linear(hidden, w, None, dtype, out=out, out_dtype=out_dtype, epilogue=epi,
                          aux=cond, aux_rows=cond.numel() // cond.shape[-1])
    epi = nh.EPI_ACCUMULATE if acc else nh.EPI_STORE
    return ops.linear(hidden, w, None, dtype, out=out, out_dtype=out_dtype, epilogue=epi)


def _check_accumulate(out, x):
    if out is not None and (not out.is_contiguous() or out.shape != x.shape):
        raise ValueError("accumulate_into must be a contiguous tensor shaped like x")


def diffusion_transition_hip(module: nn.Module, x: torch.Tensor, single_cond=None,
                             accumulate_into: Optional[torch.Tensor] = None, *,
                             _cond: Optional[tuple] = None) -> torch.Tensor:
    """``DiffusionTransition.forward`` (``diffusion_transformer.py:124-128``). ``_cond`` =
    (scale, shift, zero_cond) precomputed by :func:`_block_conditioning`."""
    nh.check_gpu_inference(x, single_cond)
    nh.check_module(module)
    w1 = nh.param(module, "transition1")
    dtype = nh.compute_dtype(x, w1)
    _check_accumulate(accumulate_into, x)
    aln, zero = module._modules["adaptive_layernorm"], module._modules["adaptive_zero_init"]
    stacked = weights = None
    if _cond is None and aln.use_single_cond and zero.use_single_cond and w1.dtype != dtype and not w1.is_inference():
        # A call of its own under autocast: every plain weight in one entry, copied by one call.
        *scale_shift, bias = _scale_shift_sources(aln)
        others = nh.params(zero, ("transition2", "adaptive_zero_cond"))
        stacked = nh.derived_weight(
            module, f"conditioned:{dtype}", [*scale_shift, *others] if bias is None else [*scale_shift, *others, bias],
            lambda scale, shift, *ts: _scale_shift_weights(dtype, scale, shift, bias, ts[:2]))
        weights = stacked[2:]
    xn = _adaptive_layer_norm(aln, x, single_cond, dtype, cond=None if _cond is None else _cond[:2], stacked=stacked)
    hidden = ops.gated_linear_unit(xn, nh.linear_weight(module, "transition1", dtype, "glu"), w1.shape[0] // 2, dtype)
    return _ada_ln_zero(zero, hidden, single_cond, dtype, accumulate_into, cond=None if _cond is None else _cond[2],
                        weights=weights)


_QKV = ("q_projection", "k_projection", "v_projection")


def _projection_bias(module: nn.Module, c: int, parts: int, device: torch.device) -> Optional[torch.Tensor]:
    """fp32 bias of the stacked [q | k | v (| gate)] projection: q_projection's bias, zeros
    for the rest (k, v and the gate have none), cached while the bias is unchanged."""
    q_bias = module.q_projection.bias
    if q_bias is None:
        return None

    def build(bias):
        full = torch.zeros(parts * c, dtype=torch.float32, device=device)
        full[:c] = bias.detach().to(torch.float32)
        return full
    return nh.derived_weight(module, f"projection_bias{parts}", [q_bias], build)


def qkvg_weights(module: nn.Module, dtype: torch.dtype):
    """[Wq; Wk; Wv; Wgate] in ``dtype`` and its fp32 bias (or None)."""
    w = nh.fused_linear_weight(module, _QKV + ("gating_query",), dtype)
    return w, _projection_bias(module, w.shape[0] // 4, 4, w.device)


_LOG2E = 1.4426950408889634


def self_attention_hip(module: nn.Module, x: torch.Tensor, mask: Optional[torch.Tensor],
                       pair_logits: Optional[torch.Tensor] = None,
                       single_cond: Optional[torch.Tensor] = None,
                       accumulate_into: Optional[torch.Tensor] = None, *,
                       _cond: Optional[tuple] = None,
                       _operands: Optional[ops.AttentionOperands] = None) -> torch.Tensor:
    """``SelfAttention.forward`` (``diffusion_transformer.py:184-217``) for x [N, c] or
    [S, N, c]; pair_logits [H, N, N] is the attention bias, mask [N] the key mask.
    ``_cond`` = (scale, shift, zero_cond) precomputed by :func:`_block_conditioning`.

    With bf16, a packed bias and head dims the pipelined kernel takes, the q/k/v and gating
    projections are one GEMM writing the attention kernel's layouts, and the gate is applied
    at the attention's store. ``_operands`` (an :class:`ops.AttentionOperands` of this shape,
    its mask words already set) lets a caller reuse one set of buffers over many blocks."""
    logits_t = pair_logits.tensor if isinstance(pair_logits, ops.PackedBias) else pair_logits
    nh.check_gpu_inference(x, mask, logits_t, single_cond)
    nh.check_module(module)
    sources = [*nh.params(module, _QKV + ("gating_query",)), nh.param(module, "q_projection", "bias")]
    dtype = nh.compute_dtype(x, *sources[:4])
    _check_accumulate(accumulate_into, x)
    if x.dim() not in (2, 3):
        raise ValueError("SelfAttention expects x [N, c] or [S, N, c]")
    samples = 1 if x.dim() == 2 else x.shape[0]
    n, c = x.shape[-2], x.shape[-1]
    heads = module.num_head
    d = c // heads
    xn = _adaptive_layer_norm(module.adaptive_layernorm, x, single_cond, dtype,
                              cond=None if _cond is None else _cond[:2])
    if dtype == torch.bfloat16 and isinstance(pair_logits, ops.PackedBias) and c % 32 == 0 and \
            ops.AttentionOperands.supported(n, heads, d) and \
            (mask is None or tuple(mask.shape) in ((n,), (samples, n))):
        operands = _operands
        if operands is None or not operands.matches(samples, n, heads, d, x.device):
            operands = ops.shared_attention_operands(samples, n, heads, d, x.device)
        operands.set_mask(mask)
        _, (w_all, b_all) = nh.gather(module, "qkvg", sources, 4, x, lambda dt: qkvg_weights(module, dt), dtype)
        ops.attention_project(xn, w_all, b_all, operands, d ** -0.5 * _LOG2E)
        o = ops.attention_on_operands(operands, pair_logits, torch.empty((samples, n, c), dtype=dtype, device=x.device))
        return _ada_ln_zero(module.adaptive_zero_init, o.reshape(x.shape), single_cond, dtype, accumulate_into,
                            cond=None if _cond is None else _cond[2])
    w_qkv = nh.fused_linear_weight(module, _QKV, dtype)
    bias_qkv = _projection_bias(module, c, 3, x.device)
    qkv = ops.linear(xn, w_qkv, bias_qkv, dtype)                     # [.., N, 3c]
    qkv = qkv.reshape(samples, n, 3 * c)
    row = 3 * c
    views = [torch.as_strided(qkv, (samples, heads, n, d), (n * row, d, row, 1), i * c)
             for i in range(3)]
    o = torch.empty((samples, n, c), dtype=dtype, device=x.device)
    o_view = torch.as_strided(o, (samples, heads, n, d), (n * c, d, c, 1), 0)
    bias = None
    if isinstance(pair_logits, ops.PackedBias):
        bias = pair_logits
    elif pair_logits is not None:
        bias = pair_logits if pair_logits.dim() == 4 else pair_logits.unsqueeze(0)
    ops.attention(views[0], views[1], views[2], mask, bias, out=o_view)
    ops.linear(xn.reshape(samples, n, c), nh.linear_weight(module, "gating_query", dtype), None, dtype,
               out=o, epilogue=nh.EPI_SIGMOID_MUL_AUX, aux=o)
    o = o.reshape(x.shape)
    return _ada_ln_zero(module.adaptive_zero_init, o, single_cond, dtype, accumulate_into,
                        cond=None if _cond is None else _cond[2])


def _conditioning_weights(module: nn.Module, alns, zeros, dtype: torch.dtype):
    """Stacked conditioning weights of every block (a cached one-time weight preparation):
    ([2A, c, c_s] scale/shift weights with the single_cond LayerNorm's weight folded into
    their input columns, [2A, c] fp32 biases, [Z, c, c_s] adaptive_zero_cond weights, [Z, c]
    biases). LayerNorm(s) = s_hat * g + b, so Linear(LayerNorm(s)) = s_hat (W g)^T + (W b + bias)."""
    linears = ("single_cond_scale", "single_cond_bias")
    norms = [nh.params(a, (), ("single_cond_layer_norm",)) for a in alns]
    conds = [[(nh.param(a, name), nh.param(a, name, "bias")) for name in linears] for a in alns]
    zero_conds = [(nh.param(z, "adaptive_zero_cond"), nh.param(z, "adaptive_zero_cond", "bias")) for z in zeros]
    srcs = [t for norm, cond in zip(norms, conds) for t in (*norm, *cond[0], *cond[1]) if t is not None]
    srcs += [t for pair in zero_conds for t in pair if t is not None]

    def build(*_):
        with torch.no_grad():
            none = torch.zeros(conds[0][0][0].shape[0], dtype=torch.float32, device=srcs[0].device)

            def bias_of(w, b):
                return b.detach().float() if b is not None else none if w.shape[0] == len(none) else w.new_zeros(w.shape[0])
            ws, bs = [], []
            for (nw, nb), cond in zip(norms, conds):
                for weight, bias in cond:
                    w = weight.detach().float()
                    b = bias_of(w, bias)
                    if nb is not None:
                        b = b + w @ nb.detach().float()
                    ws.append(w * nw.detach().float() if nw is not None else w)
                    bs.append(b)
            zw = [w.detach().float() for w, _ in zero_conds]
            zb = [bias_of(w, b) for w, (_, b) in zip(zw, zero_conds)]
            return (torch.stack(ws).to(dtype).contiguous(), torch.stack(bs).contiguous(),
                    torch.stack(zw).to(dtype).contiguous(), torch.stack(zb).contiguous())

    return nh.derived_weight(module, f"conditioning:{dtype}", srcs, build)


def _block_parts(module: nn.Module):
    """The transformer's attention and transition blocks, their AdaptiveLayerNorms and AdaLNZeros
    (every attention's first, then every transition's)."""
    att, tr = list(module.self_attention._modules.values()), list(module.transition_block._modules.values())
    alns = [b._modules["adaptive_layernorm"] for b in att + tr]
    zeros = [b._modules["adaptive_zero_init"] for b in att + tr]
    return att, tr, alns, zeros


def _block_conditioning(single_cond: torch.Tensor, alns, dtype: torch.dtype, zero_dtype: torch.dtype, weights):
    """Every block's conditioning linears (``AdaptiveLayerNorm`` scale/shift,
    ``diffusion_transformer.py:59-62``; ``AdaLNZero`` cond, ``:93``) computed up front: they
    read only single_cond, which is the same for all blocks of one call. Two batched launches
    (one over the normalised single_cond, one over single_cond itself) replace the 6 small
    GEMMs of every block. Returns the [2A, rows, c] scale/shift pairs of ``alns`` and the
    [Z, rows, c] conditions (:func:`_conditioning_weights` order)."""
    w_ss, b_ss, w_z, b_z = weights
    cln = alns[0].single_cond_layer_norm
    s_hat = ops.layer_norm(single_cond, cln.normalized_shape, None, None, cln.eps, out_dtype=dtype)
    ss = ops.linear_batched(s_hat.reshape(-1, s_hat.shape[-1]), w_ss, b_ss, dtype)
    zz = ops.linear_batched(single_cond.reshape(-1, single_cond.shape[-1]), w_z, b_z, dtype, out_dtype=zero_dtype)
    return ss, zz


def _conditioned_alike(single_cond, alns, zeros) -> bool:
    """Whether every block is conditioned on single_cond through LayerNorms of one shape and eps
    (else the conditioning runs block by block)."""
    if single_cond is None or not all(a.use_single_cond for a in alns) or not all(z.use_single_cond for z in zeros):
        return False
    norms = [a.single_cond_layer_norm for a in alns]
    return len({(n.eps, tuple(n.normalized_shape)) for n in norms}) == 1


def _block_sources(att, tr, alns, zeros):
    """The parameters of every block: q, k, v, gating and transition1 weights first (the ones
    that take part in the compute dtype), then the rest."""
    weights, rest = [], []
    for a in att:
        weights += nh.params(a, _QKV + ("gating_query",))
        rest.append(nh.param(a, "q_projection", "bias"))
    for t in tr:
        weights.append(nh.param(t, "transition1"))
    for z in zeros:
        rest += (nh.param(z, "transition2"), nh.param(z, "adaptive_zero_cond"), nh.param(z, "adaptive_zero_cond", "bias"))
    for a in alns:
        rest += nh.params(a, ("single_cond_scale", "single_cond_bias"), ("single_cond_layer_norm",))
        rest += (nh.param(a, "single_cond_scale", "bias"), nh.param(a, "single_cond_bias", "bias"))
    return weights, rest


def _stacked_logits_weight(module: nn.Module, projs, dtype: torch.dtype) -> torch.Tensor:
    """Every super-block's pair-logit projection stacked, in ``dtype``."""
    return nh.derived_weight(module, f"pair_logits:{dtype}", projs,
                             lambda *ws: torch.cat([w.detach() for w in ws], dim=0).to(dtype).contiguous())


def _block_weights(module, att, tr, alns, zeros, projs, dtype: torch.dtype) -> dict:
    """What the blocks' call needs of their parameters; ``c`` is None when the blocks differ in
    shape or the compute dtype is not bf16 (they then run one by one)."""
    out = [nh.linear_weight(z, "transition2", dtype) for z in zeros]
    glu = [nh.linear_weight(t, "transition1", dtype, "glu") for t in tr]
    c, f = out[0].shape[0], nh.param(tr[0], "transition1").shape[0] // 2
    same = dtype == torch.bfloat16 and \
        all(tuple(nh.param(a, n).shape) == (c, c) for a in att for n in _QKV + ("gating_query",)) and \
        all(tuple(nh.param(t, "transition1").shape) == (2 * f, c) for t in tr) and \
        all(tuple(w.shape) == ((c, c) if i < len(att) else (c, f)) for i, w in enumerate(out))
    return dict(conditioning=_conditioning_weights(module, alns, zeros, dtype),
                logits=_stacked_logits_weight(module, projs, dtype),
                qkvg=[qkvg_weights(a, dtype) for a in att] if same else None,
                glu=glu, out=out, c=c if same else None, f=f)


def _cached(module: nn.Module, name: str, dependencies, factory, modules):
    """``module._input_cache.get`` (``xfold/nn/diffusion_transformer.py:255-265``) when the
    module carries an input cache (this package's or the reference's InputCache, which share
    the interface), else ``factory()``."""
    cache = getattr(module, "_input_cache", None)
    if cache is None:
        return factory()
    return cache.get(name, dependencies, module, factory, modules=modules)


def _block_operands(module: nn.Module, act: torch.Tensor, mask: Optional[torch.Tensor]):
    """The attention-operand buffers (and mask words) every block of a forward uses, or None
    when the blocks' attention takes the general path."""
    samples = 1 if act.dim() == 2 else act.shape[0]
    n, c, heads = act.shape[-2], act.shape[-1], module.num_head
    if c % heads or not ops.AttentionOperands.supported(n, heads, c // heads):
        return None
    if mask is not None and tuple(mask.shape) not in ((n,), (samples, n)):
        return None
    operands = ops.shared_attention_operands(samples, n, heads, c // heads, act.device)
    operands.set_mask(mask)
    return operands


def _block_cond(conds, index: int, n: int):
    """Block ``index``'s attention and transition (scale, shift, zero condition), of n blocks."""
    if conds is None:
        return None, None
    ss, zz = conds
    return tuple((ss[2 * i], ss[2 * i + 1], zz[i]) for i in (index, n + index))


def _block_struct(i: int, n_blocks: int, weights, conds, packed: torch.Tensor, heads: int, att: nn.Module,
                  tr: nn.Module) -> "nh.DiffusionBlock":
    ss, zz = conds
    n = zz.shape[0] // 2
    w_qkvg, b_qkvg = weights["qkvg"][i]
    ss_ptr, ss_step = nh.ptr(ss), ss.stride(0) * ss.element_size()
    zz_ptr, zz_step = nh.ptr(zz), zz.stride(0) * zz.element_size()
    return nh.DiffusionBlock(
        nh.ptr(w_qkvg), nh.ptr(b_qkvg), nh.ptr(packed) + i * heads * packed.stride(0) * packed.element_size(),
        nh.ptr(weights["out"][i]), nh.ptr(weights["glu"][i]), nh.ptr(weights["out"][n + i]),
        ss_ptr + 2 * i * ss_step, ss_ptr + (2 * i + 1) * ss_step, zz_ptr + i * zz_step,
        ss_ptr + 2 * (n + i) * ss_step, ss_ptr + (2 * (n + i) + 1) * ss_step, zz_ptr + (n + i) * zz_step,
        att._modules["adaptive_layernorm"].layer_norm.eps, tr._modules["adaptive_layernorm"].layer_norm.eps)


def diffusion_transformer_hip(module: nn.Module, act: torch.Tensor, mask: torch.Tensor,
                              single_cond: torch.Tensor, pair_cond: torch.Tensor) -> torch.Tensor:
    """``DiffusionTransformer.forward`` (``diffusion_transformer.py:250-272``), updating
    ``act`` ([N, c] or [S, N, c], contiguous) in place and returning it.

    Inside an input-cache scope (``xfold_cpu_amd.nn.cache``, the reference's ``InputCache``
    rules) the packed pair logits of every super-block are kept across calls with the same
    ``pair_cond`` and weights, as the reference keeps its pair logits (``:255-265``), when
    they fit the scope's byte budget."""
    nh.check_gpu_inference(act, mask, single_cond, pair_cond)
    if not act.is_contiguous():
        raise ValueError("DiffusionTransformer (hip) updates act in place; pass a contiguous tensor")
    ln = module.pair_input_layer_norm
    heads, size = module.num_head, module.super_block_size
    n_blocks = module.num_super_blocks * size
    att, tr, alns, zeros = _block_parts(module)
    projs = [nh.param(module.pair_logits_projection, name) for name in module.pair_logits_projection._modules]
    dtype = nh.compute_dtype(act, projs[0])
    # Not input-cache entries: their key would cover ~400 parameters, whose checks cost more
    # host time than the two batched GEMMs they would save.
    conds = weights = None
    if _conditioned_alike(single_cond, alns, zeros):
        if not nh.first_pass(module, "blocks"):
            block_weights, rest = _block_sources(att, tr, alns, zeros)
            _, weights = nh.gather(
                module, "blocks", block_weights + projs + rest, len(block_weights), act,
                lambda dt: _block_weights(module, att, tr, alns, zeros, projs, dt), again=True)
        conds = _block_conditioning(single_cond, alns, dtype, act.dtype,
                                    weights["conditioning"] if weights is not None else
                                    _conditioning_weights(module, alns, zeros, dtype))
    # A packed bias (either path below) feeds the pipelined attention kernel, which takes
    # bf16, head dims <= 64 and at most attention_max_keys() keys.
    packed_bias = dtype == torch.bfloat16 and act.shape[-1] // heads <= 64 and \
        pair_cond.shape[0] <= nh.attention_max_keys()
    if packed_bias and pair_cond.shape[-1] == 128 and n_blocks * heads <= 384 and \
            tuple(ln.normalized_shape) == (128,):
        # Every super-block's pair logits in one pass over pair_cond, straight into the
        # attention kernel's bias layout; block b reads heads b*H .. b*H + H - 1.
        w_all = weights["logits"] if weights is not None else _stacked_logits_weight(module, projs, dtype)
        # bf16 logits, the dtype of the reference's autocast Linear output (half the bytes of
        # fp32: at N=768 all 24 blocks' logits take 453 MB and fit the input cache's budget).
        packed = _cached(module, "pair_logits_packed", (pair_cond, heads),
                         lambda: ops.pair_attention_bias(pair_cond, ln.weight, ln.bias, ln.eps, w_all, owner=ln,
                                                         out_dtype=torch.bfloat16),
                         modules=(ln, module.pair_logits_projection))
        operands = _block_operands(module, act, mask)
        c = act.shape[-1]
        # The whole stack in one library call when every block has the same shapes.
        if weights is not None and operands is not None and c % 32 == 0 and act.dim() in (2, 3) and \
                weights["c"] == c and conds[0].shape[-1] == conds[1].shape[-1] == c and \
                packed.shape[0] >= n_blocks * heads and tuple(packed.shape[1:]) == (act.shape[-2], operands.tpad) and \
                all(a.num_head == heads for a in att):
            blocks = (nh.DiffusionBlock * n_blocks)(*(
                _block_struct(i, n_blocks, weights, conds, packed, heads, att[i], tr[i]) for i in range(n_blocks)))
            ops.diffusion_blocks(act, operands, blocks, conds[0].shape[1], weights["f"], packed.dtype)
            return act
        for index in range(n_blocks):
            att_cond, tr_cond = _block_cond(conds, index, len(att))
            bias = ops.PackedBias(packed[index * heads:(index + 1) * heads])
            self_attention_hip(module.self_attention[index], act, mask, bias, single_cond,
                               accumulate_into=act, _cond=att_cond, _operands=operands)
            diffusion_transition_hip(module.transition_block[index], act, single_cond,
                                     accumulate_into=act, _cond=tr_cond)
        return act
    pair_act = ops.layer_norm(pair_cond, ln.normalized_shape, ln.weight, ln.bias, ln.eps,
                              out_dtype=dtype, owner=ln)
    operands = _block_operands(module, act, mask) if packed_bias else None
    for s in range(module.num_super_blocks):
        weight = nh.linear_weight(module.pair_logits_projection, str(s), dtype)
        logits = ops.linear(pair_act, weight, None, dtype)               # [N, N, size*heads]
        # 'n s (b h) -> b h n s': block j, head h reads column j*heads + h. On the pipelined
        # attention path (bf16, head dim <= 64) the super-block's biases are converted once.
        n_tok = logits.shape[0]
        if packed_bias:
            packed = ops.attention_bias_pack(logits.view(n_tok, n_tok, size, heads).permute(2, 3, 0, 1))
        for j in range(size):
            if packed_bias:
                bias = ops.PackedBias(packed[j])
            else:
                bias = logits[..., j * heads:(j + 1) * heads].permute(2, 0, 1)
            index = s * size + j
            att_cond, tr_cond = _block_cond(conds, index, len(att))
            self_attention_hip(module.self_attention[index], act, mask, bias, single_cond,
                               accumulate_into=act, _cond=att_cond, _operands=operands)
            diffusion_transition_hip(module.transition_block[index], act, single_cond,
                                     accumulate_into=act, _cond=tr_cond)
    return act


class AdaptiveLayerNorm(nn.Module):
    def __init__(self, c_x: int, c_single_cond: int, use_single_cond: bool = False) -> None:
        super().__init__()
        self.c_x = c_x
        self.c_single_cond = c_single_cond
        self.use_single_cond = use_single_cond
        if use_single_cond:
            self.layer_norm = LayerNorm(c_x, elementwise_affine=False, bias=False)
            self.single_cond_layer_norm = LayerNorm(c_single_cond, bias=False)
            self.single_cond_scale = nn.Linear(c_single_cond, c_x, bias=True)
            self.single_cond_bias = nn.Linear(c_single_cond, c_x, bias=False)
        else:
            self.layer_norm = LayerNorm(c_x)

    def forward(self, x, single_cond=None):
        _require(fastnn_config.layer_norm_implementation, "layer_norm_implementation")
        nh.check_gpu_inference(x, single_cond)
        dtype = nh.compute_dtype(x)
        # Under CUDA autocast the reference's LayerNorm output is fp32 and so is the
        # conditioned sum (fp32 * bf16 + bf16); outside autocast it is x's dtype.
        out_dtype = torch.float32 if torch.is_autocast_enabled("cuda") else x.dtype
        return _adaptive_layer_norm(self, x, single_cond, dtype, out_dtype)


class AdaLNZero(nn.Module):
    def __init__(self, c_in: int, c_out: int, c_single_cond: int, use_single_cond: bool = False):
        super().__init__()
        self.c_in = c_in
        self.c_out = c_out
        self.c_single_cond = c_single_cond
        self.use_single_cond = use_single_cond
        self.transition2 = nn.Linear(c_in, c_out, bias=False)
        if use_single_cond:
            self.adaptive_zero_cond = nn.Linear(c_single_cond, c_out, bias=True)

    def forward(self, x, single_cond=None):
        dtype = nh.compute_dtype(x, self.transition2.weight)
        return _ada_ln_zero(self, x, single_cond, dtype, None)


def _require(flag_value: str, what: str):
    if flag_value != fastnn_config.HIP:
        raise ValueError(f"Unknown {what} for xfold_cpu_amd: {flag_value!r} (only 'hip')")


class DiffusionTransition(nn.Module):
    def __init__(self, c_x: int, c_single_cond: int, num_intermediate_factor: int = 2,
                 use_single_cond: bool = False) -> None:
        super().__init__()
        self.c_x = c_x
        self.c_single_cond = c_single_cond
        self.num_intermediate_factor = num_intermediate_factor
        self.use_single_cond = use_single_cond
        self.adaptive_layernorm = AdaptiveLayerNorm(c_x, c_single_cond, use_single_cond)
        self.transition1 = nn.Linear(c_x, 2 * c_x * num_intermediate_factor, bias=False)
        self.adaptive_zero_init = AdaLNZero(num_intermediate_factor * c_x, c_x, c_single_cond,
                                            use_single_cond)

    def forward(self, x, single_cond=None):
        _require(fastnn_config.gated_linear_unit_implementation, "gated_linear_unit_implementation")
        return diffusion_transition_hip(self, x, single_cond)


class SelfAttention(nn.Module):
    def __init__(self, c_x: int = 768, c_single_cond: int = 384, num_head: int = 16,
                 use_single_cond: bool = False) -> None:
        super().__init__()
        self.c_x = c_x
        self.c_single_cond = c_single_cond
        self.num_head = num_head
        self.qkv_dim = c_x // num_head
        self.use_single_cond = use_single_cond
        self.adaptive_layernorm = AdaptiveLayerNorm(c_x, c_single_cond, use_single_cond)
        self.q_projection = nn.Linear(c_x, c_x, bias=True)
        self.k_projection = nn.Linear(c_x, c_x, bias=False)
        self.v_projection = nn.Linear(c_x, c_x, bias=False)
        self.gating_query = nn.Linear(c_x, c_x, bias=False)
        self.adaptive_zero_init = AdaLNZero(c_x, c_x, c_single_cond, use_single_cond)

    def forward(self, x, mask, pair_logits=None, single_cond=None):
        _require(fastnn_config.dot_product_attention_implementation, "dot_product_attention_implementation")
        return self_attention_hip(self, x, mask, pair_logits, single_cond)


def cross_attention_hip(module: nn.Module, x_q: torch.Tensor, x_k: torch.Tensor, mask_q: torch.Tensor,
                        mask_k: torch.Tensor, pair_logits: Optional[torch.Tensor] = None,
                        single_cond_q: Optional[torch.Tensor] = None, single_cond_k: Optional[torch.Tensor] = None,
                        accumulate_into: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``CrossAttention.forward`` (``diffusion_transformer.py:304-350``) for x_q [..., Q, c],
    x_k [..., K, c] with masks [..., Q] / [..., K] and pair_logits broadcastable to
    [..., H, Q, K]: the q/k adaptive LayerNorms, the q and fused k|v projections, one
    attention over all subsets whose fp32 bias (pair logits + the reference's positive 1e9
    on pairs of a masked query and a masked key) comes from xfh_cross_attention_bias, the
    sigmoid gate as the gating Linear's epilogue and the conditioned AdaLNZero."""
    if mask_q.dim() != x_q.dim() - 1 or mask_k.dim() != x_k.dim() - 1:
        raise ValueError(f"CrossAttention: masks must drop the channel dim of x ({tuple(mask_q.shape)}, "
                         f"{tuple(x_q.shape)}; {tuple(mask_k.shape)}, {tuple(x_k.shape)})")
    nh.check_gpu_inference(x_q, x_k, mask_q, mask_k, pair_logits, single_cond_q, single_cond_k)
    nh.check_module(module)
    sources = nh.params(module, _QKV + ("gating_query",))
    dtype = nh.compute_dtype(x_q, *sources)
    lead, nq, nk = tuple(x_q.shape[:-2]), x_q.shape[-2], x_k.shape[-2]
    if tuple(x_k.shape[:-2]) != lead:
        raise ValueError("CrossAttention: x_q and x_k must share their leading (subset) dims")
    batch = 1
    for d in lead:
        batch *= d
    h, dk, dv = module.num_head, module.key_dim_per_head, module.value_dim_per_head
    kd, vd = module.key_dim, module.value_dim
    if accumulate_into is not None and (not accumulate_into.is_contiguous() or
                                        tuple(accumulate_into.shape) != lead + (nq, vd)):
        raise ValueError("accumulate_into must be a contiguous [..., Q, value_dim] tensor")
    fused = _cross_attention_fused(module, x_q, x_k, mask_q, mask_k, pair_logits, single_cond_q, single_cond_k, dtype,
                                   lead, batch, accumulate_into)
    if fused is not None:
        return fused
    _, (w_q, w_kv, w_gate) = nh.gather(
        module, "cross_attention", sources, 4, x_q,
        lambda dt: (nh.linear_weight(module, "q_projection", dt),
                    nh.fused_linear_weight(module, ("k_projection", "v_projection"), dt),
                    nh.linear_weight(module, "gating_query", dt)), dtype)
    xq = _adaptive_layer_norm(module.q_adaptive_layernorm, x_q, single_cond_q, dtype)
    xk = _adaptive_layer_norm(module.k_adaptive_layernorm, x_k, single_cond_k, dtype)
    q = ops.linear(xq, w_q, nh.param(module, "q_projection", "bias"), dtype)
    kv = ops.linear(xk, w_kv, None, dtype)
    q4 = torch.as_strided(q, (batch, h, nq, dk), (nq * kd, dk, kd, 1))
    k4 = torch.as_strided(kv, (batch, h, nk, dk), (nk * (kd + vd), dk, kd + vd, 1))
    v4 = torch.as_strided(kv, (batch, h, nk, dv), (nk * (kd + vd), dv, kd + vd, 1), kd)
    mq, mq_code = nh.mask_arg(mask_q, lead + (nq,))
    mk, mk_code = nh.mask_arg(mask_k, lead + (nk,))
    bias = torch.empty((batch, h, nq, nk), dtype=torch.float32, device=x_q.device)
    pl, pl_code, strides = None, nh.F32, None
    if pair_logits is not None:
        if pair_logits.dtype not in (torch.float32, torch.bfloat16):
            raise ValueError("CrossAttention: pair_logits must be fp32 or bf16")
        pl = pair_logits.expand(*lead, h, nq, nk).reshape(batch, h, nq, nk)
        pl_code = nh.dtype_code(pl.dtype)
        strides = (ctypes.c_int64 * 4)(*pl.stride())
    nh.call("xfh_cross_attention_bias", nh.ptr(pl), pl_code, strides, nh.ptr(mq), mq_code, nh.ptr(mk), mk_code,
            batch, h, nq, nk, nh.ptr(bias), nh.stream_of(x_q.device))
    o = torch.empty(lead + (nq, vd), dtype=dtype, device=x_q.device)
    o_view = torch.as_strided(o, (batch, h, nq, dv), (nq * vd, dv, vd, 1))
    ops.attention(q4, k4, v4, None, bias, out=o_view, scale=module.q_scale)
    ops.linear(xq, w_gate, None, dtype, out=o, epilogue=nh.EPI_SIGMOID_MUL_AUX, aux=o)
    return _ada_ln_zero(module.adaptive_zero_init, o, single_cond_q, dtype, accumulate_into)


def _cross_sources(module: nn.Module):
    """Parameters of a conditioned CrossAttention: the matrices, then biases and LayerNorms."""
    m = module._modules
    alns, zero = (m["q_adaptive_layernorm"], m["k_adaptive_layernorm"]), m["adaptive_zero_init"]
    matrices = [nh.param(a, n) for a in alns for n in ("single_cond_scale", "single_cond_bias")]
    matrices += nh.params(module, _QKV + ("gating_query",)) + nh.params(zero, ("adaptive_zero_cond", "transition2"))
    rest = [nh.param(module, "q_projection", "bias"), nh.param(zero, "adaptive_zero_cond", "bias")]
    for a in alns:
        rest += (nh.param(a, "single_cond_scale", "bias"), nh.param(a, "single_cond_layer_norm"),
                 nh.param(a, "single_cond_layer_norm", "bias"))
    return matrices, rest


def _cross_values(module: nn.Module, dtype: torch.dtype):
    """The prepared weights in ``XfhCrossWeights`` order."""
    m = module._modules
    alns, zero = (m["q_adaptive_layernorm"], m["k_adaptive_layernorm"]), m["adaptive_zero_init"]
    out = []
    for a in alns:
        out += (*nh.norm_params(a, "single_cond_layer_norm"), nh.linear_weight(a, "single_cond_scale", dtype),
                nh.linear_weight(a, "single_cond_bias", dtype),
                nh.fp32_param(a, "single_cond_scale.bias", nh.param(a, "single_cond_scale", "bias")))
    out += (nh.linear_weight(module, "q_projection", dtype),
            nh.fp32_param(module, "q_projection.bias", nh.param(module, "q_projection", "bias")))
    out += (nh.linear_weight(module, n, dtype) for n in ("k_projection", "v_projection", "gating_query"))
    out += (nh.linear_weight(zero, "adaptive_zero_cond", dtype),
            nh.fp32_param(zero, "adaptive_zero_cond.bias", nh.param(zero, "adaptive_zero_cond", "bias")),
            nh.linear_weight(zero, "transition2", dtype))
    return out


def _cross_attention_fused(module: nn.Module, x_q, x_k, mask_q, mask_k, pair_logits, cond_q, cond_k,
                           dtype: torch.dtype, lead: tuple, batch: int, accumulate_into) -> Optional[torch.Tensor]:
    """The call in three launches (``xfh_cross_attention``) at the atom attention's widths: bf16
    compute, 128 channels, 4 heads, at most 128 keys, one activation dtype, every condition
    given; None otherwise. With the subsets' logits broadcast over outer leading dims the
    general path's one copy of them stays."""
    alns = (module.q_adaptive_layernorm, module.k_adaptive_layernorm)
    zero = module.adaptive_zero_init
    nq, nk = x_q.shape[-2], x_k.shape[-2]
    acts = (x_q, x_k, cond_q, cond_k)
    if (dtype != torch.bfloat16 or module.num_head != 4 or module.key_dim != 128 or module.value_dim != 128
            or cond_q is None or cond_k is None or not zero.use_single_cond
            or not all(a.use_single_cond for a in alns) or not 1 <= nk <= 128 or nq == 0
            or any(t.dtype != x_q.dtype for t in acts) or x_q.dtype not in (torch.float32, torch.bfloat16)
            or tuple(x_q.shape) != lead + (nq, 128) or tuple(x_k.shape) != lead + (nk, 128)
            or cond_q.shape != x_q.shape or cond_k.shape != x_k.shape
            or any(tuple(a.single_cond_layer_norm.normalized_shape) != (128,)
                   or tuple(a.layer_norm.normalized_shape) != (128,) for a in alns)):
        return None
    matrices, rest = _cross_sources(module)
    if any(tuple(w.shape) != (128, 128) for w in matrices) or any(nh.param(a, "single_cond_bias", "bias") is not None
                                                                  for a in alns):
        return None
    logits, code, strides = None, nh.F32, None
    if pair_logits is not None:
        if pair_logits.dtype not in (torch.float32, torch.bfloat16):
            raise ValueError("CrossAttention: pair_logits must be fp32 or bf16")
        logits = pair_logits.expand(*lead, 4, nq, nk).reshape(batch, 4, nq, nk)
        code, strides = nh.dtype_code(logits.dtype), (ctypes.c_int64 * 4)(*logits.stride())
    _, values = nh.gather(module, "fused", matrices + rest, 0, x_q, lambda dt: _cross_values(module, dt), dtype)
    mq, mq_code = nh.mask_arg(mask_q, lead + (nq,))
    mk, mk_code = nh.mask_arg(mask_k, lead + (nk,))
    acts = [t.contiguous() for t in acts]
    out = accumulate_into
    if out is None:
        out = torch.empty(lead + (nq, 128), dtype=dtype, device=x_q.device)
    if any(t.data_ptr() % 16 for t in (*acts, out)):
        return None
    eps = (ctypes.c_float * 4)(*(e for a in alns for e in (a.single_cond_layer_norm.eps, a.layer_norm.eps)))
    lib = nh.load_library()
    ws = nh.workspace(lib.xfh_cross_attention_workspace_size(batch, nq, nk), x_q.device)
    nh.call("xfh_cross_attention", *map(nh.ptr, acts), nh.dtype_code(x_q.dtype), nh.ptr(mq), mq_code, nh.ptr(mk), mk_code,
            nh.ptr(logits), code, strides, batch, nq, nk, nh.ptrs(values), eps, float(module.q_scale), nh.ptr(out),
            nh.dtype_code(out.dtype), int(accumulate_into is not None), nh.ptr(ws), ws.numel(), nh.stream_of(x_q.device))
    return out


class CrossAttention(nn.Module):
    def __init__(self, key_dim: int = 128, value_dim: int = 128, c_single_cond: int = 128,
                 num_head: int = 4) -> None:
        super().__init__()
        self.key_dim = key_dim
        self.value_dim = value_dim
        self.c_single_cond = c_single_cond
        self.num_head = num_head
        self.key_dim_per_head = key_dim // num_head
        self.value_dim_per_head = value_dim // num_head
        self.q_scale = self.key_dim_per_head ** (-0.5)
        self.q_adaptive_layernorm = AdaptiveLayerNorm(key_dim, c_single_cond, use_single_cond=True)
        self.k_adaptive_layernorm = AdaptiveLayerNorm(key_dim, c_single_cond, use_single_cond=True)
        self.q_projection = nn.Linear(key_dim, key_dim, bias=True)
        self.k_projection = nn.Linear(key_dim, key_dim, bias=False)
        self.v_projection = nn.Linear(value_dim, value_dim, bias=False)
        self.gating_query = nn.Linear(key_dim, value_dim, bias=False)
        self.adaptive_zero_init = AdaLNZero(value_dim, value_dim, key_dim, use_single_cond=True)

    def forward(self, x_q, x_k, mask_q, mask_k, pair_logits=None, single_cond_q=None, single_cond_k=None):
        _require(fastnn_config.dot_product_attention_implementation, "dot_product_attention_implementation")
        return cross_attention_hip(self, x_q, x_k, mask_q, mask_k, pair_logits, single_cond_q, single_cond_k)


class DiffusionTransformer(nn.Module):
    def __init__(self, c_act: int = 768, c_single_cond: int = 384, c_pair_cond: int = 128,
                 num_head: int = 16, num_blocks: int = 24, super_block_size: int = 4) -> None:
        super().__init__()
        self.c_act = c_act
        self.c_single_cond = c_single_cond
        self.c_pair_cond = c_pair_cond
        self.num_head = num_head
        self.num_blocks = num_blocks
        self.super_block_size = super_block_size
        self.num_super_blocks = num_blocks // super_block_size
        self.pair_input_layer_norm = LayerNorm(c_pair_cond)
        self.pair_logits_projection = nn.ModuleList(
            [nn.Linear(c_pair_cond, super_block_size * num_head, bias=False)
             for _ in range(self.num_super_blocks)])
        self.self_attention = nn.ModuleList(
            [SelfAttention(c_act, c_single_cond, use_single_cond=True) for _ in range(num_blocks)])
        self.transition_block = nn.ModuleList(
            [DiffusionTransition(c_act, c_single_cond, use_single_cond=True) for _ in range(num_blocks)])
        self._input_cache = InputCache()

    def forward(self, act, mask, single_cond, pair_cond):
        _require(fastnn_config.dot_product_attention_implementation, "dot_product_attention_implementation")
        _require(fastnn_config.gated_linear_unit_implementation, "gated_linear_unit_implementation")
        _require(fastnn_config.layer_norm_implementation, "layer_norm_implementation")
        return diffusion_transformer_hip(self, act, mask, single_cond, pair_cond)
