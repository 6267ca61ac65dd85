"""Performance cases of the Pairformer, MSA-stack and diffusion-transformer modules.

``listed()`` are the cases that are always timed, ``draw(rng)`` gives more of the same ranges.
A case names one module (its ``kind``) and its sizes; ``prepare`` builds the module with random
weights and its inputs on the GPU, ``run`` is one forward call, and ``exact`` is the same call in
64-bit torch. The modules run inference only, so there is no backward direction. Blocks update
``pair``, ``msa``, ``single`` and ``act`` in place, as a trunk or a sampler does block after block.

Kinds and their real use:
  pair_block           PairformerBlock: 48 of them per trunk pass (``single``: with its single track)
  template_block       PairformerBlock at 64 pair channels, factor 2: the template stack, per template
  triangle_mult        TriangleMultiplication returning its update (a caller with its own residual)
  triangle_attention   GridSelfAttention returning its update
  evoformer            EvoformerBlock: the MSA stack's block over ``rows`` sequences
  diffusion            DiffusionTransformer: 24 blocks over ``samples`` samples, once per denoising step
  diffusion_transition DiffusionTransition: one conditioned transition of that transformer
  cross_attention      CrossAttention of 32-atom query subsets over 128 keys: the atom encoder/decoder
"""

from __future__ import annotations

import math

import torch

from xfold_cpu_amd import nn as hnn

DEVICE = "cuda"


def listed():
    return [
        # A peptide or a small ligand complex: the smallest trunk call, where launches count.
        {"name": "pair_block_72", "kind": "pair_block", "n": 72, "pad": 5, "single": True, "dtype": "bf16"},
        # The benchmark's pair block: a typical single chain, 32 padded tokens.
        {"name": "pair_block_384", "kind": "pair_block", "n": 384, "pad": 32, "single": False, "dtype": "bf16"},
        # One block of the benchmark's trunk with its single track: a typical complex.
        {"name": "trunk_block_768", "kind": "pair_block", "n": 768, "pad": 77, "single": True, "dtype": "bf16"},
        # The fp32 mode (parity runs, debugging a checkpoint).
        {"name": "pair_block_fp32_128", "kind": "pair_block", "n": 128, "pad": 0, "single": False, "dtype": "fp32"},
        # An odd token count, the incoming direction, out of place.
        {"name": "triangle_mult_509", "kind": "triangle_mult", "n": 509, "pad": 20, "outgoing": False},
        # A large complex, odd token count, the ending node.
        {"name": "triangle_attention_1283", "kind": "triangle_attention", "n": 1283, "pad": 64, "transpose": True},
        # The template stack's block for one medium chain.
        {"name": "template_block_300", "kind": "template_block", "n": 300, "pad": 12},
        # The MSA stack's block: a crop with a moderately deep alignment.
        {"name": "evoformer_512x256", "kind": "evoformer", "rows": 512, "n": 256, "pad": 10},
        # One denoising step of the benchmark's diffusion transformer.
        {"name": "diffusion_5x768", "kind": "diffusion", "samples": 5, "n": 768, "pad": 0},
        # The same for a peptide and a single sample: the smallest denoising step.
        {"name": "diffusion_1x96", "kind": "diffusion", "samples": 1, "n": 96, "pad": 4},
        # One conditioned transition over five samples of a ragged length.
        {"name": "diffusion_transition_5x437", "kind": "diffusion_transition", "samples": 5, "n": 437},
        # One atom attention layer of a ~260-token complex: 24 atoms a token, 32 to a subset; the
        # logits are a view of a projection for three layers, heads innermost.
        {"name": "cross_attention_192", "kind": "cross_attention", "subsets": 192, "view": True},
    ]


def _spread(rng, low, high):
    """A whole number between low and high, spread evenly over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng):
    kind = rng.choice(["pair_block", "pair_block", "pair_block_fp32", "triangle_mult", "triangle_attention",
                       "template_block", "evoformer", "diffusion", "diffusion_transition", "cross_attention"])
    pad_of = lambda n: rng.randrange(0, max(1, n // 8) + 1)  # noqa: E731
    if kind == "pair_block":
        n = _spread(rng, 16, 768)
        return {"kind": kind, "n": n, "pad": pad_of(n), "single": rng.random() < 0.6, "dtype": "bf16"}
    if kind == "pair_block_fp32":
        n = _spread(rng, 16, 160)
        return {"kind": "pair_block", "n": n, "pad": pad_of(n), "single": rng.random() < 0.5, "dtype": "fp32"}
    if kind == "triangle_mult":
        n = _spread(rng, 32, 1100)
        return {"kind": kind, "n": n, "pad": pad_of(n), "outgoing": rng.random() < 0.5}
    if kind == "triangle_attention":
        n = _spread(rng, 32, 1200)
        return {"kind": kind, "n": n, "pad": pad_of(n), "transpose": rng.random() < 0.5}
    if kind == "template_block":
        n = _spread(rng, 24, 640)
        return {"kind": kind, "n": n, "pad": pad_of(n)}
    if kind == "evoformer":
        n = _spread(rng, 24, 384)
        return {"kind": kind, "rows": _spread(rng, 2, 1024), "n": n, "pad": pad_of(n)}
    if kind == "diffusion":
        n = _spread(rng, 32, 640)
        return {"kind": kind, "samples": rng.randrange(1, 6), "n": n, "pad": pad_of(n)}
    if kind == "diffusion_transition":
        return {"kind": kind, "samples": rng.randrange(1, 6), "n": _spread(rng, 32, 1100)}
    return {"kind": kind, "subsets": _spread(rng, 4, 1200), "view": rng.random() < 0.5}


# ------------------------------------------------------------------------------- preparation

def _module(case):
    kind = case["kind"]
    if kind == "pair_block":
        return hnn.PairformerBlock(with_single=case["single"])
    if kind == "template_block":
        return hnn.PairformerBlock(c_pair=64, num_intermediate_factor=2, with_single=False)
    if kind == "triangle_mult":
        return hnn.TriangleMultiplication(c_pair=128, _outgoing=case["outgoing"])
    if kind == "triangle_attention":
        return hnn.GridSelfAttention(c_pair=128, num_head=4, transpose=case["transpose"])
    if kind == "evoformer":
        return hnn.EvoformerBlock()
    if kind == "diffusion":
        return hnn.DiffusionTransformer()
    if kind == "diffusion_transition":
        return hnn.DiffusionTransition(768, 384, use_single_cond=True)
    return hnn.CrossAttention()


def _weights_(module, g):
    """Linear weights N(0, 1/fan_in), LayerNorms near the identity, biases small."""
    for name, p in module.named_parameters():
        r = torch.randn(p.shape, device=DEVICE, generator=g)
        if p.dim() == 2:
            r /= math.sqrt(p.shape[1])
        elif p.dim() == 3:
            r /= math.sqrt(p.shape[0] * p.shape[1])
        elif name.endswith("weight"):
            r = 1 + 0.1 * r
        else:
            r *= 0.1
        p.data.copy_(r)


def _dtype(case):
    return torch.float32 if case.get("dtype") == "fp32" else torch.bfloat16


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    with torch.device("meta"):
        module = _module(case)
    module = module.to_empty(device=DEVICE).eval().requires_grad_(False)
    _weights_(module, g)
    dtype, kind = _dtype(case), case["kind"]
    randn = lambda *s: torch.randn(s, device=DEVICE, generator=g)  # noqa: E731
    state = {"case": case, "module": module}

    def token_mask(n):
        m = torch.ones(n, device=DEVICE)
        m[n - case.get("pad", 0):] = 0
        return m

    if kind in ("pair_block", "template_block", "triangle_mult", "triangle_attention"):
        n, c = case["n"], 64 if kind == "template_block" else 128
        seq = token_mask(n)
        state.update(pair=randn(n, n, c).to(dtype), pair_mask=seq[:, None] * seq[None, :], seq_mask=seq)
        if case.get("single"):
            state["single"] = randn(n, 384).to(dtype)
    elif kind == "evoformer":
        n, rows = case["n"], case["rows"]
        seq = token_mask(n)
        gaps = (torch.rand(rows, n, device=DEVICE, generator=g) > 0.1).float() * seq
        gaps[0] = seq                                    # the query sequence covers every token
        state.update(msa=randn(rows, n, 64).to(dtype), msa_mask=gaps, pair=randn(n, n, 128).to(dtype),
                     pair_mask=seq[:, None] * seq[None, :])
    elif kind == "diffusion":
        n = case["n"]
        state.update(act=randn(case["samples"], n, 768).to(dtype), mask=token_mask(n),
                     single_cond=randn(n, 384).to(dtype), pair_cond=randn(n, n, 128).to(dtype))
    elif kind == "diffusion_transition":
        state.update(act=randn(case["samples"], case["n"], 768).to(dtype),
                     single_cond=randn(case["n"], 384).to(dtype))
    else:
        s = case["subsets"]
        logits = randn(s, 32, 128, 12).to(dtype)[..., 4:8].permute(0, 3, 1, 2)
        state.update(x_q=randn(s, 32, 128).to(dtype), x_k=randn(s, 128, 128).to(dtype),
                     mask_q=(torch.rand(s, 32, device=DEVICE, generator=g) > 0.1).float(),
                     mask_k=(torch.rand(s, 128, device=DEVICE, generator=g) > 0.1).float(),
                     pair_logits=logits if case["view"] else logits.contiguous(),
                     cond_q=randn(s, 32, 128).to(dtype), cond_k=randn(s, 128, 128).to(dtype))
    return state


def run(state):
    case, module, kind = state["case"], state["module"], state["case"]["kind"]
    with torch.inference_mode(), torch.autocast("cuda", dtype=torch.bfloat16, enabled=_dtype(case) != torch.float32):
        if kind == "pair_block" and case["single"]:
            return module(state["pair"], state["pair_mask"], state["single"], state["seq_mask"])
        if kind in ("pair_block", "template_block", "triangle_mult", "triangle_attention"):
            return module(state["pair"], state["pair_mask"])
        if kind == "evoformer":
            return module(state["msa"], state["pair"], state["msa_mask"], state["pair_mask"])
        if kind == "diffusion":
            return module(state["act"], state["mask"], state["single_cond"], state["pair_cond"])
        if kind == "diffusion_transition":
            return module(state["act"], state["single_cond"])
        return module(state["x_q"], state["x_k"], state["mask_q"], state["mask_k"], state["pair_logits"],
                      state["cond_q"], state["cond_k"])


# --------------------------------------------------------------------------- bytes and operations

def _pair_ops(n, c, f):
    """Matrix-product flops of the five pair updates at c channels and f transition features."""
    p = n * n
    triangle_mult = 2 * p * c * (2 * c + 2 * c + c + c) + 2 * c * n ** 3
    attention = 2 * p * c * (5 * c + 4) + 4 * c * n ** 3
    transition = 2 * p * c * 3 * f
    return triangle_mult, attention, transition


def work(case):
    kind, eb = case["kind"], 4 if case.get("dtype") == "fp32" else 2
    n = case.get("n", 0)
    if kind in ("pair_block", "template_block"):
        c, f = (64, 128) if kind == "template_block" else (128, 512)
        t, a, tr = _pair_ops(n, c, f)
        flops, bytes_ = 2 * t + 2 * a + tr, 2 * n * n * c * eb + 4 * n * n + (24 * c * c + 3 * c * f) * 4
        if case.get("single"):
            flops += 2 * n * n * 128 * 16 + 2 * n * 384 * (5 * 384 + 3 * 1536) + 4 * n * n * 384
            bytes_ += 2 * n * 384 * eb + (5 * 384 * 384 + 3 * 384 * 1536) * 4
        return {"bytes": bytes_, "flops": flops}
    if kind in ("triangle_mult", "triangle_attention"):
        t, a, _ = _pair_ops(n, 128, 512)
        return {"bytes": 2 * n * n * 128 * eb + 4 * n * n + 6 * 128 * 128 * 4, "flops": t if kind == "triangle_mult" else a}
    if kind == "evoformer":
        rows = case["rows"]
        t, a, tr = _pair_ops(n, 128, 512)
        opm = 2 * rows * n * 64 * 64 + 2 * n * n * 1024 * rows + 2 * n * n * 1024 * 128
        msa = 2 * n * n * 128 * 8 + 2 * rows * n * 64 * 192 + 2 * rows * n * n * 64 + 2 * rows * n * 64 * 3 * 256
        return {"bytes": 2 * rows * n * 64 * eb + 4 * rows * n + 2 * n * n * 128 * eb + 4 * n * n + 4 * 800_000,
                "flops": 2 * t + 2 * a + tr + opm + msa}
    if kind in ("diffusion", "diffusion_transition"):
        m = case["samples"] * n
        one = 2 * m * 768 * 3 * 1536
        cond = 2 * n * 384 * 768 * 3
        if kind == "diffusion_transition":
            return {"bytes": 2 * m * 768 * eb + n * 384 * eb + (3 * 768 * 1536 + 3 * 384 * 768) * 4, "flops": one + cond}
        attention = 2 * m * 768 * 5 * 768 + 4 * m * n * 768
        weights = 24 * (5 * 768 * 768 + 3 * 768 * 1536 + 6 * 384 * 768) * 4
        return {"bytes": 2 * m * 768 * eb + n * 384 * eb + n * n * 128 * eb + weights,
                "flops": 24 * (one + attention + 2 * cond) + 2 * n * n * 128 * 384}
    s = case["subsets"]
    return {"bytes": s * ((3 * 32 + 2 * 128) * 128 + 4 * 32 * 128) * eb + s * 160 * 4 + 12 * 128 * 128 * 4,
            "flops": s * (2 * 32 * 128 * 128 * 6 + 2 * 128 * 128 * 128 * 4 + 4 * 32 * 128 * 128)}


def tolerance(case):
    """About four times the distance from ``exact``: single layers and blocks in bf16 are 5e-3 to
    6.3e-3 off it, the 24-block transformer 1.2e-2, the fp32 block 4e-7 (sums of up to 512 terms)."""
    if case.get("dtype") == "fp32":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 3e-2, "max": 0.5} if case["kind"] == "diffusion" else {"rel": 2.5e-2, "max": 0.25}


# ------------------------------------------------------------------------------- 64-bit reference

def _ln(x, m, prefix, eps=1e-5):
    x = x - x.mean(-1, keepdim=True)
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    w, b = m.get(prefix + ".weight"), m.get(prefix + ".bias")
    x = x if w is None else x * w
    return x if b is None else x + b


def _lin(x, m, name):
    y = x @ m[name + ".weight"].T
    return y + m[name + ".bias"] if name + ".bias" in m else y


def _silu(x):
    return x * torch.sigmoid(x)


def _sub(m, name):
    return {k[len(name) + 1:]: v for k, v in m.items() if k.startswith(name + ".")}


def _x_triangle_mult(m, pair, mask, outgoing):
    z = _ln(pair, m, "left_norm_input")
    p = _lin(z, m, "projection") * mask[..., None] * torch.sigmoid(_lin(z, m, "gate"))
    a, b = p[..., 0::2].permute(2, 0, 1).contiguous(), p[..., 1::2].permute(2, 0, 1).contiguous()
    del p
    if outgoing:
        x = torch.bmm(a, b.transpose(1, 2).contiguous())
    else:                                        # x[c, i, j] = sum_k b[c, k, i] a[c, k, j]
        x = torch.bmm(b.transpose(1, 2).contiguous(), a)
    del a, b
    x = _ln(x.permute(1, 2, 0).contiguous(), m, "center_norm")
    return _lin(x, m, "output_projection") * torch.sigmoid(_lin(z, m, "gating_linear"))


def _attend(q, k, v, bias, fill, value=-1e9):
    """[B, H, T, D] attention; bias broadcast to the logits, which are ``value`` where ``fill`` is set."""
    s = torch.matmul(q * q.shape[-1] ** -0.5, k.transpose(-1, -2).contiguous()) + bias
    s = s.masked_fill(fill, value)
    return torch.matmul(torch.softmax(s, -1), v)


def _heads(x, h):
    return x.unflatten(-1, (h, x.shape[-1] // h)).transpose(-2, -3).contiguous()


def _x_triangle_attention(m, pair, mask, transpose, h=4):
    z = _ln(pair, m, "act_norm")
    bias = _lin(z, m, "pair_bias_projection").permute(2, 0, 1).contiguous()
    z = z.transpose(0, 1).contiguous() if transpose else z
    out, n = torch.empty_like(z), z.shape[0]
    step = max(1, 200_000_000 // (h * n * n))
    for i in range(0, n, step):
        x = z[i:i + step]
        o = _attend(*(_heads(_lin(x, m, w + "_projection"), h) for w in "qkv"), bias,
                    (mask[i:i + step] == 0)[:, None, None, :])
        out[i:i + step] = _lin(o.transpose(1, 2).flatten(-2) * torch.sigmoid(_lin(x, m, "gating_query")), m,
                               "output_projection")
    return out.transpose(0, 1) if transpose else out


def _x_transition(m, x):
    a, b = _lin(_ln(x, m, "input_layer_norm"), m, "transition1").chunk(2, -1)
    return _lin(_silu(a) * b, m, "transition2")


def _x_pair_updates(m, pair, mask):
    pair = pair + _x_triangle_mult(_sub(m, "triangle_multiplication_outgoing"), pair, mask, True)
    pair = pair + _x_triangle_mult(_sub(m, "triangle_multiplication_incoming"), pair, mask, False)
    pair = pair + _x_triangle_attention(_sub(m, "pair_attention1"), pair, mask, False)
    pair = pair + _x_triangle_attention(_sub(m, "pair_attention2"), pair, mask, True)
    tr = _sub(m, "pair_transition")
    for i in range(0, pair.shape[0], 64):                # rows are independent; bounds the hidden features
        pair[i:i + 64] += _x_transition(tr, pair[i:i + 64])
    return pair


def _x_adaptive_ln(m, x, cond):
    if cond is None:
        return _ln(x, m, "layer_norm")
    c = _ln(cond, m, "single_cond_layer_norm")
    return torch.sigmoid(_lin(c, m, "single_cond_scale")) * _ln(x, m, "layer_norm") + _lin(c, m, "single_cond_bias")


def _x_zero(m, x, cond):
    y = _lin(x, m, "transition2")
    return y if cond is None else torch.sigmoid(_lin(cond, m, "adaptive_zero_cond")) * y


def _x_self_attention(m, x, mask, logits, cond, h=16):
    a = _x_adaptive_ln(_sub(m, "adaptive_layernorm"), x, cond)
    q, k, v = (_heads(_lin(a, m, w + "_projection"), h) for w in "qkv")
    o = _attend(q, k, v, logits, mask == 0)
    o = o.transpose(1, 2).flatten(-2) * torch.sigmoid(_lin(a, m, "gating_query"))
    return _x_zero(_sub(m, "adaptive_zero_init"), o, cond)


def _x_diffusion_transition(m, x, cond):
    a, b = _lin(_x_adaptive_ln(_sub(m, "adaptive_layernorm"), x, cond), m, "transition1").chunk(2, -1)
    return _x_zero(_sub(m, "adaptive_zero_init"), _silu(a) * b, cond)


def _x_outer_product_mean(m, msa, mask):
    z = _ln(msa, m, "layer_norm_input")
    left, right = (_lin(z, m, w) * mask[..., None] for w in ("left_projection", "right_projection"))
    (s, n, c), f = left.shape, m["output_w"].shape[-1]
    out, r = torch.empty(n, n, f, dtype=z.dtype, device=z.device), right.reshape(s, n * c)
    for i in range(0, n, 32):
        o = left[:, i:i + 32].reshape(s, -1).T.contiguous() @ r
        o = o.view(-1, c, n, c).permute(0, 2, 1, 3).reshape(-1, n, c * c)
        out[i:i + 32] = o @ m["output_w"].reshape(c * c, f) + m["output_b"]
    return out / (1e-3 + mask.T @ mask)[..., None]


def _x_msa_attention(m, msa, mask, pair, h=8):
    z = _ln(msa, m, "act_norm")
    w = _lin(_ln(pair, m, "pair_norm"), m, "pair_logits").permute(2, 0, 1) + 1e9 * (mask.max(0).values - 1)
    w = torch.softmax(w, -1)
    v = _heads(_lin(z, m, "v_projection"), h)                                  # [S, H, K, D]
    (s, _, n, d) = v.shape
    avg = torch.matmul(w, v.permute(1, 2, 0, 3).reshape(h, n, s * d).contiguous())
    avg = avg.view(h, n, s, d).permute(2, 1, 0, 3).reshape(s, n, h * d)
    return _lin(avg * torch.sigmoid(_lin(z, m, "gating_query")), m, "output_projection")


def _x_cross_attention(m, st, h=4):
    xq = _x_adaptive_ln(_sub(m, "q_adaptive_layernorm"), st["x_q"], st["cond_q"])
    xk = _x_adaptive_ln(_sub(m, "k_adaptive_layernorm"), st["x_k"], st["cond_k"])
    q, k, v = (_heads(_lin(x, m, w + "_projection"), h) for x, w in ((xq, "q"), (xk, "k"), (xk, "v")))
    both = (st["mask_q"] == 0)[:, None, :, None] & (st["mask_k"] == 0)[:, None, None, :]
    # The module adds 1e9 to these logits in 32 bits, where a step is 64: nothing else is left of them.
    o = _attend(q, k, v, st["pair_logits"], both, 1e9)
    o = o.transpose(1, 2).flatten(-2) * torch.sigmoid(_lin(xq, m, "gating_query"))
    return _x_zero(_sub(m, "adaptive_zero_init"), o, st["cond_q"])


def exact(case, seed):
    st, kind = prepare(case, seed), case["kind"]
    m = {k: v.double() for k, v in st["module"].state_dict().items()}
    st = {k: v.double() for k, v in st.items() if isinstance(v, torch.Tensor)}
    if kind in ("pair_block", "template_block"):
        pair = _x_pair_updates(m, st["pair"], st["pair_mask"])
        if not case.get("single"):
            return pair
        logits = _lin(_ln(pair, m, "single_pair_logits_norm"), m, "single_pair_logits_projection").permute(2, 0, 1)
        single = st["single"]
        single = single + _x_self_attention(_sub(m, "single_attention_"), single[None], st["seq_mask"], logits, None)[0]
        return pair, single + _x_transition(_sub(m, "single_transition"), single)
    if kind == "triangle_mult":
        return _x_triangle_mult(m, st["pair"], st["pair_mask"], case["outgoing"])
    if kind == "triangle_attention":
        return _x_triangle_attention(m, st["pair"], st["pair_mask"], case["transpose"])
    if kind == "evoformer":
        msa, pair, mask = st["msa"], st["pair"], st["msa_mask"]
        pair = pair + _x_outer_product_mean(_sub(m, "outer_product_mean"), msa, mask)
        msa = msa + _x_msa_attention(_sub(m, "msa_attention1"), msa, mask, pair)
        msa = msa + _x_transition(_sub(m, "msa_transition"), msa)
        return msa, _x_pair_updates(m, pair, st["pair_mask"])
    if kind == "diffusion":
        act, pair = st["act"], _ln(st["pair_cond"], m, "pair_input_layer_norm")
        for b in range(24):
            logits = (pair @ m[f"pair_logits_projection.{b // 4}.weight"][b % 4 * 16:b % 4 * 16 + 16].T).permute(2, 0, 1)
            act = act + _x_self_attention(_sub(m, f"self_attention.{b}"), act, st["mask"], logits, st["single_cond"])
            act = act + _x_diffusion_transition(_sub(m, f"transition_block.{b}"), act, st["single_cond"])
        return act
    if kind == "diffusion_transition":
        return _x_diffusion_transition(m, st["act"], st["single_cond"])
    return _x_cross_attention(m, st)
