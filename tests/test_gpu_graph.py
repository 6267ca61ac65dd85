"""HIP-graph capture of the HIP modules (torch.cuda.CUDAGraph): a bf16 PairformerBlock
(xfold/nn/pairformer.py:77-114) and a DiffusionTransformer forward
(xfold/nn/diffusion_transformer.py:250-272) are captured once and replayed several times, with
eager work and synchronisations between the replays; every replay must equal the eager
result bit for bit (the kernels are deterministic and the path records no memset, host copy
or synchronisation). The replayed Pairformer block is also held to the fp32 CPU oracle
(oracle/restatement.py) and its bf16 floor, the bar of the eager tests."""

import pytest
import torch

from tests.helpers import assert_parity_bf16, floor_of, residual
from tests.test_gpu_ops import announce, autocast, pair_of
from xfold_cpu_amd.synthetic import pair_block_inputs

pytestmark = pytest.mark.gpu


def capture(fn):
    """Warm up on a side stream (weight caches are built outside the capture), then capture."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    return graph


def replay_and_check(graph, reset, outputs, wants, replays=3, check=None):
    """Replays `graph` after `reset()`; every replay's outputs must equal `wants` bit for bit
    and pass `check(outputs)` when one is given."""
    for rep in range(replays):
        reset()
        graph.replay()
        torch.cuda.synchronize()
        # Eager work on the same stream between replays.
        scratch = torch.randn(1 << 16, device=outputs[0].device).sum()
        torch.cuda.synchronize()
        assert torch.isfinite(scratch)
        for got, want in zip(outputs, wants):
            assert torch.equal(got, want), f"replay {rep} differs from the eager result"
        if check is not None:
            check(outputs)


@pytest.mark.parametrize("n", [48, 100])
def test_pairformer_block_graph_replay(device, n):
    announce("graph pairformer_block", n)
    args = dict(n_heads=16, c_pair=128, c_single=384, n_heads_pair=4)
    ref, hip = pair_of("PairformerBlock", args, seed=n, device=device)
    inp = pair_block_inputs(n, pad=3, seed=n)
    pair0, single0 = inp.pair.bfloat16().to(device), inp.single.bfloat16().to(device)
    pm, sm = inp.pair_mask.to(device), inp.seq_mask.to(device)
    pair, single = pair0.clone(), single0.clone()

    def oracle(wrap=lambda t: t):
        return ref(wrap(inp.pair.bfloat16().float()), inp.pair_mask, wrap(inp.single.bfloat16().float()),
                   inp.seq_mask)
    with torch.inference_mode():
        want_pair_ref, want_single_ref = oracle()
    floor_pair, floor_single = floor_of(lambda: oracle(residual))

    def against_oracle(outputs):
        got_pair, got_single = outputs
        assert_parity_bf16(got_pair, want_pair_ref, f"graph replay PairformerBlock N={n} pair", floor=floor_pair)
        assert_parity_bf16(got_single, want_single_ref, f"graph replay PairformerBlock N={n} single",
                           floor=floor_single)

    def reset():
        pair.copy_(pair0)
        single.copy_(single0)

    def block():
        hip(pair, pm, single, sm)

    with torch.inference_mode(), autocast(True):
        block()                                    # eager result
        torch.cuda.synchronize()
        want_pair, want_single = pair.clone(), single.clone()
        reset()
        graph = capture(block)
        replay_and_check(graph, reset, (pair, single), (want_pair, want_single), check=against_oracle)


def test_diffusion_transformer_graph_replay(device):
    announce("graph diffusion_transformer")
    args = dict(c_act=256, c_single_cond=64, c_pair_cond=128, num_head=16, num_blocks=4, super_block_size=2)
    _, hip = pair_of("DiffusionTransformer", args, seed=5, device=device)
    torch.manual_seed(5)
    n, samples = 40, 3
    act0 = torch.randn(samples, n, 256).bfloat16().to(device)
    mask = torch.ones(n)
    mask[-3:] = 0
    mask = mask.to(device)
    scond, pcond = torch.randn(n, 64).to(device), torch.randn(n, n, 128).to(device)
    act = act0.clone()
    out = {}

    def reset():
        act.copy_(act0)

    def forward():
        out["act"] = hip(act, mask, scond, pcond)

    with torch.inference_mode(), autocast(True):
        forward()
        torch.cuda.synchronize()
        want = out["act"].clone()
        reset()
        graph = capture(forward)
        replay_and_check(graph, reset, (out["act"],), (want,))


def linear_inputs(kind, n, device):
    """A module's inputs at n tokens, one of them updated in place or none."""
    g = torch.Generator().manual_seed(n)
    randn = lambda *s: torch.randn(s, generator=g).to(device)  # noqa: E731
    if kind == "DiffusionTransition":
        return randn(2, n, 256), randn(n, 64)
    if kind == "SelfAttention":
        return randn(2, n, 256), torch.ones(n, device=device), randn(16, n, n), randn(n, 64)
    return (randn(3, n, 128), randn(3, 2 * n, 128), torch.ones(3, n, device=device), torch.ones(3, 2 * n, device=device),
            randn(3, 4, n, 2 * n), randn(3, n, 128), randn(3, 2 * n, 128))


@pytest.mark.parametrize("kind,args,bf16", [
    ("DiffusionTransition", dict(c_x=256, c_single_cond=64, use_single_cond=True), True),
    ("SelfAttention", dict(c_x=256, num_head=16, c_single_cond=64, use_single_cond=True), True),
    ("CrossAttention", dict(), False), ("CrossAttention", dict(), True)])
def test_capture_after_one_eager_pass(device, kind, args, bf16):
    """One eager pass, then two captures of other lengths: the eager module before the first replay, and
    the second graph replayed before the first, equal the eager results of a module of its own."""
    announce("graph after one pass", kind, bf16)
    _, twin = pair_of(kind, args, seed=3, device=device)
    _, hip = pair_of(kind, args, seed=3, device=device)
    inputs = [linear_inputs(kind, n, device) for n in (33, 48, 20)]
    with torch.inference_mode(), autocast(bf16):
        wants = [twin(*i).clone() for i in inputs]
        hip(*inputs[0])
        torch.cuda.synchronize()
        graphs, outs = [], []
        for i in inputs[1:]:
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                outs.append(hip(*i))
            graphs.append(graph)
        assert torch.equal(hip(*inputs[0]), wants[0])
        for _ in range(3):
            for k in (1, 0):
                outs[k].zero_()
                graphs[k].replay()
                torch.cuda.synchronize()
                assert torch.equal(outs[k], wants[1 + k])
                assert torch.equal(hip(*inputs[0]), wants[0])


def test_graphs_of_one_shape_share_no_buffers(device):
    """Two captures of one shape and mask: the second is replayed before the first, then eager calls with
    another mask run between the replays on the captures' own stream."""
    announce("graphs of one shape")
    args = dict(c_act=256, c_single_cond=64, c_pair_cond=128, num_head=16, num_blocks=4, super_block_size=2)
    _, hip = pair_of("DiffusionTransformer", args, seed=6, device=device)
    torch.manual_seed(6)
    n = 40
    acts = [torch.randn(2, n, 256).to(device) for _ in range(2)]
    masks = [torch.ones(n, device=device), (torch.arange(n, device=device) % 3 > 0).float()]
    scond, pcond = torch.randn(n, 64).to(device), torch.randn(n, n, 128).to(device)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.inference_mode(), autocast(True), torch.cuda.stream(stream):
        run = lambda act, mask: hip(act.clone(), mask, scond, pcond)  # noqa: E731
        run(acts[0], masks[0])
        wants = [[run(a, m) for m in masks] for a in acts]
        torch.cuda.synchronize()
        graphs, outs = [], []
        for act in acts:
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                outs.append(run(act, masks[0]))
            graphs.append(graph)
        for _ in range(3):
            for k in (1, 0):
                outs[k].zero_()
                graphs[k].replay()
                torch.cuda.synchronize()
                assert torch.equal(outs[k], wants[k][0])
                assert torch.equal(run(acts[k], masks[1]), wants[k][1])
