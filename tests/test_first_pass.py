"""What a module prepares of its weights, and when (CPU, the library's calls stubbed): everything on
its first pass, so that a second pass may be a graph capture, and nothing that is made while a
stream is captured outlives the call."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from xfold_cpu_amd import nn as hnn
from xfold_cpu_amd.fastnn import native_hip as nh
from xfold_cpu_amd.nn.cache import InputCache, input_cache_scope


class Library:
    def __getattr__(self, name):
        return {"xfh_glu_packed_rows": lambda f: 2 * f, "xfh_attention_max_keys": lambda: 4096}.get(name, lambda *a: 256)


def stub_call(name, *args):
    if name == "xfh_attention_operands_size":
        B, T, H, Dh, sizes = args
        dp, tpad = 32 if Dh <= 32 else 64, (T + 63) // 64 * 64
        sizes[:] = [dp, tpad, B * H * T * dp, B * H * tpad * dp, B * H * dp * tpad]


@pytest.fixture
def stubbed(monkeypatch):
    library = Library()
    monkeypatch.setattr(nh, "load_library", lambda path=None: library)
    monkeypatch.setattr(nh, "attention_max_keys", lambda: 4096)
    monkeypatch.setattr(nh, "call", stub_call)
    monkeypatch.setattr(nh, "ptr", lambda t: None if t is None else t.data_ptr())
    monkeypatch.setattr(nh, "stream_of", lambda device: 0)
    monkeypatch.setattr(nh, "check_gpu_inference", lambda *tensors: None)
    monkeypatch.setattr(torch, "is_autocast_enabled", lambda device="cuda": True)
    monkeypatch.setattr(torch, "get_autocast_dtype", lambda device="cuda": torch.bfloat16)


def bf16(*shape):
    return torch.randn(shape).bfloat16()


MODULES = {
    "diffusion_transition": (lambda: hnn.DiffusionTransition(64, 32, use_single_cond=True),
                             lambda: (bf16(5, 64), bf16(5, 32))),
    "self_attention": (lambda: hnn.SelfAttention(c_x=64, num_head=2, c_single_cond=32, use_single_cond=True),
                       lambda: (bf16(5, 64), torch.ones(5), bf16(2, 5, 5), bf16(5, 32))),
    "cross_attention": (lambda: hnn.CrossAttention(key_dim=64, value_dim=64, c_single_cond=64, num_head=2),
                        lambda: (bf16(3, 4, 64), bf16(3, 6, 64), torch.ones(3, 4), torch.ones(3, 6), bf16(3, 2, 4, 6),
                                 bf16(3, 4, 64), bf16(3, 6, 64))),
    "cross_attention_fused": (hnn.CrossAttention,
                              lambda: (bf16(3, 4, 128), bf16(3, 6, 128), torch.ones(3, 4), torch.ones(3, 6),
                                       bf16(3, 4, 4, 6), bf16(3, 4, 128), bf16(3, 6, 128))),
    "pairformer": (lambda: hnn.PairformerBlock(c_single=64), lambda: (bf16(5, 5, 128), torch.ones(5, 5), bf16(5, 64),
                                                                     torch.ones(5))),
    "evoformer": (hnn.EvoformerBlock, lambda: (bf16(3, 5, 64), bf16(5, 5, 128), torch.ones(3, 5), torch.ones(5, 5))),
    "diffusion_transformer": (lambda: hnn.DiffusionTransformer(c_act=64, c_single_cond=32, num_head=16, num_blocks=4,
                                                               super_block_size=2),
                              lambda: (bf16(2, 5, 64), torch.ones(5), bf16(5, 32), bf16(5, 5, 128))),
}


class Computed(TorchDispatchMode):
    """The operators that write new memory."""

    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if not func.is_view and "empty" not in func.name():
            self.names.append(func.name())
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("kind", MODULES)
def test_the_first_pass_prepares_every_weight(stubbed, kind):
    make, inputs = MODULES[kind]
    module, args, passes = make().eval(), inputs(), []
    with torch.inference_mode(False), torch.no_grad():
        for _ in range(3):
            with Computed() as computed:
                module(*args)
            passes.append(computed.names)
    assert passes[0] and passes[1] == passes[2]


def test_an_operators_weights_are_copied_together(stubbed):
    """The four plain weights of a triangle multiplication and the six of a grid attention, in one call and
    one allocation each: a block's first pass is bound by this host work."""
    make, inputs = MODULES["pairformer"]
    module, args = make().eval(), inputs()
    with torch.no_grad(), Computed() as computed:
        module(*args)
    assert computed.names.count("aten::_foreach_copy_") == 4
    # What is left: both transitions' two, the pair logits' one, the attention's four and output.
    assert computed.names.count("aten::_to_copy") == 10
    make, inputs = MODULES["diffusion_transition"]
    transition, args = make().eval(), inputs()
    with torch.no_grad(), Computed() as computed:
        transition(*args)
    # scale, shift, the condition and transition2 in one call; transition1 is packed.
    assert computed.names.count("aten::_foreach_copy_") == 1 and computed.names.count("aten::_to_copy") == 1
    weights = nh.linear_weights(module.pair_attention1, ("q_projection", "pair_bias_projection", "k_projection"), torch.bfloat16)
    for name, w in zip(("q_projection", "pair_bias_projection", "k_projection"), weights):
        assert torch.equal(w, getattr(module.pair_attention1, name).weight.detach().bfloat16()) and w.is_contiguous()
        assert (w.data_ptr() - weights[0].data_ptr()) % 256 == 0


def test_the_fused_cross_attention_prepares_its_own_weights_only(stubbed):
    """No stacked k and v for the general path beside the fused kernels' separate ones."""
    make, inputs = MODULES["cross_attention_fused"]
    module, args = make().eval(), inputs()
    with torch.no_grad():
        module(*args)
        module(*args)
    assert set(module.__dict__["_hip_weight_groups"]) == {"fused"}
    assert not [tag for tag in module.__dict__["_hip_weight_caches"] if tag.startswith("fused:")]


@pytest.mark.parametrize("kind", MODULES)
def test_nothing_made_in_a_capture_is_kept(stubbed, monkeypatch, kind):
    make, inputs = MODULES[kind]
    module, args = make().eval(), inputs()
    with torch.no_grad():
        monkeypatch.setattr(nh, "capturing", lambda: True)
        module(*args)
        module(*args)
        for m in module.modules():
            assert all(c._key is None for c in m.__dict__.get("_hip_weight_caches", {}).values())
            assert all(g.values is None for g in m.__dict__.get("_hip_weight_groups", {}).values())
        monkeypatch.setattr(nh, "capturing", lambda: False)
        module(*args)
        assert any(c._key is not None for m in module.modules() for c in m.__dict__.get("_hip_weight_caches", {}).values())


def test_a_memo_entry_is_not_made_in_a_capture(monkeypatch):
    from xfold_cpu_amd.fastnn import config
    from xfold_cpu_amd.nn import cache as cache_module
    monkeypatch.setattr(config, "input_cache_enabled", True)
    owner, cache, feature = torch.nn.Linear(3, 3).eval(), InputCache(), torch.randn(2, 3)
    with torch.no_grad(), input_cache_scope():
        monkeypatch.setattr(cache_module, "capturing", lambda: True)
        cache.get("x", (feature,), owner, lambda: owner(feature))
        assert not cache._entries
        monkeypatch.setattr(cache_module, "capturing", lambda: False)
        kept = cache.get("x", (feature,), owner, lambda: owner(feature))
        monkeypatch.setattr(cache_module, "capturing", lambda: True)
        assert cache.get("x", (feature,), owner, lambda: owner(feature)) is kept


def test_each_capture_has_attention_operands_of_its_own(stubbed, monkeypatch):
    """The buffers' zero fill and mask words are recorded in the graph that makes them."""
    from xfold_cpu_amd.fastnn import ops
    monkeypatch.setattr(ops, "_SHARED_OPERANDS", type(ops._SHARED_OPERANDS)())
    capture = 0
    monkeypatch.setattr(nh, "capture_id", lambda device: capture, raising=False)
    get = lambda T=40: ops.shared_attention_operands(1, T, 4, 32, torch.device("cpu"))  # noqa: E731
    eager = get()
    capture = 7
    first = get()
    assert first is not eager and get() is first and get(50) is not first
    capture = 8
    second = get()
    assert second is not first and second is not eager and get() is second
    capture = 0
    assert get() is eager
    assert [k[-1] for k in ops._SHARED_OPERANDS] == [0]      # the captures' sets are given back


def test_a_single_weight_is_checked_once(stubbed, monkeypatch):
    """A conditioned transition's later passes take each weight's key once, without a group around it."""
    make, inputs = MODULES["diffusion_transition"]
    module, args = make().eval(), inputs()
    seen, stamp = [], nh.stamp
    monkeypatch.setattr(nh, "stamp", lambda t: seen.append(t) or stamp(t))
    with torch.no_grad():
        for _ in range(2):
            del seen[:]
            module(*args)
            assert len(seen) == len({id(t) for t in seen}) == 6     # (three Linears, scale, shift and its bias)
    assert not any("_hip_weight_groups" in m.__dict__ for m in module.modules())


def test_weights_that_cannot_be_kept_are_not_stacked(stubbed, monkeypatch):
    """Inference tensors carry no version: their copies are made on every call, where scale and shift take two
    products of plain copies rather than one of a stack."""
    make, inputs = MODULES["diffusion_transition"]
    made, prepare, calls = [], nh._prepare, []
    monkeypatch.setattr(nh, "_prepare", lambda *args: made.append(args) or prepare(*args))
    monkeypatch.setattr(nh, "call", lambda name, *args: calls.append(name))
    with torch.inference_mode():
        module, args = make().eval(), inputs()
        for _ in range(2):
            del made[:], calls[:]
            module(*args)
            assert len(made) == 5 and "xfh_linear_batched" not in calls
    for m in module.modules():
        assert all(c._key is None for c in m.__dict__.get("_hip_weight_caches", {}).values())


def test_weights_on_two_devices_are_refused():
    """One call copies several weights: a weight that lies elsewhere is not brought along."""
    from xfold_cpu_amd.nn.diffusion_transformer import _scale_shift_weights
    here, elsewhere = torch.randn(8, 8), torch.empty(8, 8, device="meta")
    with pytest.raises(ValueError, match="one device"):
        nh._copies((here, elsewhere), torch.bfloat16)
    for weights in ((here, elsewhere), (here, here, None, (elsewhere,))):
        with pytest.raises(ValueError, match="one device"):
            _scale_shift_weights(torch.bfloat16, *weights)
