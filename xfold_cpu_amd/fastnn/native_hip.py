"""ctypes bridge to libxfold_hip.so (the MI355X backend), mirroring the reference's
native bridge ``xfold/fastnn/native.py:1-70``:

* :func:`load_library`    ~ ``load_native_operator`` (``native.py:7-18``): loads once,
                            checks the ABI version and every exported symbol, and fails
                            loudly (RuntimeError) when the library is missing. There is no
                            fallback to another implementation.
* :func:`check_gpu_inference` ~ ``check_cpu_inference`` (``native.py:21-28``) for ROCm
                            tensors (``device.type == 'cuda'`` under PyTorch-ROCm).
* :func:`compute_dtype`   ~ ``compute_dtype`` (``native.py:31-43``) with the CUDA/HIP
                            autocast state instead of the CPU one.
* :class:`HipWeightCache` ~ ``GLUWeightCache`` (``xfold/fastnn/gated_linear_unit.py:6-48``):
                            one device copy per weight version in the compute dtype, and
                            the packed GLU layout.

Torch is used here only for device memory, streams and dtype bookkeeping; all arithmetic
runs in the library's HIP kernels.
"""

from __future__ import annotations

import ctypes
import functools
import os
from pathlib import Path
from typing import Optional

import torch

LIBRARY_PATH = Path(__file__).resolve().parent.parent / "lib" / "libxfold_hip.so"
ABI_VERSION = 11

F32, BF16, BOOL = 0, 1, 2
BIAS_PACKED = 3                 # bias 'dtype' of a packed fp32 block (times log2(e))
BIAS_PACKED_BF16 = 4            # bias 'dtype' of a packed bf16 block (natural units)
EPI_STORE, EPI_MUL_SIGMOID_AUX, EPI_SIGMOID_MUL_AUX, EPI_ACCUMULATE, EPI_MUL_SIGMOID_AUX_ACCUMULATE = range(5)

_p, _i, _i64, _f = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float
_pi64 = ctypes.POINTER(ctypes.c_int64)

# name -> (restype, argtypes); must match include/xfold_hip.h.
SIGNATURES = {
    "xfh_abi_version": (_i, []),
    "xfh_runtime_info": (ctypes.c_char_p, []),
    "xfh_last_error": (ctypes.c_char_p, []),
    "xfh_set_kernel_timing": (None, [_i]),
    "xfh_kernel_timing_read": (_i, [ctypes.c_char_p, ctypes.POINTER(ctypes.c_double), _pi64]),
    "xfh_kernel_timing_read_work": (_i, [ctypes.c_char_p, ctypes.POINTER(ctypes.c_double), _pi64,
                                         ctypes.POINTER(ctypes.c_double)]),
    "xfh_layer_norm": (_i, [_p, _i, _i64, _i64, _p, _p, _f, _p, _i, _p]),
    "xfh_adaptive_layer_norm": (_i, [_p, _i, _i64, _i64, _p, _p, _i, _i64, _f, _p, _i, _p]),
    "xfh_linear": (_i, [_p, _i64, _p, _p, _i64, _i64, _i64, _i, _p, _i64, _i, _i, _p, _i64, _i64, _p]),
    "xfh_linear_batched": (_i, [_p, _i64, _i64, _p, _i64, _p, _i64, _i64, _i64, _i64, _i64, _i, _p, _i64, _i64, _i, _p]),
    "xfh_glu_packed_rows": (_i64, [_i64]),
    "xfh_glu_pack_weight": (_i, [_p, _i64, _i64, _i, _p, _p]),
    "xfh_gated_linear_unit": (_i, [_p, _p, _i64, _i64, _i64, _i, _p, _i, _p]),
    "xfh_dot_product_attention_workspace_size": (_i64, [_pi64, _i]),
    "xfh_dot_product_attention": (_i, [_p, _p, _p, _i, _p, _i, _p, _i, _p, _i, _pi64, _pi64, _f, _p, _i64, _p]),
    "xfh_attention_max_keys": (_i64, []),
    "xfh_attention_bias_pack": (_i, [_p, _i, _pi64, _pi64, _p, _p]),
    "xfh_attention_operands_size": (_i, [_i64, _i64, _i64, _i64, _pi64]),
    "xfh_stream_capture_id": (_i, [_p, ctypes.POINTER(ctypes.c_uint64)]),
    "xfh_attention_project": (_i, [_p, _i64, _p, _p, _i64, _i64, _i64, _i64, _i64, _f, _p, _p, _p, _p, _p]),
    "xfh_attention_mask_words": (_i, [_p, _i, _i64, _i64, _i64, _p, _p]),
    "xfh_attention_operands": (_i, [_p, _p, _p, _p, _i, _p, _i, _p, _p, _i64, _i64, _i64, _i64, _p]),
    "xfh_pair_updates_workspace_size": (_i64, [_i64, _i64, _i64, _i64, _i]),
    "xfh_pair_updates": (_i, [_p, _i, _p, _i, _i64, _i64, _i64, _i64, _p, _p, _p, _p, _i, _p, _i64, _p]),
    "xfh_pairformer_single_workspace_size": (_i64, [_i64, _i64, _i64, _i64]),
    "xfh_pairformer_single": (_i, [_p, _p, _i, _i64, _i64, _i64, _i64, _p, _p, _f, _p, _p, _p, _p, _p, _p, _i64, _p]),
    "xfh_diffusion_blocks_workspace_size": (_i64, [_i64, _i64, _i64]),
    "xfh_diffusion_blocks": (_i, [_p, _i, _i64, _i64, _i64, _i64, _i64, _i64, _p, _i64, _i, _f, _p, _p, _p, _p, _p, _i,
                                  _p, _i64, _p]),
    "xfh_pair_attention_bias": (_i, [_p, _i, _i64, _i64, _p, _p, _f, _p, _i, _i64, _p, _i, _p]),
    "xfh_triangle_multiplication_workspace_size": (_i64, [_i64, _i64, _i]),
    "xfh_triangle_multiplication": (_i, [_p, _i, _p, _i, _i64, _i64, _i, _p, _p, _f, _p, _p, _p, _p,
                                         _f, _p, _p, _i, _p, _i, _i, _p, _i64, _p]),
    "xfh_triangle_multiplication_noalloc": (_i, [_p, _i, _p, _i, _i64, _i64, _i, _p, _p, _f, _p, _p, _p, _p,
                                                 _f, _p, _p, _i, _p, _i, _i, _p]),
    "xfh_grid_self_attention_workspace_size": (_i64, [_i64, _i64, _i64, _i]),
    "xfh_grid_self_attention": (_i, [_p, _i, _p, _i, _i64, _i64, _i64, _i, _p, _p, _f, _p, _p, _p,
                                     _p, _p, _p, _i, _p, _i, _i, _p, _i64, _p]),
    "xfh_transition_workspace_size": (_i64, [_i64, _i64, _i64, _i]),
    "xfh_transition": (_i, [_p, _i, _i64, _i64, _i64, _p, _p, _f, _p, _p, _i, _p, _i, _i, _p, _i64, _p]),
    "xfh_transition_pair_bias": (_i, [_p, _i64, _i64, _i64, _p, _p, _f, _p, _p, _p, _p, _f, _p, _i64, _p, _p]),
    "xfh_outer_product_mean_workspace_size": (_i64, [_i64, _i64, _i64, _i64, _i]),
    "xfh_outer_product_mean": (_i, [_p, _i, _p, _i, _i64, _i64, _i64, _i64, _i64, _p, _p, _f, _p, _p, _p, _f,
                                    _i, _p, _i, _i, _p, _i64, _p]),
    "xfh_msa_attention_workspace_size": (_i64, [_i64, _i64, _i64, _i64, _i64, _i]),
    "xfh_msa_attention": (_i, [_p, _i, _p, _i, _p, _i, _i64, _i64, _i64, _i64, _i64, _p, _p, _f, _p, _p, _f,
                               _p, _p, _p, _p, _i, _p, _i, _i, _p, _i64, _p]),
    "xfh_cross_attention_workspace_size": (_i64, [_i64, _i64, _i64]),
    "xfh_cross_attention": (_i, [_p, _p, _p, _p, _i, _p, _i, _p, _i, _p, _i, _pi64, _i64, _i64, _i64, _p, _p, _f, _p,
                                 _i, _i, _p, _i64, _p]),
    "xfh_cross_attention_bias": (_i, [_p, _i, _pi64, _p, _i, _p, _i, _i64, _i64, _i64, _i64, _p, _p]),
    "xfh_convert": (_i, [_p, _i, _p, _i, _i64, _p]),
}


class HipBackendError(RuntimeError):
    """A libxfold_hip call returned an error status."""


@functools.lru_cache(maxsize=None)
def load_library(path: Optional[str] = None) -> ctypes.CDLL:
    """Load libxfold_hip.so once; raise RuntimeError if it is absent or incomplete."""
    lib_path = Path(path or os.environ.get("XFOLD_HIP_LIBRARY", LIBRARY_PATH))
    if not lib_path.exists():
        raise RuntimeError(
            f"The 'hip' backend needs {lib_path}; build it with `python -m xfold_cpu_amd._build` "
            "(hipcc, gfx950) before selecting 'hip'.")
    lib = ctypes.CDLL(str(lib_path))
    missing = [name for name in SIGNATURES if not hasattr(lib, name)]
    if missing:
        raise RuntimeError(f"Rebuild libxfold_hip.so: missing symbols {missing}.")
    for name, (restype, argtypes) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = restype
        fn.argtypes = argtypes
    version = lib.xfh_abi_version()
    if version != ABI_VERSION:
        raise RuntimeError(f"libxfold_hip.so ABI {version} != expected {ABI_VERSION}; rebuild it.")
    return lib


class DiffusionBlock(ctypes.Structure):
    """``XfhDiffusionBlock`` of include/xfold_hip.h."""
    _fields_ = [(name, ctypes.c_void_p) for name in
                ("w_qkvg", "b_qkvg", "logits", "w_attention_out", "w_glu", "w_transition_out",
                 "attention_scale", "attention_shift", "attention_zero",
                 "transition_scale", "transition_shift", "transition_zero")] + [
               ("attention_eps", ctypes.c_float), ("transition_eps", ctypes.c_float)]


def call(name: str, *args) -> None:
    lib = load_library()
    status = getattr(lib, name)(*args)
    if status != 0:
        message = lib.xfh_last_error().decode()
        if status in (1, 2):
            raise ValueError(f"{name}: {message}")
        raise HipBackendError(f"{name} failed ({status}): {message}")


def set_kernel_timing(enable: bool) -> None:
    load_library().xfh_set_kernel_timing(int(enable))


def kernel_timing_read(name: str):
    """(total milliseconds, launches) recorded for ``name`` since the last read."""
    total, count = ctypes.c_double(), ctypes.c_int64()
    call("xfh_kernel_timing_read", name.encode(), ctypes.byref(total), ctypes.byref(count))
    return total.value, count.value


def kernel_timing_read_work(name: str):
    """(total milliseconds, launches, total declared FLOPs) recorded for ``name`` since the
    last read."""
    total, count, work = ctypes.c_double(), ctypes.c_int64(), ctypes.c_double()
    call("xfh_kernel_timing_read_work", name.encode(), ctypes.byref(total), ctypes.byref(count), ctypes.byref(work))
    return total.value, count.value, work.value


@functools.lru_cache(maxsize=None)
def attention_max_keys() -> int:
    """Largest key count of the pipelined attention kernel, hence of a packed bias."""
    return int(load_library().xfh_attention_max_keys())


def runtime_info() -> str:
    return load_library().xfh_runtime_info().decode()


# ------------------------------------------------------------------------- tensor helpers

_FLOATS = frozenset((torch.float32, torch.bfloat16))


def dtype_code(dtype: torch.dtype) -> int:
    if dtype == torch.float32:
        return F32
    if dtype == torch.bfloat16:
        return BF16
    if dtype in (torch.bool, torch.uint8):
        return BOOL
    raise ValueError(f"The 'hip' backend supports FP32/BF16 tensors (and bool masks), got {dtype}.")


def check_gpu_inference(*tensors) -> None:
    """Device, layout and inference-only guards (reference ``native.py:21-28``)."""
    for tensor in tensors:
        if tensor is None:
            continue
        if torch.is_grad_enabled() and tensor.requires_grad:
            raise RuntimeError("The 'hip' backend supports inference only; disable gradients.")
        if tensor.device.type != "cuda" or tensor.layout != torch.strided:
            raise ValueError("The 'hip' backend requires strided ROCm (cuda) tensors.")


def compute_dtype(x: torch.Tensor, *weights: torch.Tensor) -> torch.dtype:
    """Compute dtype per reference ``native.py:31-43``, reading the CUDA autocast state."""
    return _compute_dtype(x.dtype, [w.dtype for w in weights])


def _compute_dtype(x: torch.dtype, weights) -> torch.dtype:
    if x not in _FLOATS or not _FLOATS.issuperset(weights):
        raise ValueError("The 'hip' backend supports FP32/BF16 only.")
    if torch.is_autocast_enabled("cuda"):
        dtype = torch.get_autocast_dtype("cuda")
    else:
        dtype = x
        if any(w != dtype for w in weights):
            raise ValueError("Input/weight dtypes must match outside autocast.")
    if dtype not in _FLOATS:
        raise ValueError("The 'hip' backend supports FP32/BF16 autocast only.")
    return dtype


def check_module(module: torch.nn.Module) -> None:
    """Inference-only guard for a module's parameters (reference ``native.py:21-28``): a
    parameter that requires grad matters only in grad mode, so the walk over them happens
    only then; their device is checked where their pointers are taken (:func:`ptr`)."""
    if torch.is_grad_enabled():
        check_gpu_inference(*module.parameters())


def ptr(tensor: Optional[torch.Tensor]) -> Optional[int]:
    """Device address of a tensor handed to the library; a host tensor is refused here."""
    if tensor is None:
        return None
    if not tensor.is_cuda:
        raise ValueError("The 'hip' backend requires strided ROCm (cuda) tensors.")
    return tensor.data_ptr()


def ptrs(tensors) -> ctypes.Array:
    """A host struct of device pointers (the pointer-only structs of include/xfold_hip.h)."""
    return (ctypes.c_void_p * len(tensors))(*map(ptr, tensors))


def stream_of(device: torch.device) -> int:
    """The current stream of ``device`` as a raw hipStream_t."""
    index = device.index if device.index is not None else torch.cuda.current_device()
    return torch._C._cuda_getCurrentRawStream(index)


def capture_id(device: torch.device) -> int:
    """The id of the graph capture that the current stream records, 0 when it records none."""
    if not capturing():
        return 0
    value = ctypes.c_uint64()
    call("xfh_stream_capture_id", stream_of(device), ctypes.byref(value))
    return value.value


def workspace(nbytes: int, device: torch.device) -> torch.Tensor:
    """Caller-owned scratch memory (PyTorch caching allocator); the library allocates none."""
    if nbytes < 0:
        raise ValueError("invalid workspace request")
    return torch.empty(max(int(nbytes), 1), dtype=torch.uint8, device=device)


def mask_arg(mask: Optional[torch.Tensor], shape) -> tuple:
    """(tensor, dtype code) of a contiguous mask broadcast to ``shape`` (kept alive by caller)."""
    if mask is None:
        return None, BOOL
    if mask.dtype not in (torch.float32, torch.bfloat16, torch.bool, torch.uint8):
        raise ValueError("masks must be bool/uint8/float32/bfloat16")
    if tuple(mask.shape) != tuple(shape):
        mask = mask.expand(shape)
    return mask.contiguous(), dtype_code(mask.dtype)


def stamp(t: torch.Tensor) -> tuple:
    """What changes with a tensor's storage, contents or layout (``data`` swaps leave the version
    as it is). RuntimeError for an inference tensor, which carries no version counter."""
    return (t.data_ptr(), t._version, t.shape, t.stride(), t.dtype, t.device)


_expired = torch.UntypedStorage._expired
_is_inference = torch.Tensor.is_inference


class Storages:
    """Weak references to the storages of tensors, as each was when the object was made. An address
    means the same storage only while the old one is alive: after ``p.data = a; p.data = b`` the
    parameter object and its version are the old ones, and ``b`` may sit where the first storage was.
    (Weak, so that weights moved off the device free their memory.)"""

    __slots__ = ("_refs",)

    def __init__(self, tensors):
        self._refs = [t.untyped_storage()._weak_ref() for t in tensors if t is not None]

    def alive(self) -> bool:
        return not any(map(_expired, self._refs))

    def __del__(self, _free=torch.UntypedStorage._free_weak_ref):
        for ref in self._refs:
            _free(ref)


def capturing(_stream_capturing=torch._C._cuda_isCurrentStreamCapturing) -> bool:
    """Whether the current stream records a graph. What is prepared then lives in the graph's memory
    and is written by its replays only: it serves the capture and is not kept."""
    return torch.cuda.is_initialized() and _stream_capturing()


class _Kept:
    """One kept value and what it was made from, replaced as a whole (threads may share a module);
    a copied or pickled one starts empty."""

    _entry = (None, None, None)

    def __reduce__(self):
        return type(self), ()

    @property
    def _key(self):
        return self._entry[0]

    @property
    def _value(self):
        return self._entry[2]

    def clear(self):
        self._entry = _Kept._entry

    def lookup(self, key):
        kept, storages, value = self._entry
        return value if kept == key and storages.alive() else None

    def keep(self, key, sources, value):
        if not capturing():
            self._entry = (key, Storages(sources), value)
        return value


class HipWeightCache(_Kept):
    """Device copy of one weight in a compute dtype, re-made when the weight changes.

    Keyed like the reference ``GLUWeightCache`` (``gated_linear_unit.py:15-30``) on
    (data_ptr, _version, shape, stride, dtype, device, compute dtype, layout) and on the
    storage (:class:`Storages`); tensors without a version counter (inference tensors) are
    never cached. ``layout`` is ``"plain"`` (contiguous copy) or ``"glu"`` (the packed
    gate/value layout).
    """

    def get(self, weight: torch.Tensor, dtype: torch.dtype, layout: str = "plain") -> torch.Tensor:
        if weight.is_inference():
            self.clear()
            return _prepare(weight, dtype, layout)
        key = (*stamp(weight), dtype, layout)
        value = self.lookup(key)
        return value if value is not None else self.keep(key, [weight], _prepare(weight, dtype, layout))


def _prepare(weight: torch.Tensor, dtype: torch.dtype, layout: str) -> torch.Tensor:
    w = weight.detach().to(dtype=dtype).contiguous()
    if layout == "plain":
        return w
    if layout == "glu":
        # w is transition1.weight: [2F, K], rows [0, F) = SiLU gate.
        rows2f, k = w.shape
        f = rows2f // 2
        lib = load_library()
        packed = torch.empty((lib.xfh_glu_packed_rows(f), k), dtype=dtype, device=w.device)
        call("xfh_glu_pack_weight", ptr(w), f, k, dtype_code(dtype), ptr(packed), stream_of(w.device))
        return packed
    raise ValueError(f"unknown weight layout {layout}")


def module_cache(module: torch.nn.Module, name: str) -> HipWeightCache:
    """Per-module weight caches, held outside ``state_dict`` (like ``_native_weights``)."""
    caches = module.__dict__.setdefault("_hip_weight_caches", {})
    cache = caches.get(name)
    if cache is None:
        cache = caches[name] = HipWeightCache()
    return cache


def linear_weight(module: torch.nn.Module, name: str, dtype: torch.dtype, layout: str = "plain"):
    """Device copy of ``module.<name>.weight`` ([out, in]) in ``dtype``."""
    return module_cache(module, name).get(param(module, name), dtype, layout)


class FusedWeightCache(_Kept):
    """Row-concatenation of several weights ([out_i, in] -> [sum out_i, in]) in one dtype,
    re-made when any source weight changes (same keys as :class:`HipWeightCache`)."""

    def get(self, weights, dtype: torch.dtype) -> torch.Tensor:
        build = lambda: torch.cat([w.detach().to(dtype) for w in weights], dim=0).contiguous()  # noqa: E731
        if any(map(_is_inference, weights)):
            self.clear()
            return build()
        key = (*map(stamp, weights), dtype)
        value = self.lookup(key)
        return value if value is not None else self.keep(key, weights, build())


def fused_linear_weight(module: torch.nn.Module, names, dtype: torch.dtype) -> torch.Tensor:
    caches = module.__dict__.setdefault("_hip_weight_caches", {})
    tag = "fused:" + ",".join(names)
    cache = caches.get(tag)
    if cache is None:
        cache = caches[tag] = FusedWeightCache()
    return cache.get([param(module, n) for n in names], dtype)


class DerivedWeightCache(_Kept):
    """A tensor built from several parameters by ``build(*sources)`` (a one-time weight
    preparation), re-made when any source changes (same keys as :class:`HipWeightCache`;
    never cached when a source is an inference tensor)."""

    def get(self, sources, build):
        if any(map(_is_inference, sources)):
            self.clear()
            return build(*sources)
        key = tuple(map(stamp, sources))
        value = self.lookup(key)
        return value if value is not None else self.keep(key, sources, build(*sources))


def derived_weight(module: torch.nn.Module, tag: str, sources, build):
    caches = module.__dict__.setdefault("_hip_weight_caches", {})
    cache = caches.get(tag)
    if cache is None:
        cache = caches[tag] = DerivedWeightCache()
    return cache.get(list(sources), build)


def linear_weights(module: torch.nn.Module, names, dtype: torch.dtype):
    """:func:`linear_weight` of several Linears as one cache entry: the copies are made by one call,
    into one allocation (each 256-byte aligned). A new 72-token pair block with its single track: 655 us
    with the copies made and kept one by one, 582 now."""
    return derived_weight(module, f"linears:{names}:{dtype}", [param(module, n) for n in names],
                          lambda *ws: _copies(ws, dtype))


def check_one_device(weights) -> None:
    """Copies made by one call land where the first weight is: one that lies elsewhere (a host weight, which
    :func:`ptr` refuses) must not be brought along."""
    if any(w.device != weights[0].device for w in weights):
        raise ValueError("The 'hip' backend requires strided ROCm (cuda) tensors, a module's weights on one device.")


def _copies(weights, dtype: torch.dtype) -> list:
    ws = [w.detach() for w in weights]
    if all(w.dtype == dtype and w.is_contiguous() for w in ws):
        return ws
    check_one_device(ws)
    flat = torch.empty(sum((w.numel() + 127) // 128 * 128 for w in ws), dtype=dtype, device=ws[0].device)
    out, at = [], 0
    for w in ws:
        out.append(flat.as_strided(w.shape, (w.shape[1], 1), at))
        at += (w.numel() + 127) // 128 * 128
    torch._foreach_copy_(out, ws)
    return out


def fp32_param(module: torch.nn.Module, name: str, param: Optional[torch.Tensor]):
    """LayerNorm affine parameters as contiguous fp32 (None stays None)."""
    if param is None:
        return None
    if param.dtype == torch.float32 and param.is_contiguous():
        return param.detach()
    return module_cache(module, name).get(param, torch.float32)


_MISSING = object()


def param(module: torch.nn.Module, name: str, attr: str = "weight") -> Optional[torch.Tensor]:
    """``module.<name>.<attr>`` read from the registration tables (``nn.Module.__getattr__``
    takes several times as long), or as an attribute where it is not a plain parameter."""
    sub = module._modules.get(name)
    value = _MISSING if sub is None else sub._parameters.get(attr, _MISSING)
    return getattr(getattr(module, name), attr) if value is _MISSING else value


def params(module: torch.nn.Module, names, norms=()) -> list:
    """The weights of ``names``, then weight and bias of each LayerNorm of ``norms``."""
    out = [param(module, name) for name in names]
    for name in norms:
        out += (param(module, name), param(module, name, "bias"))
    return out


class WeightGroup:
    """The prepared weights of one module call, checked as a whole: the same key and storages per
    source as :class:`HipWeightCache`, compared once. A copied or pickled module starts with an
    empty group."""

    __slots__ = ("key", "storages", "dtypes", "values")

    def __init__(self):
        self.key = self.storages = self.dtypes = self.values = None

    def __reduce__(self):
        return WeightGroup, ()


def gather(module: torch.nn.Module, tag: str, sources, weights: int, x: torch.Tensor, build,
           dtype: Optional[torch.dtype] = None, again: bool = False):
    """(compute dtype, ``build(dtype)``) of a module's ``sources`` (parameters or None), the first
    ``weights`` of which take part in :func:`compute_dtype` (unless ``dtype`` is given). ``build``
    runs again when a source or the dtype has changed; its values are kept for one dtype.

    The first pass over a module keeps nothing and takes no key: its weights are being prepared
    (each in its own cache) while the GPU waits. ``again``: the values are None on that pass and
    on the first one after a change, when a whole block's weights are prepared operator by
    operator behind the operators already queued; the block's one call starts with the next.
    Its ``build`` only collects what the operators prepared: a capture may be that next pass,
    and what it makes is not kept (:func:`capturing`)."""
    groups = module.__dict__.setdefault("_hip_weight_groups", {})
    group = groups.get(tag)
    if group is None:
        groups[tag] = WeightGroup()
        dtype = dtype or _compute_dtype(x.dtype, [p.dtype for p in sources[:weights]])
        return dtype, None if again else build(dtype)
    try:
        key = None if sources[0].is_inference() else [None if p is None else stamp(p) for p in sources]
    except RuntimeError:                             # (a mixture)
        key = None
    if key is None:                                  # inference tensors carry no version: nothing is kept
        dtype = dtype or _compute_dtype(x.dtype, [p.dtype for p in sources[:weights]])
        return dtype, None if again else build(dtype)
    changed = group.key is not None and (group.key != key or not group.storages.alive())
    if changed or group.key is None:
        group = WeightGroup()
        group.key, group.storages = key, Storages(sources)
        group.dtypes = {p.dtype for p in sources[:weights]}
        groups[tag] = group
    dtype = dtype or _compute_dtype(x.dtype, group.dtypes)
    values = group.values
    if values is None or values[0] != dtype:
        if again and changed:
            return dtype, None
        values = (dtype, build(dtype))
        if not capturing():
            group.values = values
    return values


def first_pass(module: torch.nn.Module, tag: str) -> bool:
    """Whether ``tag`` of ``module`` is met for the first time: :func:`gather` with ``again`` would
    give None, without collecting the sources of a whole block for it (100 of 690 us of a
    pair block's first pass with its single track at 72 tokens)."""
    groups = module.__dict__.setdefault("_hip_weight_groups", {})
    if tag in groups:
        return False
    groups[tag] = WeightGroup()
    return True


def norm_params(module: torch.nn.Module, name: str) -> tuple:
    """fp32 weight and bias of LayerNorm ``module.<name>``."""
    return (fp32_param(module, name + ".weight", param(module, name)),
            fp32_param(module, name + ".bias", param(module, name, "bias")))
