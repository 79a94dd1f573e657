"""The operator boundary: ``alexdremov_streaming_attention::forward`` / ``::backward``.

Same dispatcher names, argument lists, fake implementations and autograd registration as
the reference (src/streaming_attention/kernel.py:1270-1530).  The ops, their GPU implementation (which enqueues the HIP
kernels of libstreaming_attention.so on the current stream instead of launching Triton kernels) and their autograd are
native code (csrc/sa_torch.cpp, module ``_native``); this file holds the fake implementations and the argument checks.
``autotune``, ``prescale_qk`` and ``precision`` are accepted for signature
compatibility and do not change the result: kernel variants are read from a table measured
on MI355X (head dimension, context_size class, window class), all accumulation is fp32, and
where the scale is applied is fixed per kernel: in float32 inside the exp2 argument in the forward
and dQ kernels and in all float32 ones (at least as accurate as either setting of ``prescale_qk``), folded into K and
rounded to the element type in the 16-bit dK/dV kernels at head dimensions 32 and up (what the
reference does under ``prescale_qk=True``, kernel.py:1065-1066).
"""
from __future__ import annotations

import torch

try:
    from ._native import kernel_layout as _kernel_layout  # noqa: F401  (the module registers the ops)
except ImportError as e:
    raise ImportError(
        "streaming_attention._native cannot be loaded: build it with `make -C kernels_amd/csrc` "
        "(or `python -c 'import __graft_entry__ as g; g.build()'`). There is no fallback implementation."
    ) from e

_HEAD_DIMS = (16, 32, 64, 128, 256)


def _validate_placement(q, k, v, lens, *others):
    """The kernels index k, v (and o, dO) with q's batch and head counts and dereference every
    pointer on q's device, so a tensor that lives elsewhere or has fewer batches / heads (an
    un-expanded grouped-query k or v) must be refused before any ``data_ptr()`` is taken."""
    assert q.ndim == 4 and k.ndim == 4 and v.ndim == 4
    assert k.shape[:2] == q.shape[:2] and v.shape[:2] == q.shape[:2], "k and v need q's batch and head sizes"
    assert k.device == q.device and v.device == q.device, "q, k and v must be on one device"
    assert lens is None or lens.device == q.device, "lens must be on the device of q"
    for t in others:
        assert t.shape == q.shape, "o and dO need q's shape"
        assert t.device == q.device, "o and dO must be on the device of q"


def _validate(q, k, v, lens, context_size, back_contexts, sm_scale, *others):
    # same conditions, same exception type as kernel.py:1288-1295
    shape, dev = q.shape, q.device
    plain = (len(shape) == 4 and k.shape == shape and v.shape == shape
             and k.device == dev and v.device == dev and (lens is None or lens.device == dev))
    for t in others:
        plain = plain and t.shape == shape and t.device == dev
    if not plain:   # name the condition that failed
        _validate_placement(q, k, v, lens, *others)
    batch, _, T, head_dim = shape
    assert back_contexts >= 0 and context_size >= 1
    assert head_dim in _HEAD_DIMS
    assert head_dim == k.shape[-1] and head_dim == v.shape[-1]
    assert T == k.shape[-2] and T == v.shape[-2]
    assert sm_scale is not None
    assert lens is None or (lens.dtype == torch.int32 and lens.ndim == 1 and batch == lens.shape[0])
    assert q.dtype == k.dtype == v.dtype
    assert q.device.type != "cuda" or q.dtype in (torch.float32, torch.float16, torch.bfloat16), \
        f"unsupported dtype {q.dtype}: expected float32, float16 or bfloat16"


@torch.library.register_fake("alexdremov_streaming_attention::forward")
def attention_forward_adapter_abstract(
    q, k, v, lens, context_size, back_contexts, sm_scale, autotune, return_lse, prescale_qk, precision
):
    return (
        torch.empty_like(q, memory_format=torch.contiguous_format),
        torch.empty(q.shape[:3], dtype=torch.float32, device=q.device) if return_lse else torch.empty(0),
    )


@torch.library.register_fake("alexdremov_streaming_attention::backward")
def attention_backward_adapter_abstract(
    q, k, v, lens, o, lse, do, context_size, back_contexts, sm_scale, autotune, prescale_qk, precision
):
    return (
        torch.empty_like(q, memory_format=torch.contiguous_format),
        torch.empty_like(k, memory_format=torch.contiguous_format),
        torch.empty_like(v, memory_format=torch.contiguous_format),
    )
