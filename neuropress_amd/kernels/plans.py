"""What the lowered modules hand to the native call path (``csrc/host/call_plan.cpp``).

A module that has decided which kernel serves a call describes that call here once -- the entry point's constant
arguments as a *template*, the token counts it serves as *routes* -- and later calls are issued by the plan without
Python argument checks.  A plan is valid while the module's buffers, the attributes and thresholds that the decision
read, and the wrapper functions of ``kernels`` are what they were; otherwise it declines and the module decides again.
"""

from __future__ import annotations

import torch
import torch.nn.modules.module as nn_module

from .. import _lib

_TORCH_CALL = torch.nn.Module.__call__
_TORCH_LINEAR = torch.nn.functional.linear

(SLICED, VQ_GEMV, VQ_GEMV_PERM, VQ_TILE, VQ_DENSE, RVQ_GEMV, RVQ_TILE, RVQ_DENSE,
 Q_GEMV, Q_TILE, Q_DENSE, RMS_NORM, VQ_EMBEDDING, Q_EMBEDDING, VQ_SLICE, VQ_BLOCKS, RVQ_BLOCKS, Q_BLOCKS) = range(18)  # fmt: skip

DTYPE_CODES = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16, torch.float32: _lib.F32, torch.int64: 3}


def make(module, attributes, thresholds=None, names=(), holders=(), sources=()):
    """An empty plan for *module*, or None where it cannot have one (a tensor off the module's GPU, or with gaps).

    *attributes*: names in the module's ``__dict__`` the dispatch reads; *thresholds* / *names*: the globals of the
    module's file it reads (next to the band lines of ``nn.backends``); *holders*: further modules whose buffers are used (shared codebooks); *sources*: the
    buffers themselves.
    """
    from .. import kernels
    from ..nn import backends

    device = None
    for t in sources:
        if t is None:
            continue
        if not t.is_cuda or not t.is_contiguous() or (device is not None and t.device != device):
            return None
        device = t.device
    if device is None:
        return None
    plan = _lib.host().CallPlan(device.index)
    own = module.__dict__
    plan.guard_module({name: own[name] for name in (*attributes, "_buffers") if name in own})
    for holder in (module, *holders):
        plan.guard(holder._buffers, dict(holder._buffers), False)
    if names:
        plan.guard(thresholds, {name: thresholds[name] for name in names}, False)
        plan.guard(backends.__dict__, {name: getattr(backends, name) for name in backends.BAND_LINES}, False)
    plan.guard(kernels.__dict__, kernels.WRAPPERS, True)
    plan.guard(torch.nn.functional.__dict__, {"linear": _TORCH_LINEAR}, True)
    plan.guard(kernels.SlicedCallPlan, {"run": kernels.SLICED_RUN}, True)
    for t in sources:
        plan.source(t)
    _call_directly(plan, module)
    return plan


_HOOKS = ("_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks")


def _call_directly(plan, module) -> None:
    """Let ``module(x)`` go to the plan without ``torch.nn.Module.__call__`` and ``forward`` in between.

    For the classes that declare their ``forward`` to do nothing but ask the plan first (``_planned_forward``), and
    only while that call would find nothing else to do: no hooks, no compiled call, neither function replaced."""
    cls, call = type(module), _lib.host().module_call
    if vars(cls).get("_planned_forward") is None:
        return
    if "__call__" not in vars(cls):
        cls.__call__ = call
    if vars(cls)["__call__"] is not call:
        return
    every = tuple(getattr(nn_module, "_global" + name) for name in _HOOKS)
    own = {name: module.__dict__.get(name) for name in _HOOKS}
    if any(hooks is None for hooks in own.values()):
        return
    plan.direct(
        cls,
        {**own, "forward": ..., "_compiled_call_impl": ...},
        ((cls, {"forward": cls._planned_forward, "__call__": call}), (torch.nn.Module, {"__call__": _TORCH_CALL})),
        (*own.values(), *every),
    )


def template(plan, kind, n, k, args, dtype, *, f=0.0, k_in=None, perm=None, bias=None, leaf=None, own=False):
    """Template number of one call shape.  *args*: its constant arguments, tensors standing for their addresses (the
    plan keeps them alive); *dtype*: of the output; *perm*: columns of x to gather first; *k_in*: columns of x where the
    kernel contracts more (rows padded with zeros); *own*: the dense product is the package's own (*bias* in float32); *leaf*: the
    module's bias itself, for dense products: the plan declines while it asks for a gradient."""
    ints = tuple(a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args)
    keep = tuple(a for a in args if isinstance(a, torch.Tensor))
    return plan.template(kind, n, k, k if k_in is None else k_in, ints, f, DTYPE_CODES[dtype], perm, bias, leaf, own, keep)


def tile_scratch(m: int, n: int, k: int) -> int:
    """Bytes of scratch a tile GEMM of this shape can use."""
    return max(0, int(_lib.load().npamd_gemm_tile_workspace_bytes(m, n, k))) // 4 * 4


def slice_scratch(m: int, n: int, k: int, num_centroids: int) -> int:
    """Bytes of scratch a slice GEMM of this shape needs."""
    return int(_lib.load().npamd_vq_slice_workspace_bytes(m, n, k, num_centroids))


def product_scratch(m: int, n: int, k: int) -> int:
    """Bytes of scratch the package's own dense product of this shape can use, next to the decoded weight."""
    return int(_lib.load().npamd_dense_gemm_workspace_bytes(m, n, k))
