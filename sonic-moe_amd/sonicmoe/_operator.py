"""Operators of the `sonicmoe::` namespace and how the layer calls them.

Every operator is a torch custom op: what traces, transforms or intercepts PyTorch calls sees it.  The dispatcher's way
to such an op costs about 20 us of host time per call, more than most of its kernels take on a few tokens; where none of
the observers below looks on, `run` calls the operator's Python body (its argument checks and the C entry point) directly.
An ExecutionTraceObserver without a profiler around it gives no sign of itself: its trace lacks the operators.
"""

from __future__ import annotations

import torch
from torch.fx.experimental.proxy_tensor import get_proxy_mode

from . import _lib
from ._lib import NoMemory
from .enums import LIBRARY_NAME

# The dispatcher would do nothing but call the body for these values and for tensors that are no subclass, have memory (a
# meta tensor stops at the fake implementation, a zero tensor without memory is filled) and hold their values as they are
# (a lazily negated view is resolved).  A zero tensor is told where its pointer is taken, before the C entry point: asking
# every tensor cost 7 us of host time per forward pass.
_TENSORS = (torch.Tensor, torch.nn.Parameter)
_VALUES = frozenset((type(None), int, float, bool, str))

# Dispatch keys of a plain tensor under which somebody else may register an implementation of an operator (the operator's
# own registrations are under alias keys), and the names, "namespace/operator/key", of all that Python code has registered
# (a torch without that record: every call takes the dispatcher).
_KEYS = ("CUDA", "AutogradCUDA", "AutocastCUDA", "CPU", "AutogradCPU", "AutocastCPU", "BackendSelect",
         "CompositeImplicitAutograd")
_REGISTERED = getattr(torch.library, "_impls", None)


def _names(library: str, *names: str) -> frozenset:
    return frozenset(f"{library}/{name}/{key}" for name in names for key in _KEYS)


def operator(name: str, mutates_args: set[str]):
    """torch.library.custom_op in this package's namespace; the undecorated function is kept as `.body`."""

    def register(body):
        op = torch.library.custom_op(f"{LIBRARY_NAME}::{name}", mutates_args=mutates_args)(body)
        op.body = body
        op.elsewhere = _names(LIBRARY_NAME, name)
        return op

    return register


def elsewhere(*ops) -> frozenset:
    """The names under which somebody else may register an implementation of one of these operators."""
    return frozenset().union(*(op.elsewhere for op in ops))


def torch_elsewhere(*names: str) -> frozenset:
    """The same of these torch operations."""
    return _names("aten", *names)


def on_gpu(names: frozenset) -> frozenset:
    """Those of the names that matter for tensors on a GPU (each costs some 25 ns per question)."""
    return frozenset(name for name in names if not name.endswith("CPU"))


def registered(names: frozenset) -> bool:
    """Whether somebody has registered an implementation under one of these names (or nobody can say)."""
    return _REGISTERED is None or not _REGISTERED.isdisjoint(names)


def untraced() -> bool:
    """Whether no mode, transformation or trace stands between a torch call and its tensors.  For eager code only."""
    return (
        torch._C._len_torch_dispatch_stack() == 0  # dispatch modes: fake tensors, make_fx, profiling counters
        and torch._C._functorch.peek_interpreter_stack() is None  # vmap, grad, functionalization
        and not torch._C._is_torch_function_mode_enabled()
        and torch._C._get_tracing_state() is None  # torch.jit.trace
    )


def untransformed() -> bool:
    """Whether torch calls do what they say, whoever looks on: no vmap, grad or functionalization around them and no trace
    being recorded.  For eager code only."""
    return (
        torch._C._functorch.peek_interpreter_stack() is None
        and torch._C._get_tracing_state() is None
        and (torch._C._len_torch_dispatch_stack() == 0 or get_proxy_mode() is None)
    )


def in_memory(*tensors) -> bool:
    """Whether a kernel launched now may be given the addresses of all these tensors (or None): plain ones, which have an
    address that means something, in memory of the current GPU (the torch operation that the kernel stands in for would refuse
    tensors of several, and run where theirs are)."""
    gpu = _lib.current_gpu()
    for t in tensors:
        if t is not None and (type(t) not in _TENSORS or t.get_device() != gpu or t.is_neg()):
            return False
    return True


def unobserved(names: frozenset, *tensors) -> bool:
    """Whether nobody looks on the calls of the operators behind `names` (`elsewhere`) in a row and these tensors are
    `in_memory`: the questions of `run`, asked once.  For eager code only."""
    return (
        untraced()
        and not torch.autograd._profiler_enabled()
        and not registered(names)
        and in_memory(*tensors)
    )


def stands_in(replaced: frozenset, *tensors) -> bool:
    """Whether an operator may stand in for the operations behind `replaced` (`elsewhere`, `torch_elsewhere`) on these
    tensors: whoever traces or transforms torch calls keeps them, and can see through them, as does who has registered an
    implementation of one; and so do tensors without an address to ask for.  (Profilers see the operator.)"""
    return not torch.compiler.is_compiling() and untraced() and not registered(replaced) and in_memory(*tensors)


def run(op, *args) -> None:
    """op(*args) for outputs that were allocated for this call and that nothing has saved yet (the dispatcher would also
    count the mutation in their version counters)."""
    if torch.compiler.is_compiling():
        op(*args)
        return
    if (
        untraced()
        and not torch.autograd._profiler_enabled()  # its rows come from the dispatcher
        and not args[0].is_meta  # (every operator's first argument is a tensor, and all of one call are on one device)
    ):
        for a in args:
            kind = type(a)
            if kind not in _VALUES and (kind not in _TENSORS or a.is_neg()):
                break
        else:
            # (a plain function put in an operator's place is called as it is)
            if hasattr(op, "body") and not registered(op.elsewhere):
                try:
                    return op.body(*args)
                except NoMemory:
                    pass
    op(*args)
