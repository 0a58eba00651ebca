"""The token-choice layer behind (of few tokens: with) its router GEMM as one call of the HIP library per direction (smoe_layer_forward /
smoe_layer_backward: the operators' entry points in the operators' order, so the same kernels and the same results).

For the common case only: plain 16-bit tensors of one type, no autocast, no tensor of a forward-mode derivative, memory as the
operators want it (`takes`).  Whatever is not like that -- and whatever the library refuses -- takes the operators one by one,
which say what is wrong with it.  So does a call that somebody looks on (`unobserved`); what it keeps for its backward pass is
the same, because who looks on may come and go between a forward pass and its recomputation from a checkpoint.
"""

from __future__ import annotations

import struct

import torch
from torch.autograd import forward_ad

from .. import _lib
from .._operator import elsewhere, in_memory, on_gpu, unobserved, untransformed
from ..enums import ACTIVATION_CODE, is_glu
from . import backward as _b
from . import forward as _f

# All of a step's operators run in one call, so nothing it needs for a while can be given back in between: the gathered
# rows of both GEMMs are held while the output is written, the logits while all gradients are.  Up to this many bytes of them
# that is no matter; beyond it a step takes milliseconds, to which the calls (0.1 ms) add nothing, and memory is what counts.
MAX_TRANSIENT_BYTES = 1 << 30

_FORWARD = struct.Struct("33q")
_BACKWARD = struct.Struct("45q")
_FORWARD_OPERATORS = (_f._router_logits, _f._softmax_topk_fwd, _f._topk_fwd, _f._up_projection_forward, _f._down_projection_forward,
                      _f._router_forward, _f._switch_loss_fwd)
_BACKWARD_OPERATORS = (_b._down_projection_backward, _b._up_projection_backward, _b._token_broadcast_backward, _b._token_broadcast_backward_router,
                       _b._switch_loss_bwd, _b._router_logit_grad, _b._router_weight_grad, _b._sum_chunks)
_BACKWARD_NAMES = on_gpu(elsewhere(*_BACKWARD_OPERATORS)) | _b.ROUTER_DX
_ELEMENTS = (torch.bfloat16, torch.float16)


class Refused(Exception):
    """The library does not take the layer: the operators tell why."""


# smoe_status of arguments or shapes that the kernels do not take (bad argument, unsupported)
_NOT_TAKEN = (1, 2)


def _taken(rc: int, what: str) -> bool:
    """Whether the library did it; a launch that failed or a workspace that does not suffice is told, and not tried again."""
    if rc in _NOT_TAKEN:
        return False
    _lib.check(rc, what)
    return True


def forward_names(routing_metadata) -> frozenset:
    return on_gpu(elsewhere(*_FORWARD_OPERATORS, routing_metadata)) | _f.ROUTER_LINEAR


class Indices:
    """Where the routing's outputs lie in one int32 tensor, each at a multiple of 256 bytes."""

    __slots__ = ("T", "E", "K", "at", "words")

    def __init__(self, T: int, E: int, K: int):
        pad = lambda n: (n + 63) // 64 * 64
        tk = pad(T * K)
        self.T, self.E, self.K = T, E, K
        # scores (fp32), indices, x_gather_idx, s_scatter_idx, s_reverse_scatter_idx, off, tok_off, loss_acc (fp32)
        self.at = at = [0, tk, 2 * tk, 3 * tk, 4 * tk, 5 * tk, 5 * tk + pad(E + 1), 5 * tk + pad(E + 1) + pad(T + 1)]
        self.words = at[7] + pad(E)

    def views(self, t: torch.Tensor):
        """(scores (T, K), indices (T, K), gidx, sidx, ridx, off, tok_off, loss_acc) as tensors"""
        T, E, K = self.T, self.E, self.K
        sizes = (T * K,) * 5 + (E + 1, T + 1, E)
        scores, indices, gidx, sidx, ridx, off, tok_off, acc = (t[a:a + n] for a, n in zip(self.at, sizes))
        return (scores.view(torch.float32).view(T, K), indices.view(T, K), gidx, sidx, ridx, off, tok_off,
                acc.view(torch.float32))


def takes(x, router_w, w1, b1, w2, b2, K: int, activation, stream_id: int, quiet: bool) -> bool:
    """Whether `forward` takes this layer; if not `quiet`, whether it would, were the operators `unobserved`.  (Sizes that the
    kernels refuse are told by the library.)"""
    dtype = x.dtype
    if not (
        (quiet or untransformed())
        and in_memory(x, router_w, w1, b1, w2, b2)
        and dtype in _ELEMENTS
        and router_w.dtype == dtype and w1.dtype == dtype and w2.dtype == dtype
        and x.dim() == 2 and router_w.dim() == 2 and w1.dim() == 3 and w2.dim() == 3
        and forward_ad._current_level < 0
        and not torch.is_autocast_enabled("cuda")
        and stream_id == _lib.current_stream_handle()
    ):
        return False
    T, H = x.shape
    E = router_w.size(0)
    I = w2.size(1)
    N1 = 2 * I if is_glu(activation) else I
    if not (
        T > 0 and 0 < K <= E and (T * K * (H + I) + T * E) * 2 <= MAX_TRANSIENT_BYTES
        and router_w.size(1) == H and w1.shape == (N1, H, E) and w2.shape == (H, I, E)
        and w1.stride(1) == 1 and w2.stride(1) == 1
        and x.data_ptr() != 0 and w1.data_ptr() != 0 and w2.data_ptr() != 0 and router_w.data_ptr() != 0
    ):
        return False
    if b1 is None:
        return b2 is None
    return (b2 is not None and b1.dtype == dtype and b2.dtype == dtype and b1.shape == (E, N1) and b2.shape == (E, H)
            and b1.is_contiguous() and b2.is_contiguous() and b1.data_ptr() != 0 and b2.data_ptr() != 0)


def forward(x, router_w, w1, b1, w2, b2, K: int, activation, stream_id: int, keep_z: bool, with_loss: bool):
    """(o, logits, z or None, freq, the routing's int32 tensor, loss or None), or None where the library refuses."""
    T, H = x.shape
    E, I = router_w.size(0), w2.size(1)
    dev, dtype = x.device, x.dtype
    own_logits = _f.router_logits_takes(x, router_w)
    if own_logits:
        logits = torch.empty(T, E, dtype=dtype, device=dev)
    else:
        logits = torch.nn.functional.linear(x, router_w)
        if logits.dtype != dtype or logits.stride(1) != 1:
            return None
    L = _lib.lib(dtype)
    where = Indices(T, E, K)
    need = L.smoe_layer_forward_workspace_bytes(T, H, I, E, K)
    if need == 0:
        return None
    o = torch.empty(T, H, dtype=dtype, device=dev)
    z = torch.empty(T * K, w1.size(0), dtype=dtype, device=dev) if keep_z else None
    freq = torch.empty(E, dtype=torch.int32, device=dev)
    ints = torch.empty(where.words, dtype=torch.int32, device=dev)
    loss = torch.empty((), dtype=torch.float32, device=dev) if with_loss else None
    scratch = torch.empty(need, dtype=torch.uint8, device=dev)
    s1, s2, base, at = w1.stride(), w2.stride(), ints.data_ptr(), where.at
    rc = L.smoe_layer_forward(
        _FORWARD.pack(
            x.data_ptr(), router_w.data_ptr() if own_logits else 0, logits.data_ptr(), w1.data_ptr(), 0 if b1 is None else b1.data_ptr(), w2.data_ptr(),
            0 if b2 is None else b2.data_ptr(),
            s1[2], s1[0], s2[2], s2[0], _lib.DT_CODE[dtype], logits.stride(0), T, H, I, E, K, ACTIVATION_CODE[activation],
            z.data_ptr() if keep_z else 0, o.data_ptr(),
            base, base + 4 * at[1], freq.data_ptr(), base + 4 * at[5], base + 4 * at[2], base + 4 * at[3], base + 4 * at[4],
            base + 4 * at[6],
            base + 4 * at[7], loss.data_ptr() if with_loss else 0, scratch.data_ptr(), need,
        ),
        stream_id,
    )
    return (o, logits, z, freq, ints, loss) if _taken(rc, "layer_forward") else None


def backward(x, dout, z, w1, w2, b2, has_b1: bool, ints, freq, logits, K: int, activation, stream_id: int, loss_grad,
             outside, chunks: int, router_w):
    """(dx, dlogits, dwr or None, dw1, db1, dw2, db2), or None where the operators have to do it.  chunks: token chunks of the
    router's weight gradient (0: the caller forms it).  router_w: None leaves the router's share of dx to the caller.  freq
    and logits: with loss_grad only."""
    dtype = x.dtype
    if torch.compiler.is_compiling() or not (
        unobserved(_BACKWARD_NAMES, x, dout, z, w1, w2, b2, ints, freq, logits, loss_grad, outside, router_w)
        and dout.dtype == dtype and dout.layout == torch.strided and stream_id == _lib.current_stream_handle()
        and (loss_grad is None or outside is None)
    ):
        return None
    dout = dout.contiguous()
    T, H = x.shape
    _, I, E = w2.shape
    if loss_grad is not None:
        loss_grad = loss_grad.reshape(1).float()
    elif outside is not None and not (outside.layout == torch.strided and outside.dtype == dtype
                                      and outside.shape == (T, E) and outside.stride(1) == 1
                                      and outside.stride(0) >= E):
        return None
    loss = () if loss_grad is None else (loss_grad, freq, logits)
    where = Indices(T, E, K)
    # (saved tensors may come back from hooks in other memory, of another type or shape)
    if not (z.dtype == w1.dtype == w2.dtype == dtype and (b2 is None or b2.dtype == dtype)
            and (router_w is None or router_w.dtype == dtype and router_w.shape == (E, H))
            and dout.shape == (T, H) and w1.shape == (z.size(1), H, E) and w2.size(0) == H
            and z.shape == (T * K, 2 * I if is_glu(activation) else I)
            and (b2 is None or b2.shape == (E, H)) and ints.dtype == torch.int32 and ints.shape == (where.words,)
            and (not loss or (freq.dtype == torch.int32 and freq.shape == (E,) and logits.dtype == dtype
                              and logits.shape == (T, E)))):
        return None
    s1, s2 = w1.stride(), w2.stride()
    if not (x.is_contiguous() and z.is_contiguous() and ints.is_contiguous() and s1[1] == 1 and s2[1] == 1
            and (b2 is None or b2.is_contiguous()) and (router_w is None or router_w.is_contiguous())
            and (not loss or (freq.is_contiguous() and logits.stride(1) == 1))):
        return None
    p_x, p_dout, p_z, p_w1, p_w2, base = given = (x.data_ptr(), dout.data_ptr(), z.data_ptr(), w1.data_ptr(), w2.data_ptr(),
                                                  ints.data_ptr())
    p_b2, p_outside, p_router = [0 if t is None else t.data_ptr() for t in (b2, outside, router_w)]
    p_loss, p_freq, p_logits = (loss_grad.data_ptr(), freq.data_ptr(), logits.data_ptr()) if loss else (0, 0, 0)
    # (null means "not given", of router_w that the caller adds its share; the dx kernel wants it aligned)
    if (0 in given or (loss and 0 in (p_loss, p_freq, p_logits)) or (p_b2 == 0) != (b2 is None)
            or (p_outside == 0) != (outside is None) or (p_router == 0) != (router_w is None) or p_router % 16 != 0):
        return None
    L = _lib.lib(dtype)
    code, dev = ACTIVATION_CODE[activation], x.device
    need = L.smoe_layer_backward_workspace_bytes(T, H, I, E, K, code, chunks)
    if need == 0:
        return None
    dw1, dw2 = torch.empty_like(w1), torch.empty_like(w2)  # (in the parameter views' layout)
    db1 = torch.empty(E, w1.size(0), dtype=dtype, device=dev) if has_b1 else None
    db2 = None if b2 is None else torch.empty_like(b2)
    dx = torch.empty(T, H, dtype=dtype, device=dev)
    dlogits = torch.empty(T, E, dtype=dtype, device=dev)
    dwr = torch.empty(E, H, dtype=dtype, device=dev) if chunks else None
    scratch = torch.empty(need, dtype=torch.uint8, device=dev)
    d1, d2, at = dw1.stride(), dw2.stride(), where.at
    if d1[1] != 1 or d2[1] != 1:
        return None
    rc = L.smoe_layer_backward(
        _BACKWARD.pack(
            p_x, p_dout, p_z, p_w1, p_w2, p_b2, s1[2], s1[0], s2[2], s2[0],
            base, base + 4 * at[1], p_freq, base + 4 * at[5], base + 4 * at[2], base + 4 * at[3], base + 4 * at[4],
            p_logits, _lib.DT_CODE[dtype], logits.stride(0) if loss else 0, base + 4 * at[7], p_loss,
            p_outside, 0 if outside is None else outside.stride(0), T, H, I, E, K, code,
            dw1.data_ptr(), dw2.data_ptr(), d1[2], d1[0], d2[2], d2[0],
            0 if db1 is None else db1.data_ptr(), 0 if db2 is None else db2.data_ptr(), dx.data_ptr(), dlogits.data_ptr(),
            p_router, 0 if dwr is None else dwr.data_ptr(), chunks, scratch.data_ptr(), need,
        ),
        stream_id,
    )
    return (dx, dlogits, dwr, dw1, db1, dw2, db2) if _taken(rc, "layer_backward") else None
