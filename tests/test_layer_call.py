"""The layer as one call of the library per direction: the packed arguments against the declared structs, and the same bits
as operator by operator."""

import re

import pytest
import torch

from test_abi import HEADER


@pytest.mark.parametrize("name, packed", [("smoe_layer_forward_args", "_FORWARD"), ("smoe_layer_backward_args", "_BACKWARD")])
def test_packed_arguments_fill_the_struct(name, packed):
    from sonicmoe.functional import layer_call

    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    fields = re.search(r"typedef struct \{([^}]*)\} " + name, text).group(1)
    assert getattr(layer_call, packed).size == 8 * sum(decl.count(",") + 1 for decl in fields.split(";") if decl.strip())


@pytest.mark.parametrize("T, E, K", [(1, 8, 1), (63, 5, 3), (777, 48, 4), (64, 4096, 64)])
def test_index_views_do_not_overlap(T, E, K):
    from sonicmoe.functional.layer_call import Indices

    where = Indices(T, E, K)
    spans = sorted((v.storage_offset(), v.storage_offset() + v.numel())
                   for v in where.views(torch.zeros(where.words, dtype=torch.int32)))
    assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:])) and spans[-1][1] <= where.words
    assert all(a % 64 == 0 for a, _ in spans)


@pytest.mark.parametrize("with_loss", [False, True])
def test_what_the_layer_keeps_for_its_backward(monkeypatch, with_loss):
    """Counts and logits are the caller's to change in place: without the loss the backward pass does without them."""
    from sonicmoe.enums import ActivationType
    from sonicmoe.functional import layer_call, layer_with_loss

    T, H, I, E, K = 6, 16, 8, 4, 2
    asked = []

    def forward(x, router_w, w1, b1, w2, b2, K, activation, stream_id, keep_z, loss):
        return (torch.zeros(T, H), torch.zeros(T, E), torch.zeros(T * K, 2 * I), torch.zeros(E, dtype=torch.int32),
                torch.zeros(layer_call.Indices(T, E, K).words, dtype=torch.int32), torch.zeros(()) if loss else None)

    def backward(x, dout, z, w1, w2, b2, has_b1, ints, freq, logits, *rest):
        asked.append((freq is not None, logits is not None))
        return torch.zeros(T, H), torch.zeros(T, E), torch.zeros(E, H), torch.empty_like(w1), None, torch.empty_like(w2), None

    monkeypatch.setattr(layer_call, "takes", lambda *a: True)
    monkeypatch.setattr(layer_call, "forward", forward)
    monkeypatch.setattr(layer_call, "backward", backward)
    x, wr = torch.randn(T, H, requires_grad=True), torch.randn(E, H, requires_grad=True)
    w1, w2 = torch.randn(E, 2 * I, H, requires_grad=True), torch.randn(E, H, I, requires_grad=True)
    o, logits, freq, loss = layer_with_loss(x, wr, w1.permute(1, 2, 0), None, w2.permute(1, 2, 0), None, K, 0,
                                            ActivationType.SWIGLU, False, with_loss)
    assert (loss is not None) == with_loss
    if not with_loss:
        logits.mul_(2)
        freq.add_(1)
    torch.autograd.grad([o, logits], [x, wr, w1, w2], [torch.ones_like(o), torch.ones_like(logits)])
    assert asked == [(with_loss, with_loss)]


@pytest.mark.parametrize("T, H, I, E, K, chunks", [(300000, 128, 64, 1024, 1, 4), (65536, 768, 256, 4096, 1, 8),
                                                   (6001, 1536, 256, 128, 8, 12), (64, 512, 64, 4096, 2, 0)])
def test_scratch_of_the_backward_does_not_grow_with_the_logits(T, H, I, E, K, chunks):
    """dz or the chunks of the router's gradient, y1 or dx_expanded beside it; the loss's share of the logits' gradient is
    formed where that gradient goes."""
    from sonicmoe import _lib

    need = _lib.lib().smoe_layer_backward_workspace_bytes(T, H, I, E, K, 0, chunks)
    TK = T * K
    rows = max(TK * 2 * I, chunks * E * H) * 2 + TK * max(2 * H, 2 * I + 4 * _lib.lib().smoe_dz_partial_cols(I))
    small = 2 * _lib.lib().smoe_gemm_workspace_bytes(TK, E) + 4 * (TK + E)
    assert need <= rows + small + 8 * 256


@pytest.fixture
def on_the_cpu(monkeypatch):
    """layer_call with CPU tensors (device number -1), as far as the library: on_the_cpu(library)"""
    from sonicmoe import _lib

    monkeypatch.setattr(_lib, "current_gpu", lambda: -1)
    monkeypatch.setattr(_lib, "current_stream_handle", lambda: 0)
    return lambda library: monkeypatch.setattr(_lib, "lib", library)


def _arguments():
    """(of the forward call, of the backward call)"""
    from sonicmoe.enums import ActivationType
    from sonicmoe.functional import layer_call

    T, H, I, E, K = 6, 32, 8, 4, 2
    bf16 = lambda *shape: torch.zeros(*shape, dtype=torch.bfloat16)
    both = dict(x=bf16(T, H), router_w=bf16(E, H), w1=bf16(E, 2 * I, H).permute(1, 2, 0), w2=bf16(E, H, I).permute(1, 2, 0),
                b2=bf16(E, H), K=K, activation=ActivationType.SWIGLU, stream_id=0)
    return (dict(both, b1=bf16(E, 2 * I), keep_z=True, with_loss=True),
            dict(both, dout=bf16(T, H), z=bf16(T * K, 2 * I), has_b1=True, logits=bf16(T, E), loss_grad=torch.zeros(()),
                 ints=torch.zeros(layer_call.Indices(T, E, K).words, dtype=torch.int32), freq=torch.zeros(E, dtype=torch.int32),
                 outside=None, chunks=0))


@pytest.mark.parametrize("status, told", [(0, False), (1, False), (2, False), (3, True), (4, True)])
def test_status_of_the_library(on_the_cpu, status, told):
    """What the kernels do not take goes to the operators, which tell why; a failed launch or a workspace that does not suffice
    is told at once."""
    from sonicmoe.functional import layer_call

    class Library:
        smoe_last_error = staticmethod(lambda: b"planted")

        def __getattr__(self, name):
            return lambda *args: 256 if name.endswith("workspace_bytes") else status

    from sonicmoe import _lib

    on_the_cpu(lambda *dtype: setattr(_lib._TLS, "last", Library()) or Library())
    try:
        for call, given in zip((layer_call.forward, layer_call.backward), _arguments()):
            if told:
                with pytest.raises(RuntimeError, match="planted"):
                    call(**given)
            else:
                assert (call(**given) is None) == (status != 0)
    finally:
        del _lib._TLS.last


@pytest.mark.parametrize("what", ["plain", "lazily negated", "without memory", "subclass", "other GPU", "wider type",
                                  "longer"])
def test_the_backward_asks_about_every_tensor_it_passes_on(monkeypatch, on_the_cpu, what):
    """Saved-tensor hooks decide what comes back: for each tensor that is not as the library needs it, the operators do it."""
    from sonicmoe import _operator
    from sonicmoe.functional import layer_call

    class Asked(Exception):
        pass

    class Tagged(torch.Tensor):
        pass

    class Elsewhere(torch.Tensor):
        def get_device(self):
            return 1

    def reached(dtype):
        raise Asked

    on_the_cpu(reached)
    monkeypatch.setattr(_operator, "_TENSORS", (torch.Tensor, Elsewhere))
    given = _arguments()[1]
    if what == "plain":
        with pytest.raises(Asked):
            layer_call.backward(**given)
        return
    changed = {"lazily negated": torch._neg_view, "subclass": lambda t: t.as_subclass(Tagged),
               "other GPU": lambda t: t.as_subclass(Elsewhere), "wider type": lambda t: t.double(),
               "longer": lambda t: torch.cat([t, t]),
               "without memory": lambda t: torch._efficientzerotensor(t.shape, dtype=t.dtype)}[what]
    for name, t in given.items():
        if isinstance(t, torch.Tensor) and (name != "loss_grad" or what not in ("wider type", "longer")):
            assert layer_call.backward(**{**given, name: changed(t)}) is None, name


@pytest.mark.parametrize("sparse", [False, True])
def test_gradients_of_the_loss_and_of_the_logits_add_up(monkeypatch, sparse):
    """Operator by operator: the logits' own gradient may be a sparse one (an embedding lookup in the logits)."""
    from types import SimpleNamespace

    from sonicmoe import functional
    from sonicmoe.enums import ActivationType

    T, H, I, E, K = 6, 16, 8, 4, 2
    seen = []
    monkeypatch.setattr(functional, "run", lambda op, *args: args[-1].fill_(3.0))
    monkeypatch.setattr(functional.layer_call, "backward", lambda *a: None)
    monkeypatch.setattr(functional, "_tc_layer_backward", lambda ctx, dout, dlogits, *a: seen.append(dlogits) or ())
    ints = torch.zeros(functional.layer_call.Indices(T, E, K).words, dtype=torch.int32)
    ctx = SimpleNamespace(cfg=(K, ActivationType.SWIGLU, 0, False), needs_input_grad=(True,) * 6, saved_tensors=(
        torch.zeros(T, H), torch.zeros(E, H), None, torch.zeros(H, I, E), None, None, ints, torch.zeros(E, dtype=torch.int32),
        torch.zeros(T, E)))
    own = torch.eye(T, E)
    functional._OneCallLayerFunction.backward(ctx, torch.zeros(T, H), own.to_sparse() if sparse else own, None, torch.ones(()))
    assert torch.equal(seen[0], own + 3)


def _module(T, H, I, E, K, act, bias, dtype, dev):
    from sonicmoe import MoE
    from sonicmoe.enums import ActivationType

    torch.manual_seed(T + H)
    moe = MoE(E, K, H, I, ActivationType(act), bias, 0.02).to(device=dev, dtype=dtype)
    if bias:
        for p in (moe.c_fc.bias, moe.c_proj.bias):
            torch.nn.init.normal_(p, 0, 0.1)
    return moe, torch.randn(T, H, device=dev).to(dtype), torch.randn(T, H, device=dev).to(dtype)


def _both(monkeypatch, step):
    """step() in one call per direction and operator by operator; how often the library was asked for the whole"""
    from sonicmoe.functional import layer_call

    asked = []
    for name in ("forward", "backward"):
        real = getattr(layer_call, name)
        monkeypatch.setattr(layer_call, name, lambda *a, _n=name, _r=real: (r := _r(*a), asked.append((_n, r is not None)))[0])
    one = step()
    calls = list(asked)
    monkeypatch.setattr(layer_call, "MAX_TRANSIENT_BYTES", -1)
    asked.clear()
    each = step()
    assert not asked
    for a, b in zip(one, each):
        assert (a is None) == (b is None) and (a is None or torch.equal(a, b))
    return calls


# one token; few rows and an idle expert; borders of the token chunks of the router's gradient; odd expert counts
SHAPES = [(1, 128, 64, 8, 2), (37, 192, 128, 16, 5), (255, 256, 64, 12, 3), (512, 512, 192, 8, 2), (1000, 320, 256, 33, 4)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("act, bias, dtype", [("swiglu", False, torch.bfloat16), ("geglu", True, torch.float16),
                                              ("relu_sq", True, torch.bfloat16), ("silu", False, torch.float16)])
def test_module_step(dev, monkeypatch, shape, act, bias, dtype):
    moe, x, dy = _module(*shape, act, bias, dtype, dev)

    def step():
        xx = x.clone().requires_grad_()
        out, aux = moe(xx)
        grads = torch.autograd.grad([out, aux], [xx, *moe.parameters()], grad_outputs=[dy, torch.tensor(0.3, device=dev)])
        with torch.no_grad():
            still, aux2 = moe(x)
            moe.eval()
            quiet, aux3 = moe(x)
            moe.train()
        return [out.detach(), aux.detach(), *grads, still, aux2, quiet, aux3]

    assert _both(monkeypatch, step) == [("forward", True), ("backward", True), ("forward", True), ("forward", True)]


# tile maps from the metadata's last launch (above 4096 slots, to 256 experts; above 16 rows per expert) and the experts'
# order from the backward's (from 64 rows per expert): either side of each line, one expert, remainders, and
# weight-gradient streams that walk it
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(4096, 128, 64, 1, 1), (1020, 128, 64, 255, 4), (1021, 128, 64, 255, 4),
                                   (4097, 128, 64, 1, 1), (1366, 128, 64, 63, 3), (1100, 128, 64, 65, 4), (8191, 128, 128, 256, 2),
                                   (8192, 128, 128, 256, 2), (8230, 128, 64, 257, 2), (8200, 256, 128, 8, 2),
                                   (4100, 768, 256, 128, 8)])
def test_maps_written_on_the_way(dev, monkeypatch, shape):
    moe, x, dy = _module(*shape, "swiglu", False, torch.bfloat16, dev)

    def step():
        xx = x.clone().requires_grad_()
        out, aux = moe(xx)
        return [out.detach(), *torch.autograd.grad([out, aux], [xx, *moe.parameters()],
                                                   grad_outputs=[dy, torch.tensor(0.3, device=dev)])]

    assert _both(monkeypatch, step) == [("forward", True), ("backward", True)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["loss only", "output only", "logits too", "logits transposed", "router frozen", "x frozen",
                                  "x strided", "dout strided", "weights strided", "hooks", "twice", "outputs changed", "router misaligned"])
def test_functional_forms(dev, monkeypatch, case):
    from sonicmoe.functional import moe_TC_softmax_topk_layer, switch_loss

    T, H, I, E, K = 300, 256, 128, 16, 4
    moe, x, dy = _module(T, H, I, E, K, "swiglu", False, torch.bfloat16, dev)
    parts = [p.detach() for p in moe.parameters()]
    if case == "weights strided":  # every other row of wider matrices
        parts[1:] = [torch.stack([p, p], 2).flatten(1, 2)[:, ::2] for p in parts[1:]]
    if case == "x strided":
        x = torch.stack([x, x], 1).flatten(0, 1)[::2]
    if case == "router misaligned":  # (not for the kernel that adds its share of dx)
        parts[0] = torch.cat([parts[0].new_zeros(4), parts[0].flatten()])[4:].view(E, H)
    if case == "dout strided":
        dy = dy.t().contiguous().t()
    dl = (torch.randn(E, T, device=dev) * 0.01).bfloat16()

    def step():
        xx = x.detach().requires_grad_(case != "x frozen")
        ps = [p.detach().requires_grad_(case != "router frozen" or i > 0) for i, p in enumerate(parts)]
        ins = [t for t in [xx, *ps] if t.requires_grad]

        def forward():
            return moe_TC_softmax_topk_layer(xx, ps[0], ps[1].permute(1, 2, 0), None, ps[2].permute(1, 2, 0), None, K,
                                             torch.cuda.current_stream().cuda_stream)

        if case == "hooks":
            with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.to(dev)):
                o, logits, freq = forward()
        else:
            o, logits, freq = forward()
        outs, grads = [o], [dy]
        if case == "loss only":
            outs, grads = [switch_loss(logits, freq)], [torch.tensor(2.0, device=dev)]
        elif case == "outputs changed":
            logits.mul_(2)
            freq.add_(1)
            outs.append(logits)
            grads.append(dl.t().contiguous())
        elif case.startswith("logits"):
            outs.append(logits)
            grads.append(dl.t() if case == "logits transposed" else dl.t().contiguous())
        got = torch.autograd.grad(outs, ins, grad_outputs=grads, retain_graph=case == "twice")
        again = torch.autograd.grad(outs, ins, grad_outputs=grads) if case == "twice" else ()
        return [o.detach(), logits.detach(), freq, *got, *again]

    calls = _both(monkeypatch, step)
    assert calls[0] == ("forward", True)
    assert all(done == (case != "logits transposed") for name, done in calls[1:]) and len(calls) == 2 + (case == "twice")


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(20000, 128, 64, 1024, 1), (20000, 128, 64, 1000, 2), (2000, 1024, 64, 16, 8)])
def test_memory_of_a_step(dev, monkeypatch, shape):
    """What the one call holds longer than the operators is counted: the rows of both GEMMs, and the logits."""
    T, H, I, E, K = shape
    moe, x, dy = _module(*shape, "swiglu", False, torch.bfloat16, dev)
    xx = x.clone().requires_grad_()
    peaks = []

    def step():
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        out, aux = moe(xx)
        grads = torch.autograd.grad([out, aux], [xx, *moe.parameters()], grad_outputs=[dy, torch.tensor(0.3, device=dev)])
        peaks.append(torch.cuda.max_memory_allocated() - before)
        return [out.detach(), aux.detach(), *grads]

    step()  # (workspaces that libraries keep)
    peaks.clear()
    _both(monkeypatch, step)
    # (sizes are rounded up to 512 bytes each, large ones to 2 MiB)
    assert peaks[0] - peaks[1] <= (T * K * (H + I) + T * E) * 2 + (16 << 20), peaks


@pytest.mark.gpu
def test_module_gradient_of_one_output(dev, monkeypatch):
    moe, x, dy = _module(200, 256, 128, 16, 4, "swiglu", False, torch.bfloat16, dev)

    def step():
        out = []
        for which in (0, 1):
            xx = x.clone().requires_grad_()
            got = moe(xx)[which]
            out += torch.autograd.grad(got, [xx, *moe.parameters()], grad_outputs=dy if which == 0 else None)
        return out

    _both(monkeypatch, step)


@pytest.mark.gpu
@pytest.mark.parametrize("observer", ["nobody", "profiler", "flop counter", "implementation"])
@pytest.mark.parametrize("act, bias", [("swiglu", False), ("gelu", True)])
def test_recomputed_while_somebody_looks_on(dev, observer, act, bias):
    """A checkpoint compares what a forward pass keeps with what its recomputation does; who looks on may have come since."""
    from contextlib import ExitStack

    from torch.utils.checkpoint import checkpoint
    from torch.utils.flop_counter import FlopCounterMode

    moe, x, dy = _module(300, 256, 128, 24, 4, act, bias, torch.bfloat16, dev)
    called = []

    def loss(own):
        with torch.no_grad():
            called.append(True)
            from sonicmoe.functional.forward import _switch_loss_fwd

            _switch_loss_fwd.body(*own)

    def step(observer):
        xx = x.clone().requires_grad_()
        out, aux = checkpoint(moe, xx, use_reentrant=False)
        with ExitStack() as scope:
            if observer == "profiler":
                profile = scope.enter_context(torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]))
            elif observer == "flop counter":
                scope.enter_context(FlopCounterMode(display=False))
            elif observer == "implementation":
                scope.enter_context(torch.library._scoped_library("sonicmoe", "IMPL")).impl(
                    "_switch_loss_fwd", lambda *own: loss(own), "CUDA")
            moe.zero_grad()  # (the flop counter's hooks do not run under autograd.grad)
            torch.autograd.backward([out, aux], [dy, torch.tensor(0.3, device=dev)])
        if observer == "profiler":
            rows = {e.key for e in profile.key_averages()}
            assert {"sonicmoe::_routing_metadata", "sonicmoe::_up_projection_forward", "sonicmoe::_switch_loss_fwd"} <= rows
        return [out.detach(), aux.detach(), xx.grad, *[p.grad.clone() for p in moe.parameters()]]

    for i, (a, b) in enumerate(zip(step("nobody"), step(observer))):
        if (i, observer) == (2, "flop counter"):  # dx: a mode sees the addition onto it, a second rounding of half an eps
            assert (a - b).float().norm() <= 1.5 * torch.finfo(a.dtype).eps * a.float().norm()
        else:
            assert torch.equal(a, b)
    assert bool(called) == (observer == "implementation")


@pytest.mark.gpu
def test_what_is_left_to_the_operators(dev, monkeypatch):
    """Profilers, autocast, another stream, forward-mode derivatives, odd sizes: as operator by operator, errors included."""
    from sonicmoe.functional import layer_call, moe_TC_softmax_topk_layer

    moe, x, _ = _module(64, 128, 64, 8, 2, "swiglu", False, torch.bfloat16, dev)
    real = layer_call.forward
    done = []
    monkeypatch.setattr(layer_call, "forward", lambda *a: (r := real(*a), done.append(r is not None))[0])
    with torch.no_grad():
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as profile:
            moe(x)
        assert any("_up_projection_forward" in e.key for e in profile.key_averages()) and not done
        with torch.autocast("cuda", dtype=torch.bfloat16):
            moe(x)
        assert not done
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side), pytest.raises(RuntimeError, match="stream"):
            moe(x)
        torch.cuda.current_stream().wait_stream(side)
        w = moe.c_fc.weight[:, :, :96].contiguous()  # H = 96 is no multiple of 64: told by the operator
        with pytest.raises(RuntimeError, match="multiple of 64"):
            moe_TC_softmax_topk_layer(x[:, :96].contiguous(), moe.router.weight[:, :96].contiguous(), w.permute(1, 2, 0), None,
                                      moe.c_proj.weight[:, :96].contiguous().permute(1, 2, 0), None, 2, moe.stream_id)
        assert not any(done)


@pytest.mark.gpu
def test_under_capture(dev):
    moe, x, _ = _module(16, 256, 128, 16, 4, "swiglu", False, torch.bfloat16, dev)
    moe.eval()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.no_grad():
        moe.stream_id = side.cuda_stream
        moe(x)
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            out, aux = moe(x)
    torch.cuda.current_stream().wait_stream(side)
    moe.stream_id = torch.cuda.current_stream().cuda_stream
    for seed in range(3):
        x.copy_(torch.randn(x.shape, device=dev, generator=torch.Generator(dev).manual_seed(seed)))
        graph.replay()
        torch.cuda.synchronize()
        with torch.no_grad():
            want, want_aux = moe(x)
        assert torch.equal(out, want) and torch.equal(aux, want_aux)
