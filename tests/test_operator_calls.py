"""`run` calls an operator's body directly only where nothing observes the dispatcher."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensor, FakeTensorMode
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from sonicmoe import _lib
from sonicmoe._operator import operator, run

BODY_CALLS = []


@operator("_test_copy", mutates_args={"out"})
def _test_copy(x: torch.Tensor, out: torch.Tensor, scale: float) -> None:
    BODY_CALLS.append(type(x))
    out.copy_(x * scale)


@_test_copy.register_fake
def _(x, out, scale):
    return None


class Tagged(torch.Tensor):
    pass


class Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.ops = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.ops.append(str(func))
        return func(*args, **(kwargs or {}))


@pytest.fixture(autouse=True)
def _clear():
    BODY_CALLS.clear()


def test_plain_tensors_skip_the_dispatcher(monkeypatch):
    x, out = torch.randn(3), torch.zeros(3)
    with monkeypatch.context() as m:
        m.setattr(type(_test_copy), "__call__", lambda self, *args: pytest.fail("went through the dispatcher"))
        run(_test_copy, x, out, 2.0)
        assert torch.equal(out, x * 2) and BODY_CALLS == [torch.Tensor]
        with torch.no_grad():
            run(_test_copy, torch.nn.Parameter(x), out, 3.0)
        assert torch.equal(out, x * 3)


def test_dispatch_modes_see_the_operator():
    x, out = torch.randn(3), torch.zeros(3)
    with Seen() as seen:
        run(_test_copy, x, out, 2.0)
    assert any("_test_copy" in op for op in seen.ops)
    with FakeTensorMode():
        run(_test_copy, torch.empty(3), torch.empty(3), 2.0)
    assert len(BODY_CALLS) == 1  # the fake call stopped at the fake implementation


def test_function_modes_subclasses_and_tracing_take_the_operator(monkeypatch):
    taken = []
    monkeypatch.setattr(type(_test_copy), "__call__", lambda self, *args: taken.append(args))

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    x, out = torch.randn(3), torch.zeros(3)
    with Mode():
        run(_test_copy, x, out, 2.0)
    run(_test_copy, x.as_subclass(Tagged), out, 2.0)
    torch.jit.trace(lambda t: (run(_test_copy, t, out, 2.0), t + 1)[1], x, check_trace=False)
    torch.vmap(lambda t: (run(_test_copy, t, out, 2.0), t)[1])(torch.randn(2, 3))
    assert len(taken) == 4 and not BODY_CALLS


def test_profilers_see_the_operator():
    x, out = torch.randn(3), torch.zeros(3)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], record_shapes=True) as profile:
        run(_test_copy, x, out, 2.0)
    (row,) = [r for r in profile.key_averages(group_by_input_shape=True) if r.key == "sonicmoe::_test_copy"]
    assert row.count == 1 and row.input_shapes[:2] == [[3], [3]]


@pytest.mark.parametrize("how", ["Library.impl", "register_kernel"])
def test_implementations_registered_elsewhere_are_called(how):
    @operator(f"_test_{how.split('.')[0].lower()}", mutates_args={"out"})
    def op(x: torch.Tensor, out: torch.Tensor) -> None:
        out.copy_(x)

    def sevens(x, out):
        out.fill_(7.0)

    x, out = torch.ones(3), torch.zeros(3)
    run(op, x, out)
    assert torch.equal(out, x)
    if how == "Library.impl":
        with torch.library._scoped_library("sonicmoe", "IMPL") as lib:
            lib.impl(op._name, sevens, "CPU")
            run(op, x, out)
        assert out.eq(7).all()
        run(op, x, out)
        assert torch.equal(out, x)
    else:
        torch.library.register_kernel(f"sonicmoe::{op._name}", "cpu", sevens)
        run(op, x, out)
        assert out.eq(7).all()


def test_operator_inside_an_operator():
    """The softmax router is built on the plain top-K operator; who looks on sees both."""
    from sonicmoe.functional.forward import _softmax_topk_fwd

    calls = []
    logits, scores, indices = torch.randn(4, 8), torch.empty(4, 2), torch.empty(4, 2, dtype=torch.int32)
    with torch.library._scoped_library("sonicmoe", "IMPL") as lib:
        lib.impl("_topk_fwd", lambda *args: calls.append(args[1]), "CPU")
        _softmax_topk_fwd(logits, scores, indices, 8, 2)
        run(_softmax_topk_fwd, logits, scores, indices, 8, 2)
    assert calls == [2, 2]


def test_compiled_code_keeps_the_operator():
    seen = []

    def backend(gm, _inputs):
        seen.extend(str(n.target) for n in gm.graph.nodes)
        return gm.forward

    out = torch.zeros(3)
    torch.compile(lambda t, o: (run(_test_copy, t, o, 2.0), o + 1)[1], backend=backend, fullgraph=True)(torch.ones(3), out)
    assert any("_test_copy" in t for t in seen) and torch.equal(out, torch.full((3,), 2.0))


def test_meta_tensors_stop_at_the_fake_implementation():
    run(_test_copy, torch.empty(3, device="meta"), torch.empty(3, device="meta"), 2.0)
    assert not BODY_CALLS


def test_lazily_negated_views_are_resolved():
    x, out = torch.randn(3), torch.zeros(3)
    seen = []
    body = _test_copy.body
    _test_copy.body = lambda *args: seen.append(args)
    try:
        run(_test_copy, torch._neg_view(x), out, 2.0)
    finally:
        _test_copy.body = body
    assert not seen and torch.equal(out, -x * 2)


def test_zero_tensors_without_memory_are_filled():
    pointers = []

    @operator("_test_pointers", mutates_args={"out"})
    def op(x: torch.Tensor, out: torch.Tensor) -> None:
        pointers.append((_lib.ptr(x), _lib.ptr(out)))
        out.copy_(x)

    out = torch.ones(3)
    run(op, torch._efficientzerotensor((3,)), out)
    assert len(pointers) == 1 and all(pointers[0]) and not out.any()
    run(op, torch.empty(0), torch.empty(0))
    assert len(pointers) == 2
    with pytest.raises(_lib.NoMemory):
        _lib.ptr(torch._efficientzerotensor((3,)))


def test_layer_shapes_on_the_meta_device():
    from sonicmoe import MoE
    from sonicmoe.enums import ActivationType

    with torch.device("meta"):
        moe = MoE(8, 2, 128, 64, ActivationType.SWIGLU, False, 0.02).to(torch.bfloat16)
        x = torch.empty(32, 128, dtype=torch.bfloat16, requires_grad=True)
    out, aux = moe(x)
    (dx,) = torch.autograd.grad(out, [x], torch.empty_like(out))
    assert out.shape == dx.shape == (32, 128) and aux.shape == () and out.is_meta


def _on_gpus(monkeypatch, *numbers, current=0):
    """Tensors that say they are on these GPUs, taken for ordinary ones (8 tokens; 16 router rows)"""
    from sonicmoe import _operator

    monkeypatch.setattr(_operator, "_TENSORS", (FakeTensor,))
    monkeypatch.setattr(_lib, "current_gpu", lambda: current)
    with FakeTensorMode():
        return [torch.empty(rows, 128, dtype=torch.bfloat16, device=f"cuda:{n}") for rows, n in zip((8, 16), numbers)]


@pytest.mark.parametrize("gpus, current, taken", [((0, 0), 0, True), ((0, 1), 0, False), ((1, 0), 0, False), ((1, 1), 0, False),
                                                  ((1, 1), 1, True)])
def test_kernels_in_the_place_of_torch_operations_stay_on_one_gpu(monkeypatch, gpus, current, taken):
    """F.linear refuses tensors of two GPUs and runs on theirs, not on the current one."""
    from sonicmoe._operator import stands_in, unobserved
    from sonicmoe.functional.backward import _token_broadcast_backward_router
    from sonicmoe.functional.forward import _router_logits

    x, w = _on_gpus(monkeypatch, *gpus, current=current)
    assert unobserved(frozenset(), x, None, w) == taken
    assert stands_in(frozenset(), x, w) == taken
    if gpus[0] != gpus[1]:
        with pytest.raises(RuntimeError, match="one GPU"):
            _router_logits.body(x, w, x)
        with pytest.raises(RuntimeError, match="one GPU"):
            _token_broadcast_backward_router.body(x, x, x, x, w, 2)


@pytest.mark.filterwarnings("error:Accessing the data pointer")
@pytest.mark.parametrize("tracer", ["fake tensors", "aot_function", "make_fx"])
def test_tracers_keep_the_router_gemm(monkeypatch, tracer):
    """Outside torch.compile too: no address is asked for, and the trace holds the torch operation."""
    from torch._functorch.aot_autograd import aot_function
    from torch.fx.experimental.proxy_tensor import make_fx

    from types import SimpleNamespace

    from sonicmoe.functional import _dx_with_router, moe_TC_softmax_topk_layer

    def layer(x, wr, w1, w2):
        return moe_TC_softmax_topk_layer(x, wr, w1.permute(1, 2, 0), None, w2.permute(1, 2, 0), None, 2, 0)

    monkeypatch.setattr(_lib, "current_gpu", lambda: 0)
    T, H, I, E = 8, 128, 64, 16
    graphs = []
    with FakeTensorMode(), torch.no_grad():
        args = [torch.empty(s, dtype=torch.bfloat16, device="cuda:0") for s in ((T, H), (E, H), (E, 2 * I, H), (E, H, I))]
        assert not _dx_with_router(SimpleNamespace(needs_input_grad=(True,)), args[0], args[1], torch.bfloat16, 2)
        if tracer == "aot_function":
            got = aot_function(layer, fw_compiler=lambda gm, _: (graphs.append(gm), gm)[1])(*args)
        elif tracer == "make_fx":
            graphs.append(make_fx(layer)(*args))
            got = layer(*args)
        else:
            got = layer(*args)
    assert [t.shape for t in got] == [(T, H), (T, E), (E,)]
    for graph in graphs:
        called = [str(n.target) for n in graph.graph.nodes if n.op == "call_function"]
        assert "aten.mm.default" in called and not any("_router_logits" in t for t in called)


@pytest.mark.filterwarnings("ignore:Warning only once for all operators")
@pytest.mark.parametrize("name, linear, dx", [("aten::mm", False, True), ("aten::linear", False, True), ("aten::addmm_", True, False),
                                              ("aten::addmm.out", True, False), ("aten::tanh", True, True),
                                              ("sonicmoe::_token_broadcast_backward", True, False)])
def test_implementations_registered_for_what_a_kernel_stands_in_for_are_called(monkeypatch, name, linear, dx):
    from sonicmoe._operator import stands_in, unobserved
    from sonicmoe.functional import _ONE_CALL_NAMES, ROUTER_DX, layer_call
    from sonicmoe.functional.forward import ROUTER_LINEAR

    x, w = _on_gpus(monkeypatch, 0, 0)
    with torch.library._scoped_library(name.split("::")[0], "IMPL") as lib:
        lib.impl(name.split("::")[1], lambda *args, **kwargs: pytest.fail("called"), "CUDA")
        assert stands_in(ROUTER_LINEAR, x, w) == linear and stands_in(ROUTER_DX, x, w) == dx
        assert unobserved(_ONE_CALL_NAMES, x, w) == linear and unobserved(layer_call._BACKWARD_NAMES, x, w) == dx
    assert stands_in(ROUTER_LINEAR, x, w) and stands_in(ROUTER_DX, x, w)


def test_a_function_in_the_place_of_the_reduction_is_called(monkeypatch):
    from types import SimpleNamespace

    from sonicmoe import functional

    ctx = SimpleNamespace(needs_input_grad=(True,))
    monkeypatch.setattr(functional, "stands_in", lambda *args: True)
    x, w = torch.empty(8, 64, dtype=torch.bfloat16), torch.empty(16, 64, dtype=torch.bfloat16)
    assert functional._dx_with_router(ctx, x, w, x.dtype, 2)
    monkeypatch.setattr(functional, "_token_broadcast_backward", lambda *args: None)
    assert not functional._dx_with_router(ctx, x, w, x.dtype, 2)


@pytest.mark.parametrize("T, H, E, taken", [
    (0, 512, 8, False), (1, 32, 1, True), (64, 8192, 256, True), (65, 512, 17, False), (64, 4096, 1024, True),
    (64, 4096, 1025, False), (32, 4096, 2048, True), (33, 512, 2048, False), (1, 512, 2049, False), (1, 4128, 257, False),
    (2048, 4096, 16, True), (2049, 512, 16, False), (65, 4128, 16, False), (64, 500, 8, False)])
def test_sizes_of_the_router_kernel(T, H, E, taken):
    from sonicmoe.functional.forward import router_logits_takes

    x, w = (torch.empty(n, H, dtype=torch.bfloat16, device="meta") for n in (T, E))
    assert router_logits_takes(x, w) == taken


@pytest.mark.parametrize("E, K, taken", [(8, 1, True), (128, 16, True), (136, 16, False), (256, 8, True), (512, 4, True),
                                         (512, 5, False), (520, 1, False), (8, 17, False), (12, 2, False)])
def test_sizes_of_the_dx_kernel(E, K, taken):
    from sonicmoe.functional.backward import router_dx_takes

    x, w = (torch.empty(n, 128, dtype=torch.bfloat16, device="meta") for n in (8, E))
    assert router_dx_takes(x, w, x.dtype, K) == taken
