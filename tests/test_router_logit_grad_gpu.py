"""Gradient of the router logits in one pass, and the sum of the token chunks of the router's weight gradient."""

import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0**-7, torch.float16: 2.0**-10, torch.float32: 2.0**-23}  # spacing of the values at 1 (8, 11, 24 bits)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("outside", ["none", "dense", "padded rows", "odd offset"])
@pytest.mark.parametrize("T,E,K", [(1, 8, 2), (257, 128, 8), (33, 100, 5), (19, 2056, 4), (5, 4096, 16), (700, 3, 3)])
def test_router_logit_grad(dev, T, E, K, outside, dtype):
    from sonicmoe.functional import backward as bwd

    g = torch.Generator().manual_seed(T * E + K)
    idx = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(T)]).to(torch.int32).to(dev)
    scores = torch.rand(T, K, generator=g).softmax(1).to(dev)
    ds = torch.randn(T, K, generator=g).to(dev)
    out_grad = None
    if outside != "none":
        pad, lead = {"dense": (0, 0), "padded rows": (16, 0), "odd offset": (3, 1)}[outside]
        out_grad = torch.randn(T, E + pad, generator=g).to(dtype).to(dev)[:, lead : lead + E]
    dlogits = torch.full((T, E), 7.0, dtype=dtype, device=dev)
    bwd._router_logit_grad(dlogits, out_grad, ds, scores, idx)
    ref = torch.zeros(T, E, dtype=torch.float64, device=dev) if out_grad is None else out_grad.double()
    s, d = scores.double(), ds.double()
    add = s * (d - (s * d).sum(1, keepdim=True))
    ref = ref.scatter_add(1, idx.long(), add)
    # one rounding to the stored type, and fp32 sums of K products: (K + 3) roundings of at most |s| |ds| each
    bound = EPS[dtype] * ref.abs() / 2 + (K + 3) * 2.0**-24 * (d.abs().sum(1, keepdim=True) + ref.abs()) + 1e-7
    assert ((dlogits.double() - ref).abs() <= bound).all()
    if out_grad is not None:  # what no expert was picked for passes through
        picked = torch.zeros(T, E, dtype=torch.bool, device=dev).scatter(1, idx.long(), True)
        assert torch.equal(dlogits[~picked], out_grad[~picked])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("chunks,E,H", [(1, 8, 8), (3, 8, 264), (4, 16, 128), (64, 128, 768)])
def test_sum_chunks(dev, chunks, E, H, dtype):
    from sonicmoe.functional import backward as bwd

    partial = torch.randn(chunks, E, H, generator=torch.Generator().manual_seed(chunks)).to(dtype).to(dev)
    out = torch.full((E, H), 7.0, dtype=dtype, device=dev)
    bwd._sum_chunks(partial, out)
    ref = partial.double().sum(0)
    bound = EPS[dtype] * ref.abs() / 2 + chunks * 2.0**-24 * partial.double().abs().sum(0) + 1e-7
    assert ((out.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gradient_of_fp32_router_weights(dev, dtype):
    """fp32 router weights beside 16-bit logits (autocast): the chunks' sum is not rounded to 16 bits on its way."""
    from sonicmoe.functional import _router_wgrad
    from sonicmoe.functional.backward import _router_weight_grad, router_weight_grad_chunks

    T, E, H = 1500, 16, 264
    g = torch.Generator().manual_seed(9)
    dlogits, x = torch.randn(T, E, generator=g).to(dtype).to(dev), torch.randn(T, H, generator=g).to(dtype).to(dev)
    dw = _router_wgrad(dlogits, x, torch.empty(E, H, device=dev))
    partial = torch.empty(router_weight_grad_chunks(T, E, H), E, H, dtype=dtype, device=dev)
    assert partial.size(0) > 1
    _router_weight_grad(dlogits, x, partial)
    assert dw.dtype == torch.float32
    assert ((dw.double() - partial.double().sum(0)).abs() <= partial.size(0) * 2.0**-24 * partial.double().abs().sum(0)).all()
    assert not torch.equal(dw, dw.to(dtype).float())  # more than 16 bits are there


@pytest.fixture
def layer_grads(dev):
    """Gradients of a small layer for a gradient of its output and one of its router logits."""
    from sonicmoe import MoE
    from sonicmoe.enums import ActivationType
    from sonicmoe.functional import moe_TC_softmax_topk_layer

    torch.manual_seed(3)
    moe = MoE(16, 2, 128, 64, ActivationType.SWIGLU, False, 0.02).to(device=dev, dtype=torch.bfloat16)
    x = torch.randn(64, 128, device=dev).to(torch.bfloat16)

    def grads(grad, dout=torch.ones_like):
        xi = x.clone().requires_grad_()
        out, logits, _ = moe_TC_softmax_topk_layer(xi, moe.router.weight, moe.c_fc.weight.permute(1, 2, 0), None,
                                                   moe.c_proj.weight.permute(1, 2, 0), None, 2,
                                                   torch.cuda.current_stream().cuda_stream)
        return torch.autograd.grad([out, logits], [xi, moe.router.weight], [dout(out), grad])

    return grads


def test_gradient_from_outside_in_any_layout(dev, layer_grads):
    """The gradient that reaches router_logits may be expanded, transposed or narrowed."""
    base = torch.randn(16, 64, device=dev).to(torch.bfloat16)
    row = torch.randn(16, device=dev).to(torch.bfloat16)
    for grad in (base.t(), row.expand(64, 16)):
        for a, b in zip(layer_grads(grad), layer_grads(grad.contiguous().clone())):
            assert torch.equal(a, b)


def test_zero_gradients_without_memory(dev, layer_grads):
    zero = torch._efficientzerotensor((64, 16), dtype=torch.bfloat16, device=dev)
    for a, b in zip(layer_grads(zero), layer_grads(torch.zeros(64, 16, dtype=torch.bfloat16, device=dev))):
        assert torch.equal(a, b)
    for a in layer_grads(zero, lambda out: torch._efficientzerotensor(out.shape, dtype=out.dtype, device=dev)):
        assert not a.any()


def test_sparse_gradient_from_outside(dev, layer_grads):
    """A sparse gradient (an embedding lookup on the logits, say) counts as the dense one."""
    rows = torch.tensor([5, 9, 5], device=dev)
    grad = torch.sparse_coo_tensor(rows[None], torch.randn(3, 16, device=dev).to(torch.bfloat16), (64, 16))
    dense = layer_grads(grad.to_dense())
    for a, b in zip(layer_grads(grad), dense):
        assert torch.equal(a, b)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]):  # through the dispatcher
        for a, b in zip(layer_grads(grad), dense):
            assert torch.equal(a, b)
