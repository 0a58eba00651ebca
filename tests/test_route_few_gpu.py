"""The router GEMM of few tokens and the routing fused with it, at the borders of their parts (16 tokens, 16 experts, 16 parts of
the contraction; 64 and 128 experts per lane count, 64 tokens, 1024 picks)."""

import pytest
import torch

from test_layer_call import _both, _module

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T, H, E", [(1, 32, 1), (16, 64, 16), (17, 544, 17), (33, 1472, 48), (64, 4096, 130), (5, 8224, 3),
                                     (1000, 512, 8)])
def test_router_logits(dev, T, H, E, dtype):
    from sonicmoe._operator import run
    from sonicmoe.functional.forward import _router_logits

    g = torch.Generator().manual_seed(T + H + E)
    x, w = torch.randn(T, H, generator=g).to(dtype), (torch.randn(E, H, generator=g) * 0.05).to(dtype)
    want = x.double() @ w.double().t()
    logits = torch.full((T + 2, E), -7.0, dtype=dtype, device=dev)
    run(_router_logits, x.to(dev), w.to(dev), logits[:T])
    assert (logits[T:] == -7).all()
    # rounding of the stored value, and of H products added in fp32 in some order
    bound = torch.finfo(dtype).eps / 2 * want.abs() + H * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    assert ((logits[:T].double().cpu() - want).abs() <= bound + torch.finfo(dtype).tiny).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 64, 64, 1, 1), (64, 128, 64, 256, 16), (64, 128, 64, 257, 2), (65, 128, 64, 64, 2),
                                   (17, 4160, 64, 129, 3), (48, 128, 64, 65, 21), (49, 128, 64, 65, 21), (64, 192, 64, 64, 8)])
def test_fused_routing_is_the_operators(dev, monkeypatch, shape, dtype):
    moe, x, _ = _module(*shape, "swiglu", False, dtype, dev)
    x[1::3] = x[:1]  # equal rows, and equal logits in a row
    with torch.no_grad():
        moe.router.weight[1::4] = moe.router.weight[:1]

    def step():
        xx = x.clone().requires_grad_()
        out, aux = moe(xx)
        grads = torch.autograd.grad([out, aux], [xx, *moe.parameters()], grad_outputs=[torch.ones_like(out), torch.ones_like(aux)])
        with torch.no_grad():
            return [out.detach(), aux.detach(), *grads, *moe(x)]

    _both(monkeypatch, step)
