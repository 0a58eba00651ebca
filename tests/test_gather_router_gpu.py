"""The dx reduction with the router's share formed in place, at the borders of its tiles (64 tokens, 128 columns, 64 experts)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T, H, E, K", [(1, 64, 8, 1), (63, 128, 64, 2), (64, 136, 72, 3), (65, 1472, 48, 4), (130, 256, 200, 8),
                                        (129, 320, 256, 16), (200, 64, 8, 9)])
def test_gather_sum_router(dev, T, H, E, K, dtype):
    from sonicmoe._operator import run
    from sonicmoe.functional.backward import _token_broadcast_backward_router

    g = torch.Generator().manual_seed(T * H + E)
    rows = torch.randn(T * K, H, generator=g).to(dtype)
    dlogits = (torch.randn(T, E, generator=g) * 0.1).to(dtype)
    wr = torch.randn(E, H, generator=g).to(dtype)
    ridx = torch.randperm(T * K, generator=g).int()
    picked = rows.double()[ridx.long()].view(T, K, H)
    want = picked.sum(1) + dlogits.double() @ wr.double()
    dx = torch.full((T + 1, H), -7.0, dtype=dtype, device=dev)
    run(_token_broadcast_backward_router, dx[:T], rows.to(dev), ridx.to(dev), dlogits.to(dev), wr.to(dev), K)
    assert (dx[T:] == -7).all()
    # one rounding of the stored value, and of K + E terms added in fp32 in some order
    size = picked.abs().sum(1) + dlogits.double().abs() @ wr.double().abs()
    bound = torch.finfo(dtype).eps / 2 * want.abs() + (K + E) * 2.0 ** -24 * size + torch.finfo(dtype).tiny
    assert ((dx[:T].double().cpu() - want).abs() <= bound).all()


@pytest.mark.parametrize("T, takes", [(0, False), (1, True), (65535 * 64, True), (65535 * 64 + 1, False)])
def test_token_counts_the_launch_takes(dev, T, takes):
    from sonicmoe.functional.backward import router_dx_takes

    x = torch.zeros(1, 64, dtype=torch.bfloat16, device=dev).expand(T, 64)
    assert router_dx_takes(x, torch.zeros(8, 64, dtype=x.dtype, device=dev), x.dtype, 2) == takes
