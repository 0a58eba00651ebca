"""Grouped GEMMs on 128 x 128 tiles against the 256 x 256 tile streams: the same products in the same order, so the same
bits; the score gradient is a sum of per-wavefront partial sums over other column ranges and agrees to fp32 rounding."""

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [
    ([1], 64, 64),                                  # one row, one stage, half a tile of columns
    ([0, 127, 128, 129, 0, 255, 256, 257], 320, 192),
    ([40, 0, 300], 1472, 320),                      # 320 columns: three tiles, the table of the score gradient has four
    ([513] + [3] * 30, 192, 704),
]


@pytest.mark.parametrize("act", ["swiglu", "geglu", "relu_sq"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("counts,H,I", CASES, ids=[f"rows{sum(c[0])}H{c[1]}I{c[2]}" for c in CASES])
def test_same_as_tile_streams(dev, tuning, counts, H, I, dtype, act):
    from sonicmoe.enums import ActivationType, is_glu
    from sonicmoe.functional import backward as bwd
    from sonicmoe.functional import forward as fwd

    glu = is_glu(ActivationType(act))
    E, TK, T, N = len(counts), sum(counts), 90, 2 * I if glu else I
    g = torch.Generator().manual_seed(TK + H)

    def randn(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g) * scale).to(dtype).to(dev)

    w1, b1, w2, b2 = randn(E, N, H, scale=H**-0.5), randn(E, N), randn(E, H, I, scale=I**-0.5), randn(E, H)
    x, dout, z_in, dz_in = randn(T, H), randn(T, H), randn(TK, N), randn(TK, N)
    gidx = torch.randint(T, (TK,), generator=g, dtype=torch.int32).to(dev)
    sidx = torch.randperm(TK, generator=g).to(torch.int32).to(dev)
    scores = torch.rand(TK, generator=g).to(dev)
    off = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(dev)
    stream = torch.cuda.current_stream().cuda_stream

    def run():
        z, y1, y2, dz, dxe = (torch.full((TK, n), 5.0, dtype=dtype, device=dev) for n in (N, I, H, N, H))
        ds = torch.full((TK,), 5.0, device=dev)
        fwd._up_projection_forward(x, w1.permute(1, 2, 0), z, y1, b1, off, None, gidx, stream, act, glu, False)
        fwd._down_projection_forward(w2.permute(1, 2, 0), y1, y2, b2, off, None, gidx, stream)
        bwd._down_projection_backward(dout, z_in, w2.permute(1, 2, 0), None, dz, ds, None, None, scores, off, None, gidx,
                                      sidx, stream, glu, act)
        bwd._up_projection_backward(x, w1.permute(1, 2, 0), dxe, None, dz_in, None, off, None, gidx, sidx, glu, stream)
        return z, y1, y2, dz, dxe, ds

    tuning("gemm_skinny_rows", 0)
    tuning("gemm_small_tiles", 0)
    reference = run()
    tuning("gemm_small_tiles", 2)
    *tensors, ds = run()
    for a, b in zip(tensors, reference):
        assert torch.equal(a, b)
    # fp32 sums of I products in another order: error below I * 2^-24 of the sum of magnitudes, here far below 1e-4
    assert torch.allclose(ds, reference[-1], rtol=1e-4, atol=1e-4)
