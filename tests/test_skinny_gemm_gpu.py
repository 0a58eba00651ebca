"""Forward grouped GEMM for few token rows per expert: block borders of the rows, contraction lengths that leave
wavefronts without pieces or with a remainder, more experts than rows, and every epilogue, against the oracle."""

import pytest
import torch

from helpers import rel_l2
from oracle import moe_math as M

pytestmark = pytest.mark.gpu

# one rounding of the result to 8 (bf16) resp. 11 (fp16) significand bits: 2^-9 / sqrt(3) resp. 2^-12 / sqrt(3) in the
# 2-norm, and y1 is the oracle's y1 rounded from a z of fp32 sums; twice that
TOL = {torch.bfloat16: 2.3e-3, torch.float16: 2.9e-4}

COUNTS = [
    [1],
    [0, 15, 0, 16, 17, 0],                     # both fragment heights
    [31, 32, 33, 0, 1, 2, 3, 64, 65],          # second and third blocks of an expert
    [0] * 40 + [1] + [0] * 300 + [1, 2],       # fewer rows than experts, beyond the first 256 of them
    [16] * 63 + [0] + [40],                    # as many first blocks as experts, and an overflow block
    [1] * 200 + [70] + [0] * 60 + [35],        # overflow blocks of experts in different groups of 256
]


def _ops():
    import sonicmoe  # noqa: F401
    from sonicmoe.functional import forward

    return forward


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("H,I", [(64, 64), (448, 192), (2112, 320)])
@pytest.mark.parametrize("counts", COUNTS, ids=[f"E{len(c)}rows{sum(c)}" for c in COUNTS])
def test_rows_and_contractions(dev, tuning, counts, H, I, dtype):
    tuning("gemm_skinny_rows", 1 << 20)
    fwd = _ops()
    E, TK, T = len(counts), sum(counts), 50
    g = torch.Generator().manual_seed(TK + H)
    w1 = (torch.randn(E, 2 * I, H, generator=g) * H**-0.5).to(dtype).to(dev)
    w2 = (torch.randn(E, H, I, generator=g) * I**-0.5).to(dtype).to(dev)
    x = torch.randn(T, H, generator=g).to(dtype).to(dev)
    gidx = torch.randint(T, (TK,), generator=g, dtype=torch.int32).to(dev)
    off = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(dev)
    stream = torch.cuda.current_stream().cuda_stream
    guard = 5.0  # rows behind the outputs stay as they are
    z, y1, y2 = (torch.full((TK + 40, n), guard, dtype=dtype, device=dev) for n in (2 * I, I, H))
    fwd._up_projection_forward(x, w1.permute(1, 2, 0), z[:TK], y1[:TK], None, off, None, gidx, stream, "swiglu", True, False)
    z_ref, y1_ref = M.up_projection_forward(x, w1, off, gidx)
    assert rel_l2(z[:TK], z_ref) < TOL[dtype]
    assert rel_l2(y1[:TK], y1_ref) < TOL[dtype]
    fwd._down_projection_forward(w2.permute(1, 2, 0), y1[:TK], y2[:TK], None, off, None, gidx, stream)
    assert rel_l2(y2[:TK], M.down_projection_forward(y1[:TK], w2, off)) < TOL[dtype]
    for t in (z, y1, y2):
        assert (t[TK:] == guard).all()


@pytest.mark.parametrize("H,I,E,rows,skinny", [
    (512, 256, 8, 128, (True, True)), (512, 256, 8, 129, (False, False)),  # 16 rows per expert
    # matrices that fill the chip: by the number of rows, sooner where the contraction is long
    (4096, 256, 256, 512, (True, True)), (4096, 256, 256, 513, (False, True)),
    (4096, 256, 256, 2048, (False, True)), (4096, 256, 256, 2049, (False, False)),
])
def test_where_the_line_lies(dev, monkeypatch, H, I, E, rows, skinny):
    """Only the other kernels write (a tile map) into the workspace."""
    fwd = _ops()
    off = (torch.arange(E + 1, device=dev) * rows // E).to(torch.int32)
    gidx = torch.zeros(rows, dtype=torch.int32, device=dev)
    x, y1, y2 = (torch.zeros(n, c, dtype=torch.bfloat16, device=dev) for n, c in ((1, H), (rows, I), (rows, H)))
    w1, w2 = (torch.zeros(E, *s, dtype=torch.bfloat16, device=dev).permute(1, 2, 0) for s in ((2 * I, H), (H, I)))
    stream = torch.cuda.current_stream().cuda_stream
    make, workspaces = fwd._gemm_workspace, []
    monkeypatch.setattr(fwd, "_gemm_workspace", lambda *a: workspaces.append(make(*a).fill_(0xEE)) or workspaces[-1])
    fwd._up_projection_forward(x, w1, None, y1, None, off, None, gidx, stream, "swiglu", True, True)
    fwd._down_projection_forward(w2, y1, y2, None, off, None, gidx, stream)
    assert tuple(w.eq(0xEE).all().item() for w in workspaces) == skinny


@pytest.mark.parametrize("act", ["swiglu", "geglu", "reglu", "relu_sq", "relu", "gelu", "silu"])
def test_epilogues_against_the_tile_streams(dev, tuning, act):
    """Every activation with biases, and z not stored: the same values as the other kernel of the operator up to the order
    of the fp32 sums (which moves a result across a bf16 rounding border here and there)."""
    from sonicmoe.enums import ActivationType, is_glu

    fwd = _ops()
    glu = is_glu(ActivationType(act))
    counts, H, I, T = [3, 0, 40, 17, 8, 1], 320, 128, 30
    E, TK, N = len(counts), sum(counts), 2 * I if glu else I
    g = torch.Generator().manual_seed(5)
    w1 = (torch.randn(E, N, H + 64, generator=g) * H**-0.5).to(torch.bfloat16).to(dev)[:, :, :H]  # padded rows
    b1 = torch.randn(E, N, generator=g).to(torch.bfloat16).to(dev)
    w2 = (torch.randn(E, H, I, generator=g) * I**-0.5).to(torch.bfloat16).to(dev)
    b2 = torch.randn(E, H, generator=g).to(torch.bfloat16).to(dev)
    x = torch.randn(T, H, generator=g).to(torch.bfloat16).to(dev)
    gidx = torch.randint(T, (TK,), generator=g, dtype=torch.int32).to(dev)
    off = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(dev)
    stream = torch.cuda.current_stream().cuda_stream

    def run(store_z):
        z = torch.empty(TK, N, dtype=torch.bfloat16, device=dev) if store_z else None
        y1 = torch.empty(TK, I, dtype=torch.bfloat16, device=dev)
        y2 = torch.empty(TK, H, dtype=torch.bfloat16, device=dev)
        fwd._up_projection_forward(x, w1.permute(1, 2, 0), z, y1, b1, off, None, gidx, stream, act, glu, not store_z)
        fwd._down_projection_forward(w2.permute(1, 2, 0), y1, y2, b2, off, None, gidx, stream)
        return [t for t in (z, y1, y2) if t is not None]

    tuning("gemm_skinny_rows", 1 << 20)
    mine, again = run(True), run(False)
    assert torch.equal(mine[1], again[0]) and torch.equal(mine[2], again[1])
    tuning("gemm_skinny_rows", 0)
    tuning("gemm_small_tiles", 0)
    for a, b in zip(mine, run(True)):
        assert rel_l2(a, b) < 1e-3
