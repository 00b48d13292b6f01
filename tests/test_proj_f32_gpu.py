"""Projections with fp32 products (fp32 tensors; bf16 tensors whose rows are no whole 16-byte chunks) at the edges of
their tiles: every number of low-rank tiles, ranks next to a tile's end, rows that are whole runs of 4 elements and
not, positions around a wave's 16 and 32, and enough positions for two tiles a wave.  Checked against fp64."""
import pytest
import torch

from oracle import scan_oracle as so
from tests.test_proj_gpu import N, WNAMES, make_case, reference, say

pytestmark = pytest.mark.gpu

# (B, H, W, E, R)
EDGES = [(1, 1, 1, 1, 1), (1, 3, 5, 4, 2), (1, 4, 4, 7, 3), (1, 1, 17, 17, 7), (1, 3, 21, 12, 8), (1, 13, 5, 66, 9), (2, 4, 8, 68, 15),
         (1, 1, 33, 20, 16), (1, 5, 13, 63, 17), (3, 7, 7, 100, 24), (1, 9, 9, 36, 25), (1, 10, 13, 130, 32), (1, 256, 257, 20, 2),
         (1, 300, 219, 12, 32), (2, 181, 183, 18, 9)]


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-6), (torch.bfloat16, 2e-2)], ids=["f32", "bf16"])
@pytest.mark.parametrize("shape", EDGES, ids=lambda s: "x".join(map(str, s)))
def test_fp32_products_at_the_edges(shape, dtype, tol):
    from mamba2d_amd import cabi
    say(f"\ncase proj_f32 {shape} {dtype}")
    B, H, W, E, R = shape
    _, x, w, up, _ = make_case(B, H, W, E, seed=sum(shape), dtype=dtype)
    g = torch.Generator().manual_seed(sum(shape))
    for k, s in (("x_proj_w", (2 * R + 3 * N, E)), ("dt_projT_w", (E, R)), ("dt_projL_w", (E, R))):
        w[k] = ((torch.rand(*s, generator=g) * 2 - 1) * s[1] ** -0.5).to(dtype).float()
    ref_out, ref_g = reference(x, w, up, R)
    xd, wd = x.cuda(), {k: v.cuda() for k, v in w.items()}
    low, dT, dL, BT, BL, C = cabi.proj_fwd(xd, *[wd[k] for k in WNAMES], N)
    for k, v in dict(lowrank=low, deltaT=dT, deltaL=dL, BT=BT, BL=BL, C=C).items():
        assert v.dtype == dtype and so.rel_err(v.float().cpu(), ref_out[k]) < tol, k
    dx = up["dx"].cuda()
    args = [up[k].cuda() for k in ("d_deltaT", "d_deltaL", "d_BT", "d_BL", "d_C")]
    grads = cabi.proj_bwd(xd, low, dT, dL, wd["x_proj_w"], wd["dt_projT_w"], wd["dt_projL_w"], *args, dx)
    for k, v in zip(("x",) + WNAMES, (dx, *grads)):
        assert so.rel_err(v.float().cpu(), ref_g[k]) < max(tol, 1e-5), k
