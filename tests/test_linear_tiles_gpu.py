"""The small linear layer at the edges of its tiles: an odd number of tiles of 16 outputs, slices of the outputs, rows
that end inside a wave's 16 and inside a workgroup's 64, the largest slice that fits LDS, and the stored value before the activation."""
import ctypes

import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]

# rows, inputs, outputs
SHAPES = [(1, 32, 16), (15, 64, 48), (16, 64, 80), (17, 96, 16), (63, 128, 48), (65, 128, 144), (64, 160, 112), (49, 256, 48),
          (113, 512, 80), (129, 512, 128), (77, 64, 1008), (70000, 32, 48)]


@pytest.mark.parametrize("wdtype", [torch.float32, torch.bfloat16], ids=["w_f32", "w_bf16"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_edges_of_tiles(shape, wdtype):
    from mamba2d_amd import cabi
    P, K, N = shape
    print(f"\ncase linear {shape} {wdtype}", flush=True)
    g = torch.Generator().manual_seed(P + 3 * K + N)
    x = torch.randn(P, K, generator=g).bfloat16()
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(wdtype)
    b = torch.randn(N, generator=g).to(wdtype)
    wb = w.bfloat16().double()
    exact = x.double() @ wb.t() + b.double()
    # K products of bf16 values summed in fp32 in any order, the bias, and the result's own rounding
    slack = (K + 1) * 2.0 ** -24 * (x.double().abs() @ wb.abs().t() + b.double().abs())
    xd, wd, bd = x.cuda(), w.cuda(), b.cuda()
    got = cabi.linear_fwd(xd, wd, bd).cpu().double()
    assert ((got - exact).abs() <= 2.0 ** -8 * exact.abs() + 1.01 * slack).all()
    # with a GELU and the value before it kept: the GELU reads what is stored
    z, y = (torch.full((P + 1, N), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    cabi.check(cabi.lib.m2d_linear_keep_fwd(ctypes.c_int64(P), K, N, cabi._dtype_code(wd), cabi._ptr(xd), cabi._ptr(wd), cabi._ptr(bd), cabi.ACT_GELU,
                                            cabi._ptr(None), cabi._ptr(None), cabi._ptr(z), cabi._ptr(y), cabi._stream(xd.device)))
    z, y = z.cpu(), y.cpu()
    assert (z[P] == 7).all() and (y[P] == 7).all()
    assert torch.equal(z[:P].double(), got)
    want = torch.nn.functional.gelu(z[:P].double())
    # rounding of the result; the activation's fp32 terms lose at most a few units of a value's own last place
    assert ((y[:P].double() - want).abs() <= 2.0 ** -8 * want.abs() + 8 * 2.0 ** -23 * (1 + z[:P].double().abs())).all()
