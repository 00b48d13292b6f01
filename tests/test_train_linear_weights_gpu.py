"""The gradient of a linear layer's input at sizes where the staged weight is less than, one more than, and many rounds of what a
workgroup fetches at once, and where its inputs are shared out in slices."""
import ctypes

import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("shape", [(5, 16, 32), (64, 48, 96), (65, 128, 32), (130, 144, 32), (33, 256, 64), (70, 64, 256), (200, 112, 512)],
                         ids=lambda s: "x".join(map(str, s)))
def test_input_gradient(shape):
    from mamba2d_amd import cabi
    P, K, N = shape
    print(f"\ncase linear input gradient {shape}", flush=True)
    g = torch.Generator().manual_seed(P + K + N)
    dy = torch.randn(P, N, generator=g).bfloat16()
    w = torch.randn(N, K, generator=g) / N ** 0.5
    dyd, wd = dy.cuda(), w.cuda()
    dx = torch.full((P + 1, K), 7.0, dtype=torch.bfloat16, device="cuda")
    null = cabi._ptr(None)
    cabi.check(cabi.lib.m2d_train_linear_bwd(ctypes.c_int64(P), K, N, cabi._ptr(dyd), null, 0, cabi._ptr(wd), null, 0, null, cabi._ptr(dx), null,
                                             cabi._stream(dyd.device)))
    dx = dx.cpu()
    wb = w.bfloat16().double()
    want = dy.double() @ wb
    # N products of bf16 values summed in fp32 in any order, and the result's own rounding
    slack = 1.01 * N * 2.0 ** -24 * (dy.double().abs() @ wb.abs())
    assert (dx[P] == 7).all()
    assert ((dx[:P].double() - want).abs() <= 2.0 ** -8 * want.abs() + slack).all()
