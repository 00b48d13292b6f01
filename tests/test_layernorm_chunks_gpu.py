"""LayerNorm and the residual update in front of it at the row lengths where a lane's number of 16-byte pieces
changes, and where its last pieces lie past the row: 16 lanes a row, so 1 to 16, 17 to 32, 33 to 48 and 49 to 64 pieces."""
import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def bound(want, w, dtype):
    """Rounding of the result to its type, and the row's sums in fp32: a value that has been normalised is off by at most
    a few units of the fp32 sums' last place (32 covers the longest row here), times its weight."""
    eps = 2.0 ** -8 if dtype is torch.bfloat16 else 2.0 ** -23
    return eps * want.abs() + 32 * 2.0 ** -23 * (1 + want.abs() + w.abs().max())


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 301])
@pytest.mark.parametrize("pieces", [1, 15, 16, 17, 31, 32, 33, 40, 47, 48, 49, 63, 64])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_row_lengths(pieces, rows, dtype):
    from mamba2d_amd import cabi
    C = pieces * (4 if dtype is torch.float32 else 8)
    print(f"\ncase layernorm pieces {pieces} rows {rows} {dtype}", flush=True)
    g = torch.Generator().manual_seed(64 * rows + pieces)
    x, r, r2 = (torch.randn(rows, C, generator=g).to(dtype) for _ in range(3))
    sc = torch.rand(C, generator=g) + 0.5
    w, b = torch.rand(C, generator=g) + 0.5, torch.randn(C, generator=g)

    def norm(t):
        return torch.nn.functional.layer_norm(t.double(), (C,), w.double(), b.double(), 1e-5)

    wd, bd = w.cuda(), b.cuda()
    got = cabi.layernorm_fwd(x.cuda(), wd, bd, 1e-5).cpu()
    want = norm(x)
    assert ((got.double() - want).abs() <= bound(want, w, dtype)).all()
    for second in (None, r2):
        xo, y = cabi.scale_residual_layernorm_fwd(x.cuda(), sc.cuda(), r.cuda(), None if second is None else second.cuda(), wd, bd, 1e-5)
        xo, y = xo.cpu(), y.cpu()
        total = x.double() * sc.double() + r.double() + (0 if second is None else second.double())
        size = x.double().abs() * sc.double() + r.double().abs() + (0 if second is None else second.double().abs())
        eps = 2.0 ** -8 if dtype is torch.bfloat16 else 2.0 ** -23
        # three fp32 roundings of partial sums, then the result's own
        assert ((xo.double() - total).abs() <= eps * total.abs() + 3 * 2.0 ** -23 * size).all()
        want = norm(xo)
        assert ((y.double() - want).abs() <= bound(want, w, dtype)).all()
