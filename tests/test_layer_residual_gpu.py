"""A linear layer and an MLP with the block's residual update in the same kernel, against the kernels one after the other: the same bits,
at the edges of tiles of rows and outputs; and what they refuse."""
import ctypes

import pytest
import torch

gpu = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]
on_gpu = lambda f: gpu[0](gpu[1](f))
WTYPES = pytest.mark.parametrize("wdtype", [torch.float32, torch.bfloat16], ids=["w_f32", "w_bf16"])

# rows, inputs, outputs: rows that end inside a wave's 16 and a workgroup's 64, more tiles than workgroups; an odd number of 16 outputs; slices
LINEAR = [(1, 32, 16), (15, 64, 48), (17, 32, 64), (63, 64, 64), (65, 128, 128), (130, 96, 80), (77, 128, 16), (49, 128, 112), (70001, 64, 64), (70000, 128, 128),
          (66000, 32, 48)]


@on_gpu
@WTYPES
@pytest.mark.parametrize("shape", LINEAR, ids=lambda s: "x".join(map(str, s)))
def test_linear_residual_gives_the_bits_of_two_kernels(shape, wdtype):
    from mamba2d_amd import cabi
    P, K, N = shape
    print(f"\ncase linear residual {shape} {wdtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(P + 3 * K + N)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, res, res2 = (r(P, k).bfloat16() for k in (K, N, N))
    res[0, 0], res2[P - 1, N - 1] = float("inf"), float("nan")
    w, b, s = (r(N, K) / K ** 0.5).to(wdtype), r(N).to(wdtype), r(N).to(wdtype)
    for act, second, bias in ((cabi.ACT_GELU, res2, b), (cabi.ACT_NONE, None, None)):
        layer = cabi.linear_fwd(x, w, bias, pre=act)
        want = cabi.scale_residual_fwd(res, s, layer, second)
        y = torch.full((P + 1, N), 7.0, dtype=torch.bfloat16, device="cuda")
        cabi.check(cabi.lib.m2d_linear_residual_fwd(P, K, N, cabi._dtype_code(w), cabi._ptr(x), cabi._ptr(w), cabi._ptr(bias), act, cabi._ptr(res), cabi._ptr(s),
                                                    cabi._ptr(second), cabi._ptr(y), cabi._stream(x.device)))
        assert (y[P] == 7).all()
        assert torch.equal(y[:P].isnan(), want.isnan()) and torch.equal(y[:P].nan_to_num(), want.nan_to_num())


@on_gpu
@WTYPES
@pytest.mark.parametrize("C", [32, 64])
@pytest.mark.parametrize("P", [1, 15, 16, 63, 65, 1000, 70001])
def test_mlp_residual_norm_gives_the_bits_of_two_kernels(P, C, wdtype):
    from mamba2d_amd import cabi
    print(f"\ncase mlp residual {P}x{C} {wdtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(P + C)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = (3 * r(P, C)).bfloat16()
    x[P // 2, 3] = float("inf")
    w1, w2 = (r(4 * C, C) / C ** 0.5).to(wdtype), (r(C, 4 * C) / (2 * C ** 0.5)).to(wdtype)
    b1, b2, lw, lb, s, nw, nb = (r(n).to(wdtype) for n in (4 * C, C, C, C, C, C, C))
    for ln, biases in (((lw, lb), (b1, b2)), ((None, None), (None, None))):
        branch = cabi.mlp_fwd(x, w1, biases[0], w2, biases[1], *ln, 1e-5)
        want = cabi.scale_residual_layernorm_fwd(x, s, branch, None, nw, nb, 1e-3)
        xo, y = (torch.full((P + 1, C), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
        cabi.check(cabi.lib.m2d_mlp_residual_layernorm_fwd(P, C, 4 * C, cabi._dtype_code(w1), cabi._ptr(x), cabi._ptr(ln[0]), cabi._ptr(ln[1]), 1e-5, cabi._ptr(w1),
                                                           cabi._ptr(biases[0]), cabi._ptr(w2), cabi._ptr(biases[1]), cabi._ptr(s), cabi._ptr(nw), cabi._ptr(nb), 1e-3,
                                                           cabi._ptr(xo), cabi._ptr(y), cabi._stream(x.device)))
        for got, two in zip((xo, y), want):
            assert (got[P] == 7).all()
            assert torch.equal(got[:P].isnan(), two.isnan()) and torch.equal(got[:P].nan_to_num(), two.nan_to_num())


@on_gpu
@WTYPES
@pytest.mark.parametrize("C", [32, 64])
@pytest.mark.parametrize("P", [1, 15, 65, 1000, 32769, 70001])
def test_mlp_that_keeps_its_hidden_values(P, C, wdtype):
    """The first layer's output in the bits of the layer's own kernel, the second's against fp64 sums of what it reads."""
    from mamba2d_amd import cabi
    H = 4 * C
    print(f"\ncase mlp keep {P}x{C} {wdtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(P + C)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = r(P, C).bfloat16()
    w1, w2, b1, b2 = ((r(*s) / n ** 0.5).to(wdtype) for s, n in (((H, C), C), ((C, H), H), ((H,), 1), ((C,), 1)))
    z, y = (torch.full((P + 1, k), 7.0, dtype=torch.bfloat16, device="cuda") for k in (H, C))
    cabi.check(cabi.lib.m2d_mlp_keep_fwd(P, C, H, cabi._dtype_code(w1), cabi._ptr(x), cabi._ptr(w1), cabi._ptr(b1), cabi._ptr(w2), cabi._ptr(b2), cabi._ptr(z),
                                         cabi._ptr(y), cabi._stream(x.device)))
    assert (z[P] == 7).all() and (y[P] == 7).all()
    assert torch.equal(z[:P], cabi.linear_fwd(x, w1, b1))
    eye = torch.eye(H, device="cuda").to(wdtype)
    h = cabi.linear_fwd(z[:P].contiguous(), eye, None, pre=cabi.ACT_GELU).double()      # GELU(z) as a layer's kernel rounds it
    wb = w2.bfloat16().double()
    want = h @ wb.t() + b2.double()
    slack = (H + 2) * 2.0 ** -24 * (h.abs() @ wb.abs().t() + b2.double().abs())      # fp32 sums of H products in any order, and the bias
    assert ((y[:P].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1.01 * slack).all()      # the result's rounding: half a unit in the last of 8 bits


@on_gpu
@WTYPES
@pytest.mark.parametrize("P", [1, 16, 127, 129, 1000, 66001])
def test_mlp_of_128_channels(P, wdtype):
    """Weights in slices, tiles of 128 rows: the updated stream against fp64 sums of the hidden activations that the layer's own kernel gives, its norm in
    the bits of the norm's kernel."""
    from mamba2d_amd import cabi
    C, H = 128, 512
    print(f"\ncase mlp residual {P}x{C} {wdtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(P)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = (3 * r(P, C)).bfloat16()
    w1, w2 = (r(H, C) / C ** 0.5).to(wdtype), (r(C, H) / H ** 0.5).to(wdtype)
    b1, b2, lw, lb, s, nw, nb = (r(n).to(wdtype) for n in (H, C, C, C, C, C, C))
    h = cabi.linear_fwd(x, w1, b1, post=cabi.ACT_GELU, ln=(lw, lb, 1e-5)).double()
    wb = w2.bfloat16().double()
    branch = h @ wb.t() + b2.double()
    slack = (H + 2) * 2.0 ** -24 * (h.abs() @ wb.abs().t() + b2.double().abs())      # fp32 sums of H products in any order, and the bias
    want = x.double() * s.double() + branch
    xo, y = (torch.full((P + 1, C), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    cabi.check(cabi.lib.m2d_mlp_residual_layernorm_fwd(P, C, H, cabi._dtype_code(w1), cabi._ptr(x), cabi._ptr(lw), cabi._ptr(lb), 1e-5, cabi._ptr(w1),
                                                       cabi._ptr(b1), cabi._ptr(w2), cabi._ptr(b2), cabi._ptr(s), cabi._ptr(nw), cabi._ptr(nb), 1e-3,
                                                       cabi._ptr(xo), cabi._ptr(y), cabi._stream(x.device)))
    assert (xo[P] == 7).all() and (y[P] == 7).all()
    # two roundings to bf16, each by half a unit in the last of 8 bits (2**-8 of the value): of the MLP's result and of the updated stream
    assert ((xo[:P].double() - want).abs() <= 1.02 * 2.0 ** -8 * (branch.abs() + want.abs()) + 2 * slack).all()
    same = cabi.scale_residual_layernorm_fwd(xo[:P].contiguous(), torch.ones_like(s), torch.zeros_like(x), None, nw, nb, 1e-3)
    assert torch.equal(same[0], xo[:P]) and torch.equal(same[1], y[:P])


def test_refusals():
    """Host checks only: nothing is launched."""
    from mamba2d_amd import cabi
    buf = (ctypes.c_char * 4096)()
    p = (ctypes.addressof(buf) + 255) // 256 * 256
    linear = lambda P=4, K=64, N=64, wd=1, pre=0, res=p, s=p, res2=None, y=p: cabi.lib.m2d_linear_residual_fwd(P, K, N, wd, p, p, p, pre, res, s, res2, y, None)
    ok, null, shape, unsupported, misaligned = 0, 1, 2, 3, 5
    assert [linear(res=None), linear(s=None), linear(y=None)] == [null] * 3
    assert [linear(K=160), linear(N=80), linear(K=128, N=144), linear(K=48), linear(N=40), linear(pre=cabi.ACT_STARRELU), linear(wd=7)] == [unsupported] * 7
    assert [linear(res=p + 8), linear(res2=p + 2), linear(s=p + 2), linear(y=p + 4)] == [misaligned] * 4
    assert linear(P=0) == shape
    mlp = lambda C=64, s=p, nw=p, xo=p, y=p: cabi.lib.m2d_mlp_residual_layernorm_fwd(4, C, 4 * C, 1, p, None, None, 0.0, p, p, p, p, s, nw, p, 0.0, xo, y, None)
    assert [mlp(s=None), mlp(nw=None), mlp(xo=None), mlp(y=None)] == [null] * 4
    assert [mlp(C=256), mlp(C=48)] == [unsupported] * 2
    keep = lambda C=64, z=p, y=p: cabi.lib.m2d_mlp_keep_fwd(4, C, 4 * C, 1, p, p, p, p, p, z, y, None)
    assert [keep(z=None), keep(y=None), keep(C=128), keep(C=48), keep(z=p + 8), keep(y=p + 8)] == [null] * 2 + [unsupported] * 2 + [misaligned] * 2
    assert [mlp(xo=p + 8), mlp(s=p + 2), mlp(y=p + 4)] == [misaligned] * 3


@on_gpu
@WTYPES
def test_mlp_of_32_channels_over_several_tiles_a_workgroup(wdtype):
    """More tiles of 64 rows than workgroups that are launched: the rows are what calls of a few tiles give for them, bit for bit."""
    from mamba2d_amd import cabi
    P, C = 64 * 2048 + 64 * 130 + 5, 32
    print(f"\ncase mlp {P}x{C} {wdtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(C)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = r(P, C).bfloat16()
    w = [(0.2 * r(*s)).to(wdtype) for s in ((4 * C, C), (4 * C,), (C, 4 * C), (C,), (C,), (C,))]
    y = cabi.mlp_fwd(x, *w)
    for at in (0, 64 * 2048 - 300, P - 64 * 131):
        part = x[at:at + 64 * 131].contiguous()
        same = torch.equal(cabi.mlp_fwd(part, *w), y[at:at + part.shape[0]])
        assert same
