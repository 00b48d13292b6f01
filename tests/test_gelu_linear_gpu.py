"""GELU(x W^T + b) of a wide layer (m2d_wide_linear_fwd beyond 512 positions: the tiled kernel) against float64."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

# positions, inputs, outputs, bias: the fewest the kernel takes, tiles of 128 positions that end inside a wave and between
# two, inputs that are padded to 256 or 320, one step of outputs and several slices of them, more workgroups than fit
CASES = [(513, 32, 64, True), (544, 96, 192, False), (640, 256, 64, True), (1000, 288, 1152, True), (2049, 320, 1280, False),
         (9001, 320, 1280, True), (70001, 64, 320, True)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_against_float64(case):
    from mamba2d_amd import cabi
    P, K, N, with_bias = case
    print(f"\ncase gelu_linear {case}", flush=True)
    g = torch.Generator().manual_seed(P)
    x = torch.randn(P, K, generator=g).bfloat16().cuda()
    w = (2 * torch.randn(N, K, generator=g) / K ** 0.5).bfloat16().cuda()
    b = torch.randn(N, generator=g).bfloat16().cuda() if with_bias else None
    y = cabi.wide_linear_fwd(x, w, b, gelu=True)
    pre = x.double() @ w.double().t() + (b.double() if with_bias else 0)
    want = F.gelu(pre)
    # the layer's output is rounded to bf16 (8 significant bits: half a unit in the last place is up to 2^-8 of a value; times
    # the activation's slope of at most 1.13), then the result (another 2^-8 of it, and of what the first rounding moved it
    # by: the 1 % on top); sums of K products in fp32 and the activation's 4e-7 add less than 1e-5 of the largest values met
    bound = 2.0 ** -8 * (1.13 * pre.abs() + want.abs()) * 1.01 + 1e-5 * pre.abs().max()
    assert ((y.double() - want).abs() <= bound).all()
    assert torch.equal(y, cabi.wide_linear_fwd(x, w, b, gelu=True))


def test_infinite_and_undefined_values_pass_through():
    from mamba2d_amd import cabi
    print("\ncase gelu_linear inf nan", flush=True)
    x = torch.zeros(600, 64, dtype=torch.bfloat16, device="cuda")
    x[3, 5], x[599, 0] = float("inf"), float("nan")
    w = torch.ones(64, 64, dtype=torch.bfloat16, device="cuda")
    y = cabi.wide_linear_fwd(x, w, None, gelu=True).float()
    assert torch.isinf(y[3]).all() and torch.isnan(y[599]).all() and (y[:3] == 0).all() and (y[4:599] == 0).all()


@pytest.mark.parametrize("case", [(150001, 64, 64, True), (98304, 32, 128, False), (98305, 288, 64, True), (49152, 320, 128, True)],
                         ids=lambda c: "x".join(map(str, c)))
def test_more_tiles_than_fit(case):
    """Few outputs and many positions: more tiles than the device holds workgroups, in one slice and in two."""
    test_against_float64(case)


@pytest.mark.parametrize("case", [(19700, 96, 320, True), (31999, 320, 448, True), (12700, 288, 576, False)], ids=lambda c: "x".join(map(str, c)))
def test_slices_of_unequal_length(case):
    """5, 7 and 9 steps of 64 outputs in 3, 2 and 5 slices, with tiles whose slices are on two XCDs."""
    test_against_float64(case)
