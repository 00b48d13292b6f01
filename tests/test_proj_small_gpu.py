"""GPU tests of the projections with their weights in LDS (m2d_proj_fwd, m2d_proj_bwd_parts; bf16, up to 256 channels and a rank of 16).

The products are repeated in fp64 from the operands that the kernel has: weights rounded to bf16, the low-rank inputs as bf16.
What is left is the fp32 accumulation and one rounding to bf16 of a result: half a unit in the last place, 2^-9 relative, which an
accumulation error of 1e-5 of the largest sum may carry to the next value, 2^-8.
"""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

N = 16
NAMES = ("x_proj_w", "dt_projT_w", "dt_projT_b", "dt_projL_w", "dt_projL_b")


@pytest.fixture(scope="module")
def cabi():
    from mamba2d_amd import cabi
    return cabi


def make(P, E, R, seed=0):
    g = torch.Generator().manual_seed(seed + 1000 * E + R)
    r = lambda *s: torch.rand(*s, generator=g) * 2 - 1
    w = (r(2 * R + 3 * N, E) * E ** -0.5, r(E, R) * R ** -0.5, r(E) * 3 - 2, r(E, R) * R ** -0.5, r(E) * 3 - 2)
    return torch.randn(1, P, 1, E, generator=g).bfloat16(), w


def close(got, want, scale=None):
    want = want.reshape(got.shape)
    lim = 2.0 ** -8 * want.abs() + 1e-5 * (scale if scale is not None else want.abs().max())
    bad = ((got.double() - want).abs() > lim)
    assert not bad.any(), (int(bad.sum()), float((got.double() - want).abs().max()))


def check(out, x, w):
    low, dT, dL, BT, BL, C = [t.double().cpu().flatten(0, 2) for t in out]
    x = x.double().cpu().flatten(0, 2)
    wx, wT, bT, wL, bL = [t.double() if t.dim() == 1 else t.bfloat16().double() for t in w]
    R = wT.shape[1]
    z = x @ wx.T
    close(low, z[:, :2 * R], z.abs().max())
    for k, t in enumerate((BT, BL, C)):
        close(t, z[:, 2 * R + k * N:2 * R + (k + 1) * N], z.abs().max())
    sp = torch.nn.functional.softplus
    # (an error of the sum moves a step size by less than itself; the kernel's own logarithm and exponential by 2e-6 of it and 1e-6)
    for t, wd, b, r in ((dT, wT, bT, low[:, :R]), (dL, wL, bL, low[:, R:])):
        close(t, sp(r @ wd.T + b), 1.0)


# one position, the tile's edges, a wave's edges, more tiles than a launch has workgroups; channels of every chunk count, whole and broken
# steps of 32; ranks of each number of low-rank tiles, odd ones, both sides of a whole 8-byte piece
CASES = [(1, 8, 1), (15, 16, 1), (16, 24, 2), (17, 32, 2), (63, 40, 3), (64, 64, 4), (65, 72, 5), (130, 96, 6), (200, 104, 7), (127, 128, 8),
         (129, 136, 9), (64, 160, 10), (77, 200, 13), (192, 248, 16), (333, 256, 16), (50, 64, 16), (98500, 64, 4), (98400, 16, 9), (33000, 256, 16)]


@pytest.mark.parametrize("P,E,R", CASES, ids=lambda v: str(v))
def test_products_of_the_operands(cabi, P, E, R):
    print(f"\ncase proj_small {P} {E} {R}", flush=True)
    x, w = make(P, E, R)
    xd, wd = x.cuda(), [t.cuda() for t in w]
    out = cabi.proj_fwd(xd, *wd, N)
    check(out, x, w)
    # records of fp32 B_T, B_L, C in the scan's order: the same numbers
    d = cabi.make_desc(xd, N)
    d.flags = cabi.M2D_FLAG_PACKED_BC
    low, dT, dL = torch.empty_like(out[0]), torch.empty_like(xd), torch.empty_like(xd)
    rec = torch.empty(P, 3 * N, device="cuda")
    need = cabi.lib.m2d_proj_workspace_bytes(ctypes.byref(d), R, cabi.M2D_PASS_FWD)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    cabi.check(cabi.lib.m2d_proj_fwd(ctypes.byref(d), R, *[p(t) for t in (xd, *wd, low, dT, dL, rec)], None, None, p(ws), need,
                                     ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    for a, b in ((low, out[0]), (dT, out[1]), (dL, out[2])):
        assert torch.equal(a, b)
    n = torch.arange(3 * N) % N
    slot = torch.arange(3 * N) // N * N + 4 * (n % 4) + torch.tensor([0, 2, 1, 3])[n // 4]
    assert torch.equal(rec[:, slot.cuda()], torch.cat([t.float().flatten(0, 2) for t in out[3:]], -1))


@pytest.mark.parametrize("E,R", [(64, 4), (72, 9)])
def test_values_that_are_not_finite_stay_in_their_position(cabi, E, R):
    """An infinite low-rank input of one step size must not reach the other, a NaN none of the other positions."""
    print(f"\ncase proj_small nonfinite {E} {R}", flush=True)
    x, w = make(70, E, R)
    w = [t.clone() for t in w]
    w[0][R - 1] = 0
    w[0][R - 1, 0] = 1e30      # the last low-rank input of the T step size alone overflows where x[0] is 3e38
    xb = x.clone()
    xb[0, 3, 0, 0], xb[0, 20] = 3e38, float("nan")
    wd = [t.cuda() for t in w]
    a, b = cabi.proj_fwd(x.cuda(), *wd, N), cabi.proj_fwd(xb.cuda(), *wd, N)
    torch.cuda.synchronize()
    keep = [i for i in range(70) if i not in (3, 20)]
    for u, v in zip(a, b):
        assert torch.equal(u[:, keep], v[:, keep])
    assert b[0][0, 3, 0, R - 1].isinf() and all(t[0, 20].isnan().all() for t in b)
    assert b[2][0, 3].isfinite().all()


# the same edges; channel sums of the scan in parts (0: whole arrays in bf16), whose loads go out in fours and a remainder
BWD = [(1, 8, 1, 0), (15, 16, 1, 1), (17, 32, 2, 2), (63, 40, 3, 4), (64, 64, 4, 5), (65, 72, 5, 8), (130, 96, 6, 0), (127, 128, 8, 16),
       (129, 136, 9, 3), (64, 160, 10, 0), (77, 200, 13, 7), (192, 248, 16, 4), (333, 256, 16, 9), (50, 64, 16, 0), (9000, 24, 2, 6),
       # either side of the line beyond which the widest layers go back to packed weights (256 tiles of 64 positions, where one workgroup fits a unit)
       (16384, 232, 9, 2), (16385, 232, 9, 0), (16390, 256, 16, 3), (16390, 256, 8, 3)]


@pytest.mark.parametrize("dpre", [False, True], ids=["d_delta", "dpre"])
@pytest.mark.parametrize("P,E,R,parts", BWD, ids=lambda v: str(v))
def test_input_gradient_of_the_operands(cabi, P, E, R, parts, dpre):
    """dx, against fp64 products of the operands that the kernel has.  A gradient before the second product is rounded to bf16 and may
    fall on the next value: 2^-8 of it, with the product's weights; dx itself is rounded once: 2^-8 of it."""
    print(f"\ncase proj_bwd_small {P} {E} {R} {parts} {dpre}", flush=True)
    x, w = make(P, E, R, 1)
    g = torch.Generator().manual_seed(P + E)
    bf = lambda n: torch.randn(1, P, 1, n, generator=g).bfloat16()
    low, dT, dL, ddT, ddL, dx0 = bf(2 * R), bf(E).abs(), bf(E).abs(), bf(E), bf(E), bf(E)
    if parts:
        sums = torch.randn(parts, 1, P, 1, 3 * N, generator=g)
        d3 = [sums.sum(0)[0, :, 0, k * N:(k + 1) * N].bfloat16() for k in (1, 2, 0)]      # records hold d_C, d_BT, d_BL
        given = (sums.cuda(), None, None)
    else:
        d3 = [bf(N) for _ in range(3)]
        given = tuple(t.cuda() for t in d3)
        d3 = [t[0, :, 0] for t in d3]
    dx = dx0.cuda()
    c = lambda t: t.cuda()
    gw = cabi.proj_bwd(c(x), c(low), None if dpre else c(dT), None if dpre else c(dL), c(w[0]), c(w[1]), c(w[3]), c(ddT), c(ddL), *given, dx,
                       dpre=dpre, sum_parts=parts)
    torch.cuda.synchronize()
    wx, wT, wL = [t.bfloat16().double() for t in (w[0], w[1], w[3])]
    flat = lambda t: t.double()[0, :, 0]
    pre = [flat(a) if dpre else (flat(a) * -torch.expm1(-flat(b))) for a, b in ((ddT, dT), (ddL, dL))]
    dz = torch.cat([pre[0].bfloat16().double() @ wT, pre[1].bfloat16().double() @ wL] + [t.double() for t in d3], 1)
    # d_delta times the slope is rounded to bf16 before the first product, and may fall on the next value as well
    moved = 2.0 ** -8 * torch.cat([pre[0].abs() @ wT.abs() + dz[:, :R].abs(), pre[1].abs() @ wL.abs() + dz[:, R:2 * R].abs(), dz[:, 2 * R:].abs()], 1)
    want = flat(dx0) + dz @ wx
    lim = moved @ wx.abs() + 2.0 ** -8 * want.abs() + 1e-5 * want.abs().max()
    bad = (flat(dx.cpu()) - want).abs() > lim
    assert not bad.any(), (int(bad.sum()), float((flat(dx.cpu()) - want).abs().max()))
    # the weight gradients read the dz and dpre that this kernel wrote
    for got, ref in ((gw[0], dz.T @ flat(x)), (gw[1], pre[0].T @ flat(low)[:, :R]), (gw[2], pre[0].sum(0)), (gw[3], pre[1].T @ flat(low)[:, R:]),
                     (gw[4], pre[1].sum(0))):
        assert got.shape == ref.shape and float((got.double().cpu() - ref).abs().max()) < 2e-2 * float(ref.abs().max())
