"""Both gradients of a linear layer from one kernel, for every shape it is built for: fewer positions than a tile, whole tiles, one position
more, and more tiles than workgroups."""
import ctypes

import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]

SHAPES = [(64, 64, 128), (64, 256, 64), (256, 64, 64), (64, 128, 128), (128, 64, 128), (128, 128, 64), (128, 256, 32), (256, 128, 32)]   # N, K, positions of a tile
NONE, GELU, STAR = 0, 1, 2


def gelu(v):
    return v * 0.5 * torch.erfc(-v / 2 ** 0.5)


def gelu_slope(v):
    return 0.5 * torch.erfc(-v / 2 ** 0.5) + v * torch.exp(-v * v / 2) / (2 * torch.pi) ** 0.5


@pytest.mark.parametrize("acts", [(NONE, NONE), (NONE, GELU), (GELU, NONE), (NONE, STAR)], ids=["plain", "gelu_before", "gelu_behind", "star_before"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_both_gradients(shape, acts):
    from mamba2d_amd import cabi
    N, K, T = shape
    post, pre = acts
    for P in (1, T - 1, T, T + 1, 256 * T + 7):
        print(f"\ncase both gradients {shape} {acts} P={P}", flush=True)
        g = torch.Generator().manual_seed(P + 3 * K + N)
        r = lambda *s: torch.randn(*s, generator=g)
        dy, z, x, w = r(P, N).bfloat16(), r(P, N).bfloat16(), r(P, K).bfloat16(), r(N, K) / N ** 0.5
        scale, shift = torch.tensor([0.8]), torch.tensor([-0.3])
        slices = cabi.lib.m2d_train_linear_grads_parts(ctypes.c_int64(P), N, K)
        assert slices == min(256, (P + T - 1) // T)
        dev = [t.cuda() for t in (dy, z, x, w, scale, shift)]
        dx = torch.full((P + 1, K), 7.0, dtype=torch.bfloat16, device="cuda")
        part = torch.full((slices * (N * K + N) + 64,), 7.0, device="cuda")
        star = torch.full((slices + 1, 2), 7.0, device="cuda")
        ptr, null = cabi._ptr, cabi._ptr(None)
        cabi.check(cabi.lib.m2d_train_linear_grads(ctypes.c_int64(P), N, K, ptr(dev[0]), ptr(dev[1]) if post else null, post, ptr(dev[3]), ptr(dev[2]), pre,
                                                   ptr(dev[4]), ptr(dev[5]), 1, ptr(dx), ptr(part), ptr(star), cabi._stream(dx.device)))
        dx, part, star = dx.cpu(), part.cpu(), star.cpu()
        assert (dx[P] == 7).all() and (part[slices * (N * K + N):] == 7).all() and (star[slices:] == 7).all()
        part = part[:slices * (N * K + N)].view(slices, -1).double().sum(0)
        dw, db = part[:N * K].view(N, K), part[N * K:]
        go = dy.double()
        if post:
            go = (go * gelu_slope(z.double())).bfloat16().double()
        xd = x.double()
        if pre == GELU:
            xa, slope = gelu(xd).bfloat16().double(), gelu_slope(xd)
        elif pre == STAR:
            xa, slope = (0.8 * xd.clamp(min=0) ** 2 - 0.3).bfloat16().double(), 2 * 0.8 * xd.clamp(min=0)
        else:
            xa, slope = xd, torch.ones(())
        back = go @ w.bfloat16().double()
        # An activation or slope in fp32 may round to the neighbouring bf16 value: one value in a few thousand moves by 2^-8 of itself, which 2^-14 of a
        # product's size covers; N or P products summed in fp32 in any order; a result's own rounding to bf16.
        mag = go.abs() @ w.bfloat16().double().abs()
        assert ((dx[:P].double() - back * slope).abs() <= 2.0 ** -8 * (back * slope).abs() + (N * 2.0 ** -24 + (2.0 ** -8 if post else 0)) * mag * slope.abs() + 1e-6).all()
        size = go.abs().T @ xa.abs()
        loose = 2.0 ** -8 if post or pre else 0
        near = loose * (go.abs().T.amax(1, keepdim=True) * xa.abs().amax(0, keepdim=True)) * 4
        assert ((dw - go.T @ xa).abs() <= (P * 2.0 ** -24 + 2.0 ** -14 * bool(loose)) * size + near + 1e-6).all()
        assert ((db - go.sum(0)).abs() <= (P * 2.0 ** -24 + 2.0 ** -14 * bool(post)) * go.abs().sum(0) + (2.0 ** -6 * go.abs().amax(0) if post else 0) + 1e-6).all()
        if pre == STAR:
            t = xd.clamp(min=0)
            want = torch.stack([(back * t * t).sum(), back.sum()])
            terms = torch.stack([(mag * t * t).sum(), mag.sum()])
            assert ((star[:slices].double().sum(0) - want).abs() <= (N + 64) * 2.0 ** -24 * terms + 1e-5).all()


@pytest.mark.parametrize("acts", [(NONE, NONE), (NONE, GELU), (GELU, NONE), (NONE, STAR)], ids=["plain", "gelu_before", "gelu_behind", "star_before"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}")
def test_every_tile_counts(shape, acts):
    """Workgroups that take two and three tiles, the last of them of 7 rows, so that both buffers are filled again.  Operands are -1, 0 and 1,
    and an activation or slope of those is a bf16 value that is a multiple of 2^-11 and no larger than 1.1: every product is a multiple of
    2^-11, every sum stays below 2^13, and so fp32 holds them exactly in any order.  A lost, doubled or overwritten row would show."""
    from mamba2d_amd import cabi
    N, K, T = shape
    post, pre = acts
    P = 513 * T + 7
    print(f"\ncase every tile {shape} {acts} P={P}", flush=True)
    g = torch.Generator().manual_seed(K + N)
    r = lambda *s: torch.randint(-1, 2, s, generator=g).bfloat16()
    dy, z, x, w = r(P, N), r(P, N), r(P, K), r(N, K).float()
    scale, shift = torch.tensor([0.5]), torch.tensor([-0.25])
    dev = [t.cuda() for t in (dy, z, x, w, scale, shift)]
    slices = cabi.lib.m2d_train_linear_grads_parts(ctypes.c_int64(P), N, K)
    dx = torch.empty(P, K, dtype=torch.bfloat16, device="cuda")
    part, star = torch.empty(slices, N * K + N, device="cuda"), torch.empty(slices, 2, device="cuda")
    ptr, null = cabi._ptr, cabi._ptr(None)
    cabi.check(cabi.lib.m2d_train_linear_grads(ctypes.c_int64(P), N, K, ptr(dev[0]), ptr(dev[1]) if post else null, post, ptr(dev[3]), ptr(dev[2]), pre,
                                               ptr(dev[4]), ptr(dev[5]), 1, ptr(dx), ptr(part), ptr(star), cabi._stream(dx.device)))
    part, star, dx = part.double().sum(0).cpu(), star.double().sum(0).cpu(), dx.cpu()
    go, xd = dy.double(), x.double()
    if post:
        go = (go * gelu_slope(z.double())).bfloat16().double()
    t = xd.clamp(min=0)
    xa = gelu(xd).bfloat16().double() if pre == GELU else 0.5 * t * t - 0.25 if pre == STAR else xd
    back = go @ w.double()
    assert torch.equal(part[:N * K].view(N, K), go.T @ xa)
    assert torch.equal(part[N * K:], go.sum(0))
    if pre == STAR:
        assert torch.equal(star, torch.stack([(back * t * t).sum(), back.sum()]))
    if pre != GELU:      # (its slope is no bf16 value)
        assert torch.equal(dx, (back * t if pre == STAR else back).bfloat16())
