"""Infinite values in one of the two step sizes' ranks or gradients stay with it: where the ranks of both lie in one tile of
the fp32 products, the other half must not meet them (0 x infinity is NaN)."""
import pytest
import torch

from tests.test_proj_gpu import N, WNAMES, make_case, say

pytestmark = pytest.mark.gpu

INF = float("inf")


def finite(*ts):
    return all(t.isfinite().all() for t in ts)


# (E, R): one tile for both halves, a half that ends inside the first of two, three and four tiles, whole tiles
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("E,R", [(20, 2), (100, 7), (36, 9), (66, 15), (68, 16), (100, 17), (63, 25), (130, 32)])
@pytest.mark.parametrize("half", [0, 1], ids=["T", "L"])
def test_infinite_values_stay_in_their_half(half, E, R, dtype):
    from mamba2d_amd import cabi
    if dtype == torch.bfloat16 and E % 8 == 0:
        pytest.skip("bf16 rows of whole 16-byte chunks take the bf16 products")
    say(f"\ncase proj infinite {half} {E} {R} {dtype}")
    B, H, W = 1, 5, 9
    _, x, w, up, _ = make_case(B, H, W, E, seed=E + R, dtype=dtype)
    g = torch.Generator().manual_seed(R)
    for k, s in (("x_proj_w", (2 * R + 3 * N, E)), ("dt_projT_w", (E, R)), ("dt_projL_w", (E, R))):
        w[k] = ((torch.rand(*s, generator=g) * 2 - 1) * s[1] ** -0.5).to(dtype).float()
    x[..., 0] = x[..., 0].abs() + 1
    p = dict(w)
    p["x_proj_w"] = w["x_proj_w"].clone()
    p["x_proj_w"][half * R + R - 1, 0] = INF          # the last rank of one half
    run = lambda p: cabi.proj_fwd(x.cuda(), *[p[k].cuda() for k in WNAMES], N)
    low, dT, dL, BT, BL, C = run(p)
    plain = run(w)
    assert finite(BT, BL, C) and all(torch.equal(a, b) for a, b in zip((BT, BL, C), plain[3:]))
    own, other = ((dT, dL), (dL, dT))[half]
    assert torch.equal(other, plain[2 - half]) and not finite(own) and torch.equal(low[..., (1 - half) * R:(2 - half) * R], plain[0][..., (1 - half) * R:(2 - half) * R])

    # backward: one infinite gradient of one half, at one position and channel
    args = {k: up[k].cuda() for k in ("d_deltaT", "d_deltaL", "d_BT", "d_BL", "d_C")}
    name = ("d_deltaT", "d_deltaL")[half]

    def back(args):
        dx = up["dx"].cuda()
        return dx, cabi.proj_bwd(x.cuda(), *plain[:3], *[w[k].cuda() for k in ("x_proj_w", "dt_projT_w", "dt_projL_w")], *args.values(), dx)

    dx0, g0 = back(args)
    args[name] = args[name].clone()
    args[name][0, 2, 3, E - 1] = INF
    dx1, g1 = back(args)
    there = torch.zeros(B, H, W, dtype=torch.bool)
    there[0, 2, 3] = True
    assert torch.equal(dx1.cpu()[~there], dx0.cpu()[~there]) and not dx1.cpu()[there].isfinite().any()
    rows = torch.ones(2 * R + 3 * N, dtype=torch.bool)
    rows[half * R:half * R + R] = False
    assert torch.equal(g1[0].cpu()[rows], g0[0].cpu()[rows]) and not g1[0].cpu()[~rows].isfinite().any()
    for a, b in zip(g1[3 - 2 * half:5 - 2 * half], g0[3 - 2 * half:5 - 2 * half]):      # dt weights and bias of the other half
        assert torch.equal(a, b)


@pytest.mark.parametrize("E,R", [(20, 2), (36, 9), (100, 17), (68, 16)])
def test_infinite_weight_of_the_last_rank(E, R):
    """The rows of padding behind the ranks repeat the last one."""
    from mamba2d_amd import cabi
    say(f"\ncase proj infinite weight {E} {R}")
    _, x, w, up, _ = make_case(1, 4, 7, E, seed=E, dtype=torch.float32)
    g = torch.Generator().manual_seed(R)
    for k, s in (("x_proj_w", (2 * R + 3 * N, E)), ("dt_projT_w", (E, R)), ("dt_projL_w", (E, R))):
        w[k] = (torch.rand(*s, generator=g) * 2 - 1) * s[1] ** -0.5
    plain = cabi.proj_fwd(x.cuda(), *[w[k].cuda() for k in WNAMES], N)
    w["x_proj_w"][2 * R - 1, 1] = INF
    dx = up["dx"].cuda()
    cabi.proj_bwd(x.cuda(), *plain[:3], *[w[k].cuda() for k in ("x_proj_w", "dt_projT_w", "dt_projL_w")],
                  *[up[k].cuda() for k in ("d_deltaT", "d_deltaL", "d_BT", "d_BL", "d_C")], dx)
    assert dx[..., 1].isinf().all() and finite(dx[..., 0], dx[..., 2:])
