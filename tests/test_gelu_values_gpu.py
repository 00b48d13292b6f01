"""GELU and its slope in the kernels of a block at every finite bf16 value, through layers whose weight is the identity,
against float64: what is stored must be the correctly rounded value up to the activation's own error in fp32."""
import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def values():
    """(x, Phi(x), its slope), x every finite bf16 value in rows of 64."""
    bits = torch.arange(65536, dtype=torch.int32).to(torch.int16)
    x = bits.view(torch.bfloat16)
    x = x[x.isfinite()]
    x = torch.cat([x, x[:-x.numel() % 64]]).view(-1, 64)
    d = x.double()
    cdf = 0.5 * torch.special.erfc(-d / math.sqrt(2))
    slope = cdf + torch.where(d.abs() < 50, d * torch.exp(-d * d / 2), 0.0) / math.sqrt(2 * math.pi)
    return x, cdf, slope


def check_gelu(y, x, cdf):
    # Phi's error in fp32: 1e-7 near 1 (half a unit in the last place of 1 - q, and of q before it); for negative values 2e-5
    # of Phi itself (the exponent's rounding: half a unit at up to 22, times log 2, and the fit's 4e-6), 2e-9 where that is more
    err = torch.where(x.double() < 0, torch.clamp(2e-5 * cdf, 2e-9), torch.tensor(1e-7, dtype=torch.float64))
    low, high = (x.double() * (cdf - s * err) for s in (torch.sign(x.double()), -torch.sign(x.double())))
    y = y.cpu()
    bad = ~((y >= low.bfloat16()) & (y <= high.bfloat16()))
    assert not bad.any(), (x[bad][:8], y[bad][:8], (x.double() * cdf)[bad][:8])


def train_linear_bwd(dy, z, x, K):
    """dy times the slope at z (behind the layer) or at x (in front of it), through m2d_train_linear_bwd with W = 1."""
    from mamba2d_amd import cabi
    w = torch.eye(K, device="cuda")
    dx = torch.empty_like(dy)
    p = lambda t: ctypes.c_void_p(0 if t is None else t.data_ptr())
    rc = cabi.lib.m2d_train_linear_bwd(ctypes.c_int64(dy.shape[0]), K, K, p(dy), p(z), cabi.ACT_NONE if z is None else cabi.ACT_GELU, p(w), p(x),
                                       cabi.ACT_NONE if x is None else cabi.ACT_GELU, p(None), p(dx), p(None),
                                       ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    torch.cuda.synchronize()
    return dx


@pytest.mark.parametrize("kernel", ["linear_pre", "linear_post", "wide_few", "wide_tiled"])
def test_gelu_at_every_value(values, kernel):
    from mamba2d_amd import cabi
    print(f"\ncase gelu values {kernel}", flush=True)
    x, cdf, _ = values
    w = torch.eye(64, device="cuda").bfloat16()
    d = x.cuda()
    if kernel == "wide_few":
        y = torch.cat([cabi.wide_linear_fwd(part.contiguous(), w, None, gelu=True) for part in d.split(512)])
    elif kernel == "wide_tiled":
        y = cabi.wide_linear_fwd(d, w, None, gelu=True)
    elif kernel == "linear_pre":
        y = cabi.linear_fwd(d, w, None, pre=cabi.ACT_GELU)
    else:
        y = cabi.linear_fwd(d, w, None, post=cabi.ACT_GELU)
    check_gelu(y, x, cdf)


@pytest.mark.parametrize("where", ["pre", "post"])
def test_slope_at_every_value(values, where):
    print(f"\ncase gelu slope {where}", flush=True)
    x, _, slope = values
    d = x.cuda()
    one = torch.ones_like(d)
    got = train_linear_bwd(one, d if where == "post" else None, d if where == "pre" else None, 64).cpu()
    # 6e-8 for the last rounding near 1, as much again for the two terms before it
    low, high = (slope - 1.5e-7).bfloat16(), (slope + 1.5e-7).bfloat16()
    bad = ~((got >= low) & (got <= high))
    assert not bad.any(), (x[bad][:8], got[bad][:8], slope[bad][:8])
