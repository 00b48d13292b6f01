"""Batches that fill the device with workgroups of 16 channels: a backward whose waves share 4 channels in pairs, half of
the states each (m2d_bwd2_kernel), behind a forward whose waves sweep two channels each with a quarter of the states
per lane (m2d_fwd_split_kernel; only where rows are whole 16-byte chunks).

One band and several, the shortest strides between bands (rows are read back in the blocks right behind those that send
them), last workgroups that are partly filled, snapshots every 2 and every 4 steps.  Tolerances are those of the
scan's other oracle tests (a largest error of 1e-4 of the largest element for fp32 and 2e-2 for bf16).
"""
import numpy as np
import pytest
import torch

from oracle import scan_oracle as so

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-4, torch.bfloat16: 2e-2}

CASES = [
    # B, H, W, E
    (70, 9, 5, 40),     # one band, three blocks
    (40, 28, 26, 56),   # two bands, the shortest stride
    (40, 30, 30, 56),   # ... the longest that is sent and read back by one wave
    (40, 30, 31, 56),   # ... the shortest that is not
    (40, 28, 27, 60),   # rows of whole chunks in fp32 only
    (40, 17, 29, 61),   # in neither type; the last workgroup has 13 channels
    (36, 45, 33, 72),   # four bands; the last workgroup has 8 channels
]


@pytest.mark.parametrize("interval", [0, 4], ids=["every2", "every4"])
@pytest.mark.parametrize("flip", [False, True], ids=["tl", "br"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("shape", CASES, ids=lambda c: "x".join(map(str, c)))
def test_against_the_oracle(cscan, shape, dtype, flip, interval):
    from mamba2d_amd import cabi
    B, H, W, E = shape
    inp = so.make_inputs(B, H, W, E, 16, seed=H * W + E, dtype=dtype)
    ref = {k: v.double() for k, v in inp.items()}
    turn = (lambda t: np.flip(t, axis=(1, 2)).copy()) if flip else (lambda t: t)
    if flip:
        for k in ("x", "deltaT", "deltaL", "BT", "BL", "C", "dy"):
            ref[k] = torch.flip(ref[k], dims=(1, 2)).contiguous()
    args = [ref[k] for k in so.INPUT_NAMES]
    want = {"y": turn(cscan.forward(*args)),
            **{k: turn(v) if v.ndim == 4 else v for k, v in cscan.backward(*args, ref["dy"]).items()}}
    dev = [inp[k].cuda() for k in so.INPUT_NAMES]
    print(f"\ncase {shape} {dtype} flip={flip} interval={interval}", flush=True)
    try:
        cabi.CKPT_INTERVAL = interval
        fwd, bwd = (cabi.scan_plan(B, H, W, E, dtype, which) for which in (cabi.M2D_PASS_FWD, cabi.M2D_PASS_BWD))
        if E % (8 if dtype == torch.bfloat16 else 4) == 0:
            assert fwd.startswith("m2d_fwd_split_kernel: one stream per image") and "8 waves and 4 that stage, 16 channels each" in fwd, fwd
        else:
            assert fwd.startswith("m2d_fwd_kernel: one stream per image"), fwd
        assert bwd.startswith("m2d_bwd2_kernel" if interval == 0 else "m2d_bwd_kernel") and ("in two halves" in bwd) == (interval == 0), bwd
        y_only = cabi.scan_fwd(*dev, flip=flip)
        y, ck = cabi.scan_fwd(*dev, save_ckpt=True, flip=flip)
        kept = cabi.scan_bwd(*dev, inp["dy"].cuda(), ckpt=ck, flip=flip)
        rebuilt = cabi.scan_bwd(*dev, inp["dy"].cuda(), ckpt=None, flip=flip)
        torch.cuda.synchronize()
    finally:
        cabi.CKPT_INTERVAL = 0
    for got in (y_only, y):
        assert so.rel_err(got.float().cpu(), want["y"]) < TOL[dtype]
    for grads in (kept, rebuilt):
        for k, got in zip(so.CScan.GRADS, grads):
            e = so.rel_err(got.float().cpu(), want[k])
            assert np.isfinite(e) and e < TOL[dtype], (k, e)
