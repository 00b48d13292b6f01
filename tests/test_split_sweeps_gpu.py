"""The scan kernels that split a channel's states over the lanes (csrc/m2dsplit.h), at the edges of their schedule.

Their staging waves run ahead of the sweeping ones by blocks of 4 steps and hand rows from band to band: streams of
one and two blocks, the shortest strides between bands (26 to 32 steps, where rows come back in the blocks right behind
those that send them), both sizes of workgroup, channel counts with and without whole 16-byte chunks, both forms of
the B_T, B_L, C operands.  Tolerances are those of the scan's other oracle tests (a largest error of 1e-4 of the
largest element for fp32 and 2e-2 for bf16).
"""
import numpy as np
import pytest
import torch

from oracle import scan_oracle as so

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-4, torch.bfloat16: 2e-2}

CASES = [
    # B, H, W, E, schedule, waves
    (2, 2, 2, 4, "one stream per image", 4),      # a single block
    (2, 3, 4, 5, "one stream per image", 4),      # two blocks
    (3, 9, 5, 9, "one stream per image", 4),      # one band, three workgroups, the last with one channel
    (64, 28, 26, 16, "one stream per image", 4),  # two bands, the shortest stride
    (40, 28, 27, 22, "one stream per image", 4),
    (60, 30, 30, 14, "one stream per image", 4),  # ... the longest that is sent and read back by one wave
    (60, 30, 31, 14, "one stream per image", 4),  # ... the shortest that is not
    (50, 42, 32, 20, "one stream per image", 4),
    (40, 16, 27, 40, "one stream per image", 8),
    (40, 30, 31, 41, "one stream per image", 8),
    (1, 28, 28, 12, "linked sweep", 4),           # two bands
    (1, 30, 70, 3, "linked sweep", 4),
    (1, 70, 50, 8, "linked sweep", 4),
    (3, 61, 17, 30, "linked sweep", 4),           # windows of 32 steps
    (18, 70, 50, 64, "linked sweep", 8),
    (36, 45, 40, 61, "linked sweep", 8),
]


@pytest.mark.parametrize("flip", [False, True], ids=["tl", "br"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:4])))
def test_split_states_against_the_oracle(cscan, case, dtype, flip):
    from mamba2d_amd import cabi
    B, H, W, E, schedule, waves = case
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
    print(f"\ncase {case} {dtype} flip={flip}", flush=True)
    try:
        cabi.SCHEDULE_HINT = cabi.M2D_FLAG_SPLIT_STATES
        cabi.CHECK_LINKS = True
        for which, kernel in ((cabi.M2D_PASS_FWD, "m2d_fwd_split_kernel"), (cabi.M2D_PASS_BWD, "m2d_bwd_split_kernel")):
            plan = cabi.scan_plan(B, H, W, E, dtype, which)
            assert plan.startswith(kernel) and schedule in plan and f" workgroups of {waves} waves" in plan, plan
        y_only = cabi.scan_fwd(*dev, flip=flip)
        y, ck = cabi.scan_fwd(*dev, save_ckpt=True, flip=flip)
        kept = cabi.scan_bwd(*dev, inp["dy"].cuda(), ckpt=ck, flip=flip)
        rebuilt = cabi.scan_bwd(*dev, inp["dy"].cuda(), ckpt=None, flip=flip)   # (a forward that writes snapshots and no y)
        torch.cuda.synchronize()
    finally:
        cabi.SCHEDULE_HINT = 0
        cabi.CHECK_LINKS = False
    for got in (y_only, y):
        assert so.rel_err(got.float().cpu(), want["y"]) < TOL[dtype]
    for grads in (kept, rebuilt):
        for k, got in zip(so.CScan.GRADS, grads):
            e = so.rel_err(got.float().cpu(), want[k])
            assert np.isfinite(e) and e < TOL[dtype], (k, e)
