"""m2d_fwd_rows_kernel (the forward without snapshots of batches that fill the device): every number of bands side by side and of rows a
band, one round of bands and two (rows handed on through memory), odd widths, heights that end inside a band, channel groups that
are not full, several images a workgroup, both types and directions.  Values against the oracle at the tolerances of the scan's other tests,
and against the forward that keeps snapshots: the same fp32 sums in another order, in bf16 at most one rounding of a value apart."""
import numpy as np
import pytest
import torch

from oracle import scan_oracle as so

BF16, F32 = torch.bfloat16, torch.float32
TOL = {F32: 1e-4, BF16: 2e-2}
CASES = [
    # B, H, W, E, dtype, bands side by side, rows a band
    (79, 7, 2, 52, BF16, 1, 7),       # one block of columns
    (23, 11, 2, 132, BF16, 2, 6),
    (129, 17, 9, 52, F32, 2, 6),      # two rounds, the second with one band
    (90, 14, 3, 52, F32, 2, 7),
    (154, 25, 9, 64, BF16, 2, 7),     # two rounds
    (173, 16, 2, 12, F32, 2, 8),
    (136, 29, 12, 36, BF16, 2, 8),    # two rounds
    (61, 18, 2, 36, F32, 4, 6),
    (142, 38, 11, 20, BF16, 4, 6),    # two rounds
    (259, 28, 2, 4, BF16, 4, 7),      # 4 channels, two images a workgroup, the last alone
    (131, 56, 13, 20, F32, 4, 7),     # two rounds
    (144, 32, 2, 12, F32, 4, 8),
    (142, 58, 12, 20, BF16, 4, 8),    # two rounds
    (87, 43, 2, 12, BF16, 8, 6),
    (131, 50, 2, 12, F32, 8, 7),
    (91, 60, 2, 12, BF16, 8, 8),
]
# ... with rounds of bands (rows handed on through memory, from three rounds on from more than one place of it) and images that a workgroup sweeps one after the
# other, the last workgroup not full.  The blocks of a round are as many as columns ask for, or more (padded, so that a row is stored when it is read).
HANDED = [
    # B, H, W, E, dtype, bands side by side, rows a band, rounds, images a workgroup
    (132, 33, 12, 32, BF16, 2, 6, 3, 1),
    (193, 33, 9, 48, F32, 2, 6, 3, 1),      # padded by a block
    (299, 69, 2, 48, BF16, 2, 7, 5, 2),     # one block of columns in six
    (293, 65, 2, 36, F32, 2, 7, 5, 2),
    (58, 72, 2, 36, BF16, 4, 6, 3, 1),
    (172, 65, 2, 20, F32, 4, 6, 3, 1),
    (129, 103, 2, 20, BF16, 4, 7, 4, 1),
    (261, 65, 15, 12, BF16, 4, 6, 3, 2),    # not padded
    (521, 71, 2, 12, BF16, 4, 6, 3, 3),     # the last workgroup has two images of three
    (139, 85, 2, 12, BF16, 8, 6, 2, 1),     # 8 bands: a staging wave for two of them
    (176, 136, 2, 12, F32, 8, 6, 3, 1),
    (261, 83, 7, 12, BF16, 8, 6, 2, 2),
    (293, 94, 23, 4, BF16, 8, 6, 2, 2),     # not padded
    (281, 168, 2, 12, F32, 8, 7, 3, 2),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:4])))
def test_plan_names_the_rows_kernel(case):
    from mamba2d_amd import cabi
    plan = cabi.scan_plan(*case[:5], cabi.M2D_PASS_FWD)
    assert "; without snapshots m2d_fwd_rows_kernel" in plan and plan.endswith(f"of {case[5]} bands of {case[6]} rows and {128 // case[5]} channels"), plan
    for flags in (cabi.M2D_FLAG_SPLIT_STATES, cabi.M2D_FLAG_WHOLE_STATES):      # (a lane layout that the caller asks for)
        assert "rows_kernel" not in cabi.scan_plan(*case[:5], cabi.M2D_PASS_FWD, flags=flags)


@pytest.mark.parametrize("case", HANDED, ids=lambda c: "x".join(map(str, c[:4])))
def test_plan_names_rounds_and_images(case):
    from mamba2d_amd import cabi
    plan = cabi.scan_plan(*case[:5], cabi.M2D_PASS_FWD)
    B, E, slots, rows, rounds, images = case[0], case[3], *case[5:]
    groups = -(-((E + 15) // 16) // (8 // slots))
    assert plan.endswith(f"; without snapshots m2d_fwd_rows_kernel, {-(-B // images) * groups} workgroups, {images} image{'s'[:images > 1]} and {rounds} rounds each, "
                         f"of {slots} bands of {rows} rows and {128 // slots} channels"), plan


@pytest.mark.gpu
@pytest.mark.parametrize("flip", [False, True], ids=["tl", "br"])
@pytest.mark.parametrize("case", CASES + HANDED, ids=lambda c: "x".join(map(str, c[:4])))
def test_values(cscan, case, flip):
    from mamba2d_amd import cabi
    B, H, W, E, dtype = case[:5]
    print(f"\ncase {case} flip={flip}", flush=True)
    inp = so.make_inputs(B, H, W, E, 16, seed=H * W + E, dtype=dtype)
    ref = {k: v.double() for k, v in inp.items()}
    if flip:
        for k in ("x", "deltaT", "deltaL", "BT", "BL", "C"):
            ref[k] = torch.flip(ref[k], dims=(1, 2)).contiguous()
    want = cscan.forward(*[ref[k] for k in so.INPUT_NAMES])
    want = np.flip(want, axis=(1, 2)).copy() if flip else want
    dev = [inp[k].cuda() for k in so.INPUT_NAMES]
    y = cabi.scan_fwd(*dev, flip=flip)
    y_kept, _ = cabi.scan_fwd(*dev, save_ckpt=True, flip=flip)
    again = cabi.scan_fwd(*dev, flip=flip)
    torch.cuda.synchronize()
    assert so.rel_err(y.float().cpu(), want) < TOL[dtype]
    assert torch.equal(y, again)
    y, y_kept = y.float(), y_kept.float()
    assert float((y - y_kept).abs().max() / y_kept.abs().max()) < (1e-5 if dtype == F32 else 2 ** -8)


# (with packed records two of the fp32 cases run another kernel: the rows that a workgroup hands to itself fit the scratch only where a copy of B_T, B_L and C
# is reserved too)
NOT_PACKED = [(129, 17, 9, 52), (293, 65, 2, 36)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", [c for c in CASES + HANDED if c[3] >= 20 and c[1] > 10 and c[:4] not in NOT_PACKED], ids=lambda c: "x".join(map(str, c[:4])))
def test_entry_point(case):
    """The entry point's operands: packed records, raw parameters."""
    from mamba2d_amd import cabi
    from mamba2d_amd.wavefront import wavefront_scan_cuda
    assert "m2d_fwd_rows_kernel" in cabi.scan_plan(*case[:5], cabi.M2D_PASS_FWD, flags=cabi.M2D_FLAG_PACKED_BC | cabi.M2D_FLAG_RAW_PARAMS)
    B, H, W, E, dtype = case[:5]
    print(f"\ncase entry {case}", flush=True)
    R, g = max(1, E // 16), torch.Generator(device="cuda").manual_seed(7)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    p = [0.3 * r(E, 16), 0.3 * r(E, 16), r(2 * R + 48, E) / E ** 0.5, r(E, R), r(E) - 2, r(E, R), r(E) - 2, 1 + 0.1 * r(E)]
    x = r(B, H, W, E).to(dtype)
    kept = wavefront_scan_cuda(x.clone().requires_grad_(True), *p).detach().float()
    with torch.no_grad():
        alone = wavefront_scan_cuda(x, *p).float()
    assert float((alone - kept).abs().max() / kept.abs().max()) < (1e-5 if dtype == F32 else 2 ** -8)


@pytest.mark.gpu
def test_undefined_values_stay_in_their_image_and_channel():
    """A NaN and an infinity in two images of a workgroup's three, one channel each: every other image and channel is what it is without them."""
    from mamba2d_amd import cabi
    B, H, W, E = 600, 28, 6, 32
    assert "rows_kernel" in cabi.scan_plan(B, H, W, E, F32, cabi.M2D_PASS_FWD)
    inp = so.make_inputs(B, H, W, E, 16, seed=3, dtype=F32)
    dev = [inp[k].cuda() for k in so.INPUT_NAMES]
    clean = cabi.scan_fwd(*dev)
    x = dev[0].clone()
    x[1, H - 1, W - 1, 5] = float("nan")
    x[2, 0, 0, 7] = float("inf")
    y = cabi.scan_fwd(x, *dev[1:])
    same = torch.ones_like(y, dtype=torch.bool)
    same[1, H - 1, W - 1, 5] = False
    same[2, :, :, 7] = False
    assert torch.equal(y[same], clean[same])
    assert bool(y[1, H - 1, W - 1, 5].isnan()) and not bool(torch.isfinite(y[2, 0, 0, 7]))


@pytest.mark.gpu
def test_no_link_error_is_reported():
    """Where the plan of a forward that keeps snapshots is a linked sweep, this kernel leaves the workspace's error word at 0, whatever was there."""
    import ctypes

    from mamba2d_amd import cabi
    B, H, W, E, dtype = 131, 56, 13, 20, F32
    assert cabi.scan_plan(B, H, W, E, dtype, cabi.M2D_PASS_FWD).startswith(("m2d_fwd_split_kernel: linked sweep", "m2d_fwd_kernel: linked sweep"))
    print("\ncase link error word", flush=True)
    inp = so.make_inputs(B, H, W, E, 16, seed=1, dtype=dtype)
    dev = [inp[k].cuda() for k in so.INPUT_NAMES]
    d = cabi.Desc(B=B, H=H, W=W, E=E, N=16, dtype=0)
    n = cabi.lib.m2d_scan_workspace_bytes(ctypes.byref(d), cabi.M2D_PASS_FWD, 0)
    ws, y = torch.full((n,), 255, dtype=torch.uint8, device="cuda"), torch.empty_like(dev[0])
    cabi.check(cabi.lib.m2d_scan_fwd(ctypes.byref(d), *[cabi._ptr(t) for t in dev], cabi._ptr(y), None, 0, cabi._ptr(ws), n, cabi._stream(y.device)))
    flag = ctypes.c_int(7)
    cabi.check(cabi.lib.m2d_scan_link_error(ctypes.byref(d), cabi._ptr(ws), cabi._stream(y.device), ctypes.byref(flag)))
    assert flag.value == 0
