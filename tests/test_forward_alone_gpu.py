"""Forwards that keep no snapshots and run another kernel for it than the forward of a training step: two channels per lane or the pairs
beside split states, split states beside whole ones, whole states beside the pairs.  Values against the oracle at the tolerances of the scan's other tests; the largest
(split states beside whole ones exist beyond 2 GiB of channel sums only) against the forward that keeps snapshots, the same
fp32 sums in another order."""
import numpy as np
import pytest
import torch

from oracle import scan_oracle as so

TOL = {torch.float32: 1e-4, torch.bfloat16: 2e-2}
SMALL = [
    # B, H, W, E, dtype, what runs without snapshots
    (66, 18, 15, 122, torch.bfloat16, "m2d_fwd_kernel, 132 workgroups of 64 channels"),        # rows of no whole chunks, a last workgroup of 58
    (33, 26, 6, 276, torch.bfloat16, "m2d_fwd_kernel, 165 workgroups of 64 channels"),         # a last workgroup of 20
    (249, 33, 28, 16, torch.bfloat16, "m2d_fwd_split_kernel, 249 workgroups of 16 channels"),
    (181, 12, 35, 12, torch.float32, "m2d_fwd_split_kernel, 181 workgroups of 16 channels"),   # 4 of the 16 past the end
    (228, 121, 2, 20, torch.float32, "m2d_fwd_kernel, 228 workgroups of 32 channels"),         # the pairs where snapshots are kept
]
LARGE = (12, 42, 874, 310, torch.float32, "m2d_fwd_split_kernel, 468 workgroups of 8 channels")


@pytest.mark.parametrize("case", SMALL + [LARGE], ids=lambda c: "x".join(map(str, c[:4])))
def test_plan_names_the_kernel_without_snapshots(case):
    from mamba2d_amd import cabi
    plan = cabi.scan_plan(*case[:5], cabi.M2D_PASS_FWD)
    assert plan.endswith("; without snapshots " + case[5]), plan


@pytest.mark.gpu
@pytest.mark.parametrize("flip", [False, True], ids=["tl", "br"])
@pytest.mark.parametrize("case", SMALL, ids=lambda c: "x".join(map(str, c[:4])))
def test_values_without_snapshots(cscan, case, flip):
    from mamba2d_amd import cabi
    B, H, W, E, dtype, _ = case
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
    rebuilt = cabi.scan_bwd(*dev, inp["dy"].cuda(), ckpt=None, flip=flip)      # (its own forward keeps snapshots as ever)
    y_kept, ck = cabi.scan_fwd(*dev, save_ckpt=True, flip=flip)
    kept = cabi.scan_bwd(*dev, inp["dy"].cuda(), ckpt=ck, flip=flip)
    torch.cuda.synchronize()
    for got in (y, y_kept):
        assert so.rel_err(got.float().cpu(), want) < TOL[dtype]
    for name, a, b in zip(so.CScan.GRADS, kept, rebuilt):
        assert torch.equal(a, b), name


@pytest.mark.gpu
@pytest.mark.parametrize("case", SMALL, ids=lambda c: "x".join(map(str, c[:4])))
def test_entry_point_without_snapshots(case):
    """The entry point's operands (packed records, raw parameters): the same fp32 sums in another order, in bf16 at most one rounding
    of the result apart (2^-8 of a value)."""
    from mamba2d_amd.wavefront import wavefront_scan_cuda
    B, H, W, E, dtype, _ = case
    print(f"\ncase entry {case}", flush=True)
    R, g = max(1, E // 16), torch.Generator(device="cuda").manual_seed(7)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    p = [0.3 * r(E, 16), 0.3 * r(E, 16), r(2 * R + 48, E) / E ** 0.5, r(E, R), r(E) - 2, r(E, R), r(E) - 2, 1 + 0.1 * r(E)]
    x = r(B, H, W, E).to(dtype)
    kept = wavefront_scan_cuda(x.clone().requires_grad_(True), *p).detach().float()
    with torch.no_grad():
        alone = wavefront_scan_cuda(x, *p).float()
    recomputed = wavefront_scan_cuda(x.clone().requires_grad_(True), *p, "full").detach().float()
    assert torch.equal(alone, recomputed)
    assert float((alone - kept).abs().max() / kept.abs().max()) < (1e-5 if dtype == torch.float32 else 2 ** -8)


@pytest.mark.gpu
def test_largest_without_snapshots():
    from mamba2d_amd import cabi
    B, H, W, E, dtype, _ = LARGE
    print(f"\ncase {LARGE}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(5)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    a = lambda: -torch.exp(-4 * torch.rand(E, 16, generator=g, device="cuda"))
    soft = torch.nn.functional.softplus
    dev = [r(B, H, W, E), soft(r(B, H, W, E)), soft(r(B, H, W, E)), a(), a(), r(B, H, W, 16), r(B, H, W, 16), r(B, H, W, 16), r(E)]
    y = cabi.scan_fwd(*dev)
    y_kept, _ = cabi.scan_fwd(*dev, save_ckpt=True)
    assert float((y - y_kept).abs().max() / y_kept.abs().max()) < 1e-5
