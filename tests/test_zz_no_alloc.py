"""m2d_scan_fwd_noalloc (the forward entry point whose scratch is a static device array) against
m2d_scan_fwd, through the C ABI.  Both run the same kernels on the same inputs, so the outputs must
agree bit for bit (the bar for the existing entry point itself -- 1e-4 fp32 / 2e-2 bf16 against the
oracle -- is checked here too).  Two calls in a row, the second on a smaller problem: the array keeps
the first call's contents, which must not leak into the second.  Collected last on purpose."""
import ctypes
import sys

import pytest
import torch

from oracle import scan_oracle as so



def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def one_call(cabi, cscan, B, H, W, E, dtype, seed, flip=False):
    say(f"\ncase no_alloc B={B} H={H} W={W} E={E} dtype={dtype} flip={flip} seed={seed}")
    inp = so.make_inputs(B, H, W, E, 16, seed=seed, dtype=dtype)
    a = [inp[k].cuda() for k in so.INPUT_NAMES]
    want = cabi.scan_fwd(*a, flip=flip)
    y = torch.full_like(a[0], float("nan"))
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    cabi.scan_fwd_noalloc(*a, y, flip=flip)
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() == before
    assert torch.equal(y, want), float((y.float() - want.float()).abs().max())
    ref_in = [inp[k].double() for k in so.INPUT_NAMES]
    if flip:
        ref_in = [torch.flip(t, dims=(1, 2)).contiguous() if t.dim() == 4 else t for t in ref_in]
    y_ref = torch.from_numpy(cscan.forward(*ref_in).copy())
    if flip:
        y_ref = torch.flip(y_ref, dims=(1, 2))
    e = so.rel_err(y.float().cpu(), y_ref)
    say(f"  y rel_err vs oracle {e:.3e}")
    assert e < (1e-4 if dtype == torch.float32 else 2e-2)


@pytest.mark.gpu
def test_two_calls_in_a_row_second_smaller(cscan):
    from mamba2d_amd import cabi
    # four bands back to back: uses the set-up area, the packed B/C records and the band boundary rows
    one_call(cabi, cscan, 4, 56, 56, 64, torch.bfloat16, seed=11)
    one_call(cabi, cscan, 2, 20, 9, 8, torch.float32, seed=12)
    # linked sweep (one image, five bands on workgroups of their own), then stacked images
    one_call(cabi, cscan, 1, 70, 50, 16, torch.float32, seed=13, flip=True)
    one_call(cabi, cscan, 9, 7, 7, 6, torch.bfloat16, seed=14)


def test_too_large_is_rejected_before_any_launch():
    from mamba2d_amd import cabi
    d = cabi.Desc(128, 56, 56, 64, 16, cabi.M2D_BF16, 0, 0)
    assert cabi.lib.m2d_scan_workspace_bytes(ctypes.byref(d), cabi.M2D_PASS_FWD, 0) > cabi.NOALLOC_SCRATCH_BYTES
    vp = ctypes.c_void_p
    rc = cabi.lib.m2d_scan_fwd_noalloc(ctypes.byref(d), *([vp(4096)] * 10), vp(0))
    assert rc == cabi.M2D_ERR_TOO_LARGE
    assert "M2D_NOALLOC_SCRATCH_BYTES" in cabi.status_str(rc)


# Problems whose own plan (linked sweeps of split states) needs more than the array and whose plan of whole states does not.
FIT_AS_WHOLE = [(24, 69, 123, 44, torch.bfloat16), (52, 42, 24, 144, torch.float32), (35, 627, 2, 123, torch.bfloat16), (74, 986, 20, 5, torch.bfloat16)]


@pytest.mark.parametrize("B,H,W,E,dtype", FIT_AS_WHOLE)
def test_a_problem_that_fits_with_whole_states_is_taken(B, H, W, E, dtype):
    """Host only: the output is misaligned, so that nothing is launched where there is a GPU; the check of the size comes first."""
    from mamba2d_amd import cabi
    kind = cabi.M2D_F32 if dtype == torch.float32 else cabi.M2D_BF16
    whole = cabi.Desc(B, H, W, E, 16, kind, cabi.M2D_FLAG_WHOLE_STATES, 0)
    assert cabi.lib.m2d_scan_workspace_bytes(ctypes.byref(whole), cabi.M2D_PASS_FWD, 0) <= cabi.NOALLOC_SCRATCH_BYTES
    for flags in (0, cabi.M2D_FLAG_SPLIT_STATES, cabi.M2D_FLAG_WHOLE_STATES):
        d = cabi.Desc(B, H, W, E, 16, kind, flags, 0)
        rc = cabi.lib.m2d_scan_fwd_noalloc(ctypes.byref(d), *([ctypes.c_void_p(4096)] * 9), ctypes.c_void_p(4100), ctypes.c_void_p(0))
        assert rc != cabi.M2D_ERR_TOO_LARGE, (flags, cabi.status_str(rc))


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,W,E,dtype", [FIT_AS_WHOLE[0], FIT_AS_WHOLE[1], FIT_AS_WHOLE[3]])
def test_values_of_a_problem_that_fits_with_whole_states(B, H, W, E, dtype):
    """The same sums in another order: fp32 to rounding; bf16 outputs differ by at most one rounding of the result (2^-8 of a value)
    and of the largest for sums that cancel."""
    from mamba2d_amd import cabi
    say(f"\ncase no_alloc as whole B={B} H={H} W={W} E={E} dtype={dtype}")
    inp = so.make_inputs(B, H, W, E, 16, seed=21, dtype=dtype)
    a = [inp[k].cuda() for k in so.INPUT_NAMES]
    want = cabi.scan_fwd(*a).float()
    y = torch.full_like(a[0], float("nan"))
    cabi.scan_fwd_noalloc(*a, y)
    torch.cuda.synchronize()
    assert so.rel_err(y.float().cpu(), want.cpu()) < (1e-5 if dtype == torch.float32 else 2 ** -8)
