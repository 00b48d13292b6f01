"""The order in which the workgroups of a linked launch go out, both sides of its rules against the oracle, with snapshots and without, and repeated
bit for bit: a forward whose bands, of all images, are 4 or 8 workgroups goes out in order, one of many workgroups of 16-bit tensors in units of 2."""
import pytest
import torch

from oracle import scan_oracle as so

from .test_scan_gpu import cabi, run_case, say  # noqa: F401  (cabi is a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("shape", [(1, 60, 50, 16), (2, 45, 70, 8), (1, 74, 31, 32), (2, 130, 90, 16), (1, 60, 50, 24), (1, 60, 50, 14), (3, 45, 70, 16)],
                         ids=lambda s: "x".join(map(str, s)))
def test_against_oracle(cabi, cscan, shape, dtype):
    say(f"\ncase linked order {shape} {dtype}")
    plan = cabi.scan_plan(*shape, dtype, cabi.M2D_PASS_FWD)
    assert "linked sweep" in plan and "split" in plan and "4 channels each" in plan, plan
    run_case(cabi, cscan, *shape, dtype)
    inp = so.make_inputs(*shape, 16, seed=0, dtype=dtype)
    a = [inp[k].cuda() for k in so.INPUT_NAMES]
    y = cabi.scan_fwd(*a)
    for _ in range(3):
        assert torch.equal(cabi.scan_fwd(*a), y)


# 58 and 75 workgroups a band (the last unit a single one), two images, one; 45 and 38, which only the forward of one image takes in units of 2; 30 and 46, which are not
WIDE = [((2, 37, 20, 232), 58), ((1, 30, 50, 300), 75), ((1, 60, 120, 180), 45), ((1, 75, 150, 150), 38), ((1, 60, 90, 120), 30), ((2, 37, 50, 184), 46)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("shape,groups", WIDE, ids=lambda s: "x".join(map(str, s)) if isinstance(s, tuple) else str(s))
def test_bands_of_many_workgroups(cabi, cscan, shape, groups, dtype):
    say(f"\ncase linked order, many workgroups {shape} {dtype}")
    for passes in (cabi.M2D_PASS_FWD, cabi.M2D_PASS_BWD):
        plan = cabi.scan_plan(*shape, dtype, passes)
        assert "linked sweep" in plan and f"{groups * shape[0] * ((shape[1] + 13) // 14)} workgroups" in plan, plan
    run_case(cabi, cscan, *shape, dtype)
    inp = so.make_inputs(*shape, 16, seed=1, dtype=dtype)
    a = [inp[k].cuda() for k in so.INPUT_NAMES]
    y = cabi.scan_fwd(*a)
    assert torch.equal(cabi.scan_fwd(*a), y)
