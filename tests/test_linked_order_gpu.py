"""Linked forward whose bands, of all images, are 4 or 8 workgroups: they go out in order, not in units of neighbouring channels.  Both sides
of that rule against the oracle, with snapshots and without, and repeated bit for bit."""
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
