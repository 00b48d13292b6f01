"""Gradients that are differentiated again (create_graph=True): the scan and its projections have no second derivative and
say so with a warning, as dispatched operators do; everything around them in a block has one."""
import warnings

import pytest
import torch

from tests.test_entry_gpu import problem

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def twice(f, leaves, dy):
    """y, its gradients, the gradients of their squared sum, and the warnings of the second pass."""
    y = f()
    first = torch.autograd.grad(y, leaves, dy, create_graph=True)
    plain = [t.detach().clone() for t in first]
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        second = torch.autograd.grad(sum(t.float().square().sum() for t in first), leaves, allow_unused=True)
        torch.cuda.synchronize()
    return y.detach(), plain, [t.requires_grad for t in first], second, [str(w.message) for w in seen if "autograd kernel" in str(w.message)]


@pytest.mark.parametrize("recomp", ["partial", "full"])
@pytest.mark.parametrize("params", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_entry_point_warns(recomp, params):
    from mamba2d_amd import wavefront as wf
    say(f"\ncase twice entry {recomp} {params}")
    x, p, dy = problem(2, 7, 9, 24, torch.bfloat16, params)
    leaves = [t.detach().requires_grad_(True) for t in (x, *p)]
    got = twice(lambda: wf.wavefront_scan_cuda(*leaves, recomp), leaves, dy.to(x.dtype))
    want = twice(lambda: wf.wf_cuda_fn_proj.apply(*leaves, recomp == "full", False, True), leaves, dy.to(x.dtype))
    once = torch.autograd.grad(wf.wavefront_scan_cuda(*leaves, recomp), leaves, dy.to(x.dtype))
    assert torch.equal(got[0], want[0]) and all(torch.equal(a, b) and torch.equal(a, c) for a, b, c in zip(got[1], want[1], once))
    assert got[2] == want[2] and all(got[2]) and got[4] and set(got[4]) == set(want[4])
    for a, b in zip(got[3], want[3]):
        assert (a is None) == (b is None) and (a is None or torch.equal(a, b))


@pytest.mark.parametrize("mixer,recomp,frozen", [("2D_local", "partial", None), ("2D", "full", None), ("2D_local", "full", "MLP.fc1.weight")])
def test_block_is_differentiated_twice(monkeypatch, mixer, recomp, frozen):
    from mamba2d_amd import backbone
    say(f"\ncase twice block {mixer} {recomp} {frozen}")
    torch.manual_seed(5)
    with torch.device("cuda"):
        block = backbone.ResBlock(32, mixer, res_scale_init_value=1.0, recomp=recomp, scan_start="BR")
        with torch.no_grad():
            for prm in block.parameters():
                prm.add_(0.05 * torch.randn_like(prm))
        source = torch.randn(2, 6, 5, 32, requires_grad=True)
        dy = torch.randn(2, 6, 5, 32) + 0.25
    if frozen:
        block.get_parameter(frozen).requires_grad_(False)
    leaves = [source, *(q for q in block.parameters() if q.requires_grad)]

    def f():      # the block's input hangs on one of its own parameters: gradients must not run through that twice
        x = source * block.res_scale1.scale
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert stock or block._train_parameters(x) is not None
            return block(x)

    stock = False
    got = twice(f, leaves, dy)
    once = torch.autograd.grad(f(), leaves, dy)
    stock = True
    monkeypatch.setattr(backbone.ResBlock, "_train_parameters", lambda self, x: None)
    want = twice(f, leaves, dy)
    names = ["x", *(n for n, q in block.named_parameters() if q.requires_grad)]
    rel = lambda a, b: float((a.double() - b.double()).norm() / b.double().norm().clamp(min=1e-30))
    for name, a, o, b in zip(names, got[1], once, want[1]):
        say(f"  {name:40s} first {rel(a, b):.1e}, without a graph {rel(o, b):.1e}")
        assert rel(a, b) < 1e-2 and rel(o, b) < 1e-1, name      # (bf16 branches; a StarReLU's scale is a sum that cancels)
    assert got[2] == want[2] and any(got[2]) and got[4] and set(got[4]) == set(want[4])
    for name, a, b in zip(names, got[3], want[3]):
        assert (a is None) == (b is None), name
        if a is not None:
            say(f"  {name:40s} second {rel(a, b):.1e}")
            assert rel(a, b) < 3e-2, name
