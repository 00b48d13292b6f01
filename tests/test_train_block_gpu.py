"""A residual block in bf16-mixed training (m2dscan::train_block, models/mamba2d.py:191-254) against the module's stock
operators: the block in fp32 without autocast gives the reference, and the operator's output and gradients must be as
close to it (2-norm, per tensor) as the stock operators under autocast are, up to a factor and one bf16 rounding."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def run(block, x, dy, autocast):
    leaves = [x, *block.parameters()]
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
        y = block(x)
    return (y.detach(), *torch.autograd.grad(y, leaves, dy))


# B, H, W, C, mixer, start: one tile of positions and less, rows and strips that end inside, every width the operator
# takes, more tiles than workgroups
CASES = [(1, 2, 2, 32, "2D_local", "TL"), (2, 14, 14, 32, "2D", "BR"), (1, 9, 5, 64, "2D_local", "BR"), (3, 15, 29, 96, "2D_local", "TL"),
         (2, 13, 44, 128, "2D_local", "TL"), (2, 7, 7, 128, "2D", "TL"), (11, 56, 57, 64, "2D_local", "TL")]


@pytest.mark.parametrize("recomp", ["partial", "full"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_block_matches_stock_operators(monkeypatch, case, recomp):
    from mamba2d_amd import backbone
    B, H, W, C, mixer, start = case
    if recomp == "full" and B > 3:
        pytest.skip("one recomputation mode is enough at this size")
    say(f"\ncase train_block {case} {recomp}")
    torch.manual_seed(B * H * W + C)
    with torch.device("cuda"):
        block = backbone.ResBlock(C, mixer, res_scale_init_value=1.0, scan_start=start, recomp=recomp, drop_path=0.0)
        with torch.no_grad():
            for prm in block.parameters():
                prm.add_(0.05 * torch.randn_like(prm))
        x = torch.randn(B, H, W, C, requires_grad=True)
        dy = torch.randn(B, H, W, C) + 0.25        # sums over positions that do not cancel
    assert block._train_parameters(x) is None      # no autocast: stock operators
    want = run(block, x, dy, False)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert block._train_parameters(x) is not None
    got = run(block, x, dy, True)
    again = run(block, x, dy, True)
    monkeypatch.setattr(backbone.ResBlock, "_train_parameters", lambda self, x: None)
    stock = run(block, x, dy, True)
    torch.cuda.synchronize()
    names = ["y", "dx", *(n for n, _ in block.named_parameters())]
    for name, g, a, w, s in zip(names, got, again, want, stock):
        assert g.dtype == s.dtype and g.shape == s.shape, name
        assert torch.equal(g, a), (name, "not reproducible")
        rel = lambda t: float((t.double() - w.double()).norm() / w.double().norm())
        say(f"  {name:40s} operator {rel(g):.2e} stock {rel(s):.2e}")
        bound = 1e-1 if g.numel() == 1 else 1.5e-2      # (a StarReLU's scale: one sum over everything, which cancels)
        assert rel(g) < max(bound, 1.5 * rel(s)), (name, rel(g), rel(s))


def test_block_drop_path_and_frozen_parameters():
    """A dropped sample passes through the block scaled only; a frozen parameter gets no gradient; the stock path runs
    where a hook or a foreign module asks for it."""
    from mamba2d_amd import backbone
    say("\ncase train_block drop path")
    torch.manual_seed(3)
    with torch.device("cuda"):
        block = backbone.ResBlock(64, "2D_local", res_scale_init_value=1.0, drop_path=0.5).train()
        x = torch.randn(16, 7, 9, 64, requires_grad=True)
    block.MLP.fc1.weight.requires_grad_(False)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = block(x)
    y.sum().backward()
    same = (y == x * (block.res_scale1.scale * block.res_scale2.scale)).flatten(1).all(1)
    assert 0 < int(same.sum()) < 16 and torch.isfinite(y).all()      # (a quarter of the samples drop both branches)
    dropped = (x.grad == 1).flatten(1).all(1)
    assert torch.equal(same, dropped)
    assert block.MLP.fc1.weight.grad is None and block.MLP.fc2.weight.grad is not None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        handle = block.MLP.fc1.register_forward_hook(lambda *a: None)
        assert block._train_parameters(x) is None
        handle.remove()
        assert block._train_parameters(x) is not None
        block.MLP.fc1.bias = None
        assert block._train_parameters(x) is None
