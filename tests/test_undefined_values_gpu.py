"""NaN and infinities pass through the activations of a block as the stock operators pass them (F.relu keeps a NaN):
a loss must not come out finite where a value before it was undefined."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")


def say(*a):
    print(*a, flush=True)


def run(block, x, dy):
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = block(x)
    return (y.detach(), *torch.autograd.grad(y, [x, *block.parameters()], dy))


@pytest.mark.parametrize("where", ["x", "dy", "token_mixer.local_path.pwconv1.weight", "token_mixer.local_path.dwconv.weight", "MLP.fc1.bias"])
def test_training_block_keeps_nan(monkeypatch, where):
    """One undefined value in the input, the gradient or a parameter: undefined outputs and gradients are those of the stock operators."""
    from mamba2d_amd import backbone
    say(f"\ncase nan in {where}")
    torch.manual_seed(1)
    with torch.device("cuda"):
        block = backbone.ResBlock(32, "2D_local", res_scale_init_value=1.0)
        x, dy = torch.randn(2, 9, 11, 32), torch.randn(2, 9, 11, 32)
    target = {"x": x, "dy": dy}.get(where)
    target = block.get_parameter(where).data if target is None else target[0, 5, 6]
    target.view(-1)[3] = NAN
    x.requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert block._train_parameters(x) is not None
    got = run(block, x, dy)
    monkeypatch.setattr(backbone.ResBlock, "_train_parameters", lambda self, x: None)
    want = run(block, x, dy)
    for name, g, w in zip(["y", "dx", *(n for n, _ in block.named_parameters())], got, want):
        say(f"  {name:40s} undefined {int(g.isnan().sum())} of {g.numel()}, stock {int(w.isnan().sum())}")
        assert not (w.isnan() & ~g.isnan()).any(), name
        if "dwconv" not in where:      # (an undefined filter tap also meets the zeros around the image here)
            assert torch.equal(g.isnan(), w.isnan()), name


VALUES = [NAN, INF, -INF, 0.0, -0.0, 1.5, -2.0, 3e38, -3e38, 1e-30]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_starrelu_of_undefined_values(dtype):
    from mamba2d_amd import cabi
    say(f"\ncase starrelu {dtype}")
    x = torch.tensor(VALUES * 8, dtype=dtype, device="cuda")
    s, b = torch.tensor([0.5], device="cuda"), torch.tensor([-0.25], device="cuda")
    want = (b + s * F.relu(x.float()).square()).to(dtype)
    torch.testing.assert_close(cabi.starrelu_fwd(x, s, b), want, rtol=1e-2 if dtype == torch.bfloat16 else 1e-6, atol=0, equal_nan=True)


@pytest.mark.parametrize("form", ["pre", "post", "ln_post"])
def test_linear_layers_keep_nan(form):
    from mamba2d_amd import cabi
    say(f"\ncase linear starrelu {form}")
    x = torch.randn(40, 32, device="cuda").bfloat16()
    x[17, 4] = NAN
    w = torch.randn(48, 32, device="cuda")
    par = (torch.ones(1, device="cuda"), torch.zeros(1, device="cuda"))
    act = dict(pre=cabi.ACT_STARRELU, pre_params=par) if form == "pre" else dict(post=cabi.ACT_STARRELU, post_params=par)
    ln = (torch.ones(32, device="cuda"), torch.zeros(32, device="cuda"), 1e-5) if form == "ln_post" else None
    y = cabi.linear_fwd(x, w, None, **act, ln=ln)
    assert y[17].isnan().all() and y[:17].isfinite().all() and y[18:].isfinite().all()
