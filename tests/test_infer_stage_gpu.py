"""A backbone stage at inference as one call (m2dscan::infer_stage) against the same stage module by module: the same
kernels in the same order, but for the residual updates, which narrow blocks have inside the layers in front of them in the same
bits, so the results must be the same bits (from 14000 rows on the MLP of 128 channels adds up in another order); and the cases in which the
modules run instead."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


@pytest.mark.parametrize("mode", ["bf16", "mixed"])
@pytest.mark.parametrize("shape", [(2, 64, 96), (1, 224, 224), (3, 128, 160), (1, 352, 480)], ids=lambda s: "x".join(map(str, s)))
def test_stage_in_one_call_gives_the_modules_bits(monkeypatch, shape, mode):
    from mamba2d_amd import backbone
    say(f"\ncase infer_stage {shape} {mode}")
    torch.manual_seed(sum(shape))
    with torch.device("cuda"):
        net = backbone.Mamba2DBackbone(**{**backbone.M2D_T, "n_blocks": (2, 2, 2, 1)}).eval()
        x = torch.randn(shape[0], 3, *shape[1:])
    if mode == "bf16":
        net, x = net.bfloat16(), x.bfloat16()
    seen = []
    fast = backbone._infer_stage

    def both(stage, t):      # the stage both ways on the same input (the stock convolutions in between do not repeat bits)
        got = fast(stage, t)
        seen.append(got is not None)
        if got is not None:
            monkeypatch.setattr(backbone, "_infer_stage", lambda stage, t: None)
            want = backbone.Mamba2DBackbone._run_stage(stage, t)
            monkeypatch.setattr(backbone, "_infer_stage", both)
            assert got.dtype == want.dtype == torch.bfloat16
            if len(seen) == 1:
                assert torch.equal(got, want)
            else:      # (wide layers of a few positions run in a kernel of their own in the one call)
                assert ((got.float() - want.float()).abs().max() / want.float().abs().max()).item() < 2e-2
        return got

    monkeypatch.setattr(backbone, "_infer_stage", both)
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16, enabled=mode == "mixed"):
        net(x)
    torch.cuda.synchronize()
    # the attention kernel takes grids of up to 256 cells: the third stage of the largest image is too large for it
    assert seen == [True, True, shape[1] * shape[2] <= 256 * 256, True]


def test_stage_falls_back_to_its_modules():
    from mamba2d_amd import backbone
    say("\ncase infer_stage fallback")
    with torch.device("cuda"):
        net = backbone.Mamba2DBackbone(n_blocks=(1, 1), embed_dim=(32, 64), token_mixer=("2D_local", "RopeAttention"),
                                       res_scale_init_values=(1.0, 1.0)).bfloat16().eval()
        x = torch.randn(1, 16, 16, 32, dtype=torch.bfloat16)
    mods = net.stages["0"]
    with torch.no_grad():
        assert backbone._infer_stage(mods, x) is not None
        handle = mods[0].MLP.register_forward_hook(lambda *a: None)
        assert backbone._infer_stage(mods, x) is None
        handle.remove()
        mods[0].train()
        assert backbone._infer_stage(mods, x) is None
        mods[0].eval()
        assert backbone._infer_stage(mods, x.float()) is None
        mods[0].norm1.float()
        assert backbone._infer_stage(mods, x) is None
        mods[0].norm1.bfloat16()
        y = backbone._infer_stage(mods, x)
        mods[0].norm1.weight = torch.nn.Parameter(2 * mods[0].norm1.weight)      # another parameter in the place of one
        assert not torch.equal(backbone._infer_stage(mods, x), y)
        mods[0].norm1.eps = 1.0
        z = backbone._infer_stage(mods, x)
        assert not torch.equal(z, y)
        mods[0].norm1 = backbone.LayerNorm(32).bfloat16().cuda().eval()
        assert not torch.equal(backbone._infer_stage(mods, x), z)
    assert backbone._infer_stage(mods, x) is None      # gradients of the parameters are wanted
    net.requires_grad_(False)
    assert backbone._infer_stage(mods, x) is not None


def test_widened_parameters_are_exact():
    from mamba2d_amd import wavefront as wf
    say("\ncase widen")
    g = torch.Generator().manual_seed(1)
    ts = [torch.randn(n, generator=g).bfloat16().cuda() for n in (1, 255, 256, 257, 5000)] * 14 + [torch.randn(7, generator=g).cuda()]
    out = wf.widen_op(ts)
    assert all(o.dtype == torch.float32 and torch.equal(o, t.float()) for o, t in zip(out, ts))


@pytest.mark.parametrize("grid", [(3, 28, 28), (64, 28, 28)], ids=lambda s: "x".join(map(str, s)))
def test_fp32_weights_need_autocast_beside_a_stock_product(monkeypatch, grid):
    """At 128 channels the MLP's second layer is a stock product in the modules, which refuses bf16 activations with fp32 weights: so does the one call,
    also where it has a kernel of its own for that layer."""
    from mamba2d_amd import backbone
    say(f"\ncase infer_stage fp32 weights without autocast {grid}")
    with torch.device("cuda"):
        stage = backbone.Mamba2DBackbone(n_blocks=(1,), embed_dim=(128,), token_mixer=("2D_local",), res_scale_init_values=(1.0,)).eval().stages["0"]
        x = torch.randn(*grid, 128, dtype=torch.bfloat16)
    with torch.no_grad():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert backbone._infer_stage(stage, x) is not None
        with pytest.raises(RuntimeError, match="dtype"):
            backbone._infer_stage(stage, x)
        monkeypatch.setattr(backbone, "_infer_stage", lambda stage, t: None)
        with pytest.raises(RuntimeError, match="dtype"):
            backbone.Mamba2DBackbone._run_stage(stage, x)


@pytest.mark.parametrize("mode", ["bf16", "mixed"])
@pytest.mark.parametrize("grid", [(3, 28, 28), (4, 56, 62)], ids=lambda s: "x".join(map(str, s)))
def test_stage_of_128_channels_below_the_line_of_its_one_kernel_mlp(monkeypatch, grid, mode):
    """Up to 14000 rows the MLP of 128 channels is a layer, a stock product and an update with norm, which are faster there, and the modules' own: the same
    bits (the one kernel adds the second product up in another order)."""
    from mamba2d_amd import backbone
    say(f"\ncase infer_stage 128 channels {grid} {mode}")
    torch.manual_seed(5)
    with torch.device("cuda"):
        stage = backbone.Mamba2DBackbone(n_blocks=(2,), embed_dim=(128,), token_mixer=("2D_local",), res_scale_init_values=(1.0,)).eval().stages["0"]
        x = torch.randn(*grid, 128, dtype=torch.bfloat16)
    stage = stage.bfloat16() if mode == "bf16" else stage
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16, enabled=mode == "mixed"):
        got = backbone._infer_stage(stage, x)
        monkeypatch.setattr(backbone, "_infer_stage", lambda stage, t: None)
        same = torch.equal(got, backbone.Mamba2DBackbone._run_stage(stage, x))
    assert same
