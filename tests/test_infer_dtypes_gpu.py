"""bf16 activations meet fp32 weights of a wide layer only under autocast, as the stock product has it: whether a stage takes
them must not depend on the size of the grid or of the batch."""
import pytest
import torch

from mamba2d_amd import backbone

pytestmark = pytest.mark.gpu


def stage_of(dim, mixer):
    return backbone.Mamba2DBackbone(n_blocks=(1,), embed_dim=(dim,), token_mixer=(mixer,), res_scale_init_values=(1.0,)).eval().stages["0"].cuda()


@pytest.mark.parametrize("positions", [(1, 4, 5), (2, 16, 16), (3, 16, 16)], ids=lambda p: "x".join(map(str, p)))
@pytest.mark.parametrize("dim,mixer", [(320, "2D"), (128, "2D_local"), (48, "2D"), (64, "2D_local"), (64, "RopeAttention"), (320, "RopeAttention")])
def test_fp32_weights_without_autocast(monkeypatch, dim, mixer, positions):
    print(f"\ncase fp32 weights {dim} {mixer} {positions}", flush=True)
    stage, x = stage_of(dim, mixer), torch.randn(*positions, dim, device="cuda").bfloat16()
    run = lambda: backbone.Mamba2DBackbone._run_stage(stage, x)

    def outcome():
        try:
            return run().dtype
        except RuntimeError as e:
            assert "same dtype" in str(e)
            return "refused"

    with torch.no_grad():
        got = outcome()
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert run().dtype == torch.bfloat16
        monkeypatch.setattr(backbone, "_infer_stage", lambda stage, x: None)
        want = outcome()
    assert got == want == (torch.bfloat16 if (dim, mixer) == (64, "2D_local") else "refused")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_fp16_autocast_keeps_to_the_modules(dtype):
    """Under fp16 autocast the stock products answer in fp16: no sequence of bf16 kernels."""
    print(f"\ncase fp16 autocast {dtype}", flush=True)
    stage, x = stage_of(64, "RopeAttention").to(dtype), torch.randn(2, 6, 7, 64, device="cuda").bfloat16()
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16):
        assert backbone._infer_stage(stage, x) is None
