"""Calls that go past a module's own ``forward`` (a stage as one call, a block as one function, a norm inside its reader's
kernel) are for modules that nobody watches: a hook or a ``forward`` put on an instance has to run, also when it comes
after a plan was made, and must be gone when it is taken away."""
import pytest
import torch

from mamba2d_amd import backbone

KINDS = {"scan": "2D_local", "attention": "RopeAttention"}


def stage_of(kind):
    net = backbone.Mamba2DBackbone(n_blocks=(2,), embed_dim=(32,), token_mixer=(KINDS[kind],), res_scale_init_values=(1.0,)).eval()
    return net.stages["0"]


# every module whose forward a call through the modules would run
CALLED = {"scan": ["norm1", "norm2", "MLP", "MLP.fc1", "MLP.fc2", "res_scale1", "res_scale2", "token_mixer", "token_mixer.in_proj",
                   "token_mixer.out_proj", "token_mixer.local_norm", "token_mixer.local_path", "token_mixer.local_path.pwconv1",
                   "token_mixer.local_path.act1", "token_mixer.local_path.dwconv", "token_mixer.local_path.act2",
                   "token_mixer.local_path.pwconv2"],
          "attention": ["norm1", "norm2", "MLP", "token_mixer", "token_mixer.qkv", "token_mixer.proj", "token_mixer.q_norm", "token_mixer.k_norm"]}
EVERY = [(kind, name) for kind in CALLED for name in CALLED[kind]]


@pytest.mark.parametrize("kind,name", EVERY, ids=lambda v: str(v))
@pytest.mark.parametrize("way", ["forward", "hook", "pre_hook"])
def test_stage_plan_is_for_plain_modules(kind, name, way):
    stage = stage_of(kind)
    x = torch.zeros(1, 4, 4, 32)
    with torch.no_grad():
        plan = backbone._stage_plan(stage, x)
        assert plan is not None and plan.holds(stage)
        mod = stage[0].get_submodule(name)
        if way == "forward":
            mod.forward = lambda *a, **k: None
            undo = lambda: delattr(mod, "forward")
        else:
            undo = (mod.register_forward_hook if way == "hook" else mod.register_forward_pre_hook)(lambda *a: None).remove
        assert not plan.holds(stage) and backbone._stage_plan(stage, x) is None
        undo()
        assert plan.holds(stage) and backbone._stage_plan(stage, x) is not None


@pytest.mark.parametrize("target", ["block", "end"])
def test_watched_blocks_and_norms_of_a_stage_run(target):
    """The modules of a stage: a hook on a block, or on the norm behind the last block, sees its call and may change it."""
    stage = stage_of("attention")
    x = torch.randn(1, 4, 4, 32)
    seen = []
    with torch.no_grad():
        y = backbone.Mamba2DBackbone._run_stage(stage, x)
        mod = stage[0] if target == "block" else stage[-1]
        handle = mod.register_forward_hook(lambda m, a, out: (seen.append(1), out + 1.0)[1])
        z = backbone.Mamba2DBackbone._run_stage(stage, x)
        assert seen == [1] and not torch.allclose(y, z)
        handle.remove()
        mod.forward = lambda t: (seen.append(2), t)[1]
        backbone.Mamba2DBackbone._run_stage(stage, x)
        assert seen == [1, 2]


@pytest.mark.gpu
@pytest.mark.parametrize("name", CALLED["scan"])
def test_training_block_is_for_plain_modules(name):
    with torch.device("cuda"):
        block = backbone.ResBlock(32, "2D_local", res_scale_init_value=1.0)
        x = torch.randn(1, 4, 4, 32, requires_grad=True)
    print(f"\ncase watched training block {name}", flush=True)
    seen = []
    mod = block.get_submodule(name)
    plain = mod.forward
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert block._train_parameters(x) is not None
        mod.forward = lambda *a, **k: (seen.append(1), plain(*a, **k))[1]
        assert block._train_parameters(x) is None
        block(x).sum().backward()
        del mod.forward
        assert seen == [1] and block._train_parameters(x) is not None


@pytest.mark.gpu
@pytest.mark.parametrize("name", CALLED["scan"])
@pytest.mark.parametrize("train", [False, True])
def test_hooks_of_a_stage_run(name, train):
    """bf16 inference and mixed training past the kernels that join a norm or an activation to their neighbour."""
    print(f"\ncase watched stage {name} {train}", flush=True)
    with torch.device("cuda"):
        stage = stage_of("scan")
        x = torch.randn(1, 4, 4, 32)
    if not train:
        stage, x = stage.bfloat16(), x.bfloat16()
    seen = []
    with torch.set_grad_enabled(train):
        assert train or backbone._infer_stage(stage, x) is not None      # (the plan is there before the hooks)
    for block in stage[:2]:
        block.get_submodule(name).register_forward_hook(lambda *a: seen.append(1))
    with torch.set_grad_enabled(train), torch.autocast("cuda", dtype=torch.bfloat16, enabled=train):
        backbone.Mamba2DBackbone._run_stage(stage, x)
    assert seen == [1, 1]


def test_stage_plan_is_for_registered_parameters():
    """A tensor that stands in a parameter's place as a plain attribute (as sharding tools leave one, a new one each time) is
    nothing that a plan could compare on the next call."""
    stage = stage_of("scan")
    x = torch.zeros(1, 4, 4, 32)
    with torch.no_grad():
        plan = backbone._stage_plan(stage, x)
        fc1 = stage[0].MLP.fc1
        kept = fc1.weight
        del fc1.weight
        fc1.weight = kept.detach().clone()
        assert not plan.holds(stage) and backbone._stage_plan(stage, x) is None
        del fc1.weight
        fc1.weight = kept
        assert backbone._stage_plan(stage, x) is not None


class _Watched(torch.Tensor):
    pass


def test_stage_plan_is_for_plain_parameters():
    """A parameter of another tensor class (quantized or distributed, say) goes through the dispatched operators."""
    stage = stage_of("scan")
    x = torch.zeros(1, 4, 4, 32)
    with torch.no_grad():
        fc1 = stage[0].MLP.fc1
        fc1.weight = torch.nn.Parameter(fc1.weight.detach().as_subclass(_Watched))
        assert type(fc1.weight) is not torch.nn.Parameter and backbone._stage_plan(stage, x) is None


class _Scaled(torch.nn.Linear):
    """A layer with something beside its weight, as adapters have it."""

    def forward(self, x):
        return 3 * super().forward(x)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["token_mixer.in_proj", "token_mixer.out_proj", "token_mixer.local_path.pwconv1", "token_mixer.local_path.pwconv2",
                                  "MLP.fc1", "MLP.fc2"])
@pytest.mark.parametrize("way", ["subclass", "class"])
def test_other_layers_run_their_own_forward(monkeypatch, name, way):
    print(f"\ncase other layer {name} {way}", flush=True)
    stage = stage_of("scan").cuda().bfloat16()
    x = torch.randn(1, 4, 4, 32, device="cuda").bfloat16()
    run = lambda: backbone.Mamba2DBackbone._run_stage(stage, x)
    seen = []
    with torch.no_grad():
        before = run()
        if way == "subclass":
            stage[0].get_submodule(name).__class__ = _Scaled
            assert not torch.equal(run(), before)
        else:
            plain = torch.nn.Linear.forward
            with monkeypatch.context() as m:
                m.setattr(torch.nn.Linear, "forward", lambda self, t: (seen.append(self), plain(self, t))[1])
                run()
            assert stage[0].get_submodule(name) in seen
            assert torch.equal(run(), before)
