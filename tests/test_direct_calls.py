"""When a call may be issued from C++ around the dispatched operators (wavefront._direct): not where something watches the
operators that run.  No GPU needed: the rule looks at the tensors' classes and at torch's own state."""
import pytest
import torch

from mamba2d_amd import wavefront as wf


class _Other(torch.Tensor):
    pass


def _under(enter):
    seen = []
    enter(lambda t: (seen.append(wf._direct(t)), t + 1)[1])
    return seen


def test_plain_tensors_and_parameters_go_direct():
    x = torch.ones(2)
    assert wf._direct(x, torch.nn.Parameter(x)) and not wf._direct(x, torch.ones(2).as_subclass(_Other))
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):      # (C++ functions honour these)
        assert wf._direct(x)


@pytest.mark.parametrize("name", ["vmap", "grad", "make_fx", "fake", "trace", "forward_ad", "dispatch_mode"])
def test_watched_calls_do_not(name):
    x = torch.ones(2)

    def forward_ad(f):
        with torch.autograd.forward_ad.dual_level():
            f(x)

    def fake(f):
        with torch._subclasses.FakeTensorMode():
            f(torch.empty(2))

    def dispatch_mode(f):
        from torch.utils.flop_counter import FlopCounterMode
        with FlopCounterMode(display=False):
            f(x)

    def make_fx(f):
        from torch.fx.experimental.proxy_tensor import make_fx as trace
        trace(f)(x)

    ways = {"vmap": lambda f: torch.vmap(f)(x), "grad": lambda f: torch.func.grad(lambda t: f(t).sum())(x), "make_fx": make_fx,
            "fake": fake, "trace": lambda f: torch.jit.trace(f, (x,), check_trace=False), "forward_ad": forward_ad, "dispatch_mode": dispatch_mode}
    seen = _under(ways[name])
    assert seen and not any(seen)
    assert wf._direct(x)
