"""The entry point issued from C++ (m2dscan::entry, m2dscan::scan) against the Python autograd functions over the same
kernels: the same bits, also where tensors need a copy first, and the cases in which the Python functions run instead."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def problem(B, H, W, E, dtype, params, seed=0):
    R, gen = max(1, E // 16), torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen)
    x = r(B, H, W, E).to(dtype).cuda()
    p = [0.3 * r(E, 16), 0.3 * r(E, 16), r(2 * R + 48, E) / E ** 0.5, r(E, R), r(E) - 2, r(E, R), r(E) - 2, 1 + 0.1 * r(E)]
    return x, [t.to(params).cuda() for t in p], r(B, H, W, E).cuda()


@pytest.mark.parametrize("form", ["plain", "view", "shifted"])
@pytest.mark.parametrize("recomp", ["partial", "full"])
@pytest.mark.parametrize("dtype,params", [(torch.bfloat16, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32)],
                         ids=["bf16", "bf16_bf16", "f32"])
@pytest.mark.parametrize("shape", [(2, 7, 9, 24), (1, 20, 33, 19), (40, 14, 14, 64)], ids=lambda s: "x".join(map(str, s)))
def test_entry_gives_the_functions_bits(shape, dtype, params, recomp, form):
    from mamba2d_amd import wavefront as wf
    say(f"\ncase entry {shape} {dtype} {params} {recomp} {form}")
    x, p, dy = problem(*shape, dtype, params)
    if form == "view":        # not contiguous
        x, p[2] = x.transpose(1, 2), p[2].t().contiguous().t()
        dy = dy.transpose(1, 2)
    elif form == "shifted":   # contiguous, off a 16-byte boundary
        move = lambda t: torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)
        x, p[0], p[7], dy = move(x), move(p[0]), move(p[7]), move(dy)
    leaves = [t.detach().requires_grad_(True) for t in (x, *p)]
    flip = shape[0] == 2
    y = wf.wavefront_scan_cuda(*leaves, recomp, flip=flip)
    g = torch.autograd.grad(y, leaves, dy)
    want = wf.wf_cuda_fn_proj.apply(*leaves, recomp == "full", flip, True)
    gw = torch.autograd.grad(want, leaves, dy)
    assert torch.equal(y, want) and y.dtype == dtype
    for a, b, leaf in zip(g, gw, leaves):
        assert a.dtype == b.dtype == leaf.dtype and a.shape == leaf.shape and torch.equal(a, b)
    with torch.no_grad():     # nothing kept, and for few images no set-up launch
        z = wf.wavefront_scan_cuda(*leaves, recomp, flip=flip)
        assert not z.requires_grad and torch.equal(z, wf.wf_cuda_fn_proj.apply(*leaves, recomp == "full", flip, False))
    part = [t if i != 3 else t.detach() for i, t in enumerate(leaves)]      # gradients of some inputs only
    y = wf.wavefront_scan_cuda(*part, recomp, flip=flip)
    assert torch.equal(torch.autograd.grad(y, part[0], dy)[0], gw[0])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("shape", [(1, 2, 2, 1), (1, 14, 14, 320), (3, 15, 17, 37), (1, 70, 30, 20), (70, 9, 8, 40)], ids=lambda s: "x".join(map(str, s)))
def test_scan_without_autograd_gives_the_functions_bits(shape, dtype):
    from mamba2d_amd import wavefront as wf
    from oracle import scan_oracle as so
    say(f"\ncase scan {shape} {dtype}")
    inp = so.make_inputs(*shape, 16, seed=3, dtype=dtype)
    a = [inp[k].cuda() for k in so.INPUT_NAMES]
    with torch.no_grad():
        y = wf.wf_cuda_fn_pr.apply(*a, True)
    assert not y.requires_grad and torch.equal(y, wf._ScanOnParams.apply(*a, True, False))
    kept, _ = wf.scan_fwd_op(*a, True, True)      # the forward that keeps snapshots has the set-up launch
    assert so.rel_err(y.float().cpu(), kept.float().cpu()) < (1e-2 if dtype == torch.bfloat16 else 1e-6)


def test_errors_are_those_of_the_functions():
    from mamba2d_amd import wavefront as wf
    x, p, _ = problem(1, 4, 4, 16, torch.float32, torch.float32)
    with pytest.raises(RuntimeError, match="float32 and bfloat16"):
        wf.wavefront_scan_cuda(x.half(), *p)
    with pytest.raises(RuntimeError, match="shape"):
        wf.wavefront_scan_cuda(x, *p[:2], p[2][:-1], *p[3:])
    with torch.no_grad(), pytest.raises(RuntimeError, match="dtype"):
        wf.wf_cuda_fn_pr.apply(x, x.bfloat16(), x, *[t.exp().neg() for t in p[:2]], x, x, x, p[7])
