"""Workloads of the 2-D selective scan and of the backbone around it, for timing.

Four public entry points are covered, each over the sizes it meets:

``scan``      ``wf_cuda_fn_pr.apply``: the scan on ready-made parameters, forward, or forward and backward
``entry``     ``wavefront_scan_cuda``: projections and scan as a token mixer calls them
``block``     one residual block of a scan stage in training, fp32 parameters under bf16 autocast
``backbone``  ``Mamba2DBackbone`` at inference, from images to the last stage's features

A case is a dict: ``path`` is one of the four, ``B, H, W`` the batch and the grid (of cells, or of pixels for the
backbone), ``E`` the channels, ``dtype`` the activations' type, ``train`` whether gradients are asked for, ``flip``
whether the scan starts at the bottom-right corner, ``recomp`` the recomputation mode of the entry point.
"""
import math

import torch
import torch.nn.functional as F

from mamba2d_amd import wavefront as wf
from mamba2d_amd.backbone import M2D_T, Mamba2DBackbone, ResBlock

N = 16                      # states per channel of every published configuration
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def _scan(name, B, H, W, E, dtype, train, flip=False):
    return {"name": name, "path": "scan", "B": B, "H": H, "W": W, "E": E, "dtype": dtype, "train": train, "flip": flip}


def _entry(name, B, H, W, E, dtype, train, flip=False, recomp="partial"):
    return {"name": name, "path": "entry", "B": B, "H": H, "W": W, "E": E, "dtype": dtype, "train": train, "flip": flip,
            "recomp": recomp}


def listed():
    return [
        # the smallest call: two 14x14 grids of 32 channels, forward only.  Latency and launches are what it costs
        _scan("scan-14-infer", 2, 14, 14, 32, "f32", False),
        # the headline: the first stage's scan on a batch of 128 images, forward and backward
        _scan("scan-stage1-train", 128, 56, 56, 64, "bf16", True),
        # the third stage's shape, many short anti-diagonals and many channels
        _scan("scan-stage3-train", 128, 14, 14, 320, "bf16", True),
        # the largest grid of the high-resolution series: one image, four million cells
        _scan("scan-2048-train", 1, 2048, 2048, 64, "f32", True),
        # the token mixer of the first stage at the batch per GPU of the training configurations
        _entry("entry-stage1-train", 64, 56, 56, 64, "bf16", True),
        # the second stage in a block that scans from the other corner and keeps nothing for its backward
        _entry("entry-stage2-full", 64, 28, 28, 128, "bf16", True, flip=True, recomp="full"),
        # a ragged grid with a channel count that is no multiple of 8, in fp32
        _entry("entry-odd-train", 5, 37, 45, 100, "f32", True),
        # one high-resolution grid in fp32, projections included
        _entry("entry-256-train", 1, 256, 256, 64, "f32", True),
        # the first stage on four 512x512 crops of dense prediction
        _entry("entry-crop512-train", 4, 128, 128, 64, "bf16", True),
        # a residual block of the first stage in bf16-mixed training: norms, local path, scan, MLP and their backward
        {"name": "block-stage1-train", "path": "block", "B": 64, "H": 56, "W": 56, "E": 64, "flip": False},
        # inference on a batch of images, weights in bf16
        {"name": "backbone-batch", "path": "backbone", "B": 128, "H": 224, "W": 224, "dtype": "bf16"},
        # one image at a time, as a server without batching has it: host work and launches
        {"name": "backbone-one-image", "path": "backbone", "B": 1, "H": 224, "W": 224, "dtype": "bf16"},
    ]


def _spread(rng, low, high):
    """A whole number from low to high, evenly over the logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    path = rng.choice(("scan", "scan", "entry", "entry", "entry", "block", "backbone"))
    if path == "backbone":
        H, W = _spread(rng, 96, 512), _spread(rng, 96, 512)
        most = min(128, (128 * 224 * 224) // (H * W))
        return {"path": path, "B": _spread(rng, 1, most), "H": H, "W": W, "dtype": rng.choice(("bf16", "bf16", "mixed"))}
    if path == "block":
        E = rng.choice((32, 64, 96, 128))
        H, W = _spread(rng, 14, 128), _spread(rng, 14, 128)
        most = max(1, min(64, (64 * 56 * 56 * 64) // (H * W * E)))
        return {"path": path, "B": _spread(rng, 1, most), "H": H, "W": W, "E": E, "flip": rng.random() < 0.5}
    E = _spread(rng, 16, 512)
    if rng.random() < 0.7:                     # most widths are multiples of 8, some are not
        E = max(16, E // 8 * 8)
    H = _spread(rng, 7, 1024)
    W = min(1024, max(7, round(H * math.exp(rng.uniform(-0.7, 0.7)))))
    most = max(1, min(256, (1 << 26) // (H * W * E)))
    while H * W * E > 1 << 26:
        H, W = max(7, H * 3 // 4), max(7, W * 3 // 4)
    case = {"path": path, "B": _spread(rng, 1, most), "H": H, "W": W, "E": E, "dtype": rng.choice(("bf16", "bf16", "f32")),
            "train": rng.random() < 0.7, "flip": rng.random() < 0.5}
    if path == "entry":
        case["recomp"] = rng.choice(("partial", "partial", "full"))
    return case


def _mixer_parameters(E, gen):
    """The entry point's parameters as a token mixer initialises and then trains them: A = 1..N, step sizes log-uniform
    in [1e-3, 1e-1], everything moved a little off its initial value."""
    dev = gen.device
    R = math.ceil(E / 16)
    u = lambda *s: torch.rand(*s, generator=gen, device=dev)
    r = lambda *s: torch.randn(*s, generator=gen, device=dev)
    a_log = torch.log(torch.arange(1, N + 1, dtype=torch.float32, device=dev)).repeat(E, 1)
    dt = torch.exp(u(E) * (math.log(0.1) - math.log(0.001)) + math.log(0.001)).clamp(min=1e-4)
    bias = dt + torch.log(-torch.expm1(-dt))
    return [a_log + 0.1 * r(E, N), a_log + 0.1 * r(E, N), (2 * u(2 * R + 3 * N, E) - 1) / math.sqrt(E),
            (2 * u(E, R) - 1) * R ** -0.5, bias + 0.1 * r(E), (2 * u(E, R) - 1) * R ** -0.5, bias + 0.1 * r(E), 1 + 0.1 * r(E)]


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen, device=dev)
    B, H, W = case["B"], case["H"], case["W"]
    if case["path"] == "backbone":
        mixed = case["dtype"] == "mixed"       # fp32 weights under autocast, or everything in bf16
        torch.manual_seed(seed)
        with dev:
            model = Mamba2DBackbone(**M2D_T).eval()
        if not mixed:
            model = model.to(torch.bfloat16)
        images = r(B, 3, H, W)
        return {"case": case, "model": model, "x": images if mixed else images.to(torch.bfloat16), "mixed": mixed}
    E = case["E"]
    if case["path"] == "block":
        torch.manual_seed(seed)
        with dev:
            block = ResBlock(E, "2D_local", res_scale_init_value=1.0, scan_start="BR" if case["flip"] else "TL").train()
        x = r(B, H, W, E).requires_grad_(True)             # the residual stream is fp32
        return {"case": case, "block": block, "leaves": [x, *block.parameters()], "dy": r(B, H, W, E)}
    dtype = DTYPES[case["dtype"]]
    if case["path"] == "scan":
        u = lambda *s: torch.rand(*s, generator=gen, device=dev)
        leaves = [r(B, H, W, E), F.softplus(r(B, H, W, E)), F.softplus(r(B, H, W, E)), -torch.exp(-4 * u(E, N)),
                  -torch.exp(-4 * u(E, N)), r(B, H, W, N), r(B, H, W, N), r(B, H, W, N), r(E)]
        leaves = [t.to(dtype) for t in leaves]
    else:
        leaves = [F.gelu(r(B, H, W, E)).to(dtype), *_mixer_parameters(E, gen)]
    if not case["train"]:
        return {"case": case, "leaves": leaves}
    return {"case": case, "leaves": [t.requires_grad_(True) for t in leaves], "dy": r(B, H, W, E).to(dtype)}


def run(state):
    case = state["case"]
    if case["path"] == "backbone":
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16, enabled=state["mixed"]):
            return state["model"](state["x"])
    leaves = state["leaves"]
    if case["path"] == "block":
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = state["block"](leaves[0])
        dx, *grads = torch.autograd.grad(y, leaves, state["dy"])
        return y.detach(), dx, torch.cat([g.reshape(-1) for g in grads])      # the flat bucket that is reduced and applied
    if case["path"] == "scan":
        call = lambda: wf.wf_cuda_fn_pr.apply(*leaves, case["flip"])
    else:
        call = lambda: wf.wavefront_scan_cuda(*leaves, case["recomp"], flip=case["flip"])
    if not case["train"]:
        with torch.no_grad():
            return call()
    y = call()
    return (y.detach(), *torch.autograd.grad(y, leaves, state["dy"]))


# Floating-point operations per (cell, channel, state), an exponential counted as one: two gates (a product and an
# exponential each), two inputs, the sum of two gated neighbours and two inputs halved, and the output's multiply-add;
# the backward forms the adjoint state, two gate gradients and the sums over channels, states and positions from it.
SCAN_FWD, SCAN_BWD = 14, 34


def _scan_work(P, E, s, train):
    values = P * (4 * E + 3 * N) + 2 * E * N + E                   # x, two step sizes, y; B_T, B_L, C; A_T, A_L, D
    if train:
        values += P * (4 * E + 3 * N) + 2 * E * N + E              # dy and the nine gradients
    return s * values, P * E * N * (SCAN_FWD + (SCAN_BWD if train else 0))


def _mixer_flops(P, E, train):
    R = math.ceil(E / 16)
    proj = 2 * P * E * (2 * R + 3 * N) + 2 * 2 * P * R * E
    return P * E * N * (SCAN_FWD + (SCAN_BWD if train else 0)) + proj * (3 if train else 1)


def _mixer_weights(E):
    R = math.ceil(E / 16)
    return 2 * E * N + (2 * R + 3 * N) * E + 2 * E * R + 3 * E


def work(case):
    B, H, W = case["B"], case["H"], case["W"]
    P = B * H * W
    if case["path"] == "scan":
        moved, flops = _scan_work(P, case["E"], 2 if case["dtype"] == "bf16" else 4, case["train"])
    elif case["path"] == "entry":
        E, s = case["E"], 2 if case["dtype"] == "bf16" else 4
        moved = (4 if case["train"] else 2) * s * P * E + (2 if case["train"] else 1) * 4 * _mixer_weights(E)
        flops = _mixer_flops(P, E, case["train"])
    elif case["path"] == "block":
        E = case["E"]
        dense = 2 * E * E + 4 * E * E + 8 * E * E                  # in and out projections, local path, MLP
        moved = 4 * 4 * P * E + 2 * 4 * (dense + 18 * E + _mixer_weights(E))
        flops = 3 * 2 * P * (dense + 18 * E) + _mixer_flops(P, E, True)
    else:
        s = 4 if case["dtype"] == "mixed" else 2
        h, w, cin, flops, weights = H, W, 3, 0, 0
        for i, (blocks, E, mixer) in enumerate(zip(M2D_T["n_blocks"], M2D_T["embed_dim"], M2D_T["token_mixer"])):
            k, stride, pad = (7, 4, 2) if i == 0 else (3, 2, 1)
            h, w = (h + 2 * pad - k) // stride + 1, (w + 2 * pad - k) // stride + 1
            P = B * h * w
            flops += 2 * P * k * k * cin * E
            weights += k * k * cin * E
            dense = 12 * E * E if mixer == "RopeAttention" else 14 * E * E + 18 * E
            flops += blocks * (2 * P * dense + (4 * P * h * w * E if mixer == "RopeAttention" else _mixer_flops(P, E, False)))
            weights += blocks * (dense + (0 if mixer == "RopeAttention" else _mixer_weights(E)))
            cin = E
        moved = s * (B * 3 * H * W + weights) + 2 * P * cin
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    if case["path"] == "backbone":
        return {"rel": 2e-2}                   # 18 blocks of bf16 activations
    if case["path"] == "block" or case["dtype"] == "bf16":
        return {"rel": 1e-2}
    return {"rel": 5e-5}                       # fp32 recurrences and sums over up to millions of positions
