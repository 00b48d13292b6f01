"""Sums of the workgroups' parts (m2d_train_reduce): four results to a thread where the parts are whole 16-byte pieces, one
otherwise; both add in the same order, so a sum must come out the same in either form."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


class _Seg(ctypes.Structure):
    _fields_ = [("part", ctypes.c_void_p), ("out", ctypes.c_void_p), ("stride", ctypes.c_int64), ("n", ctypes.c_int32), ("parts", ctypes.c_int32)]


def test_both_forms_against_float64():
    from mamba2d_amd import cabi
    print("\ncase train_reduce", flush=True)
    g = torch.Generator().manual_seed(1)
    segs, keep = [], []
    for n, parts, pad, off in [(1, 1, 0, 0), (4, 3, 0, 0), (64, 15, 4, 0), (68, 64, 0, 0), (132, 79, 8, 4), (67, 200, 1, 0), (64, 65, 0, 1), (2, 1024, 0, 0),
                               (1152, 112, 2, 0), (4096, 128, 64, 0)]:
        buf = torch.randn(off + parts * (n + pad), generator=g).cuda()
        out = torch.empty(n, device="cuda")
        keep.append((buf, out, n, parts, n + pad, off))
        segs.append(_Seg(buf.data_ptr() + 4 * off, out.data_ptr(), n + pad, n, parts))
    arr = (_Seg * len(segs))(*segs)
    cabi.lib.m2d_train_reduce.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
    assert cabi.lib.m2d_train_reduce(len(segs), ctypes.cast(arr, ctypes.c_void_p), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    for buf, out, n, parts, stride, off in keep:
        p = buf[off:].view(parts, stride)[:, :n]
        # at most ceil(parts / 16) + 16 additions in fp32, each off by half a unit in the last place of the sum so far
        bound = (parts // 16 + 17) * 2.0 ** -24 * p.double().abs().sum(0)
        assert ((out.double() - p.double().sum(0)).abs() <= bound).all(), (n, parts)
        shares = [torch.zeros(n, device="cuda") for _ in range(16)]
        for k in range(parts):
            shares[k % 16] = shares[k % 16] + p[k]
        total = torch.zeros(n, device="cuda")
        for s in shares:
            total = total + s
        assert torch.equal(out, total), (n, parts)
