"""The load-time kernels' 16-byte forms against their general forms: the same
call on operands one element off their alignment takes the general kernel,
and every bit has to agree (the general forms are held to the oracle by
test_gpu_w4a8.py and test_gpu_checkpoint.py)."""
import ctypes

import pytest
import torch

import phi_qlinear as Q
from phi_qlinear import synth

pytestmark = pytest.mark.gpu


def shifted(t, by=1):
    """t's values `by` elements into a buffer whose rows are `by` wider: no row keeps its 16-byte alignment."""
    rows, cols = t.shape
    buf = torch.zeros((rows * (cols + by) + by,), dtype=t.dtype, device=t.device)
    v = buf[by:].view(rows, cols + by)[:, :cols]
    v.copy_(t)
    return v


def bits(t):
    return t.contiguous().view(torch.int32)


@pytest.mark.parametrize("rows,cols", [(1, 4), (3, 252), (5, 516), (2, 3076), (70001, 4), (300, 12), (129, 2048)])
@pytest.mark.parametrize("kind", [Q.I8, Q.I4, Q.F8_E4M3, Q.F8_E5M2, Q.F16, Q.BF16, Q.F32])
def test_dequant_rows(dev, kind, rows, cols):
    g = torch.Generator().manual_seed(cols)
    dt = {Q.I8: torch.int8, Q.F16: torch.float16, Q.BF16: torch.bfloat16, Q.F32: torch.float32}.get(kind, torch.uint8)
    if dt in (torch.int8, torch.uint8):
        src = torch.randint(0, 256, (rows, cols // 2 if kind == Q.I4 else cols), generator=g, dtype=torch.uint8).view(dt)
    else:
        src = (torch.randn(rows, cols, generator=g) * 3).to(dt)
    src = src.to(dev)
    for scale in (torch.rand(rows, generator=g).to(dev), torch.rand(1, generator=g).to(dev)):
        got = Q.dequant_rows(src, kind, cols, row_scale=scale)
        want = Q.dequant_rows(shifted(src), kind, cols, row_scale=scale)
        assert torch.equal(bits(got), bits(want))


@pytest.mark.parametrize("rows,K", [(1, 256), (3, 768), (7, 5120)])
def test_convrot_rows(dev, rows, K):
    x = torch.randn(rows, K, device=dev)
    x[0, :4] = torch.tensor([float("inf"), 3e38, -3e38, 1e-40], device=dev)
    L, st = Q.load(), torch.cuda.current_stream().cuda_stream
    P, I = ctypes.c_void_p, ctypes.c_int64
    L.phi_hip_convrot_rows.argtypes = [P, P, I, I, I, P, I]
    want, got, inplace = shifted(torch.empty_like(x)), torch.empty_like(x), x.clone()
    for src, dst in ((x, want), (x, got), (inplace, inplace)):
        assert L.phi_hip_convrot_rows(st, src.data_ptr(), rows, K, src.stride(0), dst.data_ptr(), dst.stride(0)) == 0
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.nan_to_num(got, nan=0.0), torch.nan_to_num(want, nan=0.0))
    assert torch.equal(torch.nan_to_num(inplace, nan=0.0), torch.nan_to_num(got, nan=0.0))


@pytest.mark.parametrize("rows,k,rank", [(1, 4, 1), (63, 260, 4), (65, 516, 7), (130, 1024, 33), (12289, 64, 3), (3025, 260, 5),
                                         (1031, 764, 33), (260, 3076, 4)])
def test_lora_fold(dev, rows, k, rank):
    g = torch.Generator().manual_seed(rank)
    w, A, B = torch.randn(rows, k, generator=g), torch.randn(rank, k, generator=g), torch.randn(rows, rank, generator=g)
    B[:: 3, :: 2] = 0.0
    B[rows // 2] = -0.0
    w[rows // 2, :2] = -0.0
    A[0, 0] = float("inf")  # a skipped entry must not reach it
    w, A, B = w.to(dev), A.to(dev), B.to(dev)
    L, st = Q.load(), torch.cuda.current_stream().cuda_stream
    P, I = ctypes.c_void_p, ctypes.c_int64
    L.phi_hip_lora_fold.argtypes = [P, P, I, I, I, P, P, I, ctypes.c_float]
    got, want = w.clone(), shifted(w)
    for t in (got, want):
        assert L.phi_hip_lora_fold(st, t.data_ptr(), t.stride(0), rows, k, A.data_ptr(), B.data_ptr(), rank, 0.75) == 0
    torch.cuda.synchronize()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(bits(torch.nan_to_num(got, nan=7.0)), bits(torch.nan_to_num(want, nan=7.0)))


@pytest.mark.parametrize("with_cb", [False, True])
@pytest.mark.parametrize("rows,k,group", [(1, 32, 32), (5, 1056, 32), (7, 3072, 128), (2, 15360, 32), (3, 4096, 4096), (3, 1920, 32), (3, 1952, 32),
                                          (1025, 5120, 32), (2049, 7680, 32), (2049, 7712, 32)])
def test_w4a8_expand_and_prepare(dev, rows, k, group, with_cb):
    codes, s_rel, sch, corr = (t.to(dev) for t in synth.w4a8_weight(rows, k, group, seed=rows))
    codes[0] &= 0x33  # a row that uses only some of the codes
    cb = torch.linspace(-9.5, 7.25, 16, device=dev) if with_cb else None
    wide = torch.zeros((rows, k // 2 + 8), dtype=torch.uint8, device=dev)  # 8-byte rows: the general kernel
    wide[:, : k // 2] = codes
    for f in (Q.w4a8_expand, Q.w4a8_prepare):
        got, want = (f(c, s_rel, Q.F16, sch, k=k, group=group, codebook=cb, correction=corr) for c in (codes, wide))
        assert torch.equal(got[0], want[0]) and torch.equal(bits(got[1]), bits(want[1]))
