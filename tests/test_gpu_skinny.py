"""The small-problem GEMM (K split over a block's waves) against the other
kernels: the int32 sums are exact on both and the epilogue is the same, so
every output is bit-identical.  Its tiles are forced one by one over shapes
around their edges (PHI_GEMM_SKINNY=0..13; "off" keeps it out)."""
import numpy as np
import pytest
import torch

import phi_qlinear as Q
from phi_qlinear import synth

pytestmark = pytest.mark.gpu

# rows, columns around 16 .. 96, K with fewer pairs than waves, an odd number
# of them, and many; 270 rows are two K-tiled strips.
SHAPES = [(1, 8, 256), (17, 72, 768), (65, 136, 1280), (97, 56, 3072), (270, 264, 512)]


def both(monkeypatch, cfg, f):
    monkeypatch.setenv("PHI_GEMM_SKINNY", "off")
    want = f()
    monkeypatch.setenv("PHI_GEMM_SKINNY", str(cfg))
    got = f()
    torch.cuda.synchronize()
    assert got.dtype == want.dtype and torch.equal(got, want)


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("cfg", range(14))
def test_tiles_int8(dev, monkeypatch, cfg, M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    A, B = synth.int8_weight(M, K, seed=M).to(dev), synth.int8_weight(N, K, seed=N).to(dev)
    sA, sB = torch.rand(M, generator=g).to(dev), torch.rand(N, generator=g).to(dev)
    bias = torch.randn(N, generator=g).to(dev)
    gate, H = torch.randn(N, generator=g).to(dev), torch.randn(M, N, generator=g).to(dev)
    Ak, Bk = Q.pack_k_tiled(A), Q.pack_k_tiled(B)
    both(monkeypatch, cfg, lambda: Q.i8_gemm(A, B, None, None, out_dtype=torch.int32))
    both(monkeypatch, cfg, lambda: Q.i8_gemm(A, B, sA, sB, bias.bfloat16()))
    both(monkeypatch, cfg, lambda: Q.i8_gemm_kt(Ak, Bk, M, N, K, sA, sB[:1], bias, out_dtype=torch.float32))
    both(monkeypatch, cfg, lambda: Q.i8_gemm_residual(A, B, sA, sB, bias, gate, H.clone()))
    both(monkeypatch, cfg, lambda: Q.i8_gemm_residual_kt(Ak, Bk, M, N, K, sA, sB, None, gate, H.clone()))


@pytest.mark.parametrize("out", [torch.float32, torch.bfloat16, torch.int32])
@pytest.mark.parametrize("cfg", [0, 5, 8, 11])
def test_tiles_odd_columns_and_pitches(dev, monkeypatch, cfg, out):
    """Column counts and output pitches that no 16-byte store fits, operands in wider rows."""
    M, N, K = 75, 101, 640
    A = synth.int8_weight(M, K + 32, seed=1).to(dev)[:, :K]
    B = synth.int8_weight(N, K + 16, seed=2).to(dev)[:, :K]
    sA, sB = torch.rand(M, device=dev), torch.rand(N, device=dev)

    def f():
        C = torch.zeros((M, N + 2), dtype=out, device=dev)
        Q.i8_gemm(A, B, sA, sB, C=C[:, :N])
        return C

    both(monkeypatch, cfg, f)


@pytest.mark.parametrize("M,N,K", [(1, 8, 512), (33, 72, 1024), (81, 136, 2560)])
@pytest.mark.parametrize("cfg", range(14))
def test_tiles_4bit(dev, monkeypatch, cfg, M, N, K):
    g = torch.Generator().manual_seed(K)
    A = synth.int8_weight(M, K, seed=5).to(dev)
    Bw = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8).to(dev)
    sA, sB = torch.rand(M, generator=g).to(dev), torch.rand(N, generator=g).to(dev)
    both(monkeypatch, cfg, lambda: Q.i4_gemm(A, Bw, None, None, out_dtype=torch.int32))
    both(monkeypatch, cfg, lambda: Q.i4_gemm(A, Bw, sA, sB))
    x = synth.activations(M, K, seed=6).to(dev)
    for group in (64, 128, 512):
        codes, s_rel, sch, corr = (t.to(dev) for t in synth.w4a8_weight(N, K, group, seed=7))
        lut, sw = Q.w4a8_prepare(codes, s_rel, Q.F16, sch, k=K, group=group, correction=corr)
        q8 = torch.empty((M * K,), dtype=torch.int8, device=dev)
        for ws in (None, Q.w4a8_workspace(M, N, K, group, dev)):

            def f():
                """Outputs, and the activation codes in the layout of the path it stands in for."""
                y = Q.w4a8_linear(x, codes, lut, sw, group=group, out_dtype=torch.float32, q8=q8.view(M, K), workspace=ws)
                return torch.cat([y.flatten(), q8.float()])

            both(monkeypatch, cfg, f)


def test_rule_matches_oracle(dev, orc):
    """Unforced: a row, a few and an odd count through the linear, against the oracle."""
    for M, N, K in ((1, 100, 512), (9, 264, 1024), (77, 3, 768)):
        x, W, b = synth.activations(M, K, seed=M), synth.int8_weight(N, K, seed=N), synth.bias(N, seed=3)
        sW = synth.weight_scale()
        y = Q.q8_linear(x.to(dev), W.to(dev), sW.to(dev), b.to(dev))
        yq = Q.q8_linear_kq(x.to(dev), W.to(dev), sW.to(dev), b.to(dev))
        torch.cuda.synchronize()
        u16 = lambda t: t.cpu().view(torch.int16).numpy().view(np.uint16)  # noqa: E731
        want = orc.q8_linear(u16(x), W.numpy(), sW.numpy(), u16(b))[0]
        assert np.array_equal(u16(y), want) and np.array_equal(u16(yq), want)


def test_table_entry_keeps_the_persistent_kernel_and_its_bits(dev):
    M, N, K = 40, 256, 1024
    A, B = synth.int8_weight(M, K, seed=1).to(dev), synth.int8_weight(N, K, seed=2).to(dev)
    want = Q.i8_gemm(A, B, None, None, out_dtype=torch.int32)
    try:
        for kw in (dict(tile=Q.PLAN_TILE_SQUARE), dict(tile=Q.PLAN_TILE_272), dict(group_m=2), dict()):
            Q.gemm_plan_set(M, N, K, **kw)
            assert torch.equal(Q.i8_gemm(A, B, None, None, out_dtype=torch.int32), want)
    finally:
        Q.gemm_plan_clear()


@pytest.mark.parametrize("rm", [Q.ROUND_HALF_AWAY, Q.ROUND_HALF_EVEN])
@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,K,N", [(1, 256, 8), (1, 3072, 3072), (1, 12288, 96), (1, 16384, 40), (1, 5120, 4104), (2, 4096, 8200),
                                   (8, 1024, 136), (2, 3072, 1000), (7, 512, 16384), (3, 2048, 64)])
def test_few_rows_in_one_launch(dev, monkeypatch, xdt, rm, M, K, N):
    """The one-launch linear against rotate + quantise then GEMM: codes, scales
    and outputs, with rows that hold an inf, a NaN, huge and tiny values."""
    x = synth.activations(M, K, seed=M + K).to(xdt)
    if M > 2:
        x[1, 5], x[2, 7] = float("inf"), float("nan")
    if M > 4:
        x[3] *= 1e-37
        x[4, :9] = 3e38
    x = x.to(dev)
    W, b = synth.int8_weight(N, K, seed=N).to(dev), synth.bias(N, seed=3).to(dev)
    sW = torch.rand(N, device=dev) * 0.01
    Wk = Q.pack_k_tiled(W)

    def f(kt, out, bias):
        q8, s8 = torch.zeros((M * K,), dtype=torch.int8, device=dev), torch.zeros((M,), device=dev)
        kw = dict(out_dtype=out, s8=s8, round_mode=rm)
        y = Q.q8_linear_kt(x, Wk, N, sW, bias, q8=q8, **kw) if kt else Q.q8_linear(x, W, sW, bias, q8=q8.view(M, K), **kw)
        return y, q8, s8

    for kt in (False, True):
        for out, bias in ((torch.bfloat16, b), (torch.float32, None)):
            monkeypatch.setenv("PHI_ROW_LINEAR", "0")
            want = f(kt, out, bias)
            monkeypatch.delenv("PHI_ROW_LINEAR")
            got = f(kt, out, bias)
            torch.cuda.synchronize()
            for g, w in zip(got, want):
                v = {2: torch.int16, 4: torch.int32, 1: torch.int8}[g.element_size()]
                same = (g.view(v) == w.view(v)) | (torch.isnan(g.float()) & torch.isnan(w.float()))
                assert bool(same.all())


@pytest.mark.parametrize("K", [256, 3072])
def test_few_rows_in_place(dev, monkeypatch, K):
    """An output over the input takes two launches: all of x is read before the first store."""
    W, sW = synth.int8_weight(K, K, seed=2).to(dev), torch.rand(K, device=dev) * 0.01
    x = synth.activations(1, K, seed=1).to(dev)
    q8, s8 = torch.empty((1, K), dtype=torch.int8, device=dev), torch.empty((1,), device=dev)
    want = Q.q8_linear(x, W, sW, q8=q8, s8=s8)
    for _ in range(8):
        y = x.clone()
        Q.q8_linear(y, W, sW, q8=q8, s8=s8, C=y)
        torch.cuda.synchronize()
        assert torch.equal(y, want)
