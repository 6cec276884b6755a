"""GPU parity: the runtime LoRA correction out += (x A^T) B^T
(phi_hip_lora_down / _rank_add / _tail; apply_lora_tail
core/models/model_common.cpp:1667-1700).

Bar: bit-exact with the oracle, whose fp32 fma chains follow the reference's
order (k ascending from 0 for h, r ascending from out's value for the
update); the oracle itself is pinned by an exact-rational emulation of those
chains (tests/test_oracle_lora.py)."""
import numpy as np
import pytest
import torch

import phi_qlinear as Q
from phi_qlinear import synth

pytestmark = pytest.mark.gpu


def factors(M, K, R, N, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g)
    A = torch.randn(R, K, generator=g) * 0.05
    B = torch.randn(N, R, generator=g) * 0.05
    out = torch.randn(M, N, generator=g)
    return x, A, B, out


def bits(t):
    return t.cpu().contiguous().view(torch.int32).numpy()


# Ranks around 16, 32 and 64 (one, two or four waves over them), one chain a
# wave and two (above 1024 16 x 16 tiles: 8192 rows of 32 ranks, 4096 of 64),
# rows that allow four-column loads and rows that do not (K or the pitch odd).
@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,K,R", [(1, 256, 1), (37, 72, 17), (300, 3072, 64), (129, 1000, 256), (65, 33, 33),
                                   (70, 640, 37), (130, 260, 16), (130, 260, 32), (130, 260, 65), (8192, 200, 32),
                                   (8193, 200, 32), (4096, 200, 64), (4097, 200, 64), (4097, 200, 40)])
def test_lora_down_bit_exact(dev, orc, xdt, pad, M, K, R):
    x, A, _, _ = factors(M, K, R, 1, M + K + R)
    x = x.to(xdt)
    wide = torch.zeros((M, K + pad), dtype=xdt, device=dev)
    wide[:, :K] = x.to(dev)
    h = Q.lora_down(wide[:, :K], A.to(dev))
    torch.cuda.synchronize()
    want = orc.lora_down(x.float().numpy(), A.numpy())
    assert np.array_equal(bits(h), want.view(np.int32))


@pytest.mark.parametrize("cdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,R", [(1, 1, 1), (37, 1000, 17), (300, 513, 64), (129, 256, 256), (200, 130, 33), (131, 644, 16),
                                   (70, 1300, 5), (70, 1300, 17)])
def test_lora_rank_add_bit_exact(dev, orc, cdt, M, N, R):
    g = torch.Generator().manual_seed(M * N + R)
    h = torch.randn(M, R, generator=g)
    B = torch.randn(N, R, generator=g) * 0.1
    C = torch.randn(M, N, generator=g).to(cdt)
    Cd = C.to(dev)
    Q.lora_rank_add(h.to(dev), B.to(dev), Cd)
    torch.cuda.synchronize()
    want = orc.lora_rank_add(h.numpy(), B.numpy(), C.float().numpy())
    if cdt == torch.float32:
        assert np.array_equal(bits(Cd), want.view(np.int32))
    else:
        assert torch.equal(Cd.cpu().view(torch.int16), torch.from_numpy(want).to(torch.bfloat16).view(torch.int16))


def test_lora_rank_add_strided_c(dev, orc):
    M, N, R, ldc = 70, 300, 16, 320
    g = torch.Generator().manual_seed(5)
    h, B = torch.randn(M, R, generator=g), torch.randn(N, R, generator=g)
    wide = torch.randn(M, ldc, generator=g)
    Cd = wide.to(dev)
    Q.lora_rank_add(h.to(dev), B.to(dev), Cd[:, :N])
    torch.cuda.synchronize()
    want = orc.lora_rank_add(h.numpy(), B.numpy(), wide[:, :N].numpy())
    got = Cd.cpu()
    assert np.array_equal(got[:, :N].contiguous().view(torch.int32).numpy(), want.view(np.int32))
    assert torch.equal(got[:, N:], wide[:, N:])  # the padding columns are untouched


def test_lora_tail_after_the_linear(dev, orc):
    """The reference's order: linear_gemm writes fp32 out, apply_lora_tail adds
    the correction (core/models/image_dit.cpp:955-960)."""
    M, K, N, R = 333, 1024, 640, 24
    x = synth.activations(M, K, seed=31).float()
    W = synth.int8_weight(N, K, seed=32)
    sW = torch.rand(N, generator=torch.Generator().manual_seed(33)) * 0.002 + 0.001
    _, A, B, _ = factors(M, K, R, N, 34)
    xd = x.to(dev)
    y = Q.q8_linear(xd, W.to(dev), sW.to(dev), out_dtype=torch.float32)
    h = torch.empty((M, R), dtype=torch.float32, device=dev)
    Q.lora_tail(xd, A.to(dev), B.to(dev), y, h=h)
    torch.cuda.synchronize()
    y0 = orc.q8_linear(x.numpy(), W.numpy(), sW.numpy(), out="f32")[0]
    want = orc.lora_rank_add(orc.lora_down(x.numpy(), A.numpy()), B.numpy(), y0)
    assert np.array_equal(bits(y), want.view(np.int32))


def test_lora_tail_contract(dev):
    x = torch.randn(8, 256, device=dev)
    A, B = torch.randn(4, 256, device=dev), torch.randn(16, 4, device=dev)
    out = torch.zeros(8, 16, device=dev)
    with pytest.raises(Q.QLinearError) as e:
        Q.lora_tail(x, A, B, out, h=torch.empty(8 * 4 - 1, device=dev))
    assert "hidden-form scratch" in str(e.value)
    # an inactive tail (rank 0) leaves out alone
    L = Q.load()
    assert L.phi_hip_lora_tail(None, x.data_ptr(), Q.F32, 256, 8, 256, None, None, 0, 16, out.data_ptr(), Q.F32,
                               16, None, 0) == 0
    torch.cuda.synchronize()
    assert torch.count_nonzero(out) == 0


def test_lora_tail_full_size_rows_sampled(dev, orc):
    """Config 1's up-projection with a rank-64 correction; rows sampled for the oracle."""
    M, K, N, R = 4352, 3072, 12288, 64
    g = torch.Generator(device=dev).manual_seed(7)
    x = torch.randn(M, K, generator=g, device=dev)
    A = torch.randn(R, K, generator=g, device=dev) * 0.02
    B = torch.randn(N, R, generator=g, device=dev) * 0.02
    out = torch.randn(M, N, generator=g, device=dev)
    out0 = out.clone()
    Q.lora_tail(x, A, B, out)
    torch.cuda.synchronize()
    rows = torch.tensor([0, 1, 255, 256, 2049, 4095, 4096, 4351])
    xs = x[rows.to(dev)].cpu().numpy()
    want = orc.lora_rank_add(orc.lora_down(xs, A.cpu().numpy()), B.cpu().numpy(), out0[rows.to(dev)].cpu().numpy())
    assert np.array_equal(out[rows.to(dev)].cpu().contiguous().view(torch.int32).numpy(), want.view(np.int32))


def test_lora_down_both_forms_agree(dev, orc):
    """Rows whose base and pitch allow four-column loads, and the same rows 4
    bytes further on at an odd pitch (one element a load)."""
    M, K, R = 130, 512, 40
    x, A, _, _ = factors(M, K + 1, R, 1, 77)
    A = A[:, :K].contiguous()
    xd = x.to(dev)
    h_vec = Q.lora_down(xd[:, :K].contiguous(), A.to(dev))
    h_gen = Q.lora_down(xd[:, 1:], A.to(dev))  # base 4 bytes in, row pitch K + 1
    torch.cuda.synchronize()
    assert np.array_equal(bits(h_vec), orc.lora_down(x[:, :K].numpy(), A.numpy()).view(np.int32))
    assert np.array_equal(bits(h_gen), orc.lora_down(x[:, 1:].contiguous().numpy(), A.numpy()).view(np.int32))


@pytest.mark.parametrize("cdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,K,N,R", [(15, 64, 4, 4), (17, 68, 128, 16), (64, 448, 132, 20), (65, 4, 124, 32),
                                     (1031, 392, 260, 36), (2100, 260, 8, 130), (16400, 64, 12, 8)])
def test_lora_tiles_bit_exact(dev, orc, cdt, M, K, N, R):
    """Edges of the tiles: rows and ranks around 16 and 64, columns around 64
    and 128, K around the 64-column chunks, one chain a wave and two (above
    1024 16 x 16 tiles), with denormal, zero and negative-zero operands."""
    x, A, B, out = factors(M, K, R, N, M + 7 * K + R)
    x[0] *= 1e-38
    x[-1] = -0.0
    A[:, ::3] = 0.0
    B[N // 2] = -0.0
    out[-1] = -0.0
    x, out = x.to(cdt), out.to(cdt)
    y = out.to(dev)
    h = torch.empty((M, R), dtype=torch.float32, device=dev)
    Q.lora_tail(x.to(dev), A.to(dev), B.to(dev), y, h=h)
    torch.cuda.synchronize()
    hw = orc.lora_down(x.float().numpy(), A.numpy())
    assert np.array_equal(bits(h), hw.view(np.int32))
    want = orc.lora_rank_add(hw, B.numpy(), out.float().numpy())
    if cdt == torch.float32:
        assert np.array_equal(bits(y), want.view(np.int32))
    else:
        assert torch.equal(y.cpu().view(torch.int16), torch.from_numpy(want).to(torch.bfloat16).view(torch.int16))


@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,K,R", [(1, 64, 1), (65, 64, 17), (129, 64, 130), (70, 16, 5), (70, 32, 40), (70, 48, 33), (70, 144, 16), (64, 128, 16), (70, 192, 9), (1024, 192, 17), (1025, 192, 17),
                                   (16384, 256, 8), (16385, 256, 8), (16385, 1024, 3), (16385, 256, 9)])
def test_lora_down_one_row_a_lane(dev, orc, xdt, M, K, R):
    """Both sides of the lines between the chains of one row a lane and the
    matrix-core tiles: few columns, or few ranks of many rows."""
    x, A, _, _ = factors(M, K, R, 1, M + 3 * K + R)
    x[0] *= 1e-38
    x[-1] = -0.0
    A[:, ::3] = 0.0
    x = x.to(xdt)
    h = Q.lora_down(x.to(dev), A.to(dev))
    torch.cuda.synchronize()
    assert np.array_equal(bits(h), orc.lora_down(x.float().numpy(), A.numpy()).view(np.int32))


def same_values(got, want):
    """The same bits, NaN payloads and signs aside."""
    g, w = got.float().cpu().numpy(), np.asarray(want, dtype=np.float32)
    nan = np.isnan(w)
    return np.array_equal(np.isnan(g), nan) and np.array_equal(g.view(np.int32)[~nan], w.view(np.int32)[~nan])


# The matrix-core tiles (K > 64, R > 16: one and two chains a wave, with and
# without four-column loads) and the chains of one row a lane (K = 64).
@pytest.mark.parametrize("M,K,R", [(40, 328, 20), (40, 333, 20), (8200, 324, 20), (40, 64, 20)])
def test_lora_tail_non_finite(dev, orc, M, K, R):
    """Infinities, NaN, and chains that overflow on the way, in both passes."""
    N = 132
    x, A, B, out = factors(M, K, R, N, K)
    inf, big = float("inf"), 3e38
    x[1, 5], x[2, K - 1], x[M - 2, 3] = inf, float("nan"), -inf
    x[3, 0], x[3, 9] = inf, -inf          # NaN unless A's signs differ
    x[4, :4] = big
    A[3, :4] = 2.0                        # overflows to inf, then meets -inf
    A[4, :4] = torch.tensor([0.5, 0.5, 0.5, -0.5])
    A[6], A[7, 2] = 0.0, inf              # 0 * inf; finite * inf
    x[5], A[8] = 1e30, 1e10               # every product overflows
    B[2, 1], B[3, 0], B[5], B[9, R - 1] = inf, float("nan"), 0.0, -inf
    out[6], out[7, ::2], out[8, 3] = inf, -inf, float("nan")
    B[11], out[9] = 1e30, -big
    y = out.to(dev)
    h = torch.empty((M, R), dtype=torch.float32, device=dev)
    Q.lora_tail(x.to(dev), A.to(dev), B.to(dev), y, h=h)
    torch.cuda.synchronize()
    hw = orc.lora_down(x.numpy(), A.numpy())
    assert np.isinf(hw).any() and np.isnan(hw).any() and same_values(h, hw)
    want = orc.lora_rank_add(hw, B.numpy(), out.numpy())
    assert np.isinf(want).any() and same_values(y, want)
