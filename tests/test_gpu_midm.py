"""The mid-row kernel (33..128 rows, and 17..32 on wide shapes) against the oracle where its tiling
can go wrong: row counts around each 32-row tile, output widths that end inside a block, K ranges
that do not divide into the waves' steps (odd group counts, so a row's scales start in the middle of
a dword), and splits over blocks; and the layouts beside it that take other kernels."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import BF16_TOL, max_err_ratio, to_dev_bf16, to_dev_u32, to_f64, weights
import mi_qmm

pytestmark = pytest.mark.gpu

SHAPES = [(64, 64), (36, 192), (100, 960), (260, 1088), (4096, 128), (128, 7168)]


def _run(dev, M, N, K, bits, seed):
    wq, s, b = weights(1, N, K, bits, 64, seed)
    x = O.make_x_bf16(M, K, seed + 1)
    y = mi_qmm.quantized_matmul(to_dev_bf16(x, dev), to_dev_u32(wq[0], dev),
                                to_dev_bf16(s[0], dev), to_dev_bf16(b[0], dev), True, 64, bits)
    return x, (wq[0], s[0], b[0]), y


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("N,K", SHAPES)
@pytest.mark.parametrize("M", [17, 32, 33, 64, 65, 96, 97, 128])
def test_rows_and_tails(dev, M, N, K, bits):
    """(17 and 32 rows of these narrow shapes run on the few-row kernel, with the same bound.)"""
    print("CASE", dict(t="midm", M=M, N=N, K=K, bits=bits), flush=True)
    x, w, y = _run(dev, M, N, K, bits, 100 * M + N)
    truth = O.qmm_f64(x, *w, 64, bits)
    err = to_f64(y) - truth
    assert max_err_ratio(to_f64(y), truth) <= BF16_TOL
    if M <= 64:
        # exact codes and fp32 sums: what is left is one bf16 rounding of the result, half of 2^-7
        # of its binade at most (uniform: 2^-7 / sqrt(12), over values spread evenly on a log scale
        # 1.5e-3 in the 2-norm, below 2^-9), and fp32 sums 1000 times smaller
        assert np.linalg.norm(err) <= 2.0 ** -9 * 1.01 * np.linalg.norm(truth)


# Wide enough that 17..32 rows take this kernel (one 32-row tile): widths that end inside a block
# of 64 rows, K ranges that end inside a wave's steps, K splits over blocks, and (2560) blocks of
# 32 rows.
@pytest.mark.parametrize("N,K,bits", [(14340, 4224, 4), (14340, 4224, 8), (5124, 5120, 4),
                                      (4100, 14336, 8), (6148, 2560, 8)])
def test_few_rows_of_wide_shapes(dev, N, K, bits):
    G, rng = K // 64, np.random.default_rng(N + bits)
    wq = rng.integers(0, 1 << 32, size=(N, K * bits // 32), dtype=np.uint32)
    s = O.f32_to_bf16(rng.uniform(0.5, 1.5, size=(N, G)).astype(np.float32) / 2 ** bits)
    b = O.f32_to_bf16(rng.uniform(-0.6, -0.4, size=(N, G)).astype(np.float32))
    x = O.make_x_bf16(48, K, N)
    cols = np.unique(np.concatenate([np.arange(40), rng.integers(0, N, 60), np.arange(N - 70, N)]))
    truth = O.qmm_f64(x, wq[cols], s[cols], b[cols], 64, bits)
    X, W, S, B = to_dev_bf16(x, dev), to_dev_u32(wq, dev), to_dev_bf16(s, dev), to_dev_bf16(b, dev)
    for M in (17, 31, 32, 33, 48):
        print("CASE", dict(t="midm_few", M=M, N=N, K=K, bits=bits), flush=True)
        y = to_f64(mi_qmm.quantized_matmul(X[:M].contiguous(), W, S, B, True, 64, bits)[:, cols])
        # one bf16 rounding of the result, as above
        assert np.linalg.norm(y - truth[:M]) <= 2.0 ** -9 * 1.01 * np.linalg.norm(truth[:M])


@pytest.mark.parametrize("bits", [4, 8])
def test_rows_are_independent(dev, bits):
    """Infinite and NaN activations stay in their rows, and scales of the next weight row (read
    with a row's last group where the K range ends) never reach this one."""
    M, N, K = 40, 72, 320
    wq, s, b = weights(1, N, K, bits, 64, 9)
    x = O.make_x_bf16(M, K, 10)
    clean = mi_qmm.quantized_matmul(to_dev_bf16(x, dev), to_dev_u32(wq[0], dev), to_dev_bf16(s[0], dev),
                                    to_dev_bf16(b[0], dev), True, 64, bits)
    xi = x.copy()
    xi[3, 5], xi[39, 70] = 0x7F80, 0x7FC0
    si = s[0].copy()
    si[41, 0] = 0x7F80
    y = mi_qmm.quantized_matmul(to_dev_bf16(xi, dev), to_dev_u32(wq[0], dev), to_dev_bf16(si, dev),
                                to_dev_bf16(b[0], dev), True, 64, bits)
    rows = [m for m in range(M) if m not in (3, 39)]
    cols = [n for n in range(N) if n != 41]
    assert torch.equal(y[rows][:, cols], clean[rows][:, cols])
    assert not torch.isfinite(y[3].float()).any() and not torch.isfinite(y[39].float()).any()


def test_unaligned_pointers_take_another_route(dev):
    """Views that start off a 16-byte (x, w) or dword (scales, biases) boundary still give the result."""
    M, N, K = 48, 128, 512
    x, (wq, s, b), y = _run(dev, M, N, K, 4, 77)

    def off(t, n):
        buf = torch.empty(t.numel() + n, dtype=t.dtype, device=dev)
        v = buf[n:].view(t.shape)
        v.copy_(t)
        return v
    X, W, S, B = (to_dev_bf16(x, dev), to_dev_u32(wq, dev), to_dev_bf16(s, dev), to_dev_bf16(b, dev))
    truth = O.qmm_f64(x, wq, s, b, 64, 4)
    for args in ((off(X, 4), W, S, B), (X, off(W, 1), S, B), (X, W, off(S, 1), B), (X, W, S, off(B, 1))):
        assert max_err_ratio(to_f64(mi_qmm.quantized_matmul(*args, True, 64, 4)), truth) <= BF16_TOL


@pytest.mark.parametrize("bits", [4, 8])
def test_widths_off_four_columns(dev, bits):
    """33..64 rows of a wide output that is no multiple of 4 columns: two launches of the few-row
    kernel, with the bits of the separate calls."""
    N, K = 24578, 512
    rng = np.random.default_rng(bits)
    wq = rng.integers(0, 1 << 32, size=(N, K * bits // 32), dtype=np.uint32)
    s = O.f32_to_bf16(rng.uniform(0.5, 1.5, size=(N, K // 64)).astype(np.float32) / 2 ** bits)
    b = O.f32_to_bf16(rng.uniform(-0.6, -0.4, size=(N, K // 64)).astype(np.float32))
    x = O.make_x_bf16(64, K, 7)
    X, w = to_dev_bf16(x, dev), (to_dev_u32(wq, dev), to_dev_bf16(s, dev), to_dev_bf16(b, dev))
    mm = lambda t: mi_qmm.quantized_matmul(t.contiguous(), *w, True, 64, bits)
    cols = np.concatenate([np.arange(130), np.arange(N - 130, N)])
    truth = O.qmm_f64(x, wq[cols], s[cols], b[cols], 64, bits)
    for M in (34, 48, 64):
        print("CASE", dict(t="off_four", M=M, bits=bits), flush=True)
        y = mm(X[:M])
        assert torch.equal(y.view(torch.int16), torch.cat([mm(X[:32]), mm(X[32:M])]).view(torch.int16))
        assert max_err_ratio(to_f64(y[:, cols]), truth[:M]) <= BF16_TOL


@pytest.mark.parametrize("fmt", [2, 3, 5, 6, "nvfp4", "mxfp4", "mxfp8"])
@pytest.mark.parametrize("N,K", [(36, 192), (260, 1088), (4096, 128), (128, 3584)])
@pytest.mark.parametrize("M", [33, 64, 65, 128])
def test_other_formats(dev, fmt, M, N, K):
    print("CASE", dict(t="midm_fmt", fmt=fmt, M=M, N=N, K=K), flush=True)
    x = O.make_x_bf16(M, K, M + N)
    if isinstance(fmt, int):
        wq, s, b = weights(1, N, K, fmt, 64, 50 + fmt)
        y = mi_qmm.quantized_matmul(to_dev_bf16(x, dev), to_dev_u32(wq[0], dev), to_dev_bf16(s[0], dev),
                                    to_dev_bf16(b[0], dev), True, 64, fmt)
        truth = O.qmm_f64(x, wq[0], s[0], b[0], 64, fmt)
    else:
        _, bits, gs = O.FP_MODES[fmt]
        rng = np.random.default_rng(N + K)
        wq = O.pack(rng.integers(0, 1 << bits, size=(N, K)).astype(np.uint8), bits)
        lo, hi = (0x20, 0x48) if fmt == "nvfp4" else (118, 126)
        sc = rng.integers(lo, hi, size=(N, K // gs)).astype(np.uint8)
        y = mi_qmm.quantized_matmul(to_dev_bf16(x, dev), to_dev_u32(wq, dev),
                                    torch.from_numpy(sc).to(dev), None, True, gs, bits, fmt)
        truth = O.bf16_to_f32(x).astype(np.float64) @ O.dequantize_fp(wq, sc, fmt).astype(np.float64).T
    assert max_err_ratio(to_f64(y), truth) <= BF16_TOL


@pytest.mark.parametrize("mode", ["mxfp4", "mxfp8"])
@pytest.mark.parametrize("M", [33, 128, 129])
def test_scale_bytes_at_the_ends(dev, mode, M):
    """e8m0 byte 255 is infinity (the oracle's reading): a group of non-zero codes under it gives
    +-inf where every product has one sign and NaN where signs mix or a code is zero; bytes
    0..7 (down to 2^-127) give their values. Other weight rows keep theirs."""
    N, K = 36, 256
    _, bits, gs = O.FP_MODES[mode]
    rng = np.random.default_rng(5)
    top = 1 << (bits - 1)  # sign bit
    codes = rng.integers(1, top - 1, size=(N, K)).astype(np.uint8)
    sc = np.full((N, K // gs), 120, np.uint8)
    sc[0, 1] = sc[1, 7] = sc[2, 3] = sc[3, 4] = sc[35, 7] = 255
    codes[1] |= top               # -inf
    codes[2, 3 * gs + 5] = 0      # zero times infinity
    codes[3, 4 * gs + 9] |= top   # mixed signs
    sc[8:16] = np.arange(8)[:, None]
    x = np.abs(O.bf16_to_f32(O.make_x_bf16(M, K, 6))) + 0.5
    x = O.f32_to_bf16(x * np.float32(2.0 ** 30))
    y = to_f64(mi_qmm.quantized_matmul(to_dev_bf16(x, dev), to_dev_u32(O.pack(codes, bits), dev),
                                       torch.from_numpy(sc).to(dev), None, True, gs, bits, mode))
    with np.errstate(invalid="ignore"):
        w = O.dequantize_fp(O.pack(codes, bits), sc, mode).astype(np.float64)
        truth = O.bf16_to_f32(x).astype(np.float64) @ w.T
    assert np.isposinf(truth[:, [0, 35]]).all() and np.isneginf(truth[:, 1]).all()
    assert np.isnan(truth[:, 2:4]).all()
    np.testing.assert_array_equal(y[:, [0, 1, 2, 3, 35]], truth[:, [0, 1, 2, 3, 35]])
    for n in range(4, 35):  # per output column: the scales differ by orders of magnitude
        assert max_err_ratio(y[:, n:n + 1], truth[:, n:n + 1]) <= BF16_TOL, n
