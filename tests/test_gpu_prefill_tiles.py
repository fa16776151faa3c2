"""Prefill GEMM (129 rows and more) against the oracle at the edges of both of its tile heights:
row counts around 128 and 256, widths that end inside a tile, K ranges that end inside a 4-step
unit of the 128-row tiles, odd group counts (another kernel), K splits of either, and grids of more than one round of blocks."""
import pytest
import torch

import oracle as O
from helpers import BF16_TOL, max_err_ratio, to_dev_bf16, to_dev_u32, to_f64, weights
import mi_qmm

pytestmark = pytest.mark.gpu


def _check(dev, M, N, K, bits, gs):
    print("CASE", dict(t="prefill_tiles", M=M, N=N, K=K, bits=bits, gs=gs), flush=True)
    wq, s, b = weights(1, N, K, bits, gs, M + N + K)
    x = O.make_x_bf16(M, K, M + N)
    y = mi_qmm.quantized_matmul(to_dev_bf16(x, dev), to_dev_u32(wq[0], dev), to_dev_bf16(s[0], dev),
                                to_dev_bf16(b[0], dev), True, gs, bits)
    assert max_err_ratio(to_f64(y), O.qmm_f64(x, wq[0], s[0], b[0], gs, bits)) <= BF16_TOL


# 2 steps and grids of 256-row tiles; one unit, a part of one, several; 2 and 4 splits
@pytest.mark.parametrize("M,N,K", [(129, 4, 128), (129, 256, 256), (256, 260, 384), (257, 36, 640),
                                   (384, 516, 1408), (129, 100, 2816)])
@pytest.mark.parametrize("bits,gs", [(4, 32), (4, 64), (4, 128), (8, 32), (8, 64), (8, 128),
                                     (3, 64), (6, 64)])
def test_edges(dev, M, N, K, bits, gs):
    _check(dev, M, N, K, bits, gs)


# 256-row tiles: 153 of them in one round against 289 of 128 rows in two; and three K splits
@pytest.mark.parametrize("M,N,K,bits", [(2052, 4100, 640, 4), (2052, 4100, 640, 8),
                                        (2052, 4100, 640, 6), (1100, 4096, 7168, 4)])
def test_tall(dev, M, N, K, bits):
    _check(dev, M, N, K, bits, 64)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("K", [256, 640])
def test_rows_and_columns_are_independent(dev, bits, K):
    """Infinite and NaN activations stay in their rows, an infinite scale in its column."""
    M, N = 131, 264
    wq, s, b = weights(1, N, K, bits, 64, 9)
    x = O.make_x_bf16(M, K, 10)
    w = to_dev_u32(wq[0], dev)
    bd = to_dev_bf16(b[0], dev)
    clean = mi_qmm.quantized_matmul(to_dev_bf16(x, dev), w, to_dev_bf16(s[0], dev), bd, True, 64, bits)
    xi, si = x.copy(), s[0].copy()
    xi[3, 5], xi[130, K - 1] = 0x7F80, 0x7FC0
    si[41, 0] = si[257, 0] = 0x7F80
    y = mi_qmm.quantized_matmul(to_dev_bf16(xi, dev), w, to_dev_bf16(si, dev), bd, True, 64, bits)
    rows = [m for m in range(M) if m not in (3, 130)]
    cols = [n for n in range(N) if n not in (41, 257)]
    assert torch.equal(y[rows][:, cols], clean[rows][:, cols])
    assert not torch.isfinite(y[3].float()).any() and not torch.isfinite(y[130].float()).any()
