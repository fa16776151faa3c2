"""Grouped expert GEMM (sorted gather_qmm with several rows per expert) against the oracle: run
lengths around its 16-, 32- and 64-row items, output widths that end inside a block, one step
unit of K and several, and blocks of two passes over the output."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import BF16_TOL, max_err_ratio, to_dev_bf16, to_dev_u32, to_f64, weights
import mi_qmm

pytestmark = pytest.mark.gpu

RUNS = {32: [1, 15, 16, 17, 31, 32, 33, 0], 64: [1, 31, 32, 33, 63, 64, 65, 0]}


def _case(N, K, rows, seed):
    runs = RUNS[rows]
    rhs = np.repeat(np.arange(len(runs)), runs).astype(np.uint32)
    return rhs, weights(len(runs), N, K, 4, 64, seed), O.make_x_bf16(len(rhs), K, seed + 1)


@pytest.mark.parametrize("N,K", [(4, 256), (36, 768), (260, 2048), (12420, 256)])
@pytest.mark.parametrize("rows", [32, 64])
def test_runs(dev, N, K, rows):
    print("CASE", dict(t="gmm_runs", N=N, K=K, rows=rows), flush=True)
    rhs, (wq, s, b), x = _case(N, K, rows, N + K)
    y = mi_qmm.gather_qmm(to_dev_bf16(x, dev).view(len(rhs), 1, K), to_dev_u32(wq, dev),
                          to_dev_bf16(s, dev), to_dev_bf16(b, dev),
                          rhs_indices=to_dev_u32(rhs, dev), group_size=64, bits=4,
                          sorted_indices=True).view(len(rhs), N)
    truth = np.concatenate([O.qmm_f64(x[rhs == e], wq[e], s[e], b[e], 64, 4)
                            for e in range(len(wq)) if (rhs == e).any()])
    assert max_err_ratio(to_f64(y), truth) <= BF16_TOL


@pytest.mark.parametrize("N,K", [(4, 256), (100, 768)])
@pytest.mark.parametrize("rows", [32, 64])
def test_dual_matches_separate_products(dev, N, K, rows):
    """gate + up + SwiGLU in one launch: the same products, so the same bits."""
    rhs, (wq, s, b), x = _case(N, K, rows, 3 * N + K)
    up = [to_dev_u32(wq, dev), to_dev_bf16(s, dev), to_dev_bf16(b, dev)]
    gate = [t.flip(0).contiguous() for t in up]
    xd, r = to_dev_bf16(x, dev).view(len(rhs), 1, K), to_dev_u32(rhs, dev)
    kw = dict(rhs_indices=r, group_size=64, bits=4, sorted_indices=True)
    y = mi_qmm.gather_qmm_gate_up_swiglu(xd, *gate, *up, **kw)
    ref = mi_qmm.swiglu(mi_qmm.gather_qmm(xd, *gate, **kw), mi_qmm.gather_qmm(xd, *up, **kw))
    assert torch.equal(y.view(torch.int16), ref.view(torch.int16))


def test_two_passes_a_block(dev):
    """A count of blocks a little over a round (three a CU), where a block makes two passes over
    the output: 235 tiles of 128 rows x about 3.7 items of one expert; the last block has one pass
    that ends inside a tile."""
    N, K, T = 30020, 512, 200
    rng = np.random.default_rng(3)
    wq = rng.integers(0, 1 << 32, size=(1, N, K // 8), dtype=np.uint32)
    s = O.f32_to_bf16(rng.uniform(0.05, 0.1, size=(1, N, K // 64)).astype(np.float32))
    b = O.f32_to_bf16(rng.uniform(-0.6, -0.4, size=(1, N, K // 64)).astype(np.float32))
    x, rhs = O.make_x_bf16(T, K, 4), np.zeros(T, np.uint32)
    y = mi_qmm.gather_qmm(to_dev_bf16(x, dev).view(T, 1, K), to_dev_u32(wq, dev), to_dev_bf16(s, dev),
                          to_dev_bf16(b, dev), rhs_indices=to_dev_u32(rhs, dev), group_size=64,
                          bits=4, sorted_indices=True).view(T, N)
    cols = np.unique(np.concatenate([np.arange(260), rng.integers(0, N, 300), np.arange(N - 300, N)]))
    truth = O.qmm_f64(x, wq[0][cols], s[0][cols], b[0][cols], 64, 4)
    assert max_err_ratio(to_f64(y[:, cols]), truth) <= BF16_TOL


def test_scales_on_an_odd_half(dev):
    """Banks whose scales and biases start on an odd half: the same bits as aligned ones."""
    rhs, (wq, s, b), x = _case(100, 768, 64, 11)

    def off(t):
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=dev)
        v = buf[1:].view(t.shape)
        v.copy_(t)
        return v
    xd, r = to_dev_bf16(x, dev).view(len(rhs), 1, 768), to_dev_u32(rhs, dev)
    W, S, B = to_dev_u32(wq, dev), to_dev_bf16(s, dev), to_dev_bf16(b, dev)
    kw = dict(rhs_indices=r, group_size=64, bits=4, sorted_indices=True)
    ref = mi_qmm.gather_qmm(xd, W, S, B, **kw)
    y = mi_qmm.gather_qmm(xd, W, off(S), off(B), **kw)
    assert torch.equal(y.view(torch.int16), ref.view(torch.int16))
