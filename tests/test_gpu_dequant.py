"""bf16 dequantize of the formats expanded in packs of 8 codes, bit for bit against the oracle."""
import numpy as np
import pytest
import torch

import oracle as O
from helpers import bf16_bits, to_dev_u32
import mi_qmm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["nvfp4", "mxfp4", "mxfp8"])
def test_dequantize_every_scale_byte(dev, mode):
    """bf16 dequantize at all 256 scale bytes and every code, against the oracle bit for bit
    (NaN where the oracle has NaN); 5 rows, so the last block of packs is partial."""
    _, bits, gs = O.FP_MODES[mode]
    K = 256 * gs
    rng = np.random.default_rng(3)
    wq = O.pack(rng.integers(0, 1 << bits, size=(5, K)).astype(np.uint8), bits)
    sc = np.stack([rng.permutation(256) for _ in range(5)]).astype(np.uint8)
    got = bf16_bits(mi_qmm.dequantize(to_dev_u32(wq, dev), torch.from_numpy(sc).to(dev), None, mode=mode))
    want = O.dequantize_fp(wq, sc, mode, out_bf16=True)
    nan = (want & 0x7FFF) > 0x7F80
    assert np.array_equal((got & 0x7FFF) > 0x7F80, nan)
    assert np.array_equal(got[~nan], want[~nan])
