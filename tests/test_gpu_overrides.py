"""Environment overrides that pick the dense route: what was asked for runs also at the row
counts of the mid-row kernel (33..128). Each runs in a process of its own, since the library
reads its environment once."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle as O
from helpers import to_dev_bf16, to_dev_u32, to_f64, weights
import mi_qmm

pytestmark = pytest.mark.gpu

N, K = 256, 512


def _err(dev, M, bits):
    """Relative 2-norm error of one call, and the vendor GEMM calls that it made."""
    (wq, s, b), x = [a[0] for a in weights(1, N, K, bits, 64, 5)], O.make_x_bf16(M, K, 6)
    before = mi_qmm.library_gemm_calls()
    y = mi_qmm.quantized_matmul(to_dev_bf16(x, dev), to_dev_u32(wq, dev), to_dev_bf16(s, dev),
                                to_dev_bf16(b, dev), True, 64, bits)
    truth = O.qmm_f64(x, wq, s, b, 64, bits)
    return (float(np.linalg.norm(to_f64(y) - truth) / np.linalg.norm(truth)),
            mi_qmm.library_gemm_calls() - before)


def _under(env, M, bits):
    here = os.path.dirname(os.path.abspath(__file__))
    code = ("import conftest, json, torch, test_gpu_overrides as t; "
            f"print('RESULT', json.dumps(t._err(torch.device('cuda:0'), {M}, {bits})))")
    r = subprocess.run([sys.executable, "-c", code], cwd=here, env={**os.environ, **env},
                       capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout.split("RESULT")[1])


def test_vendor_gemm_on_request(dev):
    """MI_QMM_DQGEMM=1: 6-bit weights above the few-row limit go through the vendor GEMM."""
    assert _err(dev, 64, 6)[1] == 0
    err, calls = _under({"MI_QMM_DQGEMM": "1"}, 64, 6)
    assert calls == 1 and err < 5e-3


def test_prefill_from_fewer_rows(dev):
    """MI_QMM_PREFILL_MIN=64: the prefill kernel, which rounds the weights to bf16. The exact codes
    of the default route leave one rounding of the output (half of 2^-7 of its binade, about 1.6e-3
    in the 2-norm); rounded weights add an independent error of the same size (times sqrt(2))."""
    exact, _ = _err(dev, 64, 4)
    err, calls = _under({"MI_QMM_PREFILL_MIN": "64"}, 64, 4)
    assert calls == 0 and 1.2 * exact < err < 5e-3
