"""GPU parity of the q8_0 / q4_0 GEMM's tile shapes (csrc/gemm_q8.hip): MUL_MAT
with more than 16 columns, through the C ABI, against the oracle.

Block dots are exact integers; an output differs from the exact value of the
same codes by f32 rounding only. A block adds a product formed in three rounded
steps, and the additions (in any order, with K chunks and the waves' shares of
a stage) round once each, so the bound per element is (nblk + 8) * 2^-23 * sum
|w| |x|, and the oracle's own sequential sum is allowed as much again (128 /
127: the activation codes' rounding).
"""
from __future__ import annotations

import numpy as np
import pytest

from refs import NAMES, Q4_0, Q8_0, oracle
from tensorlisp_amd import native as N
from tensorlisp_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", (Q8_0, Q4_0), ids=("q8_0", "q4_0"))
@pytest.mark.parametrize("M,K,n", [(1, 32, 17), (63, 96, 32), (65, 128, 33), (64, 160, 64), (129, 2208, 31), (100, 4096, 40),
                                   (130, 224, 65), (257, 5120, 20), (70, 1024, 129)])
def test_tiles_and_tails(gpu, t, M, K, n):
    """Edges of the 64 x 32, 64 x 64 and 128 x 128 tiles in rows and tokens; K of
    part of a stage (one block) up to several K chunks."""
    import torch

    print(f"[gemm_q8] {NAMES[t]} {M}x{K} n={n}", flush=True)
    o = oracle()
    w, x = synth.random_blocks(t, 31 * M + K, M, K), synth.normal(n, (n, K))
    y = N.mul_mat(t, torch.from_numpy(w).cuda(), M, K, torch.from_numpy(x).cuda())
    torch.cuda.synchronize()
    want = o.mul_mat(t, w, M, K, x, nthreads=16)
    lim = 2 * (K // 32 + 8) * 2.0 ** -23 * (np.abs(x).astype(np.float64) @ np.abs(o.dequantize(t, w, K)).astype(np.float64).T)
    lim = lim * (128 / 127) + 1e-30
    err = np.abs(y.cpu().numpy().astype(np.float64) - want)
    assert (err <= lim).all(), f"max err {err.max():.3e}, worst {(err / lim).max():.2f} of the bound"
