"""GPU parity of the int8-plane k-quant GEMM (csrc/gemm_kq.hip): MUL_MAT with
more than 16 columns, through the C ABI, against the oracle.

The super-block sums are exact integers, so an output may differ from the exact
value of the same codes only by f32 rounding: each of its nsb super-blocks adds
a product formed in at most four rounded steps, and the additions (in any
order, with K chunks) round once each. The bound per element is therefore
(nsb + 8) * 2^-23 * sum |w| |x| over the dequantized operands, and the oracle's
own sequential f32 sum is allowed as much again.
"""
from __future__ import annotations

import numpy as np
import pytest

from refs import NAMES, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, oracle
from tensorlisp_amd import native as N
from tensorlisp_amd import synth

pytestmark = pytest.mark.gpu
TYPES = (Q2_K, Q3_K, Q4_K, Q5_K, Q6_K)


def dev(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def bound(t, w, K, x):
    o = oracle()
    wd = np.abs(o.dequantize(t, w, K)).astype(np.float64)
    if t in (Q2_K, Q4_K, Q5_K):  # scale and min terms are added apart: their sizes, not their difference's
        wd = wd + 2 * np.abs(wd).max()
    return 2 * (K // 256 + 8) * 2.0 ** -23 * (np.abs(x).astype(np.float64) @ wd.T) * (128 / 127)


def check(t, w, M, K, x, what):
    import torch

    print(f"[gemm_kq] {what}", flush=True)
    y = N.mul_mat(t, dev(w), M, K, dev(x))
    torch.cuda.synchronize()
    want = oracle().mul_mat(t, w, M, K, x, nthreads=16)
    err = np.abs(y.cpu().numpy().astype(np.float64) - want)
    lim = bound(t, w, K, x)
    assert (err <= lim).all(), f"{what}: max err {err.max():.3e}, worst {(err / lim).max():.2f} of the bound"


@pytest.mark.parametrize("t", TYPES, ids=[NAMES[t] for t in TYPES])
@pytest.mark.parametrize("M,K,n", [(1, 256, 17), (63, 512, 32), (65, 1280, 33), (64, 256, 64), (129, 768, 65),
                                   (200, 512, 128), (130, 256, 129), (96, 5120, 40), (257, 2560, 260)])
def test_tiles_and_tails(gpu, t, M, K, n):
    """Edges of the 64 x 32, 64 x 64 and 128 x 128 tiles in rows and tokens, one
    super-block up to K chunks of several."""
    w = synth.random_blocks(t, 31 * M + K, M, K)
    check(t, w, M, K, synth.normal(n, (n, K)), f"{NAMES[t]} {M}x{K} n={n}")


@pytest.mark.parametrize("t", TYPES, ids=[NAMES[t] for t in TYPES])
@pytest.mark.parametrize("n", [20, 50, 70])
def test_extreme_codes(gpu, t, n):
    """Scales and codes at the ends of their ranges (q3_K's -32 * -4 and q6_K's
    -128 * -32 are the largest scaled codes) against activation codes of +-127."""
    M, K = 70, 512
    w = synth.random_blocks(t, 5, M, K).reshape(-1, N.BLOCK[t][1]).copy()
    sc = {Q2_K: slice(0, 16), Q3_K: slice(96, 108), Q4_K: slice(4, 16), Q5_K: slice(4, 16), Q6_K: slice(192, 208)}[t]
    fill = {Q2_K: (0xFF, 0x0F), Q3_K: (0x00, 0xFF), Q4_K: (0xFF, 0x3F), Q5_K: (0xFF, 0x3F), Q6_K: (0x80, 0x7F)}[t]
    d = {Q2_K: slice(80, 84), Q3_K: slice(108, 110), Q4_K: slice(0, 4), Q5_K: slice(0, 4), Q6_K: slice(208, 210)}[t]
    keep = w[:, d].copy()
    for i in range(w.shape[0]):
        w[i] = 0x00 if i % 3 == 0 else 0xFF if i % 3 == 1 else w[i]
        w[i, sc] = fill[i % 2]
    w[:, d] = keep
    w = w.reshape(M, -1)
    x = np.sign(synth.normal(8, (n, K))).astype(np.float32)
    x[0] = 1.0
    check(t, w, M, K, x, f"{NAMES[t]} extremes n={n}")


@pytest.mark.parametrize("t", TYPES, ids=[NAMES[t] for t in TYPES])
def test_batches_broadcast_and_strided_rows(gpu, t):
    """Four src1 slices over two weight matrices (r2 = 2), weight rows padded."""
    import torch

    M, K, n = 70, 512, 21
    rb = N.row_bytes(t, K)
    w = synth.random_blocks(t, 77, 2 * M, K)
    pad = np.zeros((2 * M, rb + 6), np.uint8)
    pad[:, :rb] = w
    x = synth.normal(3, (4, n, K))
    op = N.mul_mat_op(t, M, K, n, ne2=4, w_ne2=2, w_nb=[N.BLOCK[t][1], rb + 6, M * (rb + 6), 2 * M * (rb + 6)])
    mm = N.MulMat(t, M, K, n, op=op)
    y = torch.empty((4, n, M), dtype=torch.float32, device="cuda")
    mm(dev(pad), dev(x), y)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    for b in range(4):
        wb = w[(b // 2) * M:(b // 2 + 1) * M]
        want = oracle().mul_mat(t, wb, M, K, x[b])
        assert (np.abs(got[b] - want) <= bound(t, wb, K, x[b])).all(), b


def q8_K_codes(x):
    """(scales [n, K / 256] f32, codes [n, K]) of x's q8_K rows."""
    n, K = x.shape
    b = oracle().quantize_act(Q4_K, x).reshape(n, K // 256, -1)
    return np.ascontiguousarray(b[:, :, :4]).view(np.float32)[:, :, 0], b[:, :, 4:260].copy().view(np.int8).reshape(n, K)


def short_chains(t, w, K, x, length=4):
    """(x @ w.T of the op's codes in 64 bits, the same in f32: each super-block's
    term formed in its three or four roundings and added in chains of `length`,
    the chains' sums after one another)."""
    rows, n, bb = w.shape[0], x.shape[0], N.BLOCK[t][1]
    parts = []  # the weights' scale part and min part, each exact in f32
    for drop in ((2, 4), (0, 2)):
        b = w.reshape(-1, bb).copy()
        if t in (Q4_K, Q5_K):
            b[:, drop[0]:drop[1]] = 0
        parts.append(oracle().dequantize(t, b.reshape(rows, -1), K).astype(np.float64))
    d8, q8 = q8_K_codes(x)
    f32 = np.float32
    exact = np.zeros((n, rows))
    total, chain = np.zeros((n, rows), f32), np.zeros((n, rows), f32)
    for sb in range(K // 256):
        s = slice(256 * sb, 256 * sb + 256)
        q, dy = q8[:, s].astype(np.float64), d8[:, sb, None].astype(np.float64)
        a = q @ parts[0][:, s].T
        m = q @ parts[1][:, s].T if t in (Q4_K, Q5_K) else np.zeros_like(a)
        exact += dy * (a + m)
        v = (a + m.astype(f32)).astype(f32)  # (a fused multiply-add)
        chain = (chain + dy * v).astype(f32)
        if (sb + 1) % length == 0 or sb == K // 256 - 1:
            total, chain = total + chain, np.zeros_like(chain)
    return exact, total


def check_sums(got, exact, total, what):
    """got's error, root mean square over the outputs, is total's. 5% for chance
    (8192 outputs and more: 0.8% standard deviation)."""
    rms = lambda e: np.sqrt(np.mean(e ** 2) / np.mean(exact ** 2))  # noqa: E731
    print(f"{what}: {rms(got - exact):.3e}, short chains {rms(total - exact):.3e}", flush=True)
    assert rms(got - exact) <= 1.05 * rms(total - exact)


@pytest.mark.parametrize("t", [Q3_K, Q4_K, Q5_K, Q6_K], ids=lambda t: NAMES[t])
@pytest.mark.parametrize("copies,K,n", [(1, 512, 20), (1, 512, 40), (1, 4096, 32), (28, 14336, 32), (28, 14336, 48), (63, 4096, 64), (8, 4096, 256)])
def test_sums_are_as_exact_as_short_chains(gpu, t, copies, K, n):
    """One chain over K = 14336 is 1.3 times as far off, K steps of one super-block
    finished apart 1.08 times."""
    import torch

    rows = 512 if n < 100 else 64
    w, x = synth.random_blocks(t, K + n, rows, K), synth.normal(n, (n, K))
    M = copies * rows
    y = N.mul_mat(t, dev(np.tile(w, (copies, 1))), M, K, dev(x))
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(n, copies, rows)[:, -1].astype(np.float64)
    check_sums(got, *short_chains(t, w, K, x), f"[gemm_kq] {NAMES[t]} {M}x{K} n={n}")
