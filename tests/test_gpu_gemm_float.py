"""GPU parity: the matrix-core kernels for f32 / f16 / bf16 MUL_MAT (gemm_float.hip)
at the edges of their tiles, K remainders and dispatch, against 64-bit products.

Products are exact in f32, so only the f32 sums round: with at most c additions
on any product's way (an MFMA's own; a split: a wave's blocks of 128 bytes by
fours and 3 tree levels; a tile: blocks by levels of two or four) an output is within
c * 2^-24 * sum_k |w_k x_k|; K <= 2056 gives c < 16, so 1e-6 of that sum (f32: 19,
if all of them rounded one way).
"""
from __future__ import annotations

import pytest

from tensorlisp_amd import native as N

pytestmark = pytest.mark.gpu

# M, K, N, (slices, weight slices): one row of 8; partial 16-byte chunks, blocks and
# waves; every column tile width and its remainder, 16 rows to 128 tiles of 32 and 32
# above; 64 x 64 tiles from 256 of them (N <= 16: 512; f32: N > 32); 128 x 128 tiles
# from 256 (bf16: K > 1024)
SHAPES = [(1, 8, 1, 1, 1), (33, 72, 16, 1, 1), (31, 520, 17, 3, 1), (4097, 264, 31, 1, 1), (4128, 200, 48, 1, 1),
          (100, 1032, 49, 4, 2), (65, 2056, 5, 6, 3), (1030, 40, 1000, 1, 1), (64 * 511 + 1, 24, 9, 1, 1),
          (4129, 72, 9, 1, 1), (16321, 136, 33, 1, 1), (63, 64, 65, 256, 128), (2049, 200, 2000, 1, 1), (129, 72, 127, 128, 128),
          (2049, 1032, 2000, 1, 1)]


def rows(torch, t, pad):
    """The same values in rows pad elements apart from touching."""
    buf = torch.zeros(*t.shape[:-1], t.shape[-1] + pad, dtype=t.dtype, device=t.device)
    buf[..., :t.shape[-1]] = t
    return buf[..., :t.shape[-1]]


@pytest.mark.parametrize("M,K,n,b,wb", SHAPES)
@pytest.mark.parametrize("name", ["f32", "f16", "bf16"])
def test_against_64_bits_and_the_general_kernel(gpu, name, M, K, n, b, wb):
    """Aligned rows (matrix cores; one launch, and conversion + products) and rows
    an odd number of elements apart (the element-wise kernel)."""
    import torch

    dt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[name]
    g = torch.Generator(device="cuda").manual_seed(M * 31 + K + n)
    w = torch.randn(1, wb, M, K, device="cuda", generator=g).to(dt)
    x = torch.randn(1, b, n, K, device="cuda", generator=g)
    xd = x.to(dt).double()
    wd = w.double().repeat_interleave(b // wb, 1)
    want = torch.matmul(xd, wd.transpose(2, 3).contiguous())
    bound = torch.matmul(xd.abs(), wd.abs().transpose(2, 3).contiguous()) * 1e-6
    calls = [(w, x, False), (w, x, True), (rows(torch, w, 8), rows(torch, x, 4), False), (rows(torch, w, 1), x, False),
             (w, x.to(dt), False)]
    for i, (ww, xx, split) in enumerate(calls):
        y = N.mul_mat_views(ww, xx, split=split)
        assert ((y.double() - want).abs() <= bound).all(), f"call {i}"


@pytest.mark.parametrize("name,tiny", [("f16", 1e-7), ("bf16", 1e-39)])
@pytest.mark.parametrize("n", [16, 77, 1040])
def test_src1_rounds_to_nearest_even_and_subnormals_count(gpu, name, tiny, n):
    """Through an identity matrix every output is src1 rounded to the weight
    type, exactly: over random bits, and over subnormals of the type."""
    import torch

    dt = torch.float16 if name == "f16" else torch.bfloat16
    K, M = 256, 1024
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randint(-2**31, 2**31 - 1, (n, K), device="cuda", generator=g, dtype=torch.int32).view(torch.float32)
    x = torch.where(torch.isfinite(x.to(dt).float()), x, torch.ones_like(x))
    x[::2] = torch.randn(len(x[::2]), K, device="cuda", generator=g) * tiny
    w = torch.eye(K, device="cuda").to(dt).repeat(M // K, 1)
    y = N.mul_mat_views(w.reshape(1, 1, M, K), x.reshape(1, 1, n, K)).reshape(n, M)
    assert (y == x.to(dt).float().repeat(1, M // K)).all()
    y = N.mul_mat_views((w * tiny * 3).reshape(1, 1, M, K), torch.full((1, 1, n, K), 1024.0, device="cuda"))
    assert (y == (w * tiny * 3).float().sum(1) * 1024.0).all() and (y != 0).all()


@pytest.mark.parametrize("M,K,n", [(64, 512, 1), (1024, 4096, 77), (4096, 256, 300), (16384, 64, 130)])
@pytest.mark.parametrize("name", ["f32", "f16", "bf16"])
def test_one_call_leaves_the_scratch_alone(gpu, name, M, K, n):
    """tlh_mul_mat with float weights is one launch that reads f32 src1: a scratch
    that another stream's products, or a quantize before it, use stays as it is."""
    import torch

    dt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[name]
    g = torch.Generator(device="cuda").manual_seed(n)
    w = torch.randn(M, K, device="cuda", generator=g).to(dt)
    x, other = torch.randn(2, n, K, device="cuda", generator=g)
    mm = N.MulMat({"f32": N.F32, "f16": N.F16, "bf16": N.BF16}[name], M, K, n)
    y, z = torch.empty(2, n, M, device="cuda")
    mm.quantize(x)
    before = mm.scratch.clone()
    mm(w, other, y)
    assert torch.equal(mm.scratch, before)
    mm.compute(w, z)
    mm(w, x, y)
    bound = (x.to(dt).double().abs() @ w.double().abs().T) * 2e-6
    assert ((y.double() - z.double()).abs() <= bound).all()


def lane_sums(torch, w, x):
    """x @ w.T with every output's f32 sum taken as 64 lanes would: lane l the
    elements 8 l .. 8 l + 7 of each 512, one after another, then a tree."""
    n, K = x.shape
    pad = -K % 512
    w, x = (torch.nn.functional.pad(t, (0, pad)).reshape(len(t), -1, 64, 8) for t in (w, x))
    acc = torch.zeros(n, len(w), 64, dtype=torch.float32, device=w.device)
    for i in range(w.shape[1]):
        for e in range(8):
            acc = (acc.double() + x[:, None, i, :, e] * w[None, :, i, :, e]).float()
    while acc.shape[2] > 1:
        acc = acc[:, :, ::2] + acc[:, :, 1::2]
    return acc[:, :, 0]


@pytest.mark.parametrize("copies,K,n", [(1, 256, 64), (128, 256, 64), (256, 256, 64), (1, 1000, 64), (128, 1000, 64), (1, 4096, 1), (1, 4096, 64),
                                        (128, 4096, 64), (256, 4096, 64), (1, 8192, 40), (256, 8192, 64)])
@pytest.mark.parametrize("name", ["f32", "f16", "bf16"])
def test_sums_are_as_exact_as_64_lanes(gpu, name, copies, K, n):
    """The f32 sums' error against 64 bits, root mean square over many outputs, is
    no larger than with the sums dealt over 64 lanes (one chain of MFMAs over 256
    elements is up to 1.5 times as far off). 5% for chance: 8192 outputs and more (5120 at
    n = 40), a standard deviation of 0.8% (1%)."""
    import torch

    dt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[name]
    g = torch.Generator(device="cuda").manual_seed(K + n)
    rows = 128 if n > 1 else 8192
    w = torch.randn(rows, K, device="cuda", generator=g).to(dt)
    x = torch.randn(n, K, device="cuda", generator=g)
    xd, wd = x.to(dt).double(), w.double()
    exact = xd @ wd.T
    rms = lambda y: ((y.double() - exact).square().mean().sqrt() / exact.square().mean().sqrt()).item()  # noqa: E731
    lanes = rms(torch.cat([lane_sums(torch, part, xd) for part in wd.split(128)], 1))
    ww = w.repeat(copies, 1)
    for split in (False, True):
        y = N.mul_mat_views(ww[None, None], x[None, None], split=split)[0, 0, :, -rows:]
        print(f"[float] {name} {copies * rows}x{K} n={n} split={split}: {rms(y):.3e}, lanes {lanes:.3e}", flush=True)
        assert rms(y) <= 1.05 * lanes
