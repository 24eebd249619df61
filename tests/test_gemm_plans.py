"""The tiled GEMMs' splits of K (csrc/gemm.hip), read from the library on the
CPU: no chunk may be left without a share of K, whatever the shape."""
from __future__ import annotations

import ctypes as C
import itertools

import pytest

from tensorlisp_amd import native as N

I64 = C.c_int64


def fn(name, *args):
    f = getattr(N.lib(), name)
    f.argtypes, f.restype = list(args), C.c_int
    return f


def empty_chunks(parts, ks):
    """Chunk c of ks takes parts c * share .. of ceil(parts / ks) each."""
    return ks > 1 and -(-parts // ks) * (ks - 1) >= parts


ROWS = (64, 448, 512, 1000, 1024, 1792, 4096, 14336, 32000)


def test_grouped_splits_leave_no_chunk_empty():
    """MUL_MAT_ID's tiles (448 x 14336 on 8 experts of 64 pairs each, 1792 x 14336
    on 2: nine shares of 56 super-blocks leave the last with none)."""
    split = fn("_ZN3tlh19gemm_ksplit_groupedEllll", I64, I64, I64, I64)
    seen = set()
    for M, units, n_as, per in itertools.product(ROWS, range(1, 113), (1, 2, 3, 4, 8, 64), (1, 17, 33, 64, 65, 200)):
        ks = split(M, 256 * units, per * n_as, n_as)
        assert ks >= 1 and not empty_chunks(units, ks), (M, 256 * units, n_as, per, ks)
        seen.add(ks)
    assert split(448, 14336, 512, 8) == 8 and len(seen) > 8


@pytest.mark.parametrize("t", [N.Q8_0, N.Q4_0, N.Q2_K, N.Q4_K, N.Q6_K], ids=lambda t: N.TYPE_NAMES[t])
def test_splits_leave_no_chunk_empty(t):
    split = fn("_ZN3tlh11gemm_ksplitEillll", C.c_int, I64, I64, I64, I64)
    step = N.BLOCK[t][0]
    for M, units, n, batches in itertools.product(ROWS, range(1, 113), (17, 33, 65, 129, 300, 2048), (1, 2)):
        for K in {256 * units, 256 * units - 224} if step == 32 else {256 * units}:
            ks = split(t, M, n, K, batches)
            parts = -(-K // 128) if step == 32 else units
            assert ks >= 1 and not empty_chunks(parts, ks), (M, K, n, batches, ks)


@pytest.mark.parametrize("t", [N.Q8_0, N.Q4_0, N.Q2_K, N.Q3_K, N.Q4_K, N.Q5_K, N.Q6_K, N.Q5_0, N.F16],
                         ids=lambda t: N.TYPE_NAMES[t])
def test_scratch_of_no_rows(t):
    """A MUL_MAT without weight rows has a size (it used to divide by its tiles)."""
    for n in (1, 16, 17, 40, 300):
        assert N.mul_mat_scratch_bytes(N.mul_mat_op(t, 0, 512, n)) > 0, n


def align(n):
    return -(-n // 256) * 256


def told(t, M, K, n, batches):
    """Scratch of a MUL_MAT with more than 16 columns: activation codes, scales
    and sums; f16 codes and sums (q4_K, q5_K); chunks of 128-row tiles'
    partials, or (q2_K, q3_K, q6_K) those of a 16-column slab."""
    rows = n * batches
    q8k = N.BLOCK[t][0] == 256
    act = align(align(align(rows * K) + rows * (K // (256 if q8k else 32)) * 4) + rows * K // 8)
    if t in (N.Q2_K, N.Q3_K, N.Q6_K):
        chunks = -(-K // 4096)
        return act + (align(chunks * batches * 16 * M * 4) if chunks > 1 else 0)
    if q8k:
        act += align(rows * (K + K // 16) * 2)
    wide = q8k and n > 128
    tiles = -(-n // (256 if wide else 128)) * -(-M // 128) * batches
    ks = 1 if tiles >= 256 else min(256 // tiles if wide else -(-512 // tiles), -(-K // 256) // 4, 16)
    return act + (align(ks * batches * n * M * 4) if ks > 1 else 0)


@pytest.mark.parametrize("t", [N.Q8_0, N.Q4_0, N.Q2_K, N.Q3_K, N.Q4_K, N.Q5_K, N.Q6_K], ids=lambda t: N.TYPE_NAMES[t])
def test_scratch_sizes(t):
    """The sizes, and so what the static scratch takes, stay as they were before
    the tiles and splits of the present kernels; q2_K, q3_K and q6_K, whose
    chunks are newer, may ask for more, but not past the static scratch where
    they fitted it. Whatever the size, the split has room in it."""
    static = 64 << 20
    split = fn("_ZN3tlh11gemm_ksplitEillll", C.c_int, I64, I64, I64, I64)
    for M, K, n, batches in itertools.product((1, 64, 512, 1000, 4096, 14336, 32000), (256, 512, 4096, 5120, 14336),
                                              (17, 32, 33, 64, 65, 128, 129, 512, 3584), (1, 2, 48, 100, 300)):
        got = N.mul_mat_scratch_bytes(N.mul_mat_op(t, M, K, n, ne2=batches, w_ne2=1))
        want = told(t, M, K, n, batches)
        if t in (N.Q2_K, N.Q3_K, N.Q6_K):
            assert got >= want and (got > static) == (want > static), (M, K, n, batches)
        else:
            assert got == want, (M, K, n, batches)
        ks = split(t, M, n, K, batches)
        act = align(align(align(n * batches * K) + n * batches * K // 64) + n * batches * K // 8)
        assert ks == 1 or N.BLOCK[t][0] == 32 or act + ks * batches * n * M * 4 <= got, (M, K, n, batches, ks)


@pytest.mark.parametrize("t", [N.Q4_K, N.Q5_K], ids=lambda t: N.TYPE_NAMES[t])
def test_2_to_the_31_activation_codes_are_refused(t):
    """Before anything is launched (the pointers here are never followed)."""
    op = N.mul_mat_op(t, 64, 4096, 1 << 19)
    st = N.lib().tlh_mul_mat_compute(C.byref(op), C.c_void_p(256), C.c_void_p(256), C.c_size_t(1 << 40), C.c_void_p(256), None)
    assert N.STATUS[st] == "UNSUPPORTED" and b"2^31" in N.lib().tlh_last_error()
