"""GPU parity of MUL_MAT_ID with its (expert, token) pairs grouped by expert
(csrc/gemm.hip k_group_plan; the GEMM tiles of gemm_kq.hip and the stream of
gemm_kqs.hip), through the executor, against the oracle's MUL_MAT of each pair's
expert. Bound per element as in test_gpu_gemm_kq.py."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from refs import NAMES, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, oracle
from tensorlisp_amd import graph as G
from tensorlisp_amd import native as N
from tensorlisp_amd import synth
from test_gpu_gemm_kq import bound, check_sums, dev, short_chains

pytestmark = pytest.mark.gpu


def run_case(t, M, K, n_as, used, n_b1, tokens, seed, columns=None, bad=()):
    import torch

    rng = np.random.default_rng(seed)
    w = synth.random_blocks(t, seed, n_as * M, K)
    x = synth.normal(seed + 1, (tokens, n_b1, K))
    ids = rng.integers(0, n_as - 1, (tokens, used)).astype(np.int32)  # the last expert stays unused
    for i, v in bad:
        ids.reshape(-1)[i] = v
    b = G.Builder()
    W, X, I = b.weight(t, [K, M, n_as]), b.input(N.F32, [K, n_b1, tokens]), b.input(N.I32, [used, tokens])
    y = b.mul_mat_id(W, X, I)
    b.expand(y)
    prog = G.Program(b, [y], [dev(w)])
    prog.write_input(0, dev(x))
    prog.write_input(1, dev(ids))
    labels = [label for _, ls in prog.trace() for label in ls]
    got = prog.read(y, torch.float32).reshape(tokens, used, M)
    torch.cuda.synchronize()
    got = got.cpu().numpy()
    pairs = [divmod(p, used) for p in range(tokens * used)]
    if columns is not None:
        pairs = [pairs[i] for i in sorted(set(rng.integers(0, len(pairs), columns)) | {i for i, _ in bad})]
    for tok, e in pairs:
        if not 0 <= ids[tok, e] < n_as:
            assert np.isnan(got[tok, e]).all(), (tok, e)
    for ex in range(n_as):
        mine = [(tok, e) for tok, e in pairs if ids[tok, e] == ex]
        if not mine:
            continue
        wx = w[ex * M:(ex + 1) * M]
        xs = np.stack([x[tok, e % n_b1] for tok, e in mine])
        want = oracle().mul_mat(t, wx, M, K, xs, nthreads=16)
        have = np.stack([got[tok, e] for tok, e in mine])
        err, lim = np.abs(have - want), bound(t, wx, K, xs)
        assert (err <= lim).all(), f"expert {ex}: worst {(err / lim).max():.2f} of the bound"
    return labels


@pytest.mark.parametrize("t", [Q2_K, Q3_K, Q4_K, Q5_K, Q6_K], ids=lambda t: NAMES[t])
@pytest.mark.parametrize("n_as,per_slot", [(5, False), (90, True), (200, False)])
def test_tiles(gpu, t, n_as, per_slot):
    """Tiles of 128, 64 and 32 pairs, experts of several tiles and of none, row
    tails, ids outside [0, n_as)."""
    M, K, used = 70, 512, 2
    bytes_ = M * N.row_bytes(t, K)
    tokens = int((50e6 / bytes_ + 2.25 * n_as) / used) + 8
    print(f"[mul_mat_id] {NAMES[t]} {n_as} experts, {tokens} tokens", flush=True)
    labels = run_case(t, M, K, n_as, used, used if per_slot else 1, tokens, 11 * n_as, columns=300,
                      bad=((3, -1), (2 * tokens - 1, n_as), (100, 1 << 30)))
    assert "group_plan" in labels, labels


@pytest.mark.parametrize("t", [Q2_K, Q3_K, Q4_K, Q5_K, Q6_K], ids=lambda t: NAMES[t])
@pytest.mark.parametrize("M,K,n_as,tokens,chunks", [(450, 8448, 4, 60, 7), (448, 11008, 3, 75, 9), (300, 6400, 3, 150, 5),
                                                    (450, 7168, 4, 60, 7)], ids=["32", "64", "128", "32-even"])
def test_tiles_with_k_chunks(gpu, t, M, K, n_as, tokens, chunks):
    """Tiles of 32, 64 and 128 pairs over several chunks of K, all equal or the
    last one shorter, through the partial sums: row tails, ids outside [0, n_as)."""
    split = N.lib()._ZN3tlh19gemm_ksplit_groupedEllll
    split.argtypes, split.restype = [C.c_int64] * 4, C.c_int
    assert split(M, K, 2 * tokens, n_as) == chunks
    print(f"[mul_mat_id] tiles {NAMES[t]} {n_as} x {M} x {K}, {tokens} tokens, {chunks} chunks", flush=True)
    labels = run_case(t, M, K, n_as, 2, 2 if tokens == 75 else 1, tokens, M + K, columns=24,
                      bad=((3, -1), (2 * tokens - 1, n_as)))
    assert "group_plan" in labels and "gemm_kqs" not in labels, labels


@pytest.mark.parametrize("t", [Q4_K, Q5_K], ids=lambda t: NAMES[t])
@pytest.mark.parametrize("M,K,n_as,tokens", [(1801, 4096, 9, 16), (1801, 4096, 9, 60), (450, 8448, 18, 100), (20000, 768, 6, 16)])
def test_stream(gpu, t, M, K, n_as, tokens):
    """The stream's one and two column tiles, K of one and two chunks (an odd
    number of super-blocks), row groups past M, an expert of two plan entries."""
    print(f"[mul_mat_id] stream {NAMES[t]} {n_as} x {M} x {K}, {tokens} tokens", flush=True)
    labels = run_case(t, M, K, n_as, 2, 1, tokens, M + tokens, columns=24, bad=((5, n_as + 3),))
    assert "gemm_kqs" in labels, labels


class Stream(C.Structure):
    _fields_ = [("nt", C.c_int), ("kc_elems", C.c_int), ("zc", C.c_int), ("lds", C.c_size_t)]


@pytest.mark.parametrize("t", [Q4_K, Q5_K], ids=lambda t: NAMES[t])
@pytest.mark.parametrize("M,K,n_as,tokens", [(64, 8704, 162, 190), (40, 4096, 520, 640)])
def test_stream_walks_several_entries(gpu, t, M, K, n_as, tokens):
    """More plan entries than the stream's grid has workgroups (256 over the K
    chunks): each fills its LDS again for the next one."""
    plan = N.lib()._ZN3tlh13gemm_kqs_planEllll
    plan.argtypes, plan.restype = [C.c_int64] * 4, Stream
    pairs = 2 * tokens
    p = plan(M, -(-pairs // n_as), K, min(pairs, n_as))
    ids = np.random.default_rng(M + tokens).integers(0, n_as - 1, (tokens, 2))  # (run_case's)
    entries = (-(-np.bincount(ids.reshape(-1)) // (16 * p.nt))).sum()
    print(f"[mul_mat_id] stream {NAMES[t]} {n_as} x {M} x {K}, {tokens} tokens, {entries} entries, {p.zc} chunks", flush=True)
    assert entries > 256 // p.zc
    labels = run_case(t, M, K, n_as, 2, 2 if K == 4096 else 1, tokens, M + tokens, columns=120, bad=((5, n_as + 3),))
    assert "gemm_kqs" in labels, labels


@pytest.mark.parametrize("t", [Q4_K, Q5_K], ids=lambda t: NAMES[t])
@pytest.mark.parametrize("copies,K,tokens", [(28, 8704, 16), (28, 4096, 32), (8, 8704, 60)])
def test_stream_sums_are_as_exact_as_short_chains(gpu, t, copies, K, tokens):
    """One column tile, 34 super-blocks in one chunk (one chain of them is 1.3 times
    as far off), and two, whose chunks of 17 are one chain each."""
    import torch

    rows, n_as = 512, 8
    w, x = synth.random_blocks(t, K, rows, K), synth.normal(tokens, (tokens, 1, K))
    M = copies * rows
    op = N.TlhOp()
    op.t[0], op.t[1] = N.ggml_tensor(t, [K, M, n_as]), N.ggml_tensor(N.F32, [K, 1, tokens])
    op.t[2], op.t[4] = N.ggml_tensor(N.I32, [2, tokens]), N.ggml_tensor(N.F32, [M, 2, tokens])
    need = C.c_size_t()
    N.check(N.lib().tlh_mul_mat_id_scratch_bytes(C.byref(op), C.byref(need)))
    scratch = torch.empty(need.value + 256, dtype=torch.uint8, device="cuda")
    W, X = dev(w).repeat(n_as * copies, 1), dev(x)  # every expert the same rows
    ids = torch.arange(2 * tokens, dtype=torch.int32, device="cuda") % n_as
    y = torch.empty((tokens, 2, M), device="cuda")
    N.check(N.lib().tlh_mul_mat_id(C.byref(op), N._ptr(W), N._ptr(X), N._ptr(ids), N._ptr(y),
                                   C.c_void_p(scratch.data_ptr() + -scratch.data_ptr() % 256), need, N._stream(None)))
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(tokens, 2, copies, rows)[:, 1, -1].astype(np.float64)
    exact, total = short_chains(t, w, K, x[:, 0], 17 if tokens == 60 else 4)
    check_sums(got, exact, total, f"[mul_mat_id] stream {NAMES[t]} {n_as} x {M} x {K}, {tokens} tokens")


def test_plan_of_many_experts(gpu):
    """More experts than the plan's workgroup has threads."""
    labels = run_case(Q4_K, 40, 256, 1500, 4, 4, 4200, 3, columns=200, bad=((0, 1500),))
    assert "group_plan" in labels, labels
