"""The work this framework's performance is measured on.

Each case is one call (or one compiled program's step) that a user of the
framework makes through its public entry points: quantized and float MUL_MAT
(``native.MulMat`` / ``tlh_mul_mat``) for decode, batched decode and prefill,
MUL_MAT_ID for mixture-of-experts layers (``tlh_mul_mat_id``), paged-attention
decode (``native.PagedAttention``), dense FLASH_ATTN_EXT (``native.FlashAttnExt``),
and whole decoder steps through the executor (``graph.Program``).

``listed`` names fixed cases, ``draw`` gives others of the same ranges,
``prepare`` builds what a program has in hand, ``run`` is one pass, ``work`` the
bytes and operations it cannot do without, ``exact`` the result in 64 bits by
plain torch, ``tolerance`` what another correct implementation may differ by.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from tensorlisp_amd import graph as G
from tensorlisp_amd import native as N

# the quantized weight types and the mean code that centres random blocks on zero
QUANT = {"q4_0": 8.0, "q4_1": 7.5, "q5_0": 16.0, "q5_1": 15.5, "q8_0": 0.0,
         "q2_K": 1.5, "q3_K": 0.0, "q4_K": 7.5, "q5_K": 15.5, "q6_K": 0.0}
FLOATS = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
STD = 0.02  # standard deviation of the weights


def listed():
    return [
        # the smallest call: a square projection of one token
        dict(name="decode q8_0 4096x4096 n1", path="mul_mat", wtype="q8_0", M=4096, K=4096, N=1),
        # the down projection of an 8B model decoding 8 sequences
        dict(name="decode q4_K 4096x14336 n8", path="mul_mat", wtype="q4_K", M=4096, K=14336, N=8),
        # the output matrix of a Q4_K_M file, 8 sequences
        dict(name="head q6_K 128256x4096 n8", path="mul_mat", wtype="q6_K", M=128256, K=4096, N=8),
        # a gate or up projection for 32 sequences: more columns than a GEMV, fewer than a prefill
        dict(name="batch q4_K 14336x4096 n32", path="mul_mat", wtype="q4_K", M=14336, K=4096, N=32),
        # the largest: a 2048-token prefill's gate or up projection
        dict(name="prefill q4_K 14336x4096 n2048", path="mul_mat", wtype="q4_K", M=14336, K=4096, N=2048),
        # a Q4_K_M file keeps half its down projections in q6_K
        dict(name="prefill q6_K 4096x14336 n512", path="mul_mat", wtype="q6_K", M=4096, K=14336, N=512),
        # an unquantized file, a prompt of odd length
        dict(name="prefill f16 4096x4096 n77", path="mul_mat", wtype="f16", M=4096, K=4096, N=77),
        # one expert projection of a mixture-of-experts layer over a prompt: 8 experts, 2 a token
        dict(name="experts q4_K 8x14336x4096 t99", path="mul_mat_id", wtype="q4_K", M=14336, K=4096, experts=8, used=2,
             tokens=99, per_slot=False),
        # paged decode attention of 32 sequences over contexts of 512..8192
        dict(name="paged attention 32 seqs", path="paged", seqs=32, heads=32, kv_heads=8, head_size=128, block=16,
             shortest=512, longest=8192),
        # a prompt's second chunk attending to itself and the 223 tokens before it
        dict(name="flash attention 777 of 1000", path="flash", batch=1, heads=32, kv_heads=8, head_size=128,
             queries=777, keys=1000, masked=True),
        # decode of one sequence through the executor (two layers of an 8B model and its head)
        dict(name="decoder step 1 seq", path="decode", layers=2, seqs=1, context=768, wtype="q4_K", vocab=128256),
        # a 512-token prompt through the executor, Q4_K_M's mix of q4_K and q6_K
        dict(name="decoder prompt 512", path="prompt", layers=2, tokens=512, wtype="q4_K", vocab=128256),
    ]


# ------------------------------------------------------------------ drawing
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _wtype(rng):
    # by how often files use them: Q4_K_M, Q5_K_M, Q6_K, Q8_0 and Q4_0 files first
    return rng.choices(["q4_K", "q6_K", "q8_0", "q4_0", "q5_K", "q3_K", "q2_K", "q5_0", "q4_1", "q5_1"],
                       [6, 4, 4, 3, 3, 1, 1, 1, 1, 1])[0]


def _rows(rng, lo, hi):
    m = _log(rng, lo, hi)
    return m if rng.random() < 0.25 else max(64, m // 64 * 64)


def _depth(rng, wtype, hi=14336):
    k = _log(rng, 512, hi)
    return k // 256 * 256 if N.BLOCK[N.TYPES_BY_NAME[wtype]][0] == 256 or rng.random() < 0.7 else k // 32 * 32


def draw(rng):
    kind = rng.choices(["gemv", "batch", "prefill", "float", "experts", "paged", "flash", "flash1", "decode", "prompt"],
                       [5, 3, 4, 2, 3, 3, 2, 1, 2, 1])[0]
    if kind in ("gemv", "batch", "prefill"):
        wtype = _wtype(rng)
        lo, hi = {"gemv": (1, 16), "batch": (17, 128), "prefill": (129, 2048)}[kind]
        rows = rng.choice([32000, 64128, 128256]) if kind == "gemv" and rng.random() < 0.2 else _rows(rng, 512, 14336)
        depth = _depth(rng, wtype, 4096 if rows > 14336 else 14336)
        n = _log(rng, lo, hi)
        while rows * depth * n > 14336 * 4096 * 2048:  # no larger than the largest listed
            n = n * 3 // 4
        return dict(path="mul_mat", wtype=wtype, M=rows, K=depth, N=n)
    if kind == "float":
        depth = _log(rng, 256, 8192)
        return dict(path="mul_mat", wtype=rng.choice(["f16", "f16", "bf16", "f32"]), M=_rows(rng, 256, 8192),
                    K=depth if rng.random() < 0.2 else depth // 64 * 64, N=_log(rng, 1, 512))
    if kind == "experts":
        wtype = rng.choice(["q4_K", "q4_K", "q6_K", "q8_0", "q4_0", "q5_K"])
        experts, used = rng.choice([(8, 2), (16, 4), (32, 4), (64, 8)])
        rows = _rows(rng, 512, 14336 * 8 // experts)
        depth = max(512, _log(rng, 512, 4096) // 256 * 256)
        return dict(path="mul_mat_id", wtype=wtype, M=rows, K=depth, experts=experts, used=used,
                    tokens=_log(rng, 1, 512), per_slot=rng.random() < 0.4)
    if kind == "paged":
        heads, kv_heads = rng.choice([(32, 8), (32, 32), (16, 8), (28, 4), (8, 1), (64, 8)])
        longest = _log(rng, 64, 8192)
        return dict(path="paged", seqs=_log(rng, 1, 32 if heads < 64 else 16), heads=heads, kv_heads=kv_heads,
                    head_size=rng.choice([64, 128, 128, 128, 256]) if kv_heads <= 8 else rng.choice([64, 128]),
                    block=rng.choice([16, 16, 32]), shortest=max(1, int(longest * rng.uniform(0.05, 1.0))),
                    longest=longest)
    if kind in ("flash", "flash1"):
        heads, kv_heads = rng.choice([(32, 8), (32, 32), (16, 8), (28, 4), (8, 1)])
        hs = rng.choice([64, 80, 96, 128, 128, 128, 256])
        if kind == "flash1":  # decode over dense caches
            return dict(path="flash", batch=_log(rng, 1, 16), heads=heads, kv_heads=kv_heads, head_size=hs, queries=1,
                        keys=_log(rng, 64, 4096), masked=rng.random() < 0.7)
        queries = _log(rng, 2, 1024)
        return dict(path="flash", batch=1, heads=heads, kv_heads=kv_heads, head_size=hs, queries=queries,
                    keys=queries + (0 if rng.random() < 0.4 else _log(rng, 1, 2048)), masked=True)
    if kind == "decode":
        return dict(path="decode", layers=rng.choice([1, 2]), seqs=_log(rng, 1, 32), context=_log(rng, 64, 2048),
                    wtype=rng.choice(["q4_K", "q4_K", "q8_0", "q4_0", "q5_K"]), vocab=rng.choice([32000, 128256]))
    return dict(path="prompt", layers=rng.choice([1, 2]), tokens=_log(rng, 24, 512),
                wtype=rng.choice(["q4_K", "q4_K", "q8_0", "q4_0", "q5_K"]), vocab=rng.choice([32000, 128256]))


# ------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(shape, device="cuda", generator=g).to(dtype)


def _weights(wtype, M, K, g, std=STD):
    """Random blocks (uint8 [M, row bytes]) that decode to zero-mean values of
    about the standard deviation std, or a float matrix."""
    if wtype in FLOATS:
        return (_randn(g, M, K) * std).to(FLOATS[wtype])
    be, bb = N.BLOCK[N.TYPES_BY_NAME[wtype]]
    nb = M * (K // be)
    b = torch.randint(0, 256, (nb, bb), dtype=torch.uint8, device="cuda", generator=g)
    u = 0.5 + torch.rand(nb, device="cuda", generator=g)
    rms = {"q4_0": 4.6, "q4_1": 4.6, "q5_0": 9.2, "q5_1": 9.2, "q8_0": 73.9, "q2_K": 1.1 * 8.8, "q3_K": 2.3 * 18.5,
           "q4_K": 4.6 * 36.8, "q5_K": 9.2 * 36.8, "q6_K": 18.5 * 73.9}[wtype]
    d = (u * (std / rms)).to(torch.float16)
    mean = QUANT[wtype]
    m = (d.float() * mean).to(torch.float16)
    put = lambda at, v: b[:, at:at + 2].copy_(v.view(torch.uint8).reshape(nb, 2))  # noqa: E731
    if wtype == "q8_0":
        put(0, d)
    elif wtype in ("q4_0", "q5_0"):  # the quantizer's scales have either sign
        put(0, d * (torch.randint(0, 2, (nb,), device="cuda", generator=g) * 2 - 1).half())
    elif wtype in ("q4_1", "q5_1"):
        put(0, d), put(2, -m)
    elif wtype in ("q4_K", "q5_K"):  # scale and min of a sub-block equal, d * mean as the min's unit
        s = torch.randint(1, 64, (nb, 8), device="cuda", generator=g, dtype=torch.int32)
        put(0, d), put(2, m)
        b[:, 4:8] = (s[:, :4] | ((s[:, 4:] >> 4) << 6)).to(torch.uint8)
        b[:, 8:12] = b[:, 4:8]
        b[:, 12:16] = ((s[:, 4:] & 15) * 17).to(torch.uint8)
    elif wtype == "q2_K":
        b[:, :16] = (torch.randint(1, 16, (nb, 16), device="cuda", generator=g, dtype=torch.int32) * 17).to(torch.uint8)
        put(80, d), put(82, m)
    else:  # q3_K, q6_K: signed scales
        put(bb - 2, d)
    return b.reshape(M, -1)


def _tables(g, lens, block):
    """Block tables over a shared pool whose blocks are dealt out at random."""
    per = [-(-n // block) for n in lens]
    deal = torch.randperm(sum(per), device="cuda", generator=g).to(torch.int32)
    table = torch.zeros((len(lens), max(per)), dtype=torch.int32, device="cuda")
    at = 0
    for i, n in enumerate(per):
        table[i, :n] = deal[at:at + n]
        at += n
    return table, sum(per)


def _lens(case, seed=None):
    """Context lengths spread evenly from shortest to longest; the seed deals them out."""
    lens = np.linspace(case["shortest"], case["longest"], case["seqs"] + 2)[1:-1].round().astype(int)
    lens = np.maximum(lens, 1)
    return [int(n) for n in (lens if seed is None else np.random.RandomState(seed).permutation(lens))]


def _config(case, ctx):
    t = N.TYPES_BY_NAME[case["wtype"]]
    types = {}
    if case["wtype"] == "q4_K":  # Q4_K_M: value and down projections of some layers in q6_K
        types = {"l0.wv": N.Q6_K, "l0.w_down": N.Q6_K}
    out = N.Q6_K if case["wtype"] in ("q4_K", "q5_K") else t
    return G.DecoderConfig(n_layer=case["layers"], n_vocab=case["vocab"], n_ctx=ctx, wtype=t, embd_type=t,
                           out_type=out, types=types)


def _model(c, g):
    """The decoder's weights in weight-index order: a residual stream (the
    embedding) that a layer changes by a part of it, as a trained model's does
    (its output projections are smaller than the others)."""
    std = {"tok_embd": 0.5, "wo": STD / 8, "w_down": STD / 8}
    return [1.0 + 0.1 * _randn(g, ne[0]) if ty == N.F32 else
            _weights(N.TYPE_NAMES[ty], ne[1], ne[0], g, std.get(name.split(".")[-1], STD))
            for name, ty, ne in c.weight_shapes()]


def _mul_mat_id_op(case):
    op = N.TlhOp()
    K, M, T = case["K"], case["M"], case["tokens"]
    op.t[0] = N.ggml_tensor(N.TYPES_BY_NAME[case["wtype"]], [K, M, case["experts"]])
    op.t[1] = N.ggml_tensor(N.F32, [K, case["used"] if case["per_slot"] else 1, T])
    op.t[2] = N.ggml_tensor(N.I32, [case["used"], T])
    op.t[4] = N.ggml_tensor(N.F32, [M, case["used"], T])
    return op


def _aligned(nbytes):
    """A uint8 buffer and its first 256-byte aligned address."""
    buf = torch.empty(max(nbytes, 256) + 256, dtype=torch.uint8, device="cuda")
    return buf, buf.data_ptr() + (-buf.data_ptr()) % 256


def _state_mul_mat(case, g, seed):
    M, K, n = case["M"], case["K"], case["N"]
    t = N.TYPES_BY_NAME[case["wtype"]]
    return dict(w=_weights(case["wtype"], M, K, g), x=_randn(g, n, K), y=torch.empty((n, M), device="cuda"),
                node=N.MulMat(t, M, K, n))


def _state_mul_mat_id(case, g, seed):
    M, K, E, T, used = case["M"], case["K"], case["experts"], case["tokens"], case["used"]
    w = _weights(case["wtype"], E * M, K, g)
    x = _randn(g, T, used if case["per_slot"] else 1, K)
    # a router's choice: some experts more popular than others, no expert twice for a token
    score = _randn(g, T, E) + 0.5 * _randn(g, 1, E)
    ids = score.topk(used, dim=1).indices.to(torch.int32).contiguous()
    op = _mul_mat_id_op(case)
    need = C.c_size_t()
    N.check(N.lib().tlh_mul_mat_id_scratch_bytes(C.byref(op), C.byref(need)))
    buf, ptr = _aligned(need.value)
    return dict(w=w, x=x, ids=ids, y=torch.empty((T, used, M), device="cuda"), op=op, scratch=buf,
                scratch_ptr=C.c_void_p(ptr), scratch_bytes=need.value)


def _state_paged(case, g, seed):
    S, H, KV, D, B = case["seqs"], case["heads"], case["kv_heads"], case["head_size"], case["block"]
    lens = _lens(case, seed)
    table, nblocks = _tables(g, lens, B)
    half = torch.float16
    node = N.PagedAttention(S, H, KV, D, B, table.shape[1], max(lens), D ** -0.5)
    return dict(q=_randn(g, S, H, D, dtype=half), k=_randn(g, nblocks, KV, D // 8, B, 8, dtype=half),
                v=_randn(g, nblocks, KV, D, B, dtype=half), table=table,
                lens=torch.tensor(lens, dtype=torch.int32, device="cuda"),
                out=torch.empty((S, H, D), dtype=half, device="cuda"), node=node)


def _state_flash(case, g, seed):
    nb, H, KV, D, nq, L = (case[k] for k in ("batch", "heads", "kv_heads", "head_size", "queries", "keys"))
    half = torch.float16
    q = _randn(g, nb, nq, H, D).permute(0, 2, 1, 3)  # a projection's rows, heads interleaved
    k, v = (_randn(g, nb, L, KV, D, dtype=half).permute(0, 2, 1, 3) for _ in range(2))  # cache rows
    mask = None
    if case["masked"]:
        pos = torch.arange(L - nq, L, device="cuda")[:, None]
        mask = torch.zeros((1, 1, nq, L), dtype=half, device="cuda")
        mask.masked_fill_(torch.arange(L, device="cuda")[None] > pos, float("-inf"))
    out = torch.empty((nb, nq, H, D), device="cuda")
    return dict(q=q, k=k, v=v, mask=mask, out=out, node=N.FlashAttnExt(q, k, v, mask, out, D ** -0.5))


def _state_decode(case, g, seed):
    S, ctx, block = case["seqs"], case["context"], 16
    lens = _lens(dict(shortest=max(1, ctx // 2), longest=ctx, seqs=S), seed)
    table, nblocks = _tables(g, lens, block)
    c = _config(case, 4096)
    pc = G.PagedConfig(block_size=block, n_blocks=nblocks, max_blocks=table.shape[1])
    step = G.decoder_decode_paged(c, pc, S)
    offs, total = pc.state_bytes(c)
    weights = _model(c, g)
    cache = _randn(g, total // 2, dtype=torch.float16)
    pos = np.array([n - 1 for n in lens])
    tab = table.cpu().numpy()
    slots = np.concatenate([G.paged_slots(tab[s], [p], block) for s, p in enumerate(pos)])
    dev = lambda a, ty=np.int32: torch.from_numpy(np.ascontiguousarray(a, ty)).cuda()  # noqa: E731
    tokens = torch.randint(0, c.n_vocab, (S,), device="cuda", generator=g, dtype=torch.int32)
    inputs = [tokens, dev(pos), dev(slots), table, dev(lens)]
    return dict(program=G.Program(step.builder, step.keep, weights, offs), step=step, cache=cache, inputs=inputs,
                stream=torch.cuda.Stream(), config=c, weights=weights, lens=lens, graph=True, per=total // 2 // (2 * c.n_layer))


def _state_prompt(case, g, seed):
    T, block = case["tokens"], 16
    c = _config(case, 4096)
    table, nblocks = _tables(g, [T], block)
    pc = G.PagedConfig(block_size=block, n_blocks=nblocks, max_blocks=nblocks)
    step = G.decoder_prefill_paged(c, pc, T)
    offs, total = pc.state_bytes(c)
    weights = _model(c, g)
    cache = torch.zeros(total // 2, dtype=torch.float16, device="cuda")
    pos = np.arange(T)
    dev = lambda a, ty=np.int32: torch.from_numpy(np.ascontiguousarray(a, ty)).cuda()  # noqa: E731
    tokens = torch.randint(0, c.n_vocab, (T,), device="cuda", generator=g, dtype=torch.int32)
    mask = torch.from_numpy(G.causal_mask(pos, T).view(np.int16)).cuda()
    inputs = [tokens, dev(pos), dev(G.paged_slots(table[0].cpu().numpy(), pos, block)), mask]
    return dict(program=G.Program(step.builder, step.keep, weights, offs), step=step, cache=cache, inputs=inputs,
                stream=torch.cuda.Stream(), config=c, weights=weights, graph=False)


def prepare(case, seed):
    path = case["path"]
    build = {"mul_mat": _state_mul_mat, "mul_mat_id": _state_mul_mat_id, "paged": _state_paged, "flash": _state_flash,
             "decode": _state_decode, "prompt": _state_prompt}[path]
    s = build(case, _gen(seed), seed)
    s["path"] = path
    if "stream" in s:
        s["stream"].wait_stream(torch.cuda.current_stream())
    return s


# --------------------------------------------------------------------- pass
def run(s):
    path = s["path"]
    if path == "mul_mat":
        return s["node"](s["w"], s["x"], s["y"])
    if path == "mul_mat_id":
        stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        N.check(N.lib().tlh_mul_mat_id(C.byref(s["op"]), s["w"].data_ptr(), s["x"].data_ptr(), s["ids"].data_ptr(),
                                       s["y"].data_ptr(), s["scratch_ptr"], s["scratch_bytes"], stream))
        return s["y"]
    if path == "paged":
        return s["node"](s["out"], s["q"], s["k"], s["v"], s["table"], s["lens"])
    if path == "flash":
        return s["node"](s["q"], s["k"], s["v"], s["mask"], s["out"])
    # a decoder step: this step's tokens, positions, slots and tables or mask, then the compiled program
    p, stream = s["program"], s["stream"]
    with torch.cuda.stream(stream):
        for i, a in enumerate(s["inputs"]):
            p.write_input(i, a, stream)
        p.run(s["cache"], stream, graph=s["graph"])
        logits = p.read(s["step"].logits, torch.float32, s["cache"], stream)
    torch.cuda.current_stream().wait_stream(stream)  # what reads the logits next
    return {"logits": logits, "cache": s["cache"]}


# --------------------------------------------------------------------- work
def _matrix(wtype, M, K):
    return M * (K * FLOATS[wtype].itemsize if wtype in FLOATS else N.row_bytes(N.TYPES_BY_NAME[wtype], K))


def _decoder_work(case, rows, head_rows, pairs, kv_read):
    c = _config(case, 4096)
    nbytes = flops = 0
    for name, ty, ne in c.weight_shapes():
        if ty == N.F32:
            continue
        t = N.TYPE_NAMES[ty]
        n = {"tok_embd": 0, "output": head_rows}.get(name, rows)
        nbytes += _matrix(t, rows if name == "tok_embd" else ne[1], ne[0])
        flops += 2 * ne[0] * ne[1] * n
    kv = 2 * c.n_embd_kv * 2  # key and value bytes of a token and layer
    nbytes += case["layers"] * kv * (rows + kv_read) + head_rows * c.n_vocab * 4
    return {"bytes": nbytes, "flops": flops + case["layers"] * 4 * c.n_embd * pairs}


def work(case):
    path = case["path"]
    if path == "mul_mat":
        M, K, n = case["M"], case["K"], case["N"]
        return {"bytes": _matrix(case["wtype"], M, K) + 4 * n * (K + M), "flops": 2 * M * K * n}
    if path == "mul_mat_id":
        M, K, T, used, E = case["M"], case["K"], case["tokens"], case["used"], case["experts"]
        # the experts that are chosen at all, were each as popular as the next
        touched = E * (1 - (1 - used / E) ** T)
        return {"bytes": int(_matrix(case["wtype"], M, K) * touched) + 4 * T * (K * (used if case["per_slot"] else 1) + used * M),
                "flops": 2 * M * K * T * used}
    if path == "paged":
        total = sum(_lens(case))
        H, KV, D, S = case["heads"], case["kv_heads"], case["head_size"], case["seqs"]
        return {"bytes": total * KV * D * 4 + S * H * D * 4, "flops": 4 * total * H * D}
    if path == "flash":
        nb, H, KV, D, nq, L = (case[k] for k in ("batch", "heads", "kv_heads", "head_size", "queries", "keys"))
        live = nq * L - (nq * (nq - 1) // 2 if case["masked"] else 0)
        return {"bytes": nb * (8 * nq * H * D + 4 * L * KV * D) + (2 * nq * L if case["masked"] else 0),
                "flops": 4 * nb * H * D * live}
    if path == "decode":
        total = sum(_lens(dict(shortest=max(1, case["context"] // 2), longest=case["context"], seqs=case["seqs"])))
        return _decoder_work(case, case["seqs"], case["seqs"], total, total)
    return _decoder_work(case, case["tokens"], 1, case["tokens"] * (case["tokens"] + 1) // 2, 0)


def tolerance(case):
    path = case["path"]
    if path in ("mul_mat", "mul_mat_id"):
        # the activation's codes and the products are fixed by the op; sums in 32 bits
        # (measured against exact: rel 1.5e-7, max 1.6e-6)
        return {"rel": 1e-6, "max": 1e-5}
    if path in ("paged", "flash"):
        # probabilities (and the paged output) in f16 (measured: rel 2.6e-4, max 3.4e-3)
        return {"rel": 1e-3, "max": 1.4e-2}
    # every layer rounds its activations to 8-bit codes: a last-bit difference
    # anywhere moves some codes by one, and all that follows (the norms' weights
    # changed by one unit in the last place: rel 1.6e-2, max 8.5e-2)
    return {"rel": 3e-2, "max": 3e-1}


# ----------------------------------------------------------- 64-bit results
def _f16_at(b, at):
    return b[:, at:at + 2].contiguous().view(torch.float16).double()


def _nibbles(q):  # [nb, n] -> low nibbles, then high ones
    return torch.cat([q & 15, q >> 4], 1)


def _fifth(b, at):
    shifts = torch.arange(8, device=b.device, dtype=torch.uint8)
    return ((b[:, at:at + 4, None] >> shifts) & 1).reshape(-1, 32)


def _crumbs(q):  # [nb, 64] -> the 2-bit codes of 256 elements
    q = q.reshape(-1, 2, 1, 32) >> torch.tensor([0, 2, 4, 6], device=q.device, dtype=torch.uint8)[:, None]
    return (q & 3).reshape(-1, 256)


def _decode_rows(wtype, b, K):
    """(values without the block min, block mins or None) of uint8 block rows, in 64 bits."""
    M = b.shape[0]
    be, bb = N.BLOCK[N.TYPES_BY_NAME[wtype]]
    b = b.reshape(-1, bb)
    mins = None
    if wtype == "q8_0":
        v = b[:, 2:].view(torch.int8).double() * _f16_at(b, 0)
    elif wtype == "q4_0":
        v = (_nibbles(b[:, 2:]).double() - 8) * _f16_at(b, 0)
    elif wtype == "q4_1":
        v, mins = _nibbles(b[:, 4:]).double() * _f16_at(b, 0), _f16_at(b, 2)
    elif wtype == "q5_0":
        v = ((_nibbles(b[:, 6:]) | (_fifth(b, 2) << 4)).double() - 16) * _f16_at(b, 0)
    elif wtype == "q5_1":
        v, mins = (_nibbles(b[:, 8:]) | (_fifth(b, 4) << 4)).double() * _f16_at(b, 0), _f16_at(b, 2)
    elif wtype in ("q4_K", "q5_K"):
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, bb - 128:].reshape(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32)
        if wtype == "q5_K":
            bit = (b[:, 16:48][:, None] >> torch.arange(8, device=b.device, dtype=torch.uint8)[:, None]) & 1
            q = q | (bit << 4)
        v = q.double() * (sc * _f16_at(b, 0))[:, :, None] - (mn * _f16_at(b, 2))[:, :, None]
    elif wtype == "q6_K":
        lo = b[:, :128].reshape(-1, 2, 1, 64)
        lo = torch.cat([lo & 15, lo >> 4], 2).reshape(-1, 256)
        q = (lo | (_crumbs(b[:, 128:192]) << 4)).double() - 32
        v = q.reshape(-1, 16, 16) * (b[:, 192:208].view(torch.int8).double() * _f16_at(b, 208))[:, :, None]
    elif wtype == "q2_K":
        sc, mn = (b[:, :16] & 15).double() * _f16_at(b, 80), (b[:, :16] >> 4).double() * _f16_at(b, 82)
        v = _crumbs(b[:, 16:80]).reshape(-1, 16, 16).double() * sc[:, :, None] - mn[:, :, None]
    else:  # q3_K: the third bit clear means minus 4
        bit = (b[:, None, :32] >> torch.arange(8, device=b.device, dtype=torch.uint8)[:, None]) & 1
        q = _crumbs(b[:, 32:96]).double() - 4 + 4 * bit.reshape(-1, 256).double()
        s = b[:, 96:108]
        hi = (s[:, None, 8:12] >> torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.uint8)[:, None]) & 3
        sc = (_nibbles(s[:, :8]) | (hi.reshape(-1, 16) << 4)).double() - 32
        v = q.reshape(-1, 16, 16) * (sc * _f16_at(b, 108))[:, :, None]
    return v.reshape(M, K), (mins.reshape(M, -1) if mins is not None else None)


def _codes(wtype, x):
    """(activations as the op's 8-bit codes give them, the q8_1 block sums or
    None): MUL_MAT is defined on src1 rounded to the weight type's vec_dot type."""
    n, K = x.shape
    if N.BLOCK[N.TYPES_BY_NAME[wtype]][0] == 256:  # q8_K
        b = x.reshape(n, -1, 256)
        top = b.gather(2, b.abs().argmax(2, keepdim=True))
        inv = torch.where(top == 0, 0.0, torch.full_like(top, -127.0) / top)  # (tensors: torch multiplies by 1 / a scalar)
        q = torch.round(b * inv).clamp(max=127)
        return (q.double() * torch.where(top == 0, 0.0, 1.0 / inv).double()).reshape(n, K), None
    b = x.reshape(n, -1, 32)  # q8_0 / q8_1: codes from the unrounded scale, the scale kept in f16
    d = b.abs().amax(2, keepdim=True)
    d = d / torch.full_like(d, 127.0)
    t = b * torch.where(d == 0, 0.0, 1.0 / d)
    q = torch.trunc(t + torch.copysign(torch.full_like(t, 0.5), t))
    sums = (q.sum(2) * d[:, :, 0]).half().double()
    return (q.double() * d.half().double()).reshape(n, K), sums


def _exact_mul_mat(wtype, w, x):
    if wtype in FLOATS:
        return x.to(FLOATS[wtype]).double() @ w.double().T
    K = x.shape[1]
    a, sums = _codes(wtype, x)
    out = []
    for part in w.split(16384):
        v, mins = _decode_rows(wtype, part, K)
        out.append(a @ v.T + (sums @ mins.T if mins is not None else 0))
    return torch.cat(out, 1)


def _attend(q, k, v, scale, mask=None):
    """softmax(q k^T scale + mask) v for [heads, rows, size] in 64 bits, grouped heads."""
    group = q.shape[0] // k.shape[0]
    k, v = k.repeat_interleave(group, 0), v.repeat_interleave(group, 0)
    s = q @ k.transpose(1, 2).contiguous() * scale
    return torch.softmax(s if mask is None else s + mask, 2) @ v


def _exact_decoder(s):
    """The decoder on unrounded activations in 64 bits (f16 keys and values, as the caches hold them)."""
    c, H, KV, D = s["config"], s["config"].n_head, s["config"].n_head_kv, s["config"].head_dim
    names = {name: (ty, ne, w) for (name, ty, ne), w in zip(c.weight_shapes(), s["weights"])}

    def dense(name, rows=None):
        ty, ne, w = names[name]
        w = w if rows is None else w[rows.long()]
        parts = []
        for p in w.split(16384):
            v, mins = _decode_rows(N.TYPE_NAMES[ty], p, ne[0])
            parts.append(v if mins is None else v + mins.repeat_interleave(32, 1))
        return torch.cat(parts)

    def norm(x, name):
        return x * torch.rsqrt(x.square().mean(1, keepdim=True) + c.eps) * names[name][2].double()

    def rope(t, pos):  # [T, heads, D], pairs of neighbours
        a = pos.double()[:, None, None] * c.rope_base ** (-torch.arange(0, D, 2, device="cuda").double() / D)
        x, y = t[..., 0::2], t[..., 1::2]
        return torch.stack([x * a.cos() - y * a.sin(), x * a.sin() + y * a.cos()], -1).reshape(t.shape)

    tokens, pos = s["inputs"][0], s["inputs"][1]
    T = tokens.numel()
    x = dense("tok_embd", tokens)
    for i in range(c.n_layer):
        cur = norm(x, f"l{i}.attn_norm")
        q = rope((cur @ dense(f"l{i}.wq").T).reshape(T, H, D), pos)
        k = rope((cur @ dense(f"l{i}.wk").T).reshape(T, KV, D), pos).half().double()
        v = (cur @ dense(f"l{i}.wv").T).reshape(T, KV, D).half().double()
        if s["path"] == "prompt":
            mask = torch.full((T, T), float("-inf"), device="cuda", dtype=torch.float64).triu(1)
            att = _attend(*(t.transpose(0, 1).contiguous() for t in (q, k, v)), D ** -0.5, mask).transpose(0, 1)
        else:
            kc, vc = (s["cache"][(2 * i + j) * s["per"]:(2 * i + j + 1) * s["per"]] for j in (0, 1))
            kc, vc = kc.reshape(-1, KV, D // 8, 16, 8), vc.reshape(-1, KV, D, 16)
            att = []
            for n, length in enumerate(s["lens"]):
                pages = s["inputs"][3][n, :-(-length // 16)].long()
                K = kc[pages].permute(0, 3, 1, 2, 4).reshape(-1, KV, D)[:length].double()
                V = vc[pages].permute(0, 3, 1, 2).reshape(-1, KV, D)[:length].double()
                K[length - 1], V[length - 1] = k[n], v[n]
                att.append(_attend(q[n][:, None], K.transpose(0, 1).contiguous(), V.transpose(0, 1).contiguous(),
                                   D ** -0.5)[:, 0])
            att = torch.stack(att)
        x = x + att.reshape(T, H * D) @ dense(f"l{i}.wo").T
        cur = norm(x, f"l{i}.ffn_norm")
        h = torch.nn.functional.silu(cur @ dense(f"l{i}.w_gate").T) * (cur @ dense(f"l{i}.w_up").T)
        x = x + h @ dense(f"l{i}.w_down").T
    x = norm(x[-1:] if s["path"] == "prompt" else x, "out_norm")
    return x @ dense("output").T


def exact(case, seed):
    s = prepare(case, seed)
    path = case["path"]
    if path == "mul_mat":
        return _exact_mul_mat(case["wtype"], s["w"], s["x"])
    if path == "mul_mat_id":
        M, T, used = case["M"], case["tokens"], case["used"]
        x = s["x"].expand(T, used, case["K"]).reshape(T * used, -1)
        ids = s["ids"].reshape(-1)
        out = torch.empty((T * used, M), dtype=torch.float64, device="cuda")
        for e in ids.unique().tolist():
            at = (ids == e).nonzero()[:, 0]
            out[at] = _exact_mul_mat(case["wtype"], s["w"][e * M:(e + 1) * M], x[at])
        return out.reshape(T, used, M)
    if path == "paged":
        KV, D = case["kv_heads"], case["head_size"]
        out = []
        for i, n in enumerate(s["lens"].tolist()):
            pages = s["table"][i, :-(-n // case["block"])].long()
            k = s["k"][pages].permute(1, 0, 3, 2, 4).reshape(KV, -1, D)[:, :n].double()
            v = s["v"][pages].permute(1, 0, 3, 2).reshape(KV, -1, D)[:, :n].double()
            out.append(_attend(s["q"][i][:, None].double(), k, v, D ** -0.5)[:, 0])
        return torch.stack(out)
    if path == "flash":
        mask = s["mask"][0, 0].double() if s["mask"] is not None else None
        out = [_attend(s["q"][b].half().double(), s["k"][b].double(), s["v"][b].double(), case["head_size"] ** -0.5, mask)
               for b in range(case["batch"])]
        return torch.stack(out).transpose(1, 2).contiguous()
    logits = _exact_decoder(s)
    return {"logits": logits.reshape([1, 1] + list(logits.shape)), "cache": None}
