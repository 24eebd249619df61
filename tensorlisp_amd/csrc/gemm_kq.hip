// GEMM for GGML_OP_MUL_MAT with k-quant weights and more than 16 activation
// columns on the int8 matrix cores, gfx950.
//
// What the CPU backend computes per 256-element super-block
// (ggml_vec_dot_q{2,3,4,5,6}_K_q8_K_generic, ggml-cpu/quants.c:565-904):
//   y += (d * dy) * S - (dmin * dy) * Mn,
//   S  = sum over the elements of (sc_s * q) * q8        (integer),
//   Mn = sum over the sub-blocks of m_s * (sum of q8)    (integer; q2 / q4 / q5_K).
// The scaled code sc_s * q of an element is formed once per workgroup as it
// is staged to LDS, as one or two int8 planes, so that the products of a whole
// super-block run on v_mfma_i32_32x32x32_i8 without any per-sub-block scaling
// between them, exact in int32 (the planes: kq_unit.hpp).
// Mn is one f16 MFMA per super-block (A = bsums, |.| <= 2032, B = the mins;
// exact). The f32 finalize runs once per super-block, as on the CPU.
//
// Two planes cost the matrix cores what one f16 pass costs (int8 runs at twice
// its rate), and an exact product of 13 bits has no f16 form at all (q6_K).
#include <type_traits>

#include "kernels.hpp"
#include "kq_unit.hpp"

namespace tlh {

// Tile of BM weight rows x BN tokens per workgroup of WM x WN waves: a wave owns
// BM / WM rows and BN / WN tokens in MFMA tiles of MT x MT (16 where the tile is
// too small to give every wave one of 32; waves that share a tile's K steps
// instead round each super-block's sum twice: N = 32 error 7.3e-8 -> 7.8e-8).
// K advances in stages of 128 elements through two LDS buffers: while a stage
// is multiplied, the next one's weights (fetched to registers two stages
// ahead) are scaled and written beside it with its activation codes; one
// LDS-only barrier a stage. LDS rows are 128 bytes, chunk c of row r at
// position c ^ (r & 7), so that 8 consecutive rows' operand reads hit
// distinct banks.
// GRP (MUL_MAT_ID): a column tile is an entry of the plan, its columns are
// (expert, token) pairs with activation rows and destinations of their own.
template <int MT> struct KqTileTypes;
template <> struct KqTileTypes<32> {
    using I = kq_v16i;
    using F = kq_v16f;
    using H = kq_v8h;
};
template <> struct KqTileTypes<16> {
    using I = kq_v4i;
    using F = kq_v4f;
    using H = kq_v4h;
};
__device__ __forceinline__ kq_v16i kq_mma(kq_v4i a, kq_v4i b, kq_v16i c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0); }
__device__ __forceinline__ kq_v4i kq_mma(kq_v4i a, kq_v4i b, kq_v4i c) { return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0); }
__device__ __forceinline__ kq_v16f kq_mma_min(kq_v8h a, kq_v8h b) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, (kq_v16f){}, 0, 0, 0); }
__device__ __forceinline__ kq_v4f kq_mma_min(kq_v4h a, kq_v4h b) { return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, (kq_v4f){}, 0, 0, 0); }

template <int WT, int BM, int BN, int WM, int WN, int MT, int WPE, bool GRP>
__global__ void __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) k_gemm_kq(const MatmulArgs a) {
    kernarg_prefetch<(kernarg_lines(sizeof(MatmulArgs)))>();
    constexpr int NT = 64 * WM * WN, P = kq_planes<WT>(), SB = block_bytes(WT);
    using Tile = KqTileTypes<MT>;
    constexpr int TM = BM / WM / MT, TN = BN / WN / MT, KST = MT / 8, NR = MT * MT / 64;  // tiles a wave, K steps a stage, results a lane
    constexpr int UPT = BM * 4 / NT, BPT = BN * 8 / NT;  // weight units, activation pieces a thread stages
    constexpr bool MIN = kq_has_min<WT>();
    static_assert(UPT >= 1 && BPT >= 1 && NT >= 2 * BN && TM >= 1 && TN >= 1, "tile");
    __shared__ __attribute__((aligned(16))) int8_t sW[2][P][BM][128];
    __shared__ __attribute__((aligned(16))) int8_t sX[2][BN][128];
    __shared__ __attribute__((aligned(16))) float sD[BM], sDmin[MIN ? BM : 1];
    __shared__ __attribute__((aligned(16))) uint8_t sMin[MIN ? BM : 1][16];
    __shared__ __attribute__((aligned(16))) float sDx[BN];
    __shared__ __attribute__((aligned(16))) _Float16 sBs[MIN ? BN : 1][16];
    __shared__ int64_t sOut[GRP ? BN : 1];  // byte offset of a column's outputs
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int64_t K = a.K, nsb = K / QKK;
    const uint32_t batches = GRP ? 1u : (uint32_t)(a.ne12 * a.ne13);
    const uint32_t kc = batches == 1 ? blockIdx.z : blockIdx.z / batches, batch = blockIdx.z - kc * batches;
    const MmSlice sl = mm_slice(a, batch);
    const uint8_t *W = sl.w;
    const ActView act = act_view(a.act, TLH_TYPE_Q8_K, K, mm_act_rows(a));
    const int64_t nkc = gridDim.z / batches;
    // grid x: the token tiles of a row tile next to each other (any number of rows)
    const uint32_t ntn = (uint32_t)(GRP ? a.grp_tiles : (a.N + BN - 1) / BN);
    const uint32_t tm = ntn == 1 ? blockIdx.x : blockIdx.x / ntn, tn = blockIdx.x - tm * ntn;
    const int64_t m_base = (int64_t)tm * BM;
    int64_t n_base = (int64_t)tn * BN, n_cols = a.N - n_base;
    int sg = 0;
    int64_t m0 = 0;
    const int32_t *pairs = nullptr;
    if constexpr (GRP) {
        if ((int)tn >= a.grp[0]) return;
        const int32_t *t = a.grp + 4 + 4 * (int64_t)tn;
        const int e = t[0];
        n_base = 0;
        n_cols = t[2];
        pairs = a.grp + 4 + 4 * a.grp_tiles + t[1];
        if (tid < BN) {
            const uint32_t p = (uint32_t)pairs[tid < n_cols ? tid : 0], tok = p / (uint32_t)a.ne12;
            sOut[tid] = nkc > 1 ? (int64_t)p * a.M * 4 : (int64_t)(p - tok * (uint32_t)a.ne12) * a.d_nb2 + (int64_t)tok * a.d_nb3;
        }
        lds_barrier();  // sOut, before any use: a chunk without super-blocks meets no other barrier
        if (e < 0) {  // no such expert: NaN
            char *o = nkc > 1 ? (char *)(a.part + kc * (a.ne12 * a.ne13) * a.M) : (char *)a.dst;
            for (int i = tid; i < BM * (int)n_cols; i += NT) {
                const int64_t m = m_base + i % BM;
                if (m < a.M) *(float *)(o + sOut[i / BM] + 4 * m) = __builtin_nanf("");
            }
            return;
        }
        W = a.w + (int64_t)e * a.w_nb2;
    } else if (a.nseg > 0) {  // segments: as MatmulArgs says; a tile lies in one
        sg = (int)(m_base >= a.seg_m0[1]) + (int)(a.nseg > 2 && m_base >= a.seg_m0[2]);
        m0 = a.seg_m0[sg];
        W = a.seg_w[sg];
    }
    // activation row of the tile's column c (clamped to the last one)
    auto arow = [&](int c) -> int64_t {
        const int64_t col = c < n_cols ? c : n_cols - 1;
        if constexpr (GRP) {
            const uint32_t p = (uint32_t)pairs[col], tok = p / (uint32_t)a.ne12, slot = p - tok * (uint32_t)a.ne12;
            return (int64_t)(slot % (uint32_t)a.id_b1) + a.id_b1 * (int64_t)tok;
        }
        return a.n0 + n_base + col + a.N_total * batch;
    };

    const uint8_t *wrow[UPT];
    const int u = tid & 3;
#pragma unroll
    for (int i = 0; i < UPT; ++i) {
        const int row = (tid + i * NT) >> 2;
        const int64_t grow = m_base + row < a.M ? m_base + row : a.M - 1;  // clamped: loads in bounds
        wrow[i] = W + (grow - m0) * a.w_nb1;
    }
    const int8_t *xrow[BPT];
#pragma unroll
    for (int i = 0; i < BPT; ++i) xrow[i] = act.qs + arow((tid + i * NT) >> 3) * K + 16 * (tid & 7);
    const float *dxrow = act.d + arow(tid % BN) * nsb;
    const int16_t *bsrow = act.bsums + arow((tid >> 1) % BN) * (K / 16) + 8 * (tid & 1);

    struct Regs {
        KqUnit<WT> w[UPT];
        kq_u4 x[BPT];
        float dx;
        kq_u4 bs;
    };
    Regs r0, r1;  // the next first and second half
    const int64_t share = (nsb + nkc - 1) / nkc;
    const int64_t sb0 = kc * share, sb1 = sb0 + share < nsb ? sb0 + share : nsb;
    auto fetch = [&](auto hc, int64_t sb, Regs &r) {
        constexpr int H = decltype(hc)::value;
        sb = sb < sb1 ? sb : sb1 - 1;  // past the share: the last one again, never multiplied
#pragma unroll
        for (int i = 0; i < UPT; ++i) kq_fetch<WT, H>(wrow[i] + sb * SB, u, r.w[i]);
#pragma unroll
        for (int i = 0; i < BPT; ++i) r.x[i] = *(const kq_u4 *)(xrow[i] + sb * QKK + 128 * H);
        if constexpr (H == 1) {
            r.dx = dxrow[sb];
            if constexpr (MIN) r.bs = *(const kq_u4 *)(bsrow + sb * 16);
        }
    };
    auto commit = [&](auto hc, const Regs &r) {
        constexpr int H = decltype(hc)::value;
#pragma unroll
        for (int i = 0; i < UPT; ++i) {
            const int row = (tid + i * NT) >> 2, c0 = kq_chunk<WT>(u), c1 = c0 + kq_gap<WT>();
            uint32_t o[2][2][4];
            kq_codes<WT, H>(r.w[i], u, o);
#pragma unroll
            for (int p = 0; p < P; ++p) {
                int8_t *dst = sW[H][p][row];
                *(kq_u4 *)(dst + ((c0 ^ (row & 7)) << 4)) = kq_u4{o[p][0][0], o[p][0][1], o[p][0][2], o[p][0][3]};
                *(kq_u4 *)(dst + ((c1 ^ (row & 7)) << 4)) = kq_u4{o[p][1][0], o[p][1][1], o[p][1][2], o[p][1][3]};
            }
            if (H == 1 && (!MIN || u == 0)) {  // (!MIN: the row's four threads write the same values)
                float d, dmin;
                uint32_t mn[4];
                kq_row_meta<WT>(r.w[i], d, dmin, mn);
                sD[row] = d;
                if constexpr (MIN) {
                    sDmin[row] = dmin;
                    if constexpr (WT == TLH_TYPE_Q2_K) {
                        *(kq_u4 *)sMin[row] = kq_u4{mn[0], mn[1], mn[2], mn[3]};
                    } else {  // min s belongs to bsums 2s and 2s + 1
                        *(kq_u4 *)sMin[row] = kq_u4{__builtin_amdgcn_perm(0u, mn[0], 0x01010000u),
                                                         __builtin_amdgcn_perm(0u, mn[0], 0x03030202u),
                                                         __builtin_amdgcn_perm(0u, mn[1], 0x01010000u),
                                                         __builtin_amdgcn_perm(0u, mn[1], 0x03030202u)};
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < BPT; ++i) {
            const int col = (tid + i * NT) >> 3;
            *(kq_u4 *)(sX[H][col] + (((tid & 7) ^ (col & 7)) << 4)) = r.x[i];
        }
        if constexpr (H == 1) {
            if (!MIN || tid < BN) sDx[tid % BN] = r.dx;
            if constexpr (MIN) {
                if (tid < 2 * BN) {
                    const uint32_t b[4] = {r.bs.x, r.bs.y, r.bs.z, r.bs.w};
                    kq_v8h h;
#pragma unroll
                    for (int i = 0; i < 8; ++i) h[i] = (_Float16)(float)(int16_t)(b[i >> 1] >> (16 * (i & 1)));
                    *(kq_v8h *)&sBs[tid >> 1][8 * (tid & 1)] = h;
                }
            }
        }
    };

    const int lr = lane % MT, lg = lane / MT;
    typename Tile::I S[P][TN][TM];
    typename Tile::F acc[TN][TM], tot[TN][TM];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            acc[j][i] = tot[j][i] = (typename Tile::F){};
#pragma unroll
            for (int p = 0; p < P; ++p) S[p][j][i] = (typename Tile::I){};
        }
    // without mins token tile by token tile, so that the second half's finalize
    // of one tile can run between the products of the next (the weights'
    // operands of all K steps held); the types with mins have no registers for
    // that and go K step by K step
    auto multiply = [&](auto hc) {
        constexpr int H = decltype(hc)::value;
        constexpr int G = 64 / MT;  // 16-byte chunks of a K step
        auto wop = [&](int p, int i, int t) {
            const int r = MT * (wm * TM + i) + lr;
            return *(const kq_v4i *)(sW[H][p][r] + (((G * t + lg) ^ (r & 7)) << 4));
        };
        auto xop = [&](int j, int t) {
            const int c = MT * (wn * TN + j) + lr;
            return *(const kq_v4i *)(sX[H][c] + (((G * t + lg) ^ (c & 7)) << 4));
        };
        if constexpr (!MIN) {
            kq_v4i wv[KST][P][TM];
#pragma unroll
            for (int tt = 0; tt < KST; ++tt)
#pragma unroll
                for (int p = 0; p < P; ++p)
#pragma unroll
                    for (int i = 0; i < TM; ++i) wv[tt][p][i] = wop(p, i, tt);
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int tt = 0; tt < KST; ++tt) {
                    const kq_v4i xv = xop(j, tt);
#pragma unroll
                    for (int p = 0; p < P; ++p)
#pragma unroll
                        for (int i = 0; i < TM; ++i)
                            S[p][j][i] = kq_mma(xv, wv[tt][p][i], S[p][j][i]);
                }
        } else {
#pragma unroll
            for (int tt = 0; tt < KST; ++tt) {
                kq_v4i xv[TN];
#pragma unroll
                for (int j = 0; j < TN; ++j) xv[j] = xop(j, tt);
#pragma unroll
                for (int p = 0; p < P; ++p)
#pragma unroll
                    for (int i = 0; i < TM; ++i) {
                        const kq_v4i wv = wop(p, i, tt);
#pragma unroll
                        for (int j = 0; j < TN; ++j)
                            S[p][j][i] = kq_mma(xv[j], wv, S[p][j][i]);
                    }
            }
        }
    };
    // D[token][row]: lane holds weight row lr and tokens 8 q + 4 lg + e of a tile
    auto finalize = [&]() {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int r = MT * (wm * TM + i) + lr;
            const float d = sD[r];
            float dmin = 0.0f;
            typename Tile::H mv = {};
            if constexpr (MIN) {  // of bsums lg * MT / 4 .. (k of the MFMA)
                dmin = sDmin[r];
                const kq_u2 m = *(const kq_u2 *)&sMin[r][MT == 32 ? 8 * lg : 4 * (lg & 2)];
                const uint32_t lo = MT == 32 ? m.x : lg & 1 ? m.y : m.x;
#pragma unroll
                for (int e = 0; e < MT / 4; ++e) mv[e] = (_Float16)(float)(((e < 4 ? lo : m.y) >> (8 * (e & 3))) & 0xff);
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int c0 = MT * (wn * TN + j);
                typename Tile::F Mn = {};
                if constexpr (MIN) Mn = kq_mma_min(*(const typename Tile::H *)&sBs[c0 + lr][MT / 4 * lg], mv);
#pragma unroll
                for (int q = 0; q < NR / 4; ++q) {
                    const float4 y4 = *(const float4 *)&sDx[c0 + 8 * q + 4 * lg];
                    const float dy[4] = {y4.x, y4.y, y4.z, y4.w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int k = 4 * q + e;
                        float v = kq_sum<WT>(S[0][j][i][k], S[P - 1][j][i][k]) * d;
                        if constexpr (MIN) v -= dmin * Mn[k];
                        acc[j][i][k] += dy[e] * v;
                    }
                }
#pragma unroll
                for (int p = 0; p < P; ++p) S[p][j][i] = (typename Tile::I){};
            }
        }
    };
    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;
    if (sb0 < sb1) {
        fetch(H0{}, sb0, r0);
        fetch(H1{}, sb0, r1);
        commit(H0{}, r0);
        fetch(H0{}, sb0 + 1, r0);
        lds_barrier();
        // The sums move to a second set every few super-blocks (kq_unit.hpp). Error
        // against 64 bits, rms over rms, in one chain / now: q4_K 14336 x 14336, N = 48
        // 1.10e-7 / 8.5e-8; 14336 x 4096, N = 64 7.6e-8 / 7.2e-8. In time: q4_K
        // 14336 x 4096, N = 512 107 -> 109 us.
        const int every = kq_flush_every((int)(sb1 - sb0));
        auto flush = [&]() {
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    tot[j][i] += acc[j][i];
                    acc[j][i] = (typename Tile::F){};
                }
        };
        // The 64-row tiles run to a flush and back; one inside their loop, as in the
        // 128 x 128 tiles, splits its schedule (q6_K 14336 x 4096, N = 64: 32.7 against 34.2
        // us; 128 x 128 the other way round, N = 512: 126 against 110).
        constexpr bool NEST = BM == 64;
        int64_t sb = sb0;
        int left = every;
        auto upto = [&](int64_t end) {
            for (; sb < end; ++sb) {
                multiply(H0{});
                commit(H1{}, r1);
                fetch(H1{}, sb + 1, r1);
                lds_barrier();
                multiply(H1{});
                if constexpr (MIN) finalize();
                commit(H0{}, r0);  // (past the share: read by nobody)
                fetch(H0{}, sb + 2, r0);
                if constexpr (!MIN) finalize();
                if constexpr (!NEST) {
                    if (--left == 0) {
                        flush();
                        left = every;
                    }
                }
                lds_barrier();
            }
            flush();
        };
        if constexpr (NEST) {
            while (sb < sb1) upto(sb + every < sb1 ? sb + every : sb1);
        } else {
            upto(sb1);
        }
    }

    // row m of column n goes to obase + n * ostride + 4 m (GRP: obase + sOut[n] + 4 m)
    char *obase = (char *)a.dst + sl.i12 * a.d_nb2 + sl.i13 * a.d_nb3 + a.n0 * a.d_nb1;
    int64_t ostride = a.d_nb1;
    if constexpr (GRP) {
        obase = nkc > 1 ? (char *)(a.part + kc * (a.ne12 * a.ne13) * a.M) : (char *)a.dst;
    } else if (nkc > 1 || a.keep_part) {
        obase = (char *)(a.part + (kc * batches + batch) * a.N * a.M);
        ostride = 4 * a.M;
    } else if (a.nseg > 0) {
        ostride = a.seg_d_nb1[sg];
        obase = (char *)a.seg_dst[sg] + a.n0 * ostride - 4 * m0;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int64_t m = m_base + MT * (wm * TM + i) + lr;
        if (m < a.M) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int k = 0; k < NR; ++k) {
                    const int c = MT * (wn * TN + j) + 8 * (k >> 2) + 4 * lg + (k & 3);
                    if (c < n_cols)
                        *(float *)(obase + (GRP ? sOut[c] : (n_base + c) * ostride) + 4 * m) = tot[j][i][k];
                }
        }
    }
}

template <int WT, int BM, int BN, int WM, int WN, int MT, int WPE>
static void launch_kq_tile(const MatmulArgs &a, int ks, hipStream_t stream) {
    const int64_t mt = (a.M + BM - 1) / BM, threads = 64 * WM * WN;
    if (a.ids) {
        const dim3 grid((unsigned)(a.grp_tiles * mt), 1u, (unsigned)ks);
        hipLaunchKernelGGL((k_gemm_kq<WT, BM, BN, WM, WN, MT, WPE, true>), grid, dim3(threads), 0, stream, a);
    } else {
        const dim3 grid((unsigned)((a.N + BN - 1) / BN * mt), 1u, (unsigned)(a.ne12 * a.ne13 * ks));
        hipLaunchKernelGGL((k_gemm_kq<WT, BM, BN, WM, WN, MT, WPE, false>), grid, dim3(threads), 0, stream, a);
    }
}

template <int WT> static tlh_status launch_kq(const MatmulArgs &a, int bn, int ks, hipStream_t stream) {
    switch (bn) {
    case 32: launch_kq_tile<WT, 64, 32, 4, 1, 16, 3>(a, ks, stream); break;
    case 64: launch_kq_tile<WT, 64, 64, 2, 2, 32, 2>(a, ks, stream); break;
    default: launch_kq_tile<WT, 128, 128, 4, 2, 32, 2>(a, ks, stream); break;
    }
    return check_launch(WT == TLH_TYPE_Q4_K || WT == TLH_TYPE_Q5_K ? "gemm_q4k" : "gemm_kq");
}

// Tile shapes by columns. Up to 64 columns the weights' bytes set the time:
// small tiles of 4 waves, two or three on a CU at once, keep more weight loads
// in flight and leave no products on padding (128 x 32, two a CU: q6_K 4096 x
// 4096, N = 32 21.3 against 16.3 us). Above, 128 x 128 on 8 waves (32
// rows x 64 tokens each; one workgroup's LDS fills a CU): each weight code is
// scaled once for 128 tokens. 64 x 128 tiles of 4 waves, two a CU, were slower
// (q6_K 14336 x 4096, N = 2048: 412 against 387 us).
KqTile gemm_kq_tile(int64_t N) {
    if (N <= 32) return {64, 32, 3};
    if (N <= 64) return {64, 64, 2};
    return {128, 128, 1};
}

tlh_status launch_gemm_kq(const MatmulArgs &a, int bn, int ks, hipStream_t stream) {
    switch (a.wtype) {
    case TLH_TYPE_Q2_K: return launch_kq<TLH_TYPE_Q2_K>(a, bn, ks, stream);
    case TLH_TYPE_Q3_K: return launch_kq<TLH_TYPE_Q3_K>(a, bn, ks, stream);
    case TLH_TYPE_Q4_K: return launch_kq<TLH_TYPE_Q4_K>(a, bn, ks, stream);
    case TLH_TYPE_Q5_K: return launch_kq<TLH_TYPE_Q5_K>(a, bn, ks, stream);
    case TLH_TYPE_Q6_K: return launch_kq<TLH_TYPE_Q6_K>(a, bn, ks, stream);
    default: return set_error(TLH_UNSUPPORTED, "gemm_kq: weight type %d", a.wtype);
    }
}

}  // namespace tlh
