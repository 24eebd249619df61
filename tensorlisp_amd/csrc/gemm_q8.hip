// Prefill GEMM for GGML_OP_MUL_MAT with q8_0 / q4_0 weights and more than 16
// activation columns, gfx950.
//
// The CPU backend multiplies a q8_0 / q4_0 row with a q8_0 activation row
// block by block (ggml_vec_dot_q8_0_q8_0_generic, ggml-cpu/quants.c:451-476:
// sum += sumi * (dx * dy); ggml_vec_dot_q4_0_q8_0_generic, :225-258:
// sum += (sumi * dx) * dy), where sumi is the exact integer dot product of one
// 32-element block. Here each block of a 32 x 32 output tile is one
// v_mfma_i32_32x32x32_i8 (K = 32 = one block, exact int32), and the f32 scaling
// follows per block in the CPU's rounding order (only the order of the f32
// sum over blocks differs). The per-block scaling is VALU work of the same
// order as the MFMA issue; the kernel is bound by both together, well under
// the int8 peak, but it reads each weight once per 128-token tile instead of
// once per 16 tokens.
//
// Tiling: BM weight rows x BN tokens per workgroup of 4 waves in WM x WN x WK
// parts, each in 32 x 32 MFMA tiles (WK: parts of a stage's blocks, summed in
// LDS at the end); K advances in stages of four blocks (128 elements). Weight
// codes are staged to LDS as int8 (q4_0 nibbles expanded to q - 8), activation
// codes as they are; LDS holds two stage buffers, written one stage ahead and
// fetched D + 1 stages ahead, with one barrier per stage. The tile shapes and
// what they measured are at gemm_q8_tile.
#include "kernels.hpp"

namespace tlh {

typedef int v4i32 __attribute__((ext_vector_type(4)));
typedef int v16i32 __attribute__((ext_vector_type(16)));

constexpr int QBK = 128, QSB = QBK / 32;  // K per stage, blocks per stage

// Rows of 128 code bytes = 8 chunks of 16; chunk c of row r sits at chunk
// position c ^ (r & 7), so the 16-byte operand reads of 8 consecutive rows hit
// distinct banks. Scales are block-major so 4 consecutive rows read as a float4.
template <int BM, int BN> struct __attribute__((aligned(16))) Q8GemmSmem {
    int8_t A[2][BM][QBK];
    int8_t B[2][BN][QBK];
    float dA[2][QSB][BM];
    float dB[2][QSB][BN];
};

__device__ __forceinline__ int swz16(int row, int chunk) { return (chunk ^ (row & 7)) << 4; }

__device__ __forceinline__ uint4 ld16(const void *p) {
    uint4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

// q4_0 nibble bytes -> int8 (n - 8): byte i of `v` -> elements i (low) and i + 16 (high)
// (no borrow crosses a byte: each byte is at least 0x80 before the subtraction)
__device__ __forceinline__ uint32_t nib_lo_m8(uint32_t v) {
    return (((v & 0x0f0f0f0fu) | 0x80808080u) - 0x08080808u) ^ 0x80808080u;
}
__device__ __forceinline__ uint32_t nib_hi_m8(uint32_t v) {
    return ((((v >> 4) & 0x0f0f0f0fu) | 0x80808080u) - 0x08080808u) ^ 0x80808080u;
}

// One thread's share of a stage: WI blocks of a weight row, XI of a token
// (4 / WI and 4 / XI threads a row).
template <int WI, int XI> struct Q8StageRegs {
    uint4 w[2 * WI];   // a block's 32 code bytes (q8_0) or 16 nibble bytes (q4_0: one word of the two)
    uint16_t wd[WI];   // f16 scales
    uint4 x[2 * XI];   // activation codes
    float xd[XI];
};

template <int WT, int BM, int BN, int WM, int WN, int WK, int D, int WPE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) k_gemm_q8(const MatmulArgs a) {
    constexpr int TM = BM / WM / 32, TN = BN / WN / 32;  // MFMA tiles of a wave
    constexpr int WI = BM / 64, XI = BN > 64 ? BN / 64 : 1;
    static_assert(WM * WN * WK == 4 && TM * WM * 32 == BM && TN * WN * 32 == BN && QSB % WK == 0, "4 waves");
    __shared__ Q8GemmSmem<BM, BN> sm;
    constexpr int BB = block_bytes(WT);
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wk = wave / (WM * WN), wm = wave % (WM * WN) / WN, wn = wave % WN;
    const int64_t K = a.K;
    const int64_t nblk = K / QK;
    const uint32_t batches = (uint32_t)(a.ne12 * a.ne13);
    // K chunk kc of gridDim.z / batches (one batch slice: no division)
    const uint32_t kc = batches == 1 ? blockIdx.z : blockIdx.z / batches, batch = blockIdx.z - kc * batches;
    const MmSlice sl = mm_slice(a, batch);
    const int64_t i12 = sl.i12, i13 = sl.i13;
    const uint8_t *W = sl.w;
    const ActView act = act_view(a.act, TLH_TYPE_Q8_0, K, mm_act_rows(a));
    // grid x: the token tiles of a row tile next to each other (any number of rows)
    const uint32_t ntn = (uint32_t)((a.N + BN - 1) / BN);
    const uint32_t tm = ntn == 1 ? blockIdx.x : blockIdx.x / ntn;
    const int64_t m_base = (int64_t)tm * BM;
    const int64_t n_base = (int64_t)(blockIdx.x - tm * ntn) * BN;

    const int wr = tid / (4 / WI), wb = tid % (4 / WI) * WI;  // weight row, first block of the stage's four
    const int xr = tid / (4 / XI), xb = tid % (4 / XI) * XI;  // token
    const bool xon = BN >= 64 || tid < 4 * BN;                // (whole waves)
    const int64_t grow = m_base + wr < a.M ? m_base + wr : a.M - 1;  // clamped: loads in bounds
    const int64_t gcol = n_base + xr < a.N ? n_base + xr : a.N - 1;
    const uint8_t *wrow = W + grow * a.w_nb1;
    const int64_t arow = a.n0 + gcol + a.N_total * batch;
    const int8_t *xrow = act.qs + arow * K;
    const float *xdrow = act.d + arow * nblk;

    // this workgroup's stages: chunk kc of equal shares (stage indices are global)
    const int64_t nst = (nblk + QSB - 1) / QSB, nkc = gridDim.z / batches, share = (nst + nkc - 1) / nkc;
    const int64_t g0 = kc * share, stages = g0 + share < nst ? g0 + share : nst;
    // blocks past K (the last stage of a K that is not a multiple of 128)
    // load block 0 and get zero scales
    auto fetch = [&](int64_t stage, Q8StageRegs<WI, XI> &r) {
        stage = stage < stages ? stage : stages - 1;  // past the share: the last one again, never multiplied
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            const int64_t b0 = stage * QSB + wb + i;
            const uint8_t *bp = wrow + (b0 < nblk ? b0 : 0) * BB;
            __builtin_memcpy(&r.wd[i], bp, 2);
            r.w[2 * i] = ld16(bp + 2);
            if constexpr (WT == TLH_TYPE_Q8_0) r.w[2 * i + 1] = ld16(bp + 18);
            if (b0 >= nblk) r.wd[i] = 0;
        }
        if (xon) {
#pragma unroll
            for (int i = 0; i < XI; ++i) {
                const int64_t b0 = stage * QSB + xb + i, b = b0 < nblk ? b0 : 0;
                r.x[2 * i] = *(const uint4 *)(xrow + 32 * b);
                r.x[2 * i + 1] = *(const uint4 *)(xrow + 32 * b + 16);
                r.xd[i] = b0 < nblk ? xdrow[b] : 0.0f;
            }
        }
    };

    auto commit = [&](int64_t stage, const Q8StageRegs<WI, XI> &r) {
        const int buf = (int)(stage & 1);
        int8_t *ar = sm.A[buf][wr];
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            uint4 c0 = r.w[2 * i], c1;
            if constexpr (WT == TLH_TYPE_Q8_0) {
                c1 = r.w[2 * i + 1];
            } else {
                const uint4 v = c0;
                c0 = make_uint4(nib_lo_m8(v.x), nib_lo_m8(v.y), nib_lo_m8(v.z), nib_lo_m8(v.w));
                c1 = make_uint4(nib_hi_m8(v.x), nib_hi_m8(v.y), nib_hi_m8(v.z), nib_hi_m8(v.w));
            }
            const int c = 2 * (wb + i);  // the block's first 16-byte chunk in the row
            *(uint4 *)(ar + swz16(wr, c)) = c0;
            *(uint4 *)(ar + swz16(wr, c + 1)) = c1;
            sm.dA[buf][wb + i][wr] = h2f(r.wd[i]);
        }
        if (xon) {
            int8_t *br = sm.B[buf][xr];
#pragma unroll
            for (int i = 0; i < XI; ++i) {
                const int c = 2 * (xb + i);
                *(uint4 *)(br + swz16(xr, c)) = r.x[2 * i];
                *(uint4 *)(br + swz16(xr, c + 1)) = r.x[2 * i + 1];
                sm.dB[buf][xb + i][xr] = r.xd[i];
            }
        }
    };

    float acc[TM][TN][16];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int jn = 0; jn < TN; ++jn)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][jn][r] = 0.0f;

    const int lr = lane & 31, lg = lane >> 5;  // operand row / column; k half of the block
    const v16i32 zero = {};
    auto multiply = [&](int buf) {
        // one block at a time where a wave has four tiles: its products are
        // finished before the next block's MFMAs issue (all of them in flight at
        // once would hold 256 result registers)
        constexpr int UNROLL = TM * TN > 1 ? 1 : QSB / WK;
#pragma unroll UNROLL
        for (int jj = 0; jj < QSB / WK; ++jj) {
            const int j = wk * (QSB / WK) + jj;
            v4i32 av[TM], bv[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int ra = 32 * (TM * wm + i) + lr;
                av[i] = *(const v4i32 *)&sm.A[buf][ra][swz16(ra, 2 * j + lg)];
            }
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                const int rb = 32 * (TN * wn + i) + lr;
                bv[i] = *(const v4i32 *)&sm.B[buf][rb][swz16(rb, 2 * j + lg)];
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int jn = 0; jn < TN; ++jn) {
                    const v16i32 S = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[i], bv[jn], zero, 0, 0, 0);
                    const float dy = sm.dB[buf][j][32 * (TN * wn + jn) + lr];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float4 d4 = *(const float4 *)&sm.dA[buf][j][32 * (TM * wm + i) + 8 * q + 4 * lg];
                        const float dv[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
#pragma clang fp contract(off)
                            const float s = (float)S[4 * q + e];
                            if constexpr (WT == TLH_TYPE_Q8_0)
                                acc[i][jn][4 * q + e] += s * (dv[e] * dy);
                            else
                                acc[i][jn][4 * q + e] += (s * dv[e]) * dy;
                        }
                    }
                }
        }
    };
    // the sums of D stages move to a second set, which keeps the chains of
    // f32 additions as short as more K chunks would (four tiles a wave: no registers)
    constexpr bool FLUSH = TM * TN == 1;
    float tot[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) tot[r] = 0.0f;
    if (g0 < stages) {
        // D stages of loads in flight: local stage l's registers are pre[l % D]
        Q8StageRegs<WI, XI> pre[D];
#pragma unroll
        for (int d = 0; d < D; ++d) fetch(g0 + d, pre[d]);
        commit(g0, pre[0]);
        fetch(g0 + D, pre[0]);
        lds_barrier();
        for (int64_t s0 = g0; s0 < stages; s0 += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const int64_t st = s0 + d;
                if (st < stages) {
                    multiply((int)(st & 1));
                    commit(st + 1, pre[(d + 1) % D]);  // (past the share: read by nobody)
                    fetch(st + 1 + D, pre[(d + 1) % D]);
                    lds_barrier();
                }
            }
            if constexpr (FLUSH) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    tot[r] += acc[0][0][r];
                    acc[0][0][r] = 0.0f;
                }
            }
        }
        if constexpr (FLUSH) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[0][0][r] = tot[r];
        }
    }

    if constexpr (WK > 1) {
        // the waves' shares of each stage's blocks, added in wave order through LDS
        // (the last stage's barrier is behind every read of the buffers)
        static_assert(WK == 1 || (TM == 1 && TN == 1 && sizeof(sm.A) >= (size_t)(WK - 1) * WM * WN * 4096), "merge buffer");
        float *red = (float *)&sm.A[0][0][0];
        const int part = wave % (WM * WN);
        if (wk > 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r) red[((wk - 1) * WM * WN + part) * 1024 + 64 * r + lane] = acc[0][0][r];
        }
        lds_barrier();
        if (wk > 0) return;
#pragma unroll
        for (int w = 0; w < WK - 1; ++w)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[0][0][r] += red[(w * WM * WN + part) * 1024 + 64 * r + lane];
    }

    // lane holds token n = lane % 32 of each 32 x 32 tile and rows 8q + 4 lg + (0..3)
    // (with K chunks, to this chunk's partials [chunk][batch][N][M])
    char *dbase = (char *)a.dst + i12 * a.d_nb2 + i13 * a.d_nb3;
    float *pbase = nkc > 1 ? a.part + (kc * batches + batch) * a.N * a.M : nullptr;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int jn = 0; jn < TN; ++jn) {
            const int64_t n = n_base + 32 * (TN * wn + jn) + lr;
            if (n >= a.N) continue;
            float *drow = pbase ? pbase + n * a.M : (float *)(dbase + (a.n0 + n) * a.d_nb1);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int64_t m = m_base + 32 * (TM * wm + i) + 8 * q + 4 * lg;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (m + e < a.M) drow[m + e] = acc[i][jn][4 * q + e];
            }
        }
}

template <int WT, int BM, int BN, int WM, int WN, int WK, int D, int WPE>
static void launch_q8_tile(const MatmulArgs &a, int ks, hipStream_t stream) {
    const dim3 grid((unsigned)((a.N + BN - 1) / BN * ((a.M + BM - 1) / BM)), 1u, (unsigned)(a.ne12 * a.ne13 * ks));
    hipLaunchKernelGGL((k_gemm_q8<WT, BM, BN, WM, WN, WK, D, WPE>), grid, dim3(256), 0, stream, a);
}

template <int WT> static tlh_status launch_q8(const MatmulArgs &a, int ks, hipStream_t stream) {
    switch (gemm_q8_tile(a.N).bn) {
    case 32: launch_q8_tile<WT, 64, 32, 2, 1, 2, 2, 3>(a, ks, stream); break;
    case 64: launch_q8_tile<WT, 64, 64, 2, 2, 1, 3, 2>(a, ks, stream); break;
    default: launch_q8_tile<WT, 128, 128, 2, 2, 1, 1, 2>(a, ks, stream); break;
    }
    return check_launch("gemm_q8");
}

// Tile shapes by columns. Up to 64 columns a 128 x 128 tile multiplies and scales
// mostly padding, and two workgroups a CU keep few weight loads in flight: 64-row
// tiles of 32 or 64 tokens, with two or three stages of loads in flight. In us,
// 128 x 128 tiles -> these: 14336 x 4096, N = 32 q8_0 70.4 -> 42.6, q4_0 58.3 ->
// 40.5; N = 64 q8_0 80.7 -> 56.7; q4_0 4096 x 14336, N = 57 65.1 -> 52.1; q8_0
// 1000 x 4096, N = 33 52.7 -> 26.8. Error against 64 bits, rms over rms: 1.2e-7
// -> 8.2e-8 and 9.2e-8 (64 x 64 without the second set of sums: 1.5e-7).
KqTile gemm_q8_tile(int64_t N) {
    if (N <= 32) return {64, 32, 3};
    if (N <= 64) return {64, 64, 2};
    return {128, 128, 2};
}

tlh_status launch_gemm_q8(const MatmulArgs &a, int ksplit, hipStream_t stream) {
    switch (a.wtype) {
    case TLH_TYPE_Q8_0: return launch_q8<TLH_TYPE_Q8_0>(a, ksplit, stream);
    case TLH_TYPE_Q4_0: return launch_q8<TLH_TYPE_Q4_0>(a, ksplit, stream);
    default: return set_error(TLH_UNSUPPORTED, "gemm_q8: weight type %d", a.wtype);
    }
}

}  // namespace tlh
