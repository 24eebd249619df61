// MUL_MAT_ID with q4_K / q5_K weights and up to 32 (expert, token) pairs an
// expert, as a stream over the experts' matrices, gfx950. The arithmetic is
// gemm_kq.hip's (int8 planes of scaled codes, exact super-block sums, one f32
// finalize each).
//
// With so few columns the weights' bytes set the time, and a tile staged
// through LDS spends it waiting instead: its loads, conversion, barrier,
// operand reads and finalize follow one another. Here the weights never meet
// LDS: in v_mfma_i32_16x16x64_i8's operand layout lane (row, g) holds 16 bytes
// of its row for each k group g, which is what one unit's group of 16 codes is
// (kq_unit.hpp), so a lane loads its unit straight from the row, scales it and
// multiplies. The activation codes of the workgroup's columns go to LDS once
// (one barrier), then each wave walks its 16-row groups on its own, two
// super-blocks of loads ahead. Eight q4_K experts of 14336 x 4096 (264 MB), the
// kernel alone against the LDS tiles: 32 pairs 101 -> 60 us (4.4 TB/s), 198 evenly
// dealt pairs 117 -> 68 us; as a router deals them (55 to 4 an expert) 94 us, since
// experts above 32 pairs take two plan entries and their matrix is read twice (11
// entries, 363 MB), and the blocks of an entry leave its last round part empty.
// The quantize and the plan before it take 5 us each. Not for q6_K: its 2-byte aligned units take seven loads a super-block
// (64 experts of 4096 x 2048, 128 pairs: 128 us, the tiles 101 us).
#include "kq_unit.hpp"

namespace tlh {

constexpr int KQS_WAVES = 16;

// LDS of kc elements of nt * 16 columns: codes [col][kc], scales [col][kc / 256],
// bsums as f16 [col][kc / 16 + 8] (the pad spreads the columns over the banks)
constexpr int kqs_bs_row(int kc) { return kc / 16 + 8; }
static size_t kqs_lds(int nt, int kc) { return (size_t)16 * nt * (kc + kc / 64 + 2 * kqs_bs_row(kc) + 16); }

// Grid x: about a workgroup a CU, dealt out over the plan's entries (up to 16 NT
// pairs of an expert each): the workers of an entry take its blocks of NW row
// groups in turn. The entries in use are known on the device only (experts
// above the average take two); dealt out here they all run at once, where a
// grid laid out for the average ran a second round (the whole call, 198 pairs on
// 8 experts, 11 entries: 134 -> 108 us). z: K chunks.
template <int WT, int NT>
__global__ void __launch_bounds__(64 * KQS_WAVES) k_gemm_kqs(const MatmulArgs a, int kc_elems) {
    kernarg_prefetch<(kernarg_lines(sizeof(MatmulArgs) + 4))>();
    constexpr int P = kq_planes<WT>(), SB = block_bytes(WT), BN = 16 * NT, NW = KQS_WAVES;
    static_assert(WT == TLH_TYPE_Q4_K || WT == TLH_TYPE_Q5_K, "types with eight mins");
    extern __shared__ __attribute__((aligned(16))) int8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, g = lane >> 4;
    int8_t *sX = lds;                                             // [BN][kc]
    float *sDx = (float *)(lds + BN * kc_elems);                  // [kc / 256][BN]
    int64_t *sOut = (int64_t *)(sDx + BN * (kc_elems / 256));     // [BN]
    int64_t *sRow = sOut + BN;                                    // [BN]
    _Float16 *sBs = (_Float16 *)(sRow + BN);                      // [BN][kc / 16 + 8]
    const int bs_row = kqs_bs_row(kc_elems);
    const int64_t K = a.K;
    const int nsb_all = (int)(K / QKK);
    const int kc = blockIdx.z, nkc = gridDim.z;
    const ActView act = act_view(a.act, TLH_TYPE_Q8_K, K, mm_act_rows(a));
    // this chunk's super-blocks
    const int sb_first = kc * (kc_elems / QKK);
    const int nsb = nsb_all - sb_first < kc_elems / QKK ? nsb_all - sb_first : kc_elems / QKK;
    const int entries = a.grp[0], wgs = gridDim.x;
    for (int tile = entries < wgs ? blockIdx.x % entries : blockIdx.x; tile < entries; tile += wgs) {
        const int worker = entries < wgs ? blockIdx.x / entries : 0;
        const int workers = entries < wgs ? (wgs - tile + entries - 1) / entries : 1;
        const int32_t *entry = a.grp + 4 + 4 * (int64_t)tile;
        const int expert = entry[0], n_cols = entry[2];
        const int32_t *pairs = a.grp + 4 + 4 * a.grp_tiles + entry[1];
        const uint8_t *W = a.w + (int64_t)(expert < 0 ? 0 : expert) * a.w_nb2;
        __syncthreads();  // (the last entry's codes are done with)
        {
            // the columns' activation rows (the last column again past the end) and
            // output offsets
            if (tid < BN) {
                const int cc = tid < n_cols ? tid : n_cols - 1;
                const uint32_t p = (uint32_t)pairs[cc], tok = p / (uint32_t)a.ne12, slot = p - tok * (uint32_t)a.ne12;
                sOut[tid] = nkc > 1 ? (int64_t)p * a.M * 4 : (int64_t)slot * a.d_nb2 + (int64_t)tok * a.d_nb3;
                sRow[tid] = (int64_t)(slot % (uint32_t)a.id_b1) + a.id_b1 * (int64_t)tok;
            }
            lds_barrier();
            // their codes (chunk c of a super-block's 16 at c ^ (column & 15)): wave w
            // fills columns w, w + waves, ..., 1 KB a load, eight loads in flight;
            // then bsums and scales
            constexpr int CPW = BN / NW;
            const int per_col = nsb * 16, nq = (per_col + 63) / 64, total = CPW * nq;  // 16-byte pieces; loads
            for (int first = 0; first < total; first += 8) {
                kq_u4 v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int q = first + i < total ? first + i : total - 1, col = wave + NW * (q / nq);
                    int c = q % nq * 64 + lane;
                    c = c < per_col ? c : per_col - 1;
                    v[i] = *(const kq_u4 *)(act.qs + sRow[col] * K + (int64_t)sb_first * QKK + 16 * c);
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int q = first + i, col = wave + NW * (q / nq), c = q % nq * 64 + lane;
                    if (q < total && c < per_col)
                        *(kq_u4 *)(sX + col * kc_elems + (((c & ~15) | ((c ^ col) & 15)) << 4)) = v[i];
                }
            }
            for (int k = 0; k < CPW; ++k) {
                const int col = wave + NW * k;
                for (int i = lane; i < nsb; i += 64) sDx[i * BN + col] = act.d[sRow[col] * nsb_all + sb_first + i];
                for (int i = lane; i < 2 * nsb; i += 64) {  // 8 bsums
                    const kq_u4 b = *(const kq_u4 *)(act.bsums + sRow[col] * (K / 16) + (int64_t)sb_first * 16 + 8 * i);
                    kq_v8h h;
#pragma unroll
                    for (int e = 0; e < 8; ++e) h[e] = (_Float16)(float)(int16_t)(b[e >> 1] >> (16 * (e & 1)));
                    *(kq_v8h *)(sBs + col * bs_row + 8 * i) = h;
                }
            }
        }
        __syncthreads();
        char *obase = nkc > 1 ? (char *)(a.part + kc * (a.ne12 * a.ne13) * a.M) : (char *)a.dst;
        const int64_t blocks = ((a.M + 15) / 16 + NW - 1) / NW;
        using H0 = std::integral_constant<int, 0>;
        using H1 = std::integral_constant<int, 1>;

        KqUnit<WT> r0, r1, q0, q1;  // halves of two super-blocks in flight
        const uint8_t *wrow = nullptr, *wnext = nullptr, *wnext2 = nullptr;  // this row group, the next two
        auto row_of = [&](int64_t block) {  // clamped: loads in bounds
            int64_t m = ((block < blocks ? block : blocks - 1) * NW + wave) * 16 + lr;
            m = m < a.M ? m : a.M - 1;
            return W + m * a.w_nb1 + (int64_t)sb_first * SB;
        };
        // super-block sb of this row group, run on into the next groups (their
        // rows by value: an address selected among variables puts them in memory)
        auto fetch = [&](auto hc, int sb, KqUnit<WT> &r, const uint8_t *w0, const uint8_t *w1, const uint8_t *w2) {
            constexpr int H = decltype(hc)::value;
            const uint8_t *p = w0;
            if (sb >= nsb) {
                sb -= nsb;
                p = w1;
                if (sb >= nsb) {
                    sb -= nsb;
                    p = w2;
                }
            }
            kq_fetch<WT, H>(p + (int64_t)sb * SB, g, r);
        };
        kq_v4i S[P][NT];
        // One column tile: acc moves to tot every few super-blocks (kq_unit.hpp; K = 8704 in one chunk, error against 64 bits: 1.16e-7 in one chain, 8.5e-8
        // now, a pair of its own 1.12e-7). Two have no registers for it and at most
        // 17 super-blocks a chunk (9.3e-8).
        constexpr bool FLUSH = NT == 1;
        const int every = kq_flush_every(nsb);
        int left = every;
        kq_v4f acc[NT], tot = {};
        auto multiply = [&](auto hc, int sb, const KqUnit<WT> &r) {
            constexpr int H = decltype(hc)::value;
            uint32_t o[2][2][4];
            kq_codes<WT, H>(r, g, o);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int c = 8 * H + kq_chunk<WT>(g) + s * kq_gap<WT>();
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const int col = 16 * j + lr;
                    const kq_v4i xv = *(const kq_v4i *)(sX + col * kc_elems + 256 * sb + ((c ^ (col & 15)) << 4));
#pragma unroll
                    for (int p = 0; p < P; ++p) {
                        const kq_v4i wv = {(int)o[p][s][0], (int)o[p][s][1], (int)o[p][s][2], (int)o[p][s][3]};
                        S[p][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xv, wv, S[p][j], 0, 0, 0);
                    }
                }
            }
        };
        // D[token][row]: lane holds weight row lr and tokens 4 g + e of a column tile
        auto finalize = [&](int sb, const KqUnit<WT> &r) {
            float d, dmin;
            uint32_t mn[4];
            kq_row_meta<WT>(r, d, dmin, mn);
            kq_v4h mv;  // the mins of bsums 4 g .. 4 g + 3
            const uint32_t m = __builtin_amdgcn_perm(0u, (g & 2 ? mn[1] : mn[0]) >> (16 * (g & 1)), 0x01010000u);
#pragma unroll
            for (int e = 0; e < 4; ++e) mv[e] = (_Float16)(float)((m >> (8 * e)) & 0xff);
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const kq_v4f Mn = __builtin_amdgcn_mfma_f32_16x16x16f16(
                    *(const kq_v4h *)(sBs + (16 * j + lr) * bs_row + 16 * sb + 4 * g), mv, (kq_v4f){}, 0, 0, 0);
                const float4 y4 = *(const float4 *)(sDx + sb * BN + 16 * j + 4 * g);
                const float dy[4] = {y4.x, y4.y, y4.z, y4.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float v = kq_sum<WT>(S[0][j][e], S[P - 1][j][e]) * d;
                    v -= dmin * Mn[e];
                    acc[j][e] += dy[e] * v;
                }
#pragma unroll
                for (int p = 0; p < P; ++p) S[p][j] = (kq_v4i){};
            }
        };

        if (worker < blocks) {
            wrow = row_of(worker);
            wnext = row_of(worker + workers);
            wnext2 = row_of(worker + 2 * (int64_t)workers);
            fetch(H0{}, 0, r0, wrow, wnext, wnext2);
            fetch(H1{}, 0, r1, wrow, wnext, wnext2);
            fetch(H0{}, 1, q0, wrow, wnext, wnext2);
            fetch(H1{}, 1, q1, wrow, wnext, wnext2);
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            acc[j] = (kq_v4f){};
#pragma unroll
            for (int p = 0; p < P; ++p) S[p][j] = (kq_v4i){};
        }
        // one super-block of row group (b, wave); the group's last one stores it and goes on to the next
        int64_t b = worker;
        int sb = 0;
        auto step = [&](KqUnit<WT> &u0, KqUnit<WT> &u1) {
            multiply(H0{}, sb, u0);
            fetch(H0{}, sb + 2, u0, wrow, wnext, wnext2);
            multiply(H1{}, sb, u1);
            finalize(sb, u1);
            fetch(H1{}, sb + 2, u1, wrow, wnext, wnext2);
            if (++sb < nsb) {
                if constexpr (FLUSH) {
                    if (--left == 0) {
                        tot += acc[0];
                        acc[0] = (kq_v4f){};
                        left = every;
                    }
                }
                return;
            }
            if constexpr (FLUSH) acc[0] += tot;
            const int64_t m = (b * NW + wave) * 16 + lr;
            if (m < a.M) {
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int c = 16 * j + 4 * g + e;
                        if (c < n_cols)  // (no such expert: NaN)
                            *(float *)(obase + sOut[c] + 4 * m) = expert < 0 ? __builtin_nanf("") : acc[j][e];
                    }
            }
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[j] = (kq_v4f){};
            if constexpr (FLUSH) tot = (kq_v4f){}, left = every;
            sb = 0;
            b += workers;
            wrow = wnext;
            wnext = wnext2;
            wnext2 = row_of(b + 2 * (int64_t)workers);
        };
        while (b < blocks) {
            step(r0, r1);
            if (b >= blocks) break;
            step(q0, q1);
        }
        if (entries < wgs) break;
    }
}

// Column tiles nt (16 each; two from 9 columns an expert on, since a second
// entry for the experts above the average reads their matrix again: 90 pairs on
// 8 experts of 14336 x 4096 117 us with one) and K chunks zc: of what fits LDS,
// and enough that the blocks of row groups of `tiles` entries reach every CU
// (8 experts of 3000 x 8192, 16 pairs: 64 us with one chunk).
KqsPlan gemm_kqs_plan(int64_t M, int64_t cols, int64_t K, int64_t tiles) {
    constexpr int64_t LDS = 160 * 1024;
    KqsPlan p{};
    p.nt = cols <= 8 ? 1 : 2;
    const int64_t nsb = K / 256, blocks = ((M + 15) / 16 + KQS_WAVES - 1) / KQS_WAVES * tiles;
    int64_t fill = (256 + blocks - 1) / blocks;
    if (fill > nsb / 4) fill = nsb / 4;
    for (p.zc = fill > 1 ? (int)fill : 1;; ++p.zc) {
        p.kc_elems = (int)((nsb + p.zc - 1) / p.zc * 256);
        if ((int64_t)kqs_lds(p.nt, p.kc_elems) <= LDS) break;
    }
    p.zc = (int)((nsb + p.kc_elems / 256 - 1) / (p.kc_elems / 256));  // no empty chunk
    p.lds = kqs_lds(p.nt, p.kc_elems);
    return p;
}

template <int WT> static tlh_status launch_kqs(const MatmulArgs &a, const KqsPlan &p, hipStream_t stream) {
    const int wgs = device_cus() / p.zc;
    const dim3 grid((unsigned)(wgs > 1 ? wgs : 1), 1u, (unsigned)p.zc), threads(64 * KQS_WAVES);
    if (p.nt == 1) hipLaunchKernelGGL((k_gemm_kqs<WT, 1>), grid, threads, p.lds, stream, a, p.kc_elems);
    else hipLaunchKernelGGL((k_gemm_kqs<WT, 2>), grid, threads, p.lds, stream, a, p.kc_elems);
    return check_launch("gemm_kqs");
}

tlh_status launch_gemm_kqs(const MatmulArgs &a, const KqsPlan &p, hipStream_t stream) {
    if (a.wtype == TLH_TYPE_Q4_K) return launch_kqs<TLH_TYPE_Q4_K>(a, p, stream);
    if (a.wtype == TLH_TYPE_Q5_K) return launch_kqs<TLH_TYPE_Q5_K>(a, p, stream);
    return set_error(TLH_UNSUPPORTED, "gemm_kqs: weight type %d", a.wtype);
}

}  // namespace tlh
