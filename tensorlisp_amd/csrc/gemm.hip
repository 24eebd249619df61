// Dispatch of GGML_OP_MUL_MAT with more than 16 activation columns: the tiled
// GEMMs (k-quants: gemm_kq.hip; q8_0 / q4_0: gemm_q8.hip), their split of K,
// and 16-column slabs of the few-column kernel for the other types.
#include "kernels.hpp"

namespace tlh {

int k_chunks(int64_t parts, int64_t ks) {
    if (ks < 2) return 1;
    const int64_t share = (parts + ks - 1) / ks;  // (the kernels' own)
    return (int)((parts + share - 1) / share);
}
// at least four units of 256 elements a chunk
static int ksplit_of(int64_t ks, int64_t K) {
    const int64_t units = (K + 255) / 256, min_units = 4;
    if (ks > units / min_units) ks = units / min_units;
    if (ks > 16) ks = 16;
    return ks > 1 ? (int)ks : 1;
}

// The chunks that the scratch sizes told to callers (and so what
// tlh_mul_mat_noalloc refuses) have always counted, of tiles of 128 rows:
// q8_0 / q4_0, and q4_K / q5_K up to 128 columns, two 128-column tiles a CU;
// q4_K / q5_K above, one 256-column tile.
static int ksplit_told(int wtype, int64_t M, int64_t N, int64_t K, int64_t batches) {
    constexpr int64_t CUS = 256;  // MI355X
    const bool wide = kquant_type(wtype) && N > 128;
    const int64_t bn = wide ? 256 : 128, tiles = (N + bn - 1) / bn * ((M + 127) / 128) * batches;
    if (tiles == 0 || tiles >= CUS) return 1;
    return ksplit_of(wide ? CUS / tiles : (2 * CUS + tiles - 1) / tiles, K);
}
static bool told_type(int wtype) { return wtype != TLH_TYPE_Q2_K && wtype != TLH_TYPE_Q3_K && wtype != TLH_TYPE_Q6_K; }

int gemm_ksplit(int wtype, int64_t M, int64_t N, int64_t K, int64_t batches) {
    if (!has_gemm(wtype) || N <= 16 || M == 0 || batches == 0) return 1;
    constexpr int64_t CUS = 256;
    const bool kq = kquant_type(wtype);
    const int64_t parts = kq ? K / 256 : (K + 127) / 128;  // super-blocks, or stages of four blocks
    int64_t ks = 16;
    if (kq || N <= 64) {  // as many chunks as one round of workgroups holds
        const KqTile t = kq ? gemm_kq_tile(N) : gemm_q8_tile(N);
        ks = ksplit_of(CUS * t.per_cu / ((N + t.bn - 1) / t.bn * ((M + t.bm - 1) / t.bm) * batches), K);
    }
    int64_t most;  // what gemm_partial_bytes has room for
    if (told_type(wtype)) {
        most = ksplit_told(wtype, M, N, K, batches);
    } else {
        // their chunks came with the tiled GEMM: no node that fitted the static
        // scratch of tlh_mul_mat_noalloc may outgrow it by them (q6_K 512 x 14336,
        // N = 3584: 55 MB of activations, 7 MB a chunk)
        const int64_t room = (int64_t)TLH_NOALLOC_SCRATCH_BYTES - act_layout(TLH_TYPE_Q8_K, K, N * batches).total;
        most = room < 0 ? ks : (room & ~(int64_t)255) / (batches * N * M * 4);
    }
    return k_chunks(parts, ks < most ? ks : most);
}

int gemm_ksplit_grouped(int64_t M, int64_t K, int64_t pairs, int64_t n_as) {
    const int64_t per = (pairs + n_as - 1) / n_as, used = pairs < n_as ? pairs : n_as;  // evenly chosen experts
    const KqTile t = gemm_kq_tile(per);
    const int64_t tiles = used * ((per + t.bn - 1) / t.bn) * ((M + t.bm - 1) / t.bm);
    return k_chunks(K / 256, ksplit_of(256 * t.per_cu / tiles, K));
}

int64_t gemm_partial_bytes(int wtype, int64_t M, int64_t N, int64_t K, int64_t batches) {
    if (!has_gemm(wtype) || N <= 16) return 0;
    const int64_t ks = told_type(wtype) ? ksplit_told(wtype, M, N, K, batches) : gemm_ksplit(wtype, M, N, K, batches);
    const int64_t bytes = ks > 1 ? ks * batches * N * M * 4 : 0;
    // q2_K / q3_K / q6_K: at least what their 16-column slabs took
    const int64_t slab = told_type(wtype) ? 0 : gemv_mfma_partial_bytes(K, M, N, batches);
    return bytes > slab ? bytes : slab;
}

// q4_K / q5_K activations of 2^31 codes and more: refused, as they have always been
static tlh_status check_gemm_size(const MatmulArgs &a) {
    const int64_t batches = a.ne12 * a.ne13;
    if (kquant_type(a.wtype) && told_type(a.wtype) && (double)a.N_total * (double)batches * (double)a.K >= 2147483648.0)
        return set_error(TLH_UNSUPPORTED, "gemm: %lld x %lld x %lld activation codes, 2^31 or more",
                         (long long)a.N_total, (long long)batches, (long long)a.K);
    return TLH_OK;
}

tlh_status launch_gemm_epi(const MatmulArgs &a, const GemvEpi &ep, hipStream_t stream) {
    if (!kquant_type(a.wtype) || !a.part)
        return set_error(TLH_UNSUPPORTED, "gemm: the store epilogue rides on the reduce of a k-quant GEMM");
    const int ks = gemm_ksplit(a.wtype, a.M, a.N, a.K, a.ne12 * a.ne13);
    tlh_status st = check_gemm_size(a);
    if (st == TLH_OK) st = reduce_epi_check(a, ep);
    if (st != TLH_OK) return st;
    MatmulArgs g = a;
    g.keep_part = 1;  // one chunk's sums go through the reduce's stores too
    st = launch_gemm_kq(g, gemm_kq_tile(a.N).bn, ks, stream);
    return st != TLH_OK ? st : launch_partial_reduce_epi(a, ks, ep, stream);
}

tlh_status launch_gemm(const MatmulArgs &a, hipStream_t stream) {
    const int64_t batches = a.ne12 * a.ne13;
    if (has_gemm(a.wtype)) {
        const int ks = gemm_ksplit(a.wtype, a.M, a.N, a.K, batches);
        if (ks > 1 && !a.part) return set_error(TLH_INVALID, "gemm: a K split of %d needs a partials buffer", ks);
        tlh_status st = check_gemm_size(a);
        if (st == TLH_OK) st = kquant_type(a.wtype) ? launch_gemm_kq(a, gemm_kq_tile(a.N).bn, ks, stream) : launch_gemm_q8(a, ks, stream);
        return st != TLH_OK || ks == 1 || a.keep_part ? st : launch_partial_reduce(a, ks, stream);
    }
    if (a.keep_part) return set_error(TLH_UNSUPPORTED, "gemm: no kept partials for weight type %d", a.wtype);
    for (int64_t c = 0; c < a.N; c += 16) {
        MatmulArgs s = a;
        s.n0 = a.n0 + c;
        s.N = a.N - c < 16 ? a.N - c : 16;
        const tlh_status st = launch_gemv_mfma(s, stream);
        if (st != TLH_OK) return st;
    }
    return TLH_OK;
}

// MUL_MAT_ID's (expert, token) pairs by expert: one workgroup counts the pairs
// of each expert, gives every expert its run of the pair list and its column
// tiles (bn pairs each), and deals the pairs out. The order of an expert's
// pairs is not fixed; each pair's outputs depend on its own column only.
constexpr int GP_THREADS = 1024;
__global__ void __launch_bounds__(GP_THREADS) k_group_plan(const MatmulArgs a, int bn, int32_t *plan) {
    __shared__ int cnt[GROUP_MAX_EXPERTS + 1], first[GROUP_MAX_EXPERTS + 1];
    __shared__ int wave_pairs[16], wave_tiles[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n_as = (int)a.id_nas, used = (int)a.ne12, pairs = used * (int)a.ne13;
    auto expert = [&](int p) {
        const int t = p / used, e = *(const int32_t *)(a.ids + (int64_t)(p - t * used) * a.ids_nb0 + (int64_t)t * a.ids_nb1);
        return (unsigned)e < (unsigned)n_as ? e : n_as;
    };
    for (int i = tid; i <= n_as; i += GP_THREADS) cnt[i] = 0;
    __syncthreads();
    for (int p = tid; p < pairs; p += GP_THREADS) atomicAdd(&cnt[expert(p)], 1);
    __syncthreads();
    int32_t *tile = plan + 4, *list = tile + 4 * a.grp_tiles;
    int done_pairs = 0, done_tiles = 0;
    for (int e0 = 0; e0 <= n_as; e0 += GP_THREADS) {  // exclusive sums of pairs and tiles over the experts
        const int e = e0 + tid, c = e <= n_as ? cnt[e] : 0, nt = (c + bn - 1) / bn;
        int sp = c, st = nt;
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
            const int up = __shfl_up(sp, m, 64), ut = __shfl_up(st, m, 64);
            if (lane >= m) sp += up, st += ut;
        }
        if (lane == 63) wave_pairs[wave] = sp, wave_tiles[wave] = st;
        __syncthreads();
        int bp = done_pairs, bt = done_tiles;
        for (int w = 0; w < 16; ++w) {
            if (w < wave) bp += wave_pairs[w], bt += wave_tiles[w];
            done_pairs += wave_pairs[w], done_tiles += wave_tiles[w];
        }
        if (e <= n_as) {
            first[e] = bp + sp - c;
            for (int i = 0; i < nt; ++i) {
                const int left = c - i * bn;
                int32_t *t = tile + 4 * (int64_t)(bt + st - nt + i);
                t[0] = e < n_as ? e : -1;
                t[1] = bp + sp - c + i * bn;
                t[2] = left < bn ? left : bn;
                t[3] = 0;
            }
        }
        __syncthreads();
    }
    if (tid == 0) plan[0] = done_tiles;
    for (int p = tid; p < pairs; p += GP_THREADS) list[atomicAdd(&first[expert(p)], 1)] = p;
}

tlh_status launch_group_plan(const MatmulArgs &a, int64_t bn, int32_t *plan, hipStream_t stream) {
    hipLaunchKernelGGL(k_group_plan, dim3(1), dim3(GP_THREADS), 0, stream, a, (int)bn, plan);
    return check_launch("group_plan");
}

}  // namespace tlh
