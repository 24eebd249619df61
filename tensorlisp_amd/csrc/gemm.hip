// Dispatch of GGML_OP_MUL_MAT with more than 16 activation columns: the tiled
// GEMMs (k-quants: gemm_kq.hip; q8_0 / q4_0: gemm_q8.hip), their split of K,
// and 16-column slabs of the few-column kernel for the other types.
#include "kernels.hpp"

namespace tlh {

int gemm_ksplit(int wtype, int64_t M, int64_t N, int64_t K, int64_t batches) {
    if (!has_gemm(wtype) || N <= 16) return 1;
    constexpr int64_t CUS = 256;  // MI355X
    int64_t ks;
    const int64_t units = (K + 255) / 256, min_units = 4;  // units of a chunk: 256 elements
    if (kquant_type(wtype)) {  // as many chunks as one round of workgroups holds
        const KqTile t = gemm_kq_tile(N);
        ks = CUS * t.per_cu / ((N + t.bn - 1) / t.bn * ((M + t.bm - 1) / t.bm) * batches);
    } else {  // two 128 x 128 tiles a CU
        const int64_t tiles = (N + 127) / 128 * ((M + 127) / 128) * batches;
        if (tiles >= CUS) return 1;
        ks = (2 * CUS + tiles - 1) / tiles;
    }
    if (ks > units / min_units) ks = units / min_units;
    if (ks > 16) ks = 16;
    return ks > 1 ? (int)ks : 1;
}

int64_t gemm_partial_bytes(int wtype, int64_t M, int64_t N, int64_t K, int64_t batches) {
    const int ks = gemm_ksplit(wtype, M, N, K, batches);
    return ks > 1 ? (int64_t)ks * batches * N * M * 4 : 0;
}

tlh_status launch_gemm_epi(const MatmulArgs &a, const GemvEpi &ep, hipStream_t stream) {
    if (!kquant_type(a.wtype) || !a.part)
        return set_error(TLH_UNSUPPORTED, "gemm: the store epilogue rides on the reduce of a k-quant GEMM");
    const int ks = gemm_ksplit(a.wtype, a.M, a.N, a.K, a.ne12 * a.ne13);
    tlh_status st = reduce_epi_check(a, ep);
    if (st != TLH_OK) return st;
    MatmulArgs g = a;
    g.keep_part = 1;  // one chunk's sums go through the reduce's stores too
    st = launch_gemm_kq(g, ks, stream);
    return st != TLH_OK ? st : launch_partial_reduce_epi(a, ks, ep, stream);
}

tlh_status launch_gemm(const MatmulArgs &a, hipStream_t stream) {
    const int64_t batches = a.ne12 * a.ne13;
    if (has_gemm(a.wtype)) {
        const int ks = gemm_ksplit(a.wtype, a.M, a.N, a.K, batches);
        if (ks > 1 && !a.part) return set_error(TLH_INVALID, "gemm: a K split of %d needs a partials buffer", ks);
        const tlh_status st = kquant_type(a.wtype) ? launch_gemm_kq(a, ks, stream) : launch_gemm_q8(a, ks, stream);
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

}  // namespace tlh
