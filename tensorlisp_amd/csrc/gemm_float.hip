// GGML_OP_MUL_MAT with f32, f16 or bf16 weights in 16-byte aligned rows of a
// multiple of 8 elements, on gfx950's matrix cores (mm_float.hip says what is
// computed, and takes every other layout). Products are exact in f32 and the
// sums are f32 (v_mfma_f32_16x16x32_f16 / _bf16, v_mfma_f32_16x16x4_f32);
// subnormal operands count, as on the CPU.
//
// A fragment is 16 bytes a lane: lane (r, g) = (lane & 15, lane >> 4) holds
// bytes 16 g .. 16 g + 15 of row r's 64-byte step, for W rows and X rows alike;
// an f32 step is four MFMAs over the lanes' elements 0 .. 3 (which k each takes
// is the same on both sides). Memory is read in whole 128-byte lines, 8 lanes a
// line, and turned into fragments through LDS: loads straight into the
// fragment layout touch 16 lines for every 16 lanes and ran at 14 bytes a clock
// and CU (f16 4096 x 4096, N = 77: 24 us against 16).
//
// Lane-wise fused multiply-adds on the vector ALUs, which these kernels
// replaced, took, in us (f32 src1): f16 4096 x 4096 N = 1 23.4 -> 7.2, N = 16
// 36.4 -> 7.6, N = 77 107 -> 16.7, N = 512 586 -> 49; f16 8192 x 8192 N = 512
// 2699 -> 124; bf16 1024 x 1024 N = 64 13.2 -> 7.4; f32 4096 x 4096 N = 77
// 141 -> 39, N = 1 22.1 -> 17.4; f32 512 x 128, N = 512, 32 slices 397 -> 45.
//
// Sums. An MFMA rounds several times on its way through K (once a k in f32, once
// every 8 in f16 / bf16), so a chain of them is as inexact as one of that many
// additions. Here a chain is one MFMA (f32, and f16 in the tiles: two), the chains
// of a 128-byte block are added to each other, and blocks by levels of a few (the
// kernels say how many: only as many as each type needs). Error against 64 bits,
// rms over rms, with 64 lanes' sums / chains of eight MFMAs / now: bf16 8192 x 256
// 5.5e-8 / 8.6e-8 / 5.5e-8, K = 4096 8.4e-8 / 1.15e-7 / 8.1e-8; f16 K = 256 7.6e-8
// / 1.05e-7 / 7.0e-8; f32 K = 4096 1.6e-7 / 2.3e-7 / 1.0e-7. In us, chains of eight
// and now: f16 4096 x 4096, N = 512 48 / 49, bf16 46 / 49; f32 N = 256 109 / 124.
#include "kernels.hpp"

namespace tlh {

typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));

// A fragment pair's product, f16 / bf16 on top of c; f32 by itself, in two chains of
// two MFMAs (in one of four K = 256 is at 9.2e-8 instead of 8.1e-8, in four 4096 x
// 4096, N = 256 takes 136 us instead of 124)
template <int TY> __device__ __forceinline__ f4 mma(u4 a, u4 b, f4 c = (f4)(0.0f)) {
    if constexpr (TY == TLH_TYPE_F16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c, 0, 0, 0);
    } else if constexpr (TY == TLH_TYPE_BF16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0, 0);
    } else {
        const f4 af = __builtin_bit_cast(f4, a), bf = __builtin_bit_cast(f4, b);
        f4 t[2];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            t[e >> 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[e], bf[e], e & 1 ? t[e >> 1] : (f4)(0.0f), 0, 0, 0);
        return t[0] + t[1];
    }
}

// a tile's 128-byte block: f16 in one chain (two MFMAs)
template <int TY> __device__ __forceinline__ f4 mma2(u4 a0, u4 b0, u4 a1, u4 b1) {
    if constexpr (TY == TLH_TYPE_F16) return mma<TY>(a1, b1, mma<TY>(a0, b0));
    else return mma<TY>(a0, b0) + mma<TY>(a1, b1);
}

// eight f32 values of src1 -> the weight type, to nearest even (the CPU's conversion)
template <int TY> __device__ __forceinline__ u4 round8(u4 a, u4 b) {
    u4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float lo = __uint_as_float(i < 2 ? a[2 * i] : b[2 * i - 4]);
        const float hi = __uint_as_float(i < 2 ? a[2 * i + 1] : b[2 * i - 3]);
        if constexpr (TY == TLH_TYPE_F16) {
            o[i] = f2h(lo) | (uint32_t)f2h(hi) << 16;
        } else {
            const f2 t = {lo, hi};
            o[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(t, b2));  // v_cvt_pk_bf16_f32
        }
    }
    return o;
}

// Workgroup id -> (row tile, column tile): ids go round the 8 XCDs, so the
// column tiles of one row tile take ids 8 apart and share that XCD's L2 copy
// of the weight rows.
__device__ __forceinline__ void tile_of(int id, int mt, int nt, int &tm, int &tn) {
    const int full = mt / 8 * 8 * nt;
    if (id < full) {
        const int j = id / 8;
        tm = (j / nt) * 8 + (id & 7), tn = j % nt;
    } else {
        const int rest = mt & 7, j = id - full;
        tm = mt - rest + j % rest, tn = j / rest;
    }
}

struct MmfView {
    const char *w, *x;
    char *d;
};
__device__ __forceinline__ MmfView batch_view(const FloatMM &f) {
    MmfView v{f.w, f.x, (char *)f.d};
    if (blockIdx.y != 0) {
        const int64_t i12 = blockIdx.y % f.ne12, i13 = blockIdx.y / f.ne12;
        v.w += (i12 / f.r2) * f.w_nb2 + (i13 / f.r3) * f.w_nb3;
        v.x += i12 * f.x_nb2 + i13 * f.x_nb3;
        v.d += i12 * f.d_nb2 + i13 * f.d_nb3;
    }
    return v;
}

// Few tiles: 16 MR rows x 16 NT columns a workgroup, K dealt over its KW waves in
// 128-byte blocks (wave w: blocks w, w + KW, ...), so that the chip is full from
// 256 x 16 MR rows on whatever N is. The waves share no operand: each turns its
// blocks into fragments in LDS of its own, without a barrier, adds its blocks'
// sums by fours (f16, whose products are the longest, all in one chain: K = 4096
// 1.0e-7 and 16.4 us at 4096 x 4096, N = 77, by fours 8.6e-8 and 17.0; 64 lanes
// 1.5e-7), and the waves' sums meet in a tree at the end. XF: f32 src1
// rounded to the weight type as it arrives. Bound by what a CU takes in: f16 4096
// x 4096, N = 77: 131 KB of W rows and 786 KB of f32 X rows each in about 13 us;
// 8192 x 8192, N = 1: 5.0 TB/s of weights.
constexpr int KW = 8;
template <int TY, int MR, int NT, int D, bool XF>
__global__ void __launch_bounds__(64 * KW) k_mmf_split(const FloatMM f, int mt, int nt) {
    constexpr bool LEVELS = TY != TLH_TYPE_F16;
    constexpr int R = 16 * (MR + NT), LD = R / 8;  // rows of a block, rows a lane loads
    constexpr int LQ = LD + (XF ? 2 * NT : 0);   // 16-byte loads (f32 src1: two a row)
    extern __shared__ __align__(16) char lds[];  // [KW] blocks, then part[KW][16 NT][16 MR]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int c = lane & 7, lr = lane >> 3;
    const MmfView v = batch_view(f);
    int tm, tn;
    tile_of(blockIdx.x, mt, nt, tm, tn);
    const int64_t m0 = (int64_t)tm * 16 * MR, n0 = (int64_t)tn * 16 * NT;
    const char *src[LD];
#pragma unroll
    for (int i = 0; i < LD; ++i) {  // rows past M or N: clamped, their outputs are not stored
        const bool isw = i < 2 * MR;
        const int64_t at = isw ? m0 + 8 * i + lr : n0 + 8 * (i - 2 * MR) + lr, end = isw ? f.M : f.N;
        src[i] = (isw ? v.w : v.x) + (at < end ? at : end - 1) * (isw ? f.w_nb1 : f.x_nb1);
    }
    const int64_t kb = f.K * (TY == TLH_TYPE_F32 ? 4 : 2);
    f4 acc[MR][NT], sum[MR][NT];
#pragma unroll
    for (int i = 0; i < MR; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = sum[i][j] = (f4)(0.0f);
    u4 q[D][LQ];
    // (always the same loads, so that the waits count them: past K the row's last 16 bytes)
    auto fetch = [&](u4 (&q)[LQ], int64_t off) {
        const int64_t at = off + 16 * c < kb ? off + 16 * c : kb - 16;
#pragma unroll
        for (int k = 0; k < LD; ++k) {
            if (XF && k >= 2 * MR) {
                q[k] = *(const u4 *)(src[k] + 2 * at);
                q[k + 2 * NT] = *(const u4 *)(src[k] + 2 * at + 16);
            } else {
                q[k] = *(const u4 *)(src[k] + at);
            }
        }
    };
    int chain = 0;
    char *L = lds + wave * (R * 128);
    char *st = L + lr * 128 + ((c ^ lr) * 16);
    auto mul = [&](u4 (&q)[LQ], int64_t off) {
        if constexpr (XF) {
#pragma unroll
            for (int k = 2 * MR; k < LD; ++k) q[k] = round8<TY>(q[k], q[k + 2 * NT]);
        }
        if (off + 128 > kb && off + 16 * c >= kb) {
#pragma unroll
            for (int k = 0; k < LD; ++k) q[k] = (u4)(0u);
        }
#pragma unroll
        for (int k = 0; k < LD; ++k) *(u4 *)(st + k * 1024) = q[k];
        __builtin_amdgcn_wave_barrier();
        f4 t[MR][NT];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            u4 a[MR + NT];
#pragma unroll
            for (int k = 0; k < MR + NT; ++k) a[k] = *(const u4 *)(L + r * 128 + ((4 * s + g) ^ (r & 7)) * 16 + k * 2048);
#pragma unroll
            for (int i = 0; i < MR; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const f4 p = mma<TY>(a[i], a[MR + j]);
                    if (!LEVELS) acc[i][j] += p;
                    else if (s == 0) t[i][j] = p;
                    else acc[i][j] += t[i][j] + p;
                }
        }
        __builtin_amdgcn_wave_barrier();
        if (LEVELS && (++chain & 3) == 0) {
#pragma unroll
            for (int i = 0; i < MR; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) sum[i][j] += acc[i][j], acc[i][j] = (f4)(0.0f);
        }
    };
    constexpr int64_t STEP = 128 * KW;
    int64_t off = 128 * wave;
#pragma unroll
    for (int d = 0; d < D; ++d) fetch(q[d], off + d * STEP);
    for (bool more = off < kb; more;) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            mul(q[d], off);
            fetch(q[d], off + D * STEP);
            off += STEP;
            if (off >= kb) {
                more = false;
                break;
            }
        }
    }
    __syncthreads();
    constexpr int PART = 256 * MR * NT;
    float *part = (float *)lds;
    // part[wave][n][16 MR m]: a lane's four sums are rows 4 g .. 4 g + 3 of column r
    float *mine = part + wave * (PART);
#pragma unroll
    for (int i = 0; i < MR; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) *(f4 *)(mine + (16 * j + r) * (16 * MR) + 16 * i + 4 * g) = sum[i][j] + acc[i][j];
    __syncthreads();
    for (int o = threadIdx.x; o < PART; o += 64 * KW) {
        float t[KW];
#pragma unroll
        for (int w = 0; w < KW; ++w) t[w] = part[w * (PART) + o];
#pragma unroll
        for (int h = KW / 2; h > 0; h /= 2)
#pragma unroll
            for (int w = 0; w < h; ++w) t[w] += t[w + h];
        const int64_t m = m0 + o % (16 * MR), n = n0 + o / (16 * MR);
        if (m < f.M && n < f.N) *(float *)(v.d + n * f.d_nb1 + m * 4) = t[0];
    }
}

// Many tiles: B x B outputs a workgroup of WM x WN waves, both operands staged
// through two LDS buffers of 128 bytes a row, 16-byte chunk c of row r at c ^ (r &
// 7) (reads of 8 rows touch all banks once). D blocks' loads fly while one is
// multiplied (64 x 64 tiles, f16 4096 x 4096, N = 200: D = 1 / 2 / 3 / 4 48 / 40 /
// 35 / 33 us). XF: f32 src1 rounded on its way to LDS. The blocks' sums go up LV
// levels, each the sum of RAD of the one below and the last of all the rest: f16 two
// of eights; bf16 three of fours, and to K = 1024 five of twos, since its products
// are so short that 64 lanes' first sums were exact (K = 1000: 7.0e-8 by fours,
// 6.7e-8 by twos, 6.8e-8 the lanes); f32 by twos. 128 x 128 tiles have eight waves,
// since four would hold levels of 64 results each (f16 8192 x 8192, N = 512: 390
// against 124 us, without levels 109 on converted rows). 8192 x 8192, N = 512: 555
// TFLOP/s, bound by LDS reads and by one round of tiles on the chip.
template <int TY, int B, int WM, int WN, int RAD, int LV, int D, bool XF>
__global__ void __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(2))) k_mmf_tile(const FloatMM f, int mt, int nt) {
    constexpr int FM = B / WM / 16, FN = B / WN / 16;  // fragments of a wave
    constexpr int RP = 8 * WM * WN, LB = B / RP, LD = 2 * LB;  // rows a load of all threads; rows a thread and block
    constexpr int LQ = LD + (XF ? LB : 0);  // 16-byte loads (f32 src1: two a row)
    __shared__ __align__(16) char lds[2][2 * B * 128];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const MmfView v = batch_view(f);
    int tm, tn;
    tile_of(blockIdx.x, mt, nt, tm, tn);
    const int64_t m0 = (int64_t)tm * B, n0 = (int64_t)tn * B;
    const int64_t kb = f.K * (TY == TLH_TYPE_F32 ? 4 : 2);
    const int c = threadIdx.x & 7, lr = threadIdx.x >> 3;  // chunk, row (of RP) this thread loads
    const char *src[LD];
#pragma unroll
    for (int i = 0; i < LD; ++i) {
        const int64_t t = lr + RP * (i % LB);
        const bool isw = i < LB;
        const int64_t at = (isw ? m0 : n0) + t, end = isw ? f.M : f.N;
        src[i] = (isw ? v.w : v.x) + (at < end ? at : end - 1) * (isw ? f.w_nb1 : f.x_nb1);
    }
    u4 q[D][LQ];
    auto fetch = [&](u4 (&q)[LQ], int64_t off) {
        const int64_t at = off + 16 * c < kb ? off + 16 * c : kb - 16;
#pragma unroll
        for (int i = 0; i < LD; ++i) {
            if (XF && i >= LB) {
                q[i] = *(const u4 *)(src[i] + 2 * at);
                q[i + LB] = *(const u4 *)(src[i] + 2 * at + 16);
            } else {
                q[i] = *(const u4 *)(src[i] + at);
            }
        }
    };
    const int st = lr * 128 + ((c ^ (lr & 7)) * 16);
    const int wm = wave % WM * (B / WM), wn = wave / WM * (B / WN);
    const int ra = (wm + r) * 128, rb = (B + wn + r) * 128;
    f4 lev[LV][FM][FN];
#pragma unroll
    for (int l = 0; l < LV; ++l)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) lev[l][i][j] = (f4)(0.0f);
    int buf = 0, chain = 0;
    auto block = [&](u4 (&q)[LQ], int64_t off) {
        char *L = lds[buf];
        buf ^= 1;
        if constexpr (XF) {
#pragma unroll
            for (int i = LB; i < LD; ++i) q[i] = round8<TY>(q[i], q[i + LB]);
        }
        if (off + 128 > kb && off + 16 * c >= kb) {
#pragma unroll
            for (int i = 0; i < LD; ++i) q[i] = (u4)(0u);
        }
#pragma unroll
        for (int i = 0; i < LD; ++i) *(u4 *)(L + st + i * (RP * 128)) = q[i];
        __syncthreads();
        fetch(q, off + 128 * D);
        const int s0 = (g ^ (r & 7)) * 16, s1 = ((4 + g) ^ (r & 7)) * 16;
        u4 a[2][FM], b[2][FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) a[0][i] = *(const u4 *)(L + ra + s0 + i * 2048), a[1][i] = *(const u4 *)(L + ra + s1 + i * 2048);
#pragma unroll
        for (int i = 0; i < FN; ++i) b[0][i] = *(const u4 *)(L + rb + s0 + i * 2048), b[1][i] = *(const u4 *)(L + rb + s1 + i * 2048);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) lev[0][i][j] += mma2<TY>(a[0][i], b[0][j], a[1][i], b[1][j]);
        ++chain;
        int n = RAD;
#pragma unroll
        for (int l = 0; l + 1 < LV; ++l, n *= RAD) {
            if (chain & (n - 1)) break;
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) lev[l + 1][i][j] += lev[l][i][j], lev[l][i][j] = (f4)(0.0f);
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) fetch(q[d], 128 * d);
    int64_t off = 0;
    for (bool more = true; more;) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            block(q[d], off);
            off += 128;
            if (off >= kb) {
                more = false;
                break;
            }
        }
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int64_t n = n0 + wn + 16 * j + r;
        if (n >= f.N) continue;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int64_t m = m0 + wm + 16 * i + 4 * g;
            f4 t = lev[0][i][j];
#pragma unroll
            for (int l = 1; l < LV; ++l) t = lev[l][i][j] + t;
            float *d = (float *)(v.d + n * f.d_nb1) + m;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (m + e < f.M) d[e] = t[e];
        }
    }
}

static int64_t tiles(int64_t n, int64_t b) { return (n + b - 1) / b; }
static int64_t tiles2(const FloatMM &f, int64_t bm, int64_t bn) { return tiles(f.M, bm) * tiles(f.N, bn) * f.ne12 * f.ne13; }

bool gemm_float_aligned(const FloatMM &f) {
    auto al = [](const void *p, int64_t a, int64_t b, int64_t c) {
        return (((uintptr_t)p | (uintptr_t)a | (uintptr_t)b | (uintptr_t)c) & 15) == 0;
    };
    return f.K > 0 && f.K % 8 == 0 && al(f.w, f.w_nb1, f.w_nb2, f.w_nb3) && al(f.x, f.x_nb1, f.x_nb2, f.x_nb3);
}

// The tile kernels, from one 64 x 64 tile a CU on (f16 4096 x 4096: N = 200
// 256 tiles, 35 us against 35 of the split, N = 256 34 against 38, N = 512 49
// against 77; 8192 x 4096 N = 64 128 tiles, 31 against 23). Up to 16 columns two a
// CU (32768 x 4096: 46 against 56); f32, which would multiply 64 columns at an
// eighth of the rate, above 32 columns only (4096 x 4096, N = 32: 106 against 23).
static bool gemm_float_tiled(const FloatMM &f) {
    const int64_t t = tiles2(f, 64, 64);
    return f.wtype == TLH_TYPE_F32 ? f.N > 32 && t >= 256 : t >= (f.N > 16 ? 256 : 512);
}

template <int TY, int MR, int NT, int D> static void launch_split(const FloatMM &f, hipStream_t s) {
    const int mt = (int)tiles(f.M, 16 * MR), nt = (int)tiles(f.N, 16 * NT);
    const dim3 grid((unsigned)(mt * nt), (unsigned)(f.ne12 * f.ne13));
    constexpr int bytes = KW * 16 * (MR + NT) * 128;
    if constexpr (TY != TLH_TYPE_F32) {
        if (f.xtype != TY) {
            hipLaunchKernelGGL((k_mmf_split<TY, MR, NT, D, true>), grid, dim3(64 * KW), bytes, s, f, mt, nt);
            return;
        }
    }
    hipLaunchKernelGGL((k_mmf_split<TY, MR, NT, D, false>), grid, dim3(64 * KW), bytes, s, f, mt, nt);
}

template <int TY, int B, int WM, int WN, int RAD, int LV, int D, int DX> static void launch_tile(const FloatMM &f, hipStream_t s) {
    const int mt = (int)tiles(f.M, B), nt = (int)tiles(f.N, B);
    const dim3 grid((unsigned)(mt * nt), (unsigned)(f.ne12 * f.ne13));
    if constexpr (TY != TLH_TYPE_F32) {
        if (f.xtype != TY) {
            hipLaunchKernelGGL((k_mmf_tile<TY, B, WM, WN, RAD, LV, DX, true>), grid, dim3(64 * WM * WN), 0, s, f, mt, nt);
            return;
        }
    }
    hipLaunchKernelGGL((k_mmf_tile<TY, B, WM, WN, RAD, LV, D, false>), grid, dim3(64 * WM * WN), 0, s, f, mt, nt);
}

template <int TY> static void launch_ty(const FloatMM &f, hipStream_t s) {
    if (gemm_float_tiled(f)) {
        // 128 x 128 tiles once there is one a CU (f16 8192 x 4096, N = 512: 67 us, with
        // 64 x 64 tiles 82; 4096 x 4096, N = 512, half as many: 65 against 44); f32 is
        // bound by its MFMAs (8192 x 4096, N = 512: 320 against 292), and five levels
        // have no registers there
        const bool wide = tiles2(f, 128, 128) >= 256;
        if constexpr (TY == TLH_TYPE_F16) {
            if (wide) launch_tile<TY, 128, 4, 2, 8, 2, 3, 2>(f, s);
            else launch_tile<TY, 64, 2, 2, 8, 2, 4, 4>(f, s);
        } else if constexpr (TY == TLH_TYPE_BF16) {
            // (by fours 8192 x 2048, N = 512 takes 42 us and 56 by twos)
            if (f.K <= 1024) launch_tile<TY, 64, 2, 2, 2, 5, 4, 4>(f, s);
            else if (wide) launch_tile<TY, 128, 4, 2, 4, 3, 3, 2>(f, s);
            else launch_tile<TY, 64, 2, 2, 4, 3, 4, 4>(f, s);
        } else {
            launch_tile<TY, 64, 2, 2, 2, 5, 4, 4>(f, s);
        }
        return;
    }
    // Columns a workgroup: a CU's time goes with the rows it reads (32 of W,
    // 16 NT of X, those twice as long in f32) times the workgroups it runs; the
    // least of it, and of equals the widest (f16 4096 x 4096 with f32 src1: N = 32
    // 10.2 / 11.7 / 13.8 us for NT = 1 / 2 / 3, N = 77 21.7 / 20.0 / 16.3)
    const int xs = f.xtype != f.wtype ? 2 : 1;
    int best = 1;
    int64_t least = INT64_MAX;
    for (int nt = 1; nt <= 3; ++nt) {
        const int64_t cost = (32 + 16 * nt * xs) * tiles(tiles2(f, 32, 16 * nt), 256);
        if (cost <= least) least = cost, best = nt;
    }
    if (f.N <= 16 || best == 1) {
        // 16 rows a workgroup while 32 would leave half of the CUs without one: f32 777
        // x 4096, N = 1 16.2 -> 11.8 us (25 -> 49 workgroups; the lane-wise kernel, 49 of
        // 4 waves, 14.0), f16 4096 x 4096, N = 16 9.4 -> 7.6 (128 -> 256)
        if (tiles2(f, 32, 16) <= 128) launch_split<TY, 1, 1, 2>(f, s);
        else launch_split<TY, 2, 1, 2>(f, s);
    } else if (best == 2) {
        launch_split<TY, 2, 2, 1>(f, s);
    } else {
        launch_split<TY, 2, 3, 1>(f, s);
    }
}

tlh_status launch_gemm_float(const FloatMM &f, hipStream_t stream) {
    if (f.wtype == TLH_TYPE_F16) launch_ty<TLH_TYPE_F16>(f, stream);
    else if (f.wtype == TLH_TYPE_BF16) launch_ty<TLH_TYPE_BF16>(f, stream);
    else launch_ty<TLH_TYPE_F32>(f, stream);
    return check_launch("mul_mat_float");
}

}  // namespace tlh
