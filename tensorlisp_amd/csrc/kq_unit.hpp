// K-quant weights as int8 planes of scaled codes, shared by the GEMM
// (gemm_kq.hip) and the streaming form for few columns (gemm_kqs.hip): the
// types' planes, a lane's unit of 32 elements (its loads and its codes), and a
// row's d, dmin and mins.
//   q2_K  sc * q <= 45: one plane
//   q3_K  -(sc * (q - 4)) in -128..124: one plane (negated, so that it fits)
//   q4_K  sc = 8 sh + sl: planes sh * q and sl * q (<= 105), S = 8 H + L;
//         a plane of four nibbles is one packed 16-bit multiply (no byte carries)
//   q5_K, q6_K  sc * q (13 bits): high and (signed) low byte, S = 256 H + L
#pragma once

#include <type_traits>

#include "kernels.hpp"

namespace tlh {

typedef int kq_v4i __attribute__((ext_vector_type(4)));
typedef int kq_v16i __attribute__((ext_vector_type(16)));
typedef float kq_v16f __attribute__((ext_vector_type(16)));
typedef _Float16 kq_v8h __attribute__((ext_vector_type(8)));
typedef float kq_v4f __attribute__((ext_vector_type(4)));
typedef _Float16 kq_v4h __attribute__((ext_vector_type(4)));
typedef uint32_t kq_u4 __attribute__((ext_vector_type(4)));  // (plain vectors: a struct of them stays in registers)
typedef uint32_t kq_u2 __attribute__((ext_vector_type(2)));
typedef unsigned short kq_u16x2 __attribute__((ext_vector_type(2)));

template <int WT> constexpr int kq_planes() { return WT == TLH_TYPE_Q2_K || WT == TLH_TYPE_Q3_K ? 1 : 2; }
template <int WT> constexpr bool kq_has_min() { return WT == TLH_TYPE_Q2_K || WT == TLH_TYPE_Q4_K || WT == TLH_TYPE_Q5_K; }

// A unit is 32 elements of a weight row's half super-block (128 elements): two
// groups of 16 with one scale each. Unit u of half h reads 16 code bytes (and
// 16 bytes of high bits) and fills 16-byte chunks G0 and G1 of the row's LDS
// row of 128 codes.
template <int WT> struct KqUnit {
    kq_u4 q;
    kq_u4 hi;       // q3_K hmask, q5_K qh, q6_K qh
    uint32_t s[5];  // header words: scales, d / dmin
};

__device__ __forceinline__ kq_u4 kq_ld16(const void *p) {
    kq_u4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}
template <typename T> __device__ __forceinline__ T kq_ld(const void *p) {
    T v;
    __builtin_memcpy(&v, p, sizeof v);
    return v;
}

template <int WT, int HALF> __device__ __forceinline__ void kq_fetch(const uint8_t *blk, int u, KqUnit<WT> &r) {
    if constexpr (WT == TLH_TYPE_Q4_K || WT == TLH_TYPE_Q5_K) {
        const kq_u4 h = kq_ld16(blk);
        r.s[0] = h.x, r.s[1] = h.y, r.s[2] = h.z, r.s[3] = h.w;
        r.q = kq_ld16(blk + (WT == TLH_TYPE_Q5_K ? 48 : 16) + 64 * HALF + 16 * u);
        if constexpr (WT == TLH_TYPE_Q5_K) r.hi = kq_ld16(blk + 16 + 16 * (u & 1));
    } else if constexpr (WT == TLH_TYPE_Q6_K) {
        r.q = kq_ld16(blk + 64 * HALF + 16 * u);
        r.hi = kq_ld16(blk + 128 + 32 * HALF + 16 * (u & 1));
        const kq_u2 s = kq_ld<kq_u2>(blk + 192 + 8 * HALF);
        r.s[0] = s.x, r.s[1] = s.y;
        if constexpr (HALF == 1) r.s[2] = kq_ld<uint16_t>(blk + 208);
    } else if constexpr (WT == TLH_TYPE_Q2_K) {
        const kq_u4 s = kq_ld16(blk);
        r.s[0] = s.x, r.s[1] = s.y, r.s[2] = s.z, r.s[3] = s.w;
        r.q = kq_ld16(blk + 16 + 32 * HALF + 16 * (u & 1));
        if constexpr (HALF == 1) r.s[4] = kq_ld<uint32_t>(blk + 80);
    } else {  // q3_K
        r.hi = kq_ld16(blk + 16 * (u & 1));
        r.q = kq_ld16(blk + 32 + 32 * HALF + 16 * (u & 1));
        r.s[0] = kq_ld<uint32_t>(blk + 96), r.s[1] = kq_ld<uint32_t>(blk + 100), r.s[2] = kq_ld<uint32_t>(blk + 104);
        if constexpr (HALF == 1) r.s[3] = kq_ld<uint16_t>(blk + 108);
    }
}

// The unit's first chunk (of 8 per LDS row); the second is kq_gap chunks on.
template <int WT> __device__ __forceinline__ int kq_chunk(int u) {
    return WT == TLH_TYPE_Q6_K ? u : 4 * (u >> 1) + (u & 1);
}
template <int WT> constexpr int kq_gap() { return WT == TLH_TYPE_Q6_K ? 4 : 2; }

__device__ __forceinline__ uint32_t kq_mul2(uint32_t a, uint32_t b) {  // 16-bit lanes, modulo 2^16
    return __builtin_bit_cast(uint32_t, (kq_u16x2)(__builtin_bit_cast(kq_u16x2, a) * __builtin_bit_cast(kq_u16x2, b)));
}
__device__ __forceinline__ uint32_t kq_mad2(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(uint32_t, (kq_u16x2)(__builtin_bit_cast(kq_u16x2, a) * __builtin_bit_cast(kq_u16x2, b) +
                                                    __builtin_bit_cast(kq_u16x2, c)));
}
__device__ __forceinline__ uint32_t kq_twice(int v) { return (uint32_t)(v & 0xffff) * 0x10001u; }

// Four codes c (one a byte) times sc plus `off` in 16 bits each; the results'
// high bytes to h, low bytes to l.
__device__ __forceinline__ void kq_wide(uint32_t c, uint32_t sc2, uint32_t off2, uint32_t &h, uint32_t &l) {
    const uint32_t a = __builtin_amdgcn_perm(0u, c, 0x0c010c00u), b = __builtin_amdgcn_perm(0u, c, 0x0c030c02u);
    const uint32_t va = kq_mad2(a, sc2, off2), vb = kq_mad2(b, sc2, off2);
    h = __builtin_amdgcn_perm(vb, va, 0x07050301u);
    l = __builtin_amdgcn_perm(vb, va, 0x06040200u);
}

// The unit's scaled codes: out[plane][group][dword].
template <int WT, int HALF>
__device__ __forceinline__ void kq_codes(const KqUnit<WT> &r, int u, uint32_t (&out)[2][2][4]) {
    const uint32_t q[4] = {r.q.x, r.q.y, r.q.z, r.q.w};
    const uint32_t hi[4] = {r.hi.x, r.hi.y, r.hi.z, r.hi.w};
    if constexpr (WT == TLH_TYPE_Q4_K || WT == TLH_TYPE_Q5_K) {
        // scales of the half's four sub-blocks, then of 2 (u >> 1) and the next
        const uint32_t sc4 = HALF == 0 ? r.s[1] & 0x3f3f3f3fu : (r.s[3] & 0x0f0f0f0fu) | ((r.s[1] >> 2) & 0x30303030u);
        const uint32_t two = sc4 >> (16 * (u >> 1));
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const uint32_t sc = (two >> (8 * g)) & 0xff;
            if constexpr (WT == TLH_TYPE_Q4_K) {
                const uint32_t sh2 = (sc >> 3) * 0x10001u, sl2 = (sc & 7) * 0x10001u;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t c = (g == 0 ? q[i] : q[i] >> 4) & 0x0f0f0f0fu;
                    out[0][g][i] = kq_mul2(c, sh2);
                    out[1][g][i] = kq_mul2(c, sl2);
                }
            } else {
                // the low byte as a signed one: + 128 before, its sign bit flipped after
                const uint32_t sc2 = sc * 0x10001u;
                const int bit = 4 * HALF + 2 * (u >> 1) + g;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t c = ((g == 0 ? q[i] : q[i] >> 4) & 0x0f0f0f0fu) | (((hi[i] >> bit) & 0x01010101u) << 4);
                    kq_wide(c, sc2, 0x00800080u, out[0][g][i], out[1][g][i]);
                    out[1][g][i] ^= 0x80808080u;
                }
            }
        }
    } else if constexpr (WT == TLH_TYPE_Q6_K) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const int sc = (int)(int8_t)((g == 0 ? r.s[0] : r.s[1]) >> (8 * u));
            const uint32_t sc2 = kq_twice(sc), off2 = kq_twice(128 - 32 * sc);
            const int sh = 4 * g + 2 * (u >> 1);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t c = ((g == 0 ? q[i] : q[i] >> 4) & 0x0f0f0f0fu) | (((hi[i] >> sh) & 0x03030303u) << 4);
                kq_wide(c, sc2, off2, out[0][g][i], out[1][g][i]);
                out[1][g][i] ^= 0x80808080u;
            }
        }
    } else if constexpr (WT == TLH_TYPE_Q2_K) {
        const uint32_t sc4 = ((u >> 1) ? r.s[2 * HALF + 1] : r.s[2 * HALF]) & 0x0f0f0f0fu;
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const uint32_t sc2 = ((sc4 >> (8 * ((u & 1) + 2 * g))) & 0xff) * 0x10001u;
            const int sh = 2 * (2 * (u >> 1) + g);
#pragma unroll
            for (int i = 0; i < 4; ++i) out[0][g][i] = kq_mul2((q[i] >> sh) & 0x03030303u, sc2);
        }
    } else {  // q3_K
        const uint32_t lo = (u >> 1) ? r.s[1] : r.s[0];
        const uint32_t sc4 = ((HALF ? lo >> 4 : lo) & 0x0f0f0f0fu) | (((r.s[2] >> (4 * HALF + 2 * (u >> 1))) & 0x03030303u) << 4);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const int sc = (int)((sc4 >> (8 * ((u & 1) + 2 * g))) & 0xff) - 32;
            const uint32_t sc2 = kq_twice(-sc), off2 = kq_twice(4 * sc);
            const int j = 2 * (u >> 1) + g;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t c = ((q[i] >> (2 * j)) & 0x03030303u) | (((hi[i] >> (4 * HALF + j)) & 0x01010101u) << 2);
                uint32_t h;
                kq_wide(c, sc2, off2, h, out[0][g][i]);
            }
        }
    }
}

// A row's d, dmin and the 16 mins of its bsums (q4 / q5_K: each of 8 mins
// twice), from the second half's header.
template <int WT> __device__ __forceinline__ void kq_row_meta(const KqUnit<WT> &r, float &d, float &dmin, uint32_t (&mn)[4]) {
    dmin = 0.0f;
    if constexpr (WT == TLH_TYPE_Q4_K || WT == TLH_TYPE_Q5_K) {
        d = h2f((uint16_t)(r.s[0] & 0xffff));
        dmin = h2f((uint16_t)(r.s[0] >> 16));
        mn[0] = r.s[2] & 0x3f3f3f3fu;
        mn[1] = ((r.s[3] >> 4) & 0x0f0f0f0fu) | ((r.s[2] >> 2) & 0x30303030u);
    } else if constexpr (WT == TLH_TYPE_Q6_K) {
        d = h2f((uint16_t)r.s[2]);
    } else if constexpr (WT == TLH_TYPE_Q2_K) {
        d = h2f((uint16_t)(r.s[4] & 0xffff));
        dmin = h2f((uint16_t)(r.s[4] >> 16));
#pragma unroll
        for (int i = 0; i < 4; ++i) mn[i] = (r.s[i] >> 4) & 0x0f0f0f0fu;
    } else {
        d = h2f((uint16_t)r.s[3]);
    }
}

// Super-blocks after which a chunk of n moves its f32 sums to a second set, so that
// both chains of additions stay short: about sqrt(n) equal groups. Error of such
// sums against 64 bits in 1e-8 (random terms), one chain / every 4 / every 8 / this:
// n = 5 5.1 / 5.3 / 5.1 / 5.0; 9 6.2 / 5.9 / 6.3 / 5.7; 16 7.8 / 6.3 / 6.6 / 6.3; 22 9.0
// / 6.9 / 6.8 / 6.7; 56 13.7 / 8.7 / 8.0 / 8.0.
__device__ __forceinline__ int kq_flush_every(int n) {
    if (n <= 4 || n > 30) return 8;
    int g = 2;
    while ((g + 1) * (g + 1) <= n) ++g;
    return (n + g - 1) / g;
}

// A super-block's integer sum from its planes' sums.
template <int WT> __device__ __forceinline__ float kq_sum(int h, int l) {
    if constexpr (WT == TLH_TYPE_Q4_K) return (float)(l + 8 * h);
    else if constexpr (kq_planes<WT>() == 2) return (float)(l + 256 * h);
    else if constexpr (WT == TLH_TYPE_Q3_K) return -(float)l;
    else return (float)l;
}

}  // namespace tlh
