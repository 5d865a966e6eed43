// Products of fp32 (or int8) activation rows with block-quantized weight rows
// on the matrix cores, without giving up fp32: splitmm_kernel.
//
// Weights. Every quantized format here is an integer (or e4m3) code times a
// scale shared by 16 or more consecutive K: the code is exact in bf16 (and in
// int8 for the GGUF types), so the codes are the MFMA's B operand as they are
// and the scale multiplies the 16- or 32-K partial product afterwards, in
// fp32, once per output.
// fp32 activations, times 2^40, are cut into three bf16 terms by truncation (8 +
// 8 + 8 significant bits: the three add up to the fp32 value exactly), three
// MFMAs per 16 K, smallest term first. Products are exact, the MFMA adds in fp32:
// the rounding is that of an fp32 sum over 16- or 32-K pieces.
// int8 activations use the int8 MFMA (exact int32 sums per 32 K), then the
// weight scale and the activation block's scale in fp32.
// The matrix cores' fp32 addition rounds down rather than to nearest (mean
// error of 6144-long products -6e-8 to -8e-8 of their rms with Q8_0, IQ3_XXS and
// int4 weights, against 9e-8 of spread), and a sum of many such pieces drifts:
// every second 32-K block is computed with negated activations and the scale's
// sign flipped, which leaves 4e-9 at most.
// The partial products of a chunk (256 K; 128 where a chunk is that) are
// added first, then the chunk sums: a two-level sum, whose rounding error
// (8.6e-8 to 1.15e-7 of the rms over the types at K 6144) is no larger than the
// vector kernels' (tests/test_gpu_splitmm.py holds bias and error to that).
//
// Operands: A = activations (D row = token), B = weights (D column = weight
// row), so a lane's outputs belong to one weight row and need one scale.
// A wave owns NB x 32 weight rows (gate and up rows of the same 32 features,
// or output rows) and a tile of NT tokens:
//   NT = 32, 64 (prefill): 32x32x16 MFMAs, lane = weight row l % 32 and K half
//     l / 32; D value i of half hh is token 8 (i / 4) + 4 hh + i % 4.
//   NT = 4, 8, 16 (decode): 16x16x32 MFMAs, lane = weight row l % 16 and K
//     quarter q = l / 16 (the 8 weights the lane decodes). D value i of
//     quarter q is A row 4 q + i: token NV q + i sits in that row for
//     i < NV = NT / 4, so a tile of 4 tokens costs one rescale per value of
//     D the other rows of which repeat tokens and are dropped. Half the matrix
//     time and half the activation reads of the 32-row form.
// A workgroup has RW * KW waves: RW row groups x KW shares of K (chunk c goes
// to share c % KW; the shares' sums are added in order at the end).
//   - weights: a wave loads its rows' raw bytes of the next chunk as coalesced
//     dwords into registers (16 lanes per row, the rest of the row one lane
//     per row) and parks them in its own LDS rows at the chunk's start (odd
//     dword stride: lane = row reads hit distinct banks); each lane decodes the
//     fragments of its own row. The block scales of a chunk are decoded once
//     (a lane takes some of its row's blocks) and kept in LDS.
//   - activations: the tile's rows are staged KX at a time, loaded one step
//     ahead, split once per workgroup row group and read as A fragments.
#pragma once

#include <stddef.h>

#include <type_traits>

#include "common.hpp"
#include "gguf_dec.hpp"

namespace glmmoe {

constexpr uint32_t kSmW4 = 100;    // int4, two per byte, fp32 scales per `group` K
constexpr uint32_t kSmFp8 = 101;   // e4m3, optional fp32 scale per row
enum { kSmGateUp = 0, kSmDown = 1, kSmDense = 2 };

struct SmArgs {
    const float* x;                 // fp32 rows [*, K]
    const int8_t* xq;               // int8 rows [*, K] and their scales [*, K / 32]
    const float* xs;
    const uint8_t *w0, *w1;         // gate / down / dense rows; up rows
    long rb0, rb1;                  // bytes per weight row
    const float* sc;                // W4: [out, K / group]; FP8: [out] or null
    int group;
    const float* bias;              // dense, nullable
    float* y;                       // h_act / dpart / y
    int K, out, n;                  // out: weight rows (per expert)
    int E, topk;
    const int* ids;                 // MoE: routed ids
    const int* d;                   // MoE: grouping [offsets | tile prefix | rows], or null: row g alone
};

// Tokens per tile of the large MoE launches; the small ones take 4, 8 or 16.
constexpr int kSmMidTile = 32, kSmLargeTile = 64;
// The types whose experts take tiles of 64 (the measurements: gg_sm_tile).
constexpr bool sm_large_tile(uint32_t t, bool i8) { return t == 18 || t == 23 || (t == 8 && i8); }
// The launches (splitmm_launch.hpp): tile = tokens per tile of the grouping; a tile
// the type has no kernel for is refused (-2).
template <uint32_t T>
int sm_moe(bool down, bool i8, int tile, const SmArgs& a, unsigned tiles, hipStream_t s);
template <uint32_t T>
int sm_dense(bool i8, const SmArgs& a, hipStream_t s);

// fp32 activations are split times 2^40: the matrix cores take subnormal bf16 terms
// as zero, and an activation below 2^-110 has some (rows of about 1e-36 lost three
// digits). From 2^88 the epilogue recomputes.
constexpr float kSmUp = 0x1p40f;

// Output rows a launch takes: whole blocks of 32, in the grid's second dimension.
constexpr bool sm_out_ok(int out) { return out % 32 == 0 && out / 32 <= 65535; }

constexpr bool sm_g16(uint32_t t) { return t == 11 || t == 14; }          // scale per 16 K
constexpr bool sm_min(uint32_t t) { return t == 12 || t == 13; }          // weight = ds * q - dm
// These types' codes are taken less sm_mid: weight = ds (q - mid) - (dm - mid ds). A
// checkpoint's weights centre on zero, so what is left of the offset is small and
// activations with a mean do not make two large sums cancel (fp32 rows of mean and
// spread 1, K 6144, error against 64 bits: 1.1e-7 -> 9.4e-8, vector kernels 8.3e-8;
// of mean 0: 1.2e-7 -> 1.0e-7, vector kernels 1.4e-7). Sums in 64 bits do not need
// it (MID false; int8 linears, 6144 -> 2048, 1 / 64 tokens, us: Q4_K 11.8 / 23.3 centred,
// 11.5 / 22.8 not; Q5_K 12.8 / 25.0 and 12.2 / 24.1).
constexpr uint32_t sm_mid(uint32_t t) { return t == 12 ? 8 : t == 13 ? 16 : 0; }
constexpr int sm_kc(uint32_t t) { return t == 8 || t == kSmFp8 ? 128 : 256; }   // K per chunk
constexpr int sm_cb(uint32_t t) {                                          // bytes per chunk of a row
    return t == kSmW4 || t == kSmFp8 ? 128 : sm_kc(t) / gg_be(t) * gg_bb(t);
}
constexpr int sm_ndw(uint32_t t) { return (sm_cb(t) + 2) / 4; }           // dwords that cover it (2-byte aligned)
constexpr int sm_stride(uint32_t t) { return (sm_ndw(t) | 1) * 4; }       // LDS bytes per row

typedef int sm_i32x4 __attribute__((ext_vector_type(4)));
typedef int sm_i32x2 __attribute__((ext_vector_type(2)));
typedef int sm_i32x16 __attribute__((ext_vector_type(16)));

// N dwords from / to a dword-aligned address, in pieces of 4, 2 and 1.
typedef uint32_t sm_u4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t sm_u2 __attribute__((ext_vector_type(2), aligned(4)));
template <int N>
__device__ __forceinline__ void sm_get(const uint8_t* p, uint32_t (&v)[N]) {
    static_for<N / 4>([&](auto i) {
        const u32x4 t = *reinterpret_cast<const sm_u4*>(p + 16 * i);
        v[4 * i] = t.x; v[4 * i + 1] = t.y; v[4 * i + 2] = t.z; v[4 * i + 3] = t.w;
    });
    constexpr int r = N & ~3;
    if constexpr (N & 2) {
        const u32x2 t = *reinterpret_cast<const sm_u2*>(p + 4 * r);
        v[r] = t.x; v[r + 1] = t.y;
    }
    if constexpr (N & 1) v[N - 1] = *reinterpret_cast<const uint32_t*>(p + 4 * (N - 1));
}
template <int N>
__device__ __forceinline__ void sm_put(uint8_t* p, const uint32_t (&v)[N]) {
    static_for<N / 4>([&](auto i) {
        *reinterpret_cast<sm_u4*>(p + 16 * i) = sm_u4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
    });
    constexpr int r = N & ~3;
    if constexpr (N & 2) *reinterpret_cast<sm_u2*>(p + 4 * r) = sm_u2{v[r], v[r + 1]};
    if constexpr (N & 1) *reinterpret_cast<uint32_t*>(p + 4 * (N - 1)) = v[N - 1];
}

// LDS writes of the wave done, then the workgroup's barrier; loads in flight
// to registers stay in flight.
__device__ __forceinline__ void sm_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n s_barrier" ::: "memory");
}

__device__ __forceinline__ float sm_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double sm_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }

__device__ __forceinline__ uint32_t sm_bf16_int(int v) { return __float_as_uint((float)v) >> 16; }
__device__ __forceinline__ uint32_t sm_hi2(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
// Four signed bytes as bf16 pairs (exact).
__device__ __forceinline__ void sm_i8_bf16(uint32_t w, uint32_t& p0, uint32_t& p1) {
    p0 = sm_hi2((float)(int8_t)w, (float)(int8_t)(w >> 8));
    p1 = sm_hi2((float)(int8_t)(w >> 16), (float)(int8_t)(w >> 24));
}

// Lookup tables in LDS. IQ3_XXS fp32: the codebook as 4 bf16 (signs are
// or-ed in); int8: codebook entry x 4 sign bits as 4 signed bytes. IQ4_XS / W4
// fp32: two 4-bit codes of one byte as a bf16 pair (low nibble low).
template <uint32_t T, bool I8>
struct SmTables {
    uint32_t a[I8 ? (T == 18 ? 4096 : 1) : T == 18 ? 512 : T == 23 || T == kSmW4 ? 256 : 1];
};

template <uint32_t T, bool I8>
__device__ __forceinline__ void sm_init_tables(SmTables<T, I8>& L, int tid, int nt) {
    if constexpr (T == 18 && I8) {
        for (int i = tid; i < 4096; i += nt) {
            const uint32_t g = c_iq3xxs_grid[i & 255], m = gg_bytemask4((uint32_t)i >> 8);
            L.a[i] = (g ^ m) + (m & 0x01010101u);   // no carry: every magnitude is at least 4
        }
    } else {
        for (int i = tid; i < 256; i += nt) {
            if constexpr (T == 18) {
                const uint32_t g = c_iq3xxs_grid[i];
                L.a[2 * i] = sm_bf16_int(g & 255) | (sm_bf16_int((g >> 8) & 255) << 16);
                L.a[2 * i + 1] = sm_bf16_int((g >> 16) & 255) | (sm_bf16_int(g >> 24) << 16);
            } else if constexpr (!I8 && T == 23) {
                L.a[i] = sm_bf16_int(kIq4nl[i & 15]) | (sm_bf16_int(kIq4nl[i >> 4]) << 16);
            } else if constexpr (!I8 && T == kSmW4) {
                L.a[i] = sm_bf16_int((i & 15) - 8) | (sm_bf16_int((i >> 4) - 8) << 16);
            }
        }
    }
}

__device__ __forceinline__ uint32_t sm_ld16(const uint8_t* p) { return *reinterpret_cast<const uint16_t*>(p); }
__device__ __forceinline__ uint32_t sm_ld32u(const uint8_t* p) {   // 2-byte aligned
    return sm_ld16(p) | (sm_ld16(p + 2) << 16);
}
__device__ __forceinline__ uint32_t sm_ld32(const uint8_t* p) { return *reinterpret_cast<const uint32_t*>(p); }

// Four bytes at b (2-byte aligned; skew = b & 2, uniform) as one read.
__device__ __forceinline__ uint32_t sm_ld32s(const uint8_t* b, uint32_t skew) {
    const uint32_t* p = reinterpret_cast<const uint32_t*>(b - skew);
    return __builtin_amdgcn_alignbyte(p[1], p[0], skew);
}

// Scale (and offset) of the weights at K = 32 ib + 16 j of a chunk:
// weight = ds * code - dm. b: the row's chunk in LDS. (W4: the caller's.)
template <uint32_t T>
__device__ __forceinline__ void sm_scale(const uint8_t* b, int ib, int j, float& ds, float& dm) {
    dm = 0.0f;
    if constexpr (T == 18) {
        ds = gg_rdf16<true>(b) * (0.5f + (float)(sm_ld16(b + 68 + 4 * ib) >> 12)) * 0.5f;
    } else if constexpr (T == kSmFp8 || T == kSmW4) {
        ds = 1.0f;
    } else {
        int w0, w1;
        gg_dec8i<T, true>(T, b, 32 * ib + 16 * j, nullptr, nullptr, w0, w1, ds, dm);
    }
}

// Codes K = 32 ib + 8 f + [0, 8) of a chunk as 8 int8 (the types whose codes
// are plain bit fields), the integers of gg_dec8i (MID: less sm_mid). skew: b & 2.
template <uint32_t T, bool MID>
__device__ __forceinline__ void sm_codes(const uint8_t* b, int ib, int f, uint32_t skew, uint32_t& w0,
                                         uint32_t& w1) {
    if constexpr (T == 8) {   // 34-byte blocks in a 4-byte aligned chunk
        const uint32_t sk = ib & 1 ? 0u : 2u;
        w0 = sm_ld32s(b + 34 * ib + 2 + 8 * f, sk);
        w1 = sm_ld32s(b + 34 * ib + 6 + 8 * f, sk);
    } else if constexpr (T == 12 || T == 13) {   // 4-byte aligned
        const uint8_t* q = b + (T == 12 ? 16 : 48) + 32 * (ib >> 1) + 8 * f;
        w0 = (sm_ld32(q) >> (4 * (ib & 1))) & 0x0f0f0f0fu;
        w1 = (sm_ld32(q + 4) >> (4 * (ib & 1))) & 0x0f0f0f0fu;
        if constexpr (T == 13) {
            w0 |= ((sm_ld32(b + 16 + 8 * f) >> ib) & 0x01010101u) << 4;
            w1 |= ((sm_ld32(b + 20 + 8 * f) >> ib) & 0x01010101u) << 4;
        }
        if constexpr (MID) {   // per byte: 0..31 with bit 7 set borrows nothing from its neighbour
            constexpr uint32_t mid = sm_mid(T) * 0x01010101u;
            w0 = ((w0 | 0x80808080u) - mid) ^ 0x80808080u;
            w1 = ((w1 | 0x80808080u) - mid) ^ 0x80808080u;
        }
    } else if constexpr (T == 14) {
        const int half = ib >> 2, qr = ib & 3;
        const uint8_t* ql = b + 64 * half + 32 * (qr & 1) + 8 * f;
        const uint8_t* qh = b + 128 + 32 * half + 8 * f;
        // (lo | hi << 4) - 32 per byte: each byte is 0..63, so with bit 7 set no
        // byte borrows from its neighbour
        const uint32_t u0 = ((sm_ld32s(ql, skew) >> (4 * (qr >> 1))) & 0x0f0f0f0fu) |
                            (((sm_ld32s(qh, skew) >> (2 * qr)) & 0x03030303u) << 4);
        const uint32_t u1 = ((sm_ld32s(ql + 4, skew) >> (4 * (qr >> 1))) & 0x0f0f0f0fu) |
                            (((sm_ld32s(qh + 4, skew) >> (2 * qr)) & 0x03030303u) << 4);
        w0 = ((u0 | 0x80808080u) - 0x20202020u) ^ 0x80808080u;
        w1 = ((u1 | 0x80808080u) - 0x20202020u) ^ 0x80808080u;
    } else {
        int a, c;
        float ds, dm;
        gg_dec8i<T, true>(T, b, 32 * ib + 8 * f, nullptr, nullptr, a, c, ds, dm);
        w0 = (uint32_t)a;
        w1 = (uint32_t)c;
    }
}

// Codes K = 32 ib + 8 f + [0, 8) of a chunk as a bf16 B operand. skew: b & 2.
template <uint32_t T>
__device__ __forceinline__ u32x4 sm_codes_bf16(const uint8_t* b, int ib, int f, uint32_t skew,
                                               const SmTables<T, false>& L) {
    u32x4 w;
    if constexpr (T == 18) {
        const uint32_t i7 = (sm_ld32s(b + 66 + 4 * ib, skew ^ 2u) >> (7 * f)) & 127u;
        // the 8 sign bits (bit 7: the parity of the 7), twice, 15 apart: one
        // shift brings a pair's two signs to bits 15 and 31
        const uint32_t sg = (i7 | ((uint32_t)__builtin_popcount(i7) << 7)) & 255u;
        const uint32_t s2 = sg | (sg << 15);
        const uint32_t qs = sm_ld16(b + 2 + 8 * ib + 2 * f);
        const uint2 g0 = *reinterpret_cast<const uint2*>(&L.a[2 * (qs & 255u)]);
        const uint2 g1 = *reinterpret_cast<const uint2*>(&L.a[2 * (qs >> 8)]);
        w.x = ((s2 << 15) & 0x80008000u) | g0.x;
        w.y = ((s2 << 13) & 0x80008000u) | g0.y;
        w.z = ((s2 << 11) & 0x80008000u) | g1.x;
        w.w = ((s2 << 9) & 0x80008000u) | g1.y;
    } else if constexpr (T == 23) {
        const uint8_t* q = b + 8 + 16 * ib + 8 * (f & 1);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t c = (sm_ld32(q + 4 * u) >> (4 * (f >> 1))) & 0x0f0f0f0fu;
            const uint32_t t = c | (c >> 4);   // code pairs in bytes 0 and 2
            w[2 * u] = L.a[t & 255u];
            w[2 * u + 1] = L.a[(t >> 16) & 255u];
        }
    } else if constexpr (T == kSmW4) {
        const uint32_t c = sm_ld32(b + 16 * ib + 4 * f);
#pragma unroll
        for (int u = 0; u < 4; ++u) w[u] = L.a[(c >> (8 * u)) & 255u];
    } else if constexpr (T == kSmFp8) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t c = sm_ld32(b + 32 * ib + 8 * f + 4 * u);
            const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)c, false);
            const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)c, true);
            w[2 * u] = sm_hi2(lo.x, lo.y);
            w[2 * u + 1] = sm_hi2(hi.x, hi.y);
        }
    } else {
        uint32_t w0, w1, a0, a1, a2, a3;
        sm_codes<T, true>(b, ib, f, skew, w0, w1);
        sm_i8_bf16(w0, a0, a1);
        sm_i8_bf16(w1, a2, a3);
        w = u32x4{a0, a1, a2, a3};
    }
    return w;
}

// IQ4_NL values of the four codes q >> sh (bits 0..3 of each byte): the byte
// select picks among 8, a mask byte (v_perm: 0x0c gives 0x00, 0x0d 0xff) the half.
__device__ __forceinline__ uint32_t sm_iq4nl4(uint32_t q) {
    const uint32_t sel = q & 0x07070707u;
    const uint32_t lo = __builtin_amdgcn_perm(iq4nl_word(1), iq4nl_word(0), sel);
    const uint32_t hi = __builtin_amdgcn_perm(iq4nl_word(3), iq4nl_word(2), sel);
    const uint32_t m = __builtin_amdgcn_perm(0u, 0u, ((q >> 3) & 0x01010101u) | 0x0c0c0c0cu);
    return (hi & m) | (lo & ~m);
}

// The same codes as 8 int8.
template <uint32_t T, bool MID>
__device__ __forceinline__ sm_i32x2 sm_codes_i8(const uint8_t* b, int ib, int f, uint32_t skew,
                                                const SmTables<T, true>& L) {
    if constexpr (T == 18) {
        const uint32_t i7 = (sm_ld32s(b + 66 + 4 * ib, skew ^ 2u) >> (7 * f)) & 127u;
        const uint32_t sg = i7 | ((uint32_t)__builtin_popcount(i7) << 7);
        const uint32_t qs = sm_ld16(b + 2 + 8 * ib + 2 * f);
        return sm_i32x2{(int)L.a[(qs & 255u) | ((sg & 15u) << 8)],
                        (int)L.a[(qs >> 8) | ((sg & 0xf0u) << 4)]};
    } else if constexpr (T == 23) {
        const uint8_t* q = b + 8 + 16 * ib + 8 * (f & 1);
        const int sh = 4 * (f >> 1);
        return sm_i32x2{(int)sm_iq4nl4(sm_ld32(q) >> sh), (int)sm_iq4nl4(sm_ld32(q + 4) >> sh)};
    } else {
        uint32_t w0, w1;
        sm_codes<T, MID>(b, ib, f, skew, w0, w1);
        return sm_i32x2{(int)w0, (int)w1};
    }
}

// Weights k .. k + 7 (k % 8 == 0) of a row (matrix row r), dequantized.
template <uint32_t T>
__device__ __forceinline__ void sm_weights(const SmArgs& a, const uint8_t* w, int r, int k, float (&y)[8]) {
    if constexpr (T == kSmW4) {
        const uint32_t c = gg_ld32(w + k / 2);
        const float sc = a.sc[(size_t)r * (a.K / a.group) + k / a.group];
#pragma unroll
        for (int u = 0; u < 8; ++u) y[u] = (float)((int)((c >> (4 * u)) & 15u) - 8) * sc;
    } else if constexpr (T == kSmFp8) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = w[k + 2 * u] | w[k + 2 * u + 1] << 8;
            const f32x2 p = __builtin_amdgcn_cvt_pk_f32_fp8(c, false);
            y[2 * u] = p.x; y[2 * u + 1] = p.y;
        }
    } else {
        gg_dec8<T>(T, w, k, c_iq3xxs_grid, y);
    }
}

template <uint32_t T, bool I8, int RW, int KW, int NB, int NT, int KX>
struct SmLds {
    static constexpr int XS = I8 ? KX + 16 : 2 * KX + 16;     // bytes of an activation row of a plane
    static constexpr int PL = I8 ? 1 : 3;
    static constexpr int NS = sm_kc(T) / (sm_g16(T) ? 16 : 32);   // scales of a row's chunk
    SmTables<T, I8> tab;
    int src[NT], row[NT], tile[3];
    // from here on free for the shares' sums at the end
    __align__(16) uint8_t x[KW][PL][NT][XS];
    // read as float4 in the tiles of 32 and 64: rows of NT floats from 16-byte aligned starts
    __align__(16) float xsc[I8 ? KW : 1][I8 ? KX / 32 : 1][I8 ? NT : 1];           // int8 block scales
    __align__(16) float xsum[sm_min(T) ? KW : 1][sm_min(T) ? KX / 32 : 1][sm_min(T) ? NT : 1];   // block sums
    float ds[RW * KW][NB * 32][NS + 1];
    float dm[sm_min(T) ? RW * KW : 1][sm_min(T) ? NB * 32 : 1][NS + 1];
    __align__(16) uint8_t raw[RW * KW][NB * 32][sm_stride(T)];
    uint32_t past;   // sm_ld32s may read the word after a row
};

template <uint32_t T, int MODE, bool I8, int RW, int KW, int NB, int NT, int KX>
__global__ __launch_bounds__(64 * RW * KW, 2) void splitmm_kernel(SmArgs a) {
    using S = SmLds<T, I8, RW, KW, NB, NT, KX>;
    static_assert(MODE != kSmGateUp || NB == 2, "gate and up rows in one wave");
    static_assert(offsetof(S, xsc) % 16 == 0 && offsetof(S, xsum) % 16 == 0 && NT % 4 == 0, "float4 reads");
    constexpr bool SM = NT <= 16;                 // 16x16x32 MFMAs
    constexpr int TOK = NT, KC = sm_kc(T), ST = KC / KX, BX = KX / 32;
    constexpr int TB = SM ? 1 : NT / 32;          // 32-token blocks
    constexpr int NV = SM ? NT / 4 : 16;          // live D values per block
    constexpr int BR = SM ? 16 : 32;              // weight rows per block
    constexpr int NK = NB * 32 / BR;              // blocks
    constexpr int NDW = sm_ndw(T), MW = NDW / 16, TL = NDW % 16;
    constexpr int RS = sm_stride(T);
    __shared__ S L;
    const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5;
    const int lr = lane & (BR - 1), lq = lane / BR;   // row in block, K half / quarter
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rw = wave % RW, kw = wave / RW;
    const int K = a.K;

    // The tile.
    size_t e = 0;
    int nr, t0 = 0;
    if constexpr (MODE == kSmDense) {
        t0 = (int)blockIdx.x * TOK;
        nr = min(TOK, a.n - t0);
        if (tid < TOK) L.src[tid] = t0 + min(tid, nr - 1);
    } else {
        const int g = (int)blockIdx.x, E = a.E;
        if (!a.d) {
            const int id = g < a.n * a.topk ? a.ids[g] : -1;
            if (id < 0 || id >= E) return;   // routes nowhere
            e = (size_t)id;
            nr = 1;
            if (tid < TOK) {
                L.row[tid] = g;
                L.src[tid] = MODE == kSmDown ? g : g / a.topk;
            }
        } else {
            // The expert with tp[e] <= g < tp[e + 1]: every thread looks at its
            // own experts, one round trip instead of a binary search's eight.
            const int* off = a.d;
            const int* tp = a.d + E + 1;
            const int* rows = a.d + 2 * (E + 1);
            if (g >= tp[E]) return;          // the grid covers the largest possible tile count
            for (int q = tid; q < E; q += 64 * RW * KW) {
                const int p0 = tp[q], p1 = tp[q + 1], r0 = off[q], r1 = off[q + 1];
                if (p0 <= g && g < p1) {
                    L.tile[0] = q;
                    L.tile[1] = r0 + (g - p0) * TOK;
                    L.tile[2] = r1;
                }
            }
            sm_barrier();
            e = (size_t)__builtin_amdgcn_readfirstlane(L.tile[0]);
            const int r0 = __builtin_amdgcn_readfirstlane(L.tile[1]);
            nr = min(TOK, __builtin_amdgcn_readfirstlane(L.tile[2]) - r0);
            if (tid < TOK) {
                const int r = rows[r0 + min(tid, nr - 1)];
                L.row[tid] = r;
                L.src[tid] = MODE == kSmDown ? r : r / a.topk;
            }
        }
    }

    // Weight rows of this wave: block nb covers rows base[nb] + lr.
    constexpr int RWG = (MODE == kSmGateUp ? 32 : 32 * NB) * RW;   // output rows per workgroup
    const int f0 = (int)blockIdx.y * RWG + rw * (MODE == kSmGateUp ? 32 : 32 * NB);
    const uint8_t* wb[NB];
    int ob[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        // out is a multiple of 32: a block past it repeats the last one, unstored
        ob[nb] = min(MODE == kSmGateUp ? f0 : f0 + 32 * nb, a.out - 32);
        const bool up = MODE == kSmGateUp && nb == 1;
        wb[nb] = (up ? a.w1 : a.w0) + (e * (size_t)a.out + (size_t)ob[nb]) * (size_t)(up ? a.rb1 : a.rb0);
    }

    // Per-lane parts of the weight addresses.
    const long rb[2] = {a.rb0, MODE == kSmGateUp ? a.rb1 : a.rb0};
    uint32_t moff[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) moff[nb] = (uint32_t)((lane >> 4) * rb[nb] + (lane & 15) * 4 * MW);
    const bool tl_on = NB == 2 || lane < 32;
    const uint8_t* trow = (NB == 2 && hh ? wb[NB - 1] : wb[0]) + (lane & 31) * (NB == 2 && hh ? rb[1] : rb[0]) + 64 * MW;
    uint8_t* const raw = &L.raw[wave][0][0];

    const int nch = K / KC;
    uint32_t mv[NB][8][MW > 0 ? MW : 1], tv[TL > 0 ? TL : 1];
    auto load_raw = [&](int c) {
        const long off = ((long)c * sm_cb(T)) & ~3l;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const uint8_t* p = wb[nb] + off + 4 * m * rb[nb] + moff[nb];
                if constexpr (MW > 0) sm_get(p, mv[nb][m]);
            }
        if constexpr (TL > 0) {
            if (tl_on) sm_get(trow + off, tv);
        }
    };
    auto park_raw = [&]() {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int m = 0; m < 8; ++m)
                if constexpr (MW > 0)
                    sm_put(raw + (nb * 32 + 4 * m + (lane >> 4)) * RS + (lane & 15) * 4 * MW, mv[nb][m]);
        if constexpr (TL > 0) {
            if (tl_on) sm_put(raw + lane * RS + 64 * MW, tv);
        }
    };

    // The first chunk is on its way while the tables are built and the rows' ids arrive.
    load_raw(min(kw, nch - 1));
    sm_init_tables<T, I8>(L.tab, tid, 64 * RW * KW);
    sm_barrier();

    // Activations: pieces of 8 fp32 (16 int8) of the tile, per thread of the
    // K share's RW waves.
    constexpr int XP = I8 ? 16 : 8;
    constexpr int PPR = KX / XP, NP = TOK * PPR, GT = 64 * RW;
    constexpr int XN = (NP + GT - 1) / GT;
    const int gt = rw * 64 + lane;
    const size_t esz = I8 ? 1 : 4;
    const uint8_t* xp[XN];
#pragma unroll
    for (int j = 0; j < XN; ++j) {
        const int p = min(gt + j * GT, NP - 1);
        xp[j] = (I8 ? (const uint8_t*)a.xq : (const uint8_t*)a.x) +
                ((size_t)L.src[p / PPR] * K + (p % PPR) * XP) * esz;
    }
    constexpr int SN = (TOK * BX + GT - 1) / GT;   // int8: block scales per thread
    u32x4 xv[XN][I8 ? 1 : 2];
    float sv[SN];
    auto load_x = [&](int k0) {
#pragma unroll
        for (int j = 0; j < XN; ++j)
#pragma unroll
            for (int q = 0; q < (I8 ? 1 : 2); ++q) {
                // int8 rows are 4-byte aligned, fp32 rows 16-byte aligned
                const uint8_t* p = xp[j] + (size_t)k0 * esz + 16 * q;
                if constexpr (I8) xv[j][q] = *reinterpret_cast<const sm_u4*>(p);
                else xv[j][q] = *reinterpret_cast<const u32x4*>(p);
            }
        if constexpr (I8) {
#pragma unroll
            for (int j = 0; j < SN; ++j) {
                const int p = min(gt + j * GT, TOK * BX - 1);
                sv[j] = a.xs[(size_t)L.src[p / BX] * (K / 32) + k0 / 32 + p % BX];
            }
        }
    };
    auto park_x = [&](int s) {
#pragma unroll
        for (int j = 0; j < XN; ++j) {
            const int p = gt + j * GT;
            if (NP % GT != 0 && p >= NP) break;
            const int t = p / PPR, pc = p % PPR;
            if constexpr (I8) {
                *reinterpret_cast<u32x4*>(&L.x[kw][0][t][16 * pc]) = xv[j][0];
                if constexpr (sm_min(T)) {
                    int sum = 0;
#pragma unroll
                    for (int u = 0; u < 4; ++u) sum = __builtin_amdgcn_sdot4(0x01010101, (int)xv[j][0][u], sum, false);
                    sum += __shfl_xor(sum, 1);
                    if (!(pc & 1)) L.xsum[kw][pc / 2][t] = (float)sum;
                }
            } else {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = __uint_as_float(xv[j][u >> 2][u & 3]);
                if constexpr (sm_min(T)) {
                    float sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
                    sum += __shfl_xor(sum, 1);
                    sum += __shfl_xor(sum, 2);
                    if (!(pc & 3)) L.xsum[kw][pc / 4][t] = sum * kSmUp;
                }
                // odd 32-K blocks enter negated (see the head of the file)
                const float up = (s * BX + pc / 4) & 1 ? -kSmUp : kSmUp;
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] *= up;
                float m[8], l[8];   // NaN for an infinity: the epilogue recomputes what is not finite
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    m[u] = v[u] - __uint_as_float(__float_as_uint(v[u]) & 0xffff0000u);
                    l[u] = m[u] - __uint_as_float(__float_as_uint(m[u]) & 0xffff0000u);
                }
                if constexpr (T == 8 && MODE != kSmDense) {
                    // Clears what the epilogue recomputes anyway, for the branch's sake: without
                    // it the compiler no longer mixes these kernels' decode with the products
                    // (2048 x 512 x 64, top-4, 1000 tokens: 213 -> 227 us).
                    float chk = 0.0f;
#pragma unroll
                    for (int u = 0; u < 8; ++u) chk += l[u];
                    if (chk != chk) {
#pragma unroll
                        for (int u = 0; u < 8; ++u)
                            if (l[u] != l[u]) {
                                m[u] = l[u] = 0.0f;
                                if (v[u] != v[u]) v[u] = __uint_as_float(0x7fc00000u);
                            }
                    }
                }
                u32x4 ph, pm, pl;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    ph[u] = sm_hi2(v[2 * u], v[2 * u + 1]);
                    pm[u] = sm_hi2(m[2 * u], m[2 * u + 1]);
                    pl[u] = sm_hi2(l[2 * u], l[2 * u + 1]);
                }
                *reinterpret_cast<u32x4*>(&L.x[kw][0][t][16 * pc]) = ph;
                *reinterpret_cast<u32x4*>(&L.x[kw][1 % S::PL][t][16 * pc]) = pm;
                *reinterpret_cast<u32x4*>(&L.x[kw][2 % S::PL][t][16 * pc]) = pl;
            }
        }
        if constexpr (I8) {
#pragma unroll
            for (int j = 0; j < SN; ++j) {
                const int p = gt + j * GT;
                if (p < TOK * BX) L.xsc[kw][p % BX][p / BX] = sv[j];
            }
        }
    };

    // The A row of this lane holds tile token ta (+ 32 tb).
    const int ta = SM ? (lr >> 2) * NV + (lr & (NV - 1)) : lr;
    const int ntb = TB == 1 ? 1 : __builtin_amdgcn_readfirstlane((nr + 31) / 32);
    // int8 products mostly feed the int8 quantizer again, where one rounding more
    // or less moves a code: up to 16 rows per expert (gate/up) and in the linears'
    // tiles of at most 32 tokens the exact integer dots are scaled and added in
    // 64 bits (64 tokens 855 -> 873 us), so the result is the rounded exact value
    // and fewer codes move. A block of 64 tokens is 1.5e-7 from 64 bits where none
    // does and about 5e-5 where one does, on some inputs with sums in 32 bits.
    constexpr bool F64 = I8 && ((SM && MODE == kSmGateUp) || (TB == 1 && MODE == kSmDense));
    using Acc = std::conditional_t<F64, double, float>;
    Acc acc[NK][TB][NV];
    float part[NK][TB][NV];
#pragma unroll
    for (int nb = 0; nb < NK; ++nb)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
            for (int i = 0; i < NV; ++i) acc[nb][tb][i] = part[nb][tb][i] = 0.0f;

    // The floats of the lane's D tokens of one 32-K block from a [TOK] array.
    auto tokv = [&](const float* p, int tb, float (&o)[NV]) {
        if constexpr (SM) {
#pragma unroll
            for (int i = 0; i < NV; ++i) o[i] = p[lq * NV + i];
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 v = *reinterpret_cast<const float4*>(p + 32 * tb + 8 * q + 4 * hh);
                o[4 * q] = v.x; o[4 * q + 1] = v.y; o[4 * q + 2] = v.z; o[4 * q + 3] = v.w;
            }
        }
    };
    // Scales of the wave's rows of the parked chunk: rows by lane, a row's
    // scales spread over the lanes that share it.
    auto scales = [&](const uint8_t* base, int cc) {
        constexpr int RG = NB * 32 < 64 ? 32 : 64, LG = 64 / RG, PER = (S::NS + LG - 1) / LG;
        const int r = lane & (RG - 1);
        const uint8_t* b = base + r * RS;
#pragma unroll
        for (int v = 0; v < PER; ++v) {
            const int i = (lane / RG) * PER + v;
            float ds, dm;
            if constexpr (sm_g16(T)) sm_scale<T>(b, i / 2, i % 2, ds, dm);
            else sm_scale<T>(b, i, 0, ds, dm);
            if constexpr (T == kSmW4)   // group: a multiple of 32
                ds = a.sc[(size_t)(ob[r / 32] + (r & 31)) * (K / a.group) + (cc * KC + 32 * i) / a.group];
            if constexpr (sm_min(T) && !F64) dm = __builtin_fmaf(-(float)sm_mid(T), ds, dm);
            // negative for the blocks whose fp32 activations are staged negated
            L.ds[wave][r][i] = !I8 && ((sm_g16(T) ? i / 2 : i) & 1) ? -ds : ds;
            if constexpr (sm_min(T)) L.dm[wave][r][i] = dm;
        }
    };

    auto scale_of = [&](int nb, int i) {
        return T == kSmFp8 ? (i & 1 ? -1.0f : 1.0f) : L.ds[wave][nb * BR + lr][i];
    };
    // One 32-K block, 16 weight rows per MFMA.
    auto small_block = [&](int b, int ib, const uint8_t* brow, uint32_t skew) {
        const uint8_t* ax = &L.x[kw][0][ta][(I8 ? 32 : 64) * b + (I8 ? 8 : 16) * lq];
        constexpr size_t PS = sizeof(L.x[0][0]);
        float xsv[NV], sxv[NV];
        if constexpr (I8) tokv(&L.xsc[kw][b][0], 0, xsv);
        if constexpr (sm_min(T)) tokv(&L.xsum[kw][b][0], 0, sxv);
        bf16x8 A[3];
        long Ai = 0;
        if constexpr (I8) Ai = *reinterpret_cast<const long*>(ax);
        else {
#pragma unroll
            for (int p = 0; p < 3; ++p) A[p] = as_bf16x8(*reinterpret_cast<const u32x4*>(ax + p * PS));
        }
#pragma unroll
        for (int nb = 0; nb < NK; ++nb) {
            const uint8_t* rb_ = brow + nb * BR * RS;
            // sm_g16: the two 16-K halves (quarters 0-1 and 2-3) have their own
            // scale: two products with the other half's weights zeroed
            constexpr int HV = sm_g16(T) ? 2 : 1;
            float ds[HV];
#pragma unroll
            for (int h = 0; h < HV; ++h) ds[h] = scale_of(nb, HV * ib + h);
            if constexpr (I8) {
                const sm_i32x2 w = sm_codes_i8<T, !F64>(rb_, ib, lq, skew, L.tab);
                Acc v[NV];
#pragma unroll
                for (int h = 0; h < HV; ++h) {
                    const bool mine = HV == 1 || (lq >> 1) == h;
                    const long B = __builtin_bit_cast(long, (sm_i32x2){mine ? w.x : 0, mine ? w.y : 0});
                    const sm_i32x4 D = __builtin_amdgcn_mfma_i32_16x16x32_i8(Ai, B, sm_i32x4{}, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < NV; ++i) {
                        if constexpr (F64) v[i] = h ? __builtin_fma((double)ds[h], (double)D[i], v[i])
                                                    : (double)ds[h] * (double)D[i];
                        else v[i] = h ? __builtin_fmaf(ds[h], (float)D[i], v[i]) : ds[h] * (float)D[i];
                    }
                }
#pragma unroll
                for (int i = 0; i < NV; ++i) {
                    if constexpr (sm_min(T)) v[i] = sm_fma(-(Acc)L.dm[wave][nb * BR + lr][ib], (Acc)sxv[i], v[i]);
                    if constexpr (F64) acc[nb][0][i] = __builtin_fma((double)xsv[i], v[i], acc[nb][0][i]);
                    else part[nb][0][i] = __builtin_fmaf(xsv[i], v[i], part[nb][0][i]);
                }
            } else {
                const u32x4 w = sm_codes_bf16<T>(rb_, ib, lq, skew, L.tab);
                float v[NV];
#pragma unroll
                for (int h = 0; h < HV; ++h) {
                    const bool mine = HV == 1 || (lq >> 1) == h;
                    const u32x4 wh = {mine ? w.x : 0, mine ? w.y : 0, mine ? w.z : 0, mine ? w.w : 0};
                    f32x4 D = mfma16x16x32(A[2], as_bf16x8(wh), f32x4{});
                    D = mfma16x16x32(A[1], as_bf16x8(wh), D);
                    D = mfma16x16x32(A[0], as_bf16x8(wh), D);
#pragma unroll
                    for (int i = 0; i < NV; ++i) {
                        if constexpr (HV == 2) v[i] = h ? __builtin_fmaf(D[i], ds[h], v[i]) : D[i] * ds[h];
                        else if constexpr (sm_min(T))
                            v[i] = __builtin_fmaf(-L.dm[wave][nb * BR + lr][ib], sxv[i], D[i] * ds[h]);
                        else part[nb][0][i] = __builtin_fmaf(D[i], ds[h], part[nb][0][i]);
                    }
                }
                if constexpr (HV == 2 || sm_min(T)) {
#pragma unroll
                    for (int i = 0; i < NV; ++i) part[nb][0][i] += v[i];
                }
            }
        }
    };
    // One 32-K block, 32 weight rows per MFMA.
    auto large_block = [&](int b, int ib, const uint8_t* brow, uint32_t skew) {
        constexpr int HV = sm_g16(T) ? 2 : 1;
        float ds[NK][HV];
#pragma unroll
        for (int nb = 0; nb < NK; ++nb)
#pragma unroll
            for (int h = 0; h < HV; ++h) ds[nb][h] = scale_of(nb, HV * ib + h);
        if constexpr (I8) {
            sm_i32x2 w[NK][2];
#pragma unroll
            for (int nb = 0; nb < NK; ++nb)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    w[nb][j] = sm_codes_i8<T, !F64>(brow + nb * BR * RS, ib, sm_g16(T) ? 2 * j + hh : 2 * hh + j, skew, L.tab);
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) {
                if (TB > 1 && tb >= ntb) continue;
                const uint8_t* ax = &L.x[kw][0][ta + 32 * tb][32 * b];
                float xsv[NV], sxv[NV];
                tokv(&L.xsc[kw][b][0], tb, xsv);
                if constexpr (sm_min(T)) tokv(&L.xsum[kw][b][0], tb, sxv);
#pragma unroll
                for (int nb = 0; nb < NK; ++nb) {
                    Acc v[NV];
#pragma unroll
                    for (int h = 0; h < HV; ++h) {
                        sm_i32x16 D;
                        if constexpr (HV == 2)
                            D = __builtin_amdgcn_mfma_i32_32x32x16_i8(
                                *reinterpret_cast<const long*>(ax + 16 * h + 8 * hh),
                                __builtin_bit_cast(long, w[nb][h]), sm_i32x16{}, 0, 0, 0);
                        else
                            D = __builtin_amdgcn_mfma_i32_32x32x32_i8(
                                *reinterpret_cast<const sm_i32x4*>(ax + 16 * hh),
                                (sm_i32x4){w[nb][0].x, w[nb][0].y, w[nb][1].x, w[nb][1].y}, sm_i32x16{}, 0, 0, 0);
#pragma unroll
                        for (int i = 0; i < NV; ++i) {
                            if constexpr (F64) v[i] = h ? __builtin_fma((double)ds[nb][h], (double)D[i], v[i])
                                                        : (double)ds[nb][h] * (double)D[i];
                            else v[i] = h ? __builtin_fmaf(ds[nb][h], (float)D[i], v[i]) : ds[nb][h] * (float)D[i];
                        }
                    }
                    float dmv = 0.0f;
                    if constexpr (sm_min(T)) dmv = L.dm[wave][nb * BR + lr][ib];
#pragma unroll
                    for (int i = 0; i < NV; ++i) {
                        if constexpr (sm_min(T)) v[i] = sm_fma(-(Acc)dmv, (Acc)sxv[i], v[i]);
                        if constexpr (F64) acc[nb][tb][i] = __builtin_fma((double)xsv[i], v[i], acc[nb][tb][i]);
                        else part[nb][tb][i] = __builtin_fmaf(xsv[i], v[i], part[nb][tb][i]);
                    }
                }
            }
        } else {
            u32x4 w[NK][2];
#pragma unroll
            for (int nb = 0; nb < NK; ++nb)
#pragma unroll
                for (int j = 0; j < 2; ++j) w[nb][j] = sm_codes_bf16<T>(brow + nb * BR * RS, ib, 2 * j + hh, skew, L.tab);
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) {
                if (TB > 1 && tb >= ntb) continue;
                bf16x8 A[3][2];
#pragma unroll
                for (int p = 0; p < 3; ++p)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        A[p][j] = as_bf16x8(*reinterpret_cast<const u32x4*>(
                            &L.x[kw][p % S::PL][ta + 32 * tb][64 * b + 32 * j + 16 * hh]));
                float sxv[NV];
                if constexpr (sm_min(T)) tokv(&L.xsum[kw][b][0], tb, sxv);
#pragma unroll
                for (int nb = 0; nb < NK; ++nb) {
                    float v[NV];
                    float dmv = 0.0f;
                    if constexpr (sm_min(T)) dmv = L.dm[wave][nb * BR + lr][ib];
#pragma unroll
                    for (int h = 0; h < HV; ++h) {
                        f32x16 D{};
#pragma unroll
                        for (int p = 2; p >= 0; --p)
#pragma unroll
                            for (int j = 0; j < 2; ++j)
                                if (HV == 1 || j == h) D = mfma32x32x16(A[p][j], as_bf16x8(w[nb][j]), D);
#pragma unroll
                        for (int i = 0; i < NV; ++i) {
                            if constexpr (HV == 2) v[i] = h ? __builtin_fmaf(D[i], ds[nb][h], v[i]) : D[i] * ds[nb][h];
                            else if constexpr (sm_min(T)) v[i] = __builtin_fmaf(-dmv, sxv[i], D[i] * ds[nb][h]);
                            else part[nb][tb][i] = __builtin_fmaf(D[i], ds[nb][h], part[nb][tb][i]);
                        }
                    }
                    if constexpr (HV == 2 || sm_min(T)) {
#pragma unroll
                        for (int i = 0; i < NV; ++i) part[nb][tb][i] += v[i];
                    }
                }
            }
        }
    };

    const int iters = (nch + KW - 1) / KW;
    // Chunks per inner sum: 256 K, 512 where one wave walks a long K (the two
    // levels then have about as many terms).
    const int FL = (KW == 1 && K > 4096 ? 512 : 256) / KC;
    load_x(min(kw, nch - 1) * KC);
    for (int it = 0; it < iters; ++it) {
        const int c = it * KW + kw;
        const bool on = KW == 1 || c < nch;      // uniform per wave
        const int cc = min(c, nch - 1), cn = min(c + KW, nch - 1);
        park_raw();
        const uint32_t skew = (uint32_t)(cc * sm_cb(T)) & 2u;   // the chunk starts at this byte of its LDS row
        const uint8_t* const brow = raw + lr * RS + skew;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if constexpr (T != kSmFp8) scales(raw + skew, cc);
        // 32-token tiles: one step of code, or the scheduler hoists several
        // steps' decodes and spills
#pragma unroll(NT == 32 && RW > 1 ? 1 : ST)
        for (int s = 0; s < ST; ++s) {
            if constexpr (RW == 1) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            else sm_barrier();
            park_x(s);
            // the order stays: split rows, next rows, next chunk
            __builtin_amdgcn_sched_barrier(0);
            if (s + 1 < ST) load_x(cc * KC + (s + 1) * KX);
            else load_x(cn * KC);
            __builtin_amdgcn_sched_barrier(0);
            // after the next step's activations: waiting for those (loads
            // complete in order) does not wait for the chunk
            if (s == 0) load_raw(cn);
            if constexpr (RW == 1) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            else sm_barrier();
            if (KW == 1 || on) {
#pragma unroll
                for (int b = 0; b < BX; ++b) {
                    const int ib = s * BX + b;
                    if constexpr (SM) small_block(b, ib, brow, skew);
                    else large_block(b, ib, brow, skew);
                }
            }
        }
        if (!F64 && ((it + 1) % FL == 0 || it + 1 == iters)) {
#pragma unroll
            for (int nb = 0; nb < NK; ++nb)
#pragma unroll
                for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                    for (int i = 0; i < NV; ++i) {
                        acc[nb][tb][i] += part[nb][tb][i];
                        part[nb][tb][i] = 0.0f;
                    }
        }
    }

    if constexpr (KW > 1) {
        // The shares' sums, added in pairs; the staging buffers are free by then.
        constexpr int AV = NK * TB * NV;
        static_assert(sizeof(Acc) * (KW - 1) * RW * AV * 64 <= sizeof(S) - offsetof(S, x),
                      "share sums fit the staging buffers");
        Acc* red = reinterpret_cast<Acc*>(&L.x[0][0][0][0]);
        sm_barrier();
        if (kw > 0) {
#pragma unroll
            for (int v = 0; v < AV; ++v)
                red[(((kw - 1) * RW + rw) * AV + v) * 64 + lane] =
                    acc[v / (TB * NV)][v / NV % TB][v % NV];
        }
        sm_barrier();
        if (kw > 0) return;
#pragma unroll
        for (int v = 0; v < AV; ++v) {
            Acc& o = acc[v / (TB * NV)][v / NV % TB][v % NV];
            Acc p[KW];
            p[0] = o;
#pragma unroll
            for (int q = 1; q < KW; ++q) p[q] = red[(((q - 1) * RW + rw) * AV + v) * 64 + lane];
#pragma unroll
            for (int h = 1; h < KW; h *= 2)
#pragma unroll
                for (int q = 0; q + h < KW; q += 2 * h) p[q] += p[q + h];
            o = p[0];
        }
    }

    // Stores: BR lanes write BR consecutive outputs of a token.
    constexpr Acc kOut = I8 ? 1.0f : 1.0f / kSmUp;
    float z = 0.0f;   // NaN once one of the lane's sums is not finite
#pragma unroll
    for (int tb = 0; tb < TB; ++tb)
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int t = SM ? lq * NV + i : 32 * tb + 8 * (i / 4) + 4 * hh + i % 4;
            if (t >= nr) continue;
            if constexpr (MODE == kSmGateUp) {
                if (f0 + 32 > a.out) continue;
#pragma unroll
                for (int nb = 0; nb < NK / 2; ++nb) {
                    const Acc g = acc[nb][tb][i] * kOut, u = acc[nb + NK / 2][tb][i] * kOut;
                    if constexpr (!I8) z = __builtin_fmaf(g, 0.0f, __builtin_fmaf(u, 0.0f, z));
                    float& h = a.y[(size_t)L.row[t] * a.out + f0 + nb * BR + lr];
                    if constexpr (F64) h = (float)(g / (1.0 + exp(-g)) * u);
                    else h = g / (1.0f + expf(-g)) * u;
                }
            } else {
                const size_t r = MODE == kSmDown ? (size_t)L.row[t] : (size_t)(t0 + t);
#pragma unroll
                for (int nb = 0; nb < NK; ++nb) {
                    const int o = f0 + nb * BR;
                    if (f0 + 32 * (nb * BR / 32) + 32 > a.out) continue;
                    float v = (float)(acc[nb][tb][i] * kOut);
                    if constexpr (!I8) z = __builtin_fmaf(v, 0.0f, z);
                    if constexpr (MODE == kSmDense) {
                        if constexpr (T == kSmFp8) v = a.sc ? v * a.sc[o + lr] : v;
                        if (a.bias) v += a.bias[o + lr];
                    }
                    a.y[r * a.out + o + lr] = v;
                }
            }
        }

    // Outputs that are not finite, from the dequantized weights instead: an infinite
    // activation meets zeroed codes (16-K scales), a zero remainder term or the
    // offset's sum as inf * 0 or inf - inf, and sums of codes overflow before their
    // scale brings them back. The rows concerned are found among the stored outputs
    // (a sum that is not finite gives no finite output): one register through the
    // stores. With the sums themselves kept for it the compiler spilled in the main
    // loop (Q4_K experts, 2048 x 512 x 64, top-4, 1000 tokens: 282 -> 343 us).
    // A row of x at a time, lane = weight row and half of K.
    if constexpr (!I8) {
        if (__builtin_expect(__ballot(z != z) != 0, 0)) {
            __threadfence_block();   // the stores above come first
            int ln = lane;
            asm volatile("" : "+v"(ln));   // nothing of this is kept in registers through the main loop
            const int half = ln >> 5;
            constexpr int NY = MODE == kSmGateUp ? 1 : NB;   // output blocks
#pragma unroll 1
            for (int t = 0; t < nr; ++t) {
                float* y = a.y + (MODE == kSmDense ? (size_t)(t0 + t) : (size_t)L.row[t]) * a.out + f0 + (ln & 31);
                float zt = 0.0f;
#pragma unroll
                for (int nb = 0; nb < NY; ++nb)
                    if (f0 + 32 * nb + 32 <= a.out) zt = __builtin_fmaf(y[32 * nb], 0.0f, zt);
                if (!__ballot(zt != zt)) continue;
                const float* xr = a.x + (size_t)L.src[t] * K;
                float o[NB];
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    const int r = ob[nb] + (ln & 31);
                    const uint8_t* w = wb[nb] + (ln & 31) * rb[nb];
                    double sum = 0.0;
#pragma unroll 1
                    for (int k = 8 * half; k < K; k += 16) {
                        float v[8];
                        sm_weights<T>(a, w, r, k, v);
#pragma unroll
                        for (int u = 0; u < 8; ++u) sum = __builtin_fma((double)v[u], (double)xr[k + u], sum);
                    }
                    sum += __shfl_xor(sum, 32);
                    if constexpr (T == kSmFp8) sum = a.sc ? sum * a.sc[r] : sum;
                    o[nb] = (float)sum;
                }
                if constexpr (MODE == kSmGateUp) o[0] = o[0] / (1.0f + expf(-o[0])) * o[1];
                if (!half) {
#pragma unroll
                    for (int nb = 0; nb < NY; ++nb)
                        if (f0 + 32 * nb + 32 <= a.out)
                            y[32 * nb] = MODE == kSmDense && a.bias ? o[nb] + a.bias[f0 + 32 * nb + ln] : o[nb];
                }
            }
        }
    }
}

}  // namespace glmmoe
