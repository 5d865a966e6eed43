// Decode of the GGUF block types (ggml block formats, src/gguf_quant.cpp:98-262)
// on the device: 8 consecutive elements of a row as floats (gg_dec8) or as
// integers with an affine pair (gg_dec8i).
#pragma once

#include "common.hpp"

namespace glmmoe {

// ggml's IQ3_XXS codebook (256 entries of 4 magnitudes, one byte each) and
// IQ4_NL values: format data, identical to the reference's tables
// (src/gguf_quant.cpp:53-90).
static __constant__ uint32_t c_iq3xxs_grid[256] = {
    0x04040404u, 0x04040414u, 0x04040424u, 0x04040c0cu, 0x04040c1cu, 0x04040c3eu, 0x04041404u, 0x04041414u,
    0x04041c0cu, 0x04042414u, 0x04043e1cu, 0x04043e2cu, 0x040c040cu, 0x040c041cu, 0x040c0c04u, 0x040c0c14u,
    0x040c140cu, 0x040c142cu, 0x040c1c04u, 0x040c1c14u, 0x040c240cu, 0x040c2c24u, 0x040c3e04u, 0x04140404u,
    0x04140414u, 0x04140424u, 0x04140c0cu, 0x04141404u, 0x04141414u, 0x04141c0cu, 0x04141c1cu, 0x04141c3eu,
    0x04142c0cu, 0x04142c3eu, 0x04143e2cu, 0x041c040cu, 0x041c043eu, 0x041c0c04u, 0x041c0c14u, 0x041c142cu,
    0x041c3e04u, 0x04240c1cu, 0x04241c3eu, 0x04242424u, 0x04242c3eu, 0x04243e1cu, 0x04243e2cu, 0x042c040cu,
    0x042c043eu, 0x042c1c14u, 0x042c2c14u, 0x04341c2cu, 0x04343424u, 0x043e0c04u, 0x043e0c24u, 0x043e0c34u,
    0x043e241cu, 0x043e340cu, 0x0c04040cu, 0x0c04041cu, 0x0c040c04u, 0x0c040c14u, 0x0c04140cu, 0x0c04141cu,
    0x0c041c04u, 0x0c041c14u, 0x0c041c24u, 0x0c04243eu, 0x0c042c04u, 0x0c0c0404u, 0x0c0c0414u, 0x0c0c0c0cu,
    0x0c0c1404u, 0x0c0c1414u, 0x0c14040cu, 0x0c14041cu, 0x0c140c04u, 0x0c140c14u, 0x0c14140cu, 0x0c141c04u,
    0x0c143e14u, 0x0c1c0404u, 0x0c1c0414u, 0x0c1c1404u, 0x0c1c1c0cu, 0x0c1c2434u, 0x0c1c3434u, 0x0c24040cu,
    0x0c24042cu, 0x0c242c04u, 0x0c2c1404u, 0x0c2c1424u, 0x0c2c2434u, 0x0c2c3e0cu, 0x0c34042cu, 0x0c3e1414u,
    0x0c3e2404u, 0x14040404u, 0x14040414u, 0x14040c0cu, 0x14040c1cu, 0x14041404u, 0x14041414u, 0x14041434u,
    0x14041c0cu, 0x14042414u, 0x140c040cu, 0x140c041cu, 0x140c042cu, 0x140c0c04u, 0x140c0c14u, 0x140c140cu,
    0x140c1c04u, 0x140c341cu, 0x140c343eu, 0x140c3e04u, 0x14140404u, 0x14140414u, 0x14140c0cu, 0x14140c3eu,
    0x14141404u, 0x14141414u, 0x14141c3eu, 0x14142404u, 0x14142c2cu, 0x141c040cu, 0x141c0c04u, 0x141c0c24u,
    0x141c3e04u, 0x141c3e24u, 0x14241c2cu, 0x14242c1cu, 0x142c041cu, 0x142c143eu, 0x142c240cu, 0x142c3e24u,
    0x143e040cu, 0x143e041cu, 0x143e0c34u, 0x143e242cu, 0x1c04040cu, 0x1c040c04u, 0x1c040c14u, 0x1c04140cu,
    0x1c04141cu, 0x1c042c04u, 0x1c04342cu, 0x1c043e14u, 0x1c0c0404u, 0x1c0c0414u, 0x1c0c1404u, 0x1c0c1c0cu,
    0x1c0c2424u, 0x1c0c2434u, 0x1c14040cu, 0x1c14041cu, 0x1c140c04u, 0x1c14142cu, 0x1c142c14u, 0x1c143e14u,
    0x1c1c0c0cu, 0x1c1c1c1cu, 0x1c241c04u, 0x1c24243eu, 0x1c243e14u, 0x1c2c0404u, 0x1c2c0434u, 0x1c2c1414u,
    0x1c2c2c2cu, 0x1c340c24u, 0x1c341c34u, 0x1c34341cu, 0x1c3e1c1cu, 0x1c3e3404u, 0x24040424u, 0x24040c3eu,
    0x24041c2cu, 0x24041c3eu, 0x24042c1cu, 0x24042c3eu, 0x240c3e24u, 0x24141404u, 0x24141c3eu, 0x24142404u,
    0x24143404u, 0x24143434u, 0x241c043eu, 0x241c242cu, 0x24240424u, 0x24242c0cu, 0x24243424u, 0x242c142cu,
    0x242c241cu, 0x242c3e04u, 0x243e042cu, 0x243e0c04u, 0x243e0c14u, 0x243e1c04u, 0x2c040c14u, 0x2c04240cu,
    0x2c043e04u, 0x2c0c0404u, 0x2c0c0434u, 0x2c0c1434u, 0x2c0c2c2cu, 0x2c140c24u, 0x2c141c14u, 0x2c143e14u,
    0x2c1c0414u, 0x2c1c2c1cu, 0x2c240c04u, 0x2c24141cu, 0x2c24143eu, 0x2c243e14u, 0x2c2c0414u, 0x2c2c1c0cu,
    0x2c342c04u, 0x2c3e1424u, 0x2c3e2414u, 0x34041424u, 0x34042424u, 0x34042434u, 0x34043424u, 0x340c140cu,
    0x340c340cu, 0x34140c3eu, 0x34143424u, 0x341c1c04u, 0x341c1c34u, 0x34242424u, 0x342c042cu, 0x342c2c14u,
    0x34341c1cu, 0x343e041cu, 0x343e140cu, 0x3e04041cu, 0x3e04042cu, 0x3e04043eu, 0x3e040c04u, 0x3e041c14u,
    0x3e042c14u, 0x3e0c1434u, 0x3e0c2404u, 0x3e140c14u, 0x3e14242cu, 0x3e142c14u, 0x3e1c0404u, 0x3e1c0c2cu,
    0x3e1c1c1cu, 0x3e1c3404u, 0x3e24140cu, 0x3e24240cu, 0x3e2c0404u, 0x3e2c0414u, 0x3e2c1424u, 0x3e341c04u,
};
constexpr int8_t kIq4nl[16] = {-127, -104, -83, -65, -49, -35, -22, -10,
                               1,    13,   25,  38,  53,  69,  89,  113};
constexpr uint32_t iq4nl_word(int i) {
    return (uint32_t)(uint8_t)kIq4nl[4 * i] | ((uint32_t)(uint8_t)kIq4nl[4 * i + 1] << 8) |
           ((uint32_t)(uint8_t)kIq4nl[4 * i + 2] << 16) | ((uint32_t)(uint8_t)kIq4nl[4 * i + 3] << 24);
}

// IQ4_NL values of four 4-bit codes (one per byte of `codes`), packed as int8:
// two byte selects (v_perm_b32) from the table held in four constant words.
__device__ __forceinline__ uint32_t gg_iq4nl4(uint32_t codes) {
    const uint32_t sel = codes & 0x07070707u;
    const uint32_t lo = __builtin_amdgcn_perm(iq4nl_word(1), iq4nl_word(0), sel);
    const uint32_t hi = __builtin_amdgcn_perm(iq4nl_word(3), iq4nl_word(2), sel);
    const uint32_t m = ((codes >> 3) & 0x01010101u) * 0xffu;
    return (lo & ~m) | (hi & m);
}

__device__ __forceinline__ float gg_f16(const uint8_t* p) {
    const uint16_t h = (uint16_t)(p[0] | (p[1] << 8));
    return (float)__builtin_bit_cast(_Float16, h);
}

__device__ __forceinline__ uint32_t gg_ld32(const uint8_t* p) {
    return (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) | ((uint32_t)p[3] << 24);
}

// The codes of IQ4_XS elements k .. k + 7 of a block (k % 8 == 0), one per byte.
__device__ __forceinline__ void gg_iq4xs_codes(const uint8_t* b, int ib, int c, uint32_t& c0,
                                               uint32_t& c1) {
    const uint8_t* q = b + 8 + 16 * ib + (c % 16);
    const int sh = 4 * (c / 16);
    c0 = (gg_ld32(q) >> sh) & 0x0f0f0f0fu;
    c1 = (gg_ld32(q + 4) >> sh) & 0x0f0f0f0fu;
}

// Elements k .. k + 7 (k % 8 == 0) of a row of GGUF type t; grid: the IQ3_XXS
// codebook (constant memory or an LDS copy).
__device__ __forceinline__ void gg_dec8_any(uint32_t t, const uint8_t* __restrict__ row, int k,
                                            const uint32_t* __restrict__ grid, float (&y)[8]) {
    switch (t) {
        case 0: {
            const float4* p = reinterpret_cast<const float4*>(row + 4 * (size_t)k);
            const float4 a = p[0], b = p[1];
            y[0] = a.x; y[1] = a.y; y[2] = a.z; y[3] = a.w;
            y[4] = b.x; y[5] = b.y; y[6] = b.z; y[7] = b.w;
            return;
        }
        case 1: {
#pragma unroll
            for (int j = 0; j < 8; ++j) y[j] = gg_f16(row + 2 * ((size_t)k + j));
            return;
        }
        case 8: {   // d, 32 x int8
            const uint8_t* b = row + (size_t)(k / 32) * 34;
            const int p = k % 32;
            const float d = gg_f16(b);
#pragma unroll
            for (int j = 0; j < 8; ++j) y[j] = d * (float)(int8_t)b[2 + p + j];
            return;
        }
        case 11: {  // hmask[32] q[64] scales[12] d
            const uint8_t* b = row + (size_t)(k / 256) * 110;
            const int p = k % 256, half = p / 128, r = p % 128, j = r / 32, sub = (r % 32) / 16;
            const int l0 = r % 16, i = 8 * half + 2 * j + sub;
            const int lo = (b[96 + i % 8] >> (4 * (i / 8))) & 15;
            const int hi = (b[104 + i % 4] >> (2 * (i / 4))) & 3;
            const int sc = (int)(int8_t)(uint8_t)(lo | (hi << 4));
            const float dl = gg_f16(b + 108) * (float)(sc - 32);
            const int hm = 1 << (4 * half + j);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int idx = 16 * sub + l0 + e;
                const int v = (b[32 + 32 * half + idx] >> (2 * j)) & 3;
                y[e] = dl * (float)(v - ((b[idx] & hm) ? 0 : 4));
            }
            return;
        }
        case 12:
        case 13: {  // d dmin scales[12] (qh[32]) q[128]
            const int bb = t == 12 ? 144 : 176;
            const uint8_t* b = row + (size_t)(k / 256) * bb;
            const int p = k % 256, c64 = p / 64, c = p % 64, l0 = c % 32, hi = c / 32;
            const int js = 2 * c64 + hi;
            const uint8_t* s = b + 4;
            int sc, mn;
            if (js < 4) {
                sc = s[js] & 63;
                mn = s[js + 4] & 63;
            } else {
                sc = (s[js + 4] & 15) | ((s[js - 4] >> 6) << 4);
                mn = (s[js + 4] >> 4) | ((s[js] >> 6) << 4);
            }
            const float d1 = gg_f16(b) * (float)sc, m1 = gg_f16(b + 2) * (float)mn;
            const uint8_t* q = b + (t == 12 ? 16 : 48);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                int v = (q[32 * c64 + l0 + e] >> (4 * hi)) & 15;
                if (t == 13) v += (b[16 + l0 + e] & (1 << js)) ? 16 : 0;
                y[e] = d1 * (float)v - m1;
            }
            return;
        }
        case 14: {  // ql[128] qh[64] scales[16] d
            const uint8_t* b = row + (size_t)(k / 256) * 210;
            const int p = k % 256, nn = p / 128, r = p % 128, quarter = r / 32, l0 = r % 32;
            const uint8_t* ql = b + 64 * nn + 32 * (quarter & 1);
            const uint8_t* qh = b + 128 + 32 * nn;
            const float dsc = gg_f16(b + 208) * (float)(int8_t)b[192 + 8 * nn + l0 / 16 + 2 * quarter];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int lo = (ql[l0 + e] >> (4 * (quarter >> 1))) & 15;
                const int q6 = (int)(int8_t)(uint8_t)(lo | (((qh[l0 + e] >> (2 * quarter)) & 3) << 4)) - 32;
                y[e] = dsc * (float)q6;
            }
            return;
        }
        case 18: {  // d qs[64] signs+scales[32]
            const uint8_t* b = row + (size_t)(k / 256) * 98;
            const int p = k % 256, ib = p / 32, l = (p % 32) / 8;
            const uint8_t* w = b + 66 + 4 * ib;
            const uint32_t aux = (uint32_t)w[0] | ((uint32_t)w[1] << 8) | ((uint32_t)w[2] << 16) |
                                 ((uint32_t)w[3] << 24);
            const float db = gg_f16(b) * (0.5f + (float)(aux >> 28)) * 0.5f;
            const uint32_t i7 = (aux >> (7 * l)) & 127u;
            const uint32_t signs = i7 | ((uint32_t)(__builtin_popcount(i7) & 1) << 7);
            const uint32_t g0 = grid[b[2 + 8 * ib + 2 * l]];
            const uint32_t g1 = grid[b[2 + 8 * ib + 2 * l + 1]];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float mag = (float)(((e < 4 ? g0 : g1) >> (8 * (e & 3))) & 255u);
                y[e] = db * mag * ((signs & (1u << e)) ? -1.0f : 1.0f);
            }
            return;
        }
        case 23: {  // d scales_h scales_l[4] qs[128]
            const uint8_t* b = row + (size_t)(k / 256) * 136;
            const int p = k % 256, ib = p / 32, c = p % 32;
            const int sh = b[2] | (b[3] << 8);
            const int lo = (b[4 + ib / 2] >> (4 * (ib & 1))) & 15;
            const int hi = (sh >> (2 * ib)) & 3;
            const float dl = gg_f16(b) * (float)((int)(int8_t)(uint8_t)(lo | (hi << 4)) - 32);
            uint32_t c0, c1;
            gg_iq4xs_codes(b, ib, c, c0, c1);
            const uint32_t v0 = gg_iq4nl4(c0), v1 = gg_iq4nl4(c1);
#pragma unroll
            for (int e = 0; e < 8; ++e)
                y[e] = dl * (float)(int8_t)(((e < 4 ? v0 : v1) >> (8 * (e & 3))) & 255u);
            return;
        }
        default:
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = 0.0f;
    }
}

// The type as a compile-time constant (one decode body per kernel
// instantiation); kGgAny decodes by a runtime switch on t.
constexpr uint32_t kGgAny = 0xffffffffu;
template <uint32_t T>
__device__ __forceinline__ void gg_dec8(uint32_t t, const uint8_t* __restrict__ row, int k,
                                        const uint32_t* __restrict__ grid, float (&y)[8]) {
    gg_dec8_any(T == kGgAny ? t : T, row, k, grid, y);
}

// ---- int8 activations (gemm_q_i8 / moe_expert_ffn_q_i8, cuda/qgemm.cu:104-303,
// 556-587). Weights k .. k + 7 as integers with one affine pair,
// weight[j] = ds * wq[j] - dm (dm != 0 for Q4_K / Q5_K only), packed four
// per int32 for v_dot4c_i32_i8. The same bits give exactly the decode above.
__device__ __forceinline__ int gg_pk4(int a, int b, int c, int d) {
    return (a & 255) | ((b & 255) << 8) | ((c & 255) << 16) | (int)((unsigned)d << 24);
}


// A2: every 2- and 4-byte field is read as 16-bit halves (the caller's rows
// are 2-byte aligned, as in the LDS copies; block sizes are even); otherwise
// byte by byte.
template <bool A2>
__device__ __forceinline__ uint32_t gg_rd32(const uint8_t* p) {
    if constexpr (A2) {
        const uint16_t* h = reinterpret_cast<const uint16_t*>(p);
        return (uint32_t)h[0] | ((uint32_t)h[1] << 16);
    } else {
        return gg_ld32(p);
    }
}
template <bool A2>
__device__ __forceinline__ float gg_rdf16(const uint8_t* p) {
    if constexpr (A2)
        return (float)__builtin_bit_cast(_Float16, *reinterpret_cast<const uint16_t*>(p));
    else
        return gg_f16(p);
}

// Byte i of the result is 0xff where bit i of s (i < 4) is set.
__device__ __forceinline__ uint32_t gg_bytemask4(uint32_t s) {
    return (((s & 15u) * 0x00204081u) & 0x01010101u) * 0xffu;
}

// sgn (used with A2): the IQ3_XXS sign byte masks of the 128 7-bit patterns,
// two words per pattern (the LDS table of gg_dots_stream).
template <bool A2>
__device__ __forceinline__ void gg_dec8i_any(uint32_t t, const uint8_t* __restrict__ row, int k,
                                             const uint32_t* __restrict__ grid,
                                             const uint32_t* __restrict__ sgn, int& w0, int& w1,
                                             float& ds, float& dm) {
    dm = 0.0f;
    switch (t) {
        case 8: {
            const uint8_t* b = row + (size_t)(k / 32) * 34;
            ds = gg_rdf16<A2>(b);
            w0 = (int)gg_rd32<A2>(b + 2 + k % 32);
            w1 = (int)gg_rd32<A2>(b + 6 + k % 32);
            return;
        }
        case 11: {
            const uint8_t* b = row + (size_t)(k / 256) * 110;
            const int p = k % 256, half = p / 128, r = p % 128, j = r / 32, sub = (r % 32) / 16;
            const int l0 = r % 16, i = 8 * half + 2 * j + sub;
            const int lo = (b[96 + i % 8] >> (4 * (i / 8))) & 15;
            const int hi = (b[104 + i % 4] >> (2 * (i / 4))) & 3;
            ds = gg_rdf16<A2>(b + 108) * (float)((int)(int8_t)(uint8_t)(lo | (hi << 4)) - 32);
            const int idx = 16 * sub + l0, hb = 4 * half + j;
            // q - (hmask bit ? 0 : 4) per byte, q in 0..3: biased by 0x80 so no
            // byte borrows from its neighbour
            const uint32_t q0 = (gg_rd32<A2>(b + 32 + 32 * half + idx) >> (2 * j)) & 0x03030303u;
            const uint32_t q1 = (gg_rd32<A2>(b + 36 + 32 * half + idx) >> (2 * j)) & 0x03030303u;
            const uint32_t m0 = ((gg_rd32<A2>(b + idx) >> hb) & 0x01010101u) ^ 0x01010101u;
            const uint32_t m1 = ((gg_rd32<A2>(b + idx + 4) >> hb) & 0x01010101u) ^ 0x01010101u;
            w0 = (int)(((q0 | 0x80808080u) - (m0 << 2)) ^ 0x80808080u);
            w1 = (int)(((q1 | 0x80808080u) - (m1 << 2)) ^ 0x80808080u);
            return;
        }
        case 12:
        case 13: {
            const int bb = t == 12 ? 144 : 176;
            const uint8_t* b = row + (size_t)(k / 256) * bb;
            const int p = k % 256, c64 = p / 64, c = p % 64, l0 = c % 32, hi = c / 32;
            const int js = 2 * c64 + hi;
            const uint8_t* s = b + 4;
            int sc, mn;
            if (js < 4) {
                sc = s[js] & 63;
                mn = s[js + 4] & 63;
            } else {
                sc = (s[js + 4] & 15) | ((s[js - 4] >> 6) << 4);
                mn = (s[js + 4] >> 4) | ((s[js] >> 6) << 4);
            }
            ds = gg_rdf16<A2>(b) * (float)sc;
            dm = gg_rdf16<A2>(b + 2) * (float)mn;
            const uint8_t* q = b + (t == 12 ? 16 : 48) + 32 * c64 + l0;
            uint32_t a0 = (gg_rd32<A2>(q) >> (4 * hi)) & 0x0f0f0f0fu;
            uint32_t a1 = (gg_rd32<A2>(q + 4) >> (4 * hi)) & 0x0f0f0f0fu;
            if (t == 13) {
                a0 |= ((gg_rd32<A2>(b + 16 + l0) >> js) & 0x01010101u) << 4;
                a1 |= ((gg_rd32<A2>(b + 20 + l0) >> js) & 0x01010101u) << 4;
            }
            w0 = (int)a0;
            w1 = (int)a1;
            return;
        }
        case 14: {
            const uint8_t* b = row + (size_t)(k / 256) * 210;
            const int p = k % 256, nn = p / 128, r = p % 128, quarter = r / 32, l0 = r % 32;
            const uint8_t* ql = b + 64 * nn + 32 * (quarter & 1) + l0;
            const uint8_t* qh = b + 128 + 32 * nn + l0;
            ds = gg_rdf16<A2>(b + 208) * (float)(int8_t)b[192 + 8 * nn + l0 / 16 + 2 * quarter];
            const int sl = 4 * (quarter >> 1), sh = 2 * quarter;
            // q6 - 32 per byte: (lo | hi << 4) in 0..63, minus 32 by a bytewise
            // subtract with no borrow across bytes (each byte >= 0, result -32..31).
            const uint32_t u0 = ((gg_rd32<A2>(ql) >> sl) & 0x0f0f0f0fu) |
                                (((gg_rd32<A2>(qh) >> sh) & 0x03030303u) << 4);
            const uint32_t u1 = ((gg_rd32<A2>(ql + 4) >> sl) & 0x0f0f0f0fu) |
                                (((gg_rd32<A2>(qh + 4) >> sh) & 0x03030303u) << 4);
            w0 = (int)((u0 | 0x80808080u) - 0x20202020u) ^ (int)0x80808080u;
            w1 = (int)((u1 | 0x80808080u) - 0x20202020u) ^ (int)0x80808080u;
            return;
        }
        case 18: {
            const uint8_t* b = row + (size_t)(k / 256) * 98;
            const int p = k % 256, ib = p / 32, l = (p % 32) / 8;
            const uint32_t aux = gg_rd32<A2>(b + 66 + 4 * ib);
            ds = gg_rdf16<A2>(b) * (0.5f + (float)(aux >> 28)) * 0.5f;
            const uint32_t i7 = (aux >> (7 * l)) & 127u;
            uint32_t n0, n1;
            if constexpr (A2) {
                const uint2 m = *reinterpret_cast<const uint2*>(sgn + 2 * i7);
                n0 = m.x;
                n1 = m.y;
            } else {
                const uint32_t signs = i7 | ((uint32_t)(__builtin_popcount(i7) & 1) << 7);
                n0 = gg_bytemask4(signs);
                n1 = gg_bytemask4(signs >> 4);
            }
            const uint32_t qs = A2 ? *reinterpret_cast<const uint16_t*>(b + 2 + 8 * ib + 2 * l)
                                   : (uint32_t)(b[2 + 8 * ib + 2 * l] | (b[3 + 8 * ib + 2 * l] << 8));
            const uint32_t g0 = grid[qs & 255u], g1 = grid[qs >> 8];
            // negate the flagged bytes: (g ^ 0xff) + 1 per byte, with no carry
            // out of a byte since every grid magnitude is at least 4
            w0 = (int)((g0 ^ n0) + (n0 & 0x01010101u));
            w1 = (int)((g1 ^ n1) + (n1 & 0x01010101u));
            return;
        }
        case 23: {
            const uint8_t* b = row + (size_t)(k / 256) * 136;
            const int p = k % 256, ib = p / 32, c = p % 32;
            const int sh = A2 ? *reinterpret_cast<const uint16_t*>(b + 2) : (b[2] | (b[3] << 8));
            const int lo = (b[4 + ib / 2] >> (4 * (ib & 1))) & 15;
            const int hi = (sh >> (2 * ib)) & 3;
            ds = gg_rdf16<A2>(b) * (float)((int)(int8_t)(uint8_t)(lo | (hi << 4)) - 32);
            const uint8_t* q = b + 8 + 16 * ib + (c % 16);
            const int shq = 4 * (c / 16);
            w0 = (int)gg_iq4nl4((gg_rd32<A2>(q) >> shq) & 0x0f0f0f0fu);
            w1 = (int)gg_iq4nl4((gg_rd32<A2>(q + 4) >> shq) & 0x0f0f0f0fu);
            return;
        }
        default:
            ds = 0.0f;
            w0 = w1 = 0;
            return;
    }
}

template <uint32_t T, bool A2 = false>
__device__ __forceinline__ void gg_dec8i(uint32_t t, const uint8_t* __restrict__ row, int k,
                                         const uint32_t* __restrict__ grid,
                                         const uint32_t* __restrict__ sgn, int& w0, int& w1,
                                         float& ds, float& dm) {
    gg_dec8i_any<A2>(T == kGgAny ? t : T, row, k, grid, sgn, w0, w1, ds, dm);
}

constexpr int gg_be(uint32_t t) { return t == 8 ? 32 : 256; }
constexpr int gg_bb(uint32_t t) {
    return t == 8 ? 34 : t == 11 ? 110 : t == 12 ? 144 : t == 13 ? 176 : t == 14 ? 210
         : t == 18 ? 98 : t == 23 ? 136 : 0;
}

}  // namespace glmmoe
