// GGUF block-quantized weights (ggml block formats) on the reference's
// launcher signatures:
//   gg_gemv_kernel      gemm_q (cuda/kernels.cuh:63-66): y[n,out] = x[n,in] . W^T (+ bias),
//                       W [out, in] rows of GGUF blocks at qW + o * row_bytes.
//   gg_moe_kernel       moe_expert_ffn_q (cuda/kernels.cuh:117-123, cuda/qgemm.cu:1505-1639):
//                       gate/up rows [E, moe_inter, hidden], down [E, hidden, moe_inter],
//                       row o of expert e at base + (e * out + o) * row_bytes.
//                       Phase 1: h_act[r, f] = silu(gate_e[f] . x_t) * (up_e[f] . x_t) for
//                       every routed row r = t * topk + s; phase 2: dpart[r, o] =
//                       down_e[o] . h_act[r]; then out[t] = sum_s w[t, s] * dpart[t*topk+s]
//                       in slot order (the reference's fixed-order reduce,
//                       cuda/qgemm.cu:943-955).
// Element decode restates src/gguf_quant.cpp:98-262 per 8 consecutive elements
// with the same float operations in the same order, so the dequantized
// weights equal the reference's bit for bit; products and sums are fp32.
//
// Aligned shapes of whole K chunks go to the matrix cores (splitmm.hpp, see
// gg_gemm and gg_sm_tile); the kernels here take the rest.
// Work: a workgroup (4 waves) owns 16 output rows (4 per wave) and a tile of
// up to 8 input rows. With the caller's `dispatch` scratch the routed rows are
// first grouped by expert (counting pass, one workgroup), so a tile holds up
// to 8 rows of one expert and each weight row is read once per tile; without
// it every routed row is a tile of its own (the reference's token-major path).
// K is walked in chunks: the tile's input rows of a chunk are staged in LDS
// (shared by the waves); each lane takes 8 consecutive K of the wave's weight
// rows and accumulates 8-element dot products; lane partials are added by a
// fixed xor butterfly. For the block types with dword-aligned rows the weight
// bytes are streamed one chunk ahead (gg_dots_stream); otherwise each lane
// reads its blocks' bytes directly (gg_dots / gg_dots_i8).
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "gguf_dec.hpp"
#include "kernels.hpp"
#include "splitmm.hpp"

namespace glmmoe {

int gguf_block_elems(uint32_t t) {
    switch (t) {
        case 0: case 1: return 1;
        case 8: return 32;
        case 11: case 12: case 13: case 14: case 18: case 23: return 256;
        default: return 0;
    }
}

int gguf_block_bytes(uint32_t t) {
    switch (t) {
        case 0: return 4;
        case 1: return 2;
        case 8: return 34;
        case 11: return 110;
        case 12: return 144;
        case 13: return 176;
        case 14: return 210;
        case 18: return 98;
        case 23: return 136;
        default: return 0;
    }
}

constexpr int kGgWaves = 4;                // waves per workgroup
constexpr int kGgThreads = 64 * kGgWaves;
constexpr int kGgRows = 4 * kGgWaves;      // weight rows per workgroup (4 per wave)
constexpr int kGgKC = 512;    // K per staged chunk
// Input rows per tile (TT): 8 for prefill-sized groups, fewer when an expert
// holds a row or a few (decode), so no FMAs go to empty rows.

__device__ __forceinline__ float gg_wave_sum(float v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m);
    return v;
}

__device__ __forceinline__ float gg_silu(float v) { return v / (1.0f + expf(-v)); }

// The input rows of a tile (up to TT, indices into src) and its expert.
template <int TT>
struct GgTile {
    int e, nr;
    int row[TT];    // output row index (routed row r, or the token for gemm_q)
    int src[TT];    // input row index into src
};

// Stages rows srcs[0..nr) x [k0, k0 + kc) of a [*, K] fp32 matrix into xs
// (srcs: the tile's input rows, in LDS so that they index dynamically).
template <int TT>
__device__ __forceinline__ void gg_stage(float (*xs)[kGgKC], const float* __restrict__ src, int K,
                                         const int* srcs, int nr, int k0, int kc) {
    for (int i = threadIdx.x; i < TT * (kGgKC / 4); i += blockDim.x) {
        const int t = i / (kGgKC / 4), c4 = i % (kGgKC / 4);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (t < nr && 4 * c4 < kc)
            v = *reinterpret_cast<const float4*>(src + (size_t)srcs[t] * K + k0 + 4 * c4);
        *reinterpret_cast<float4*>(&xs[t][4 * c4]) = v;
    }
}

// Dot products of NM weight matrices' rows o0 .. o0 + 3 with the tile's input
// rows over K: acc[m][r][t].
template <uint32_t T, int NM, int TT>
__device__ __forceinline__ void gg_dots(float (*xs)[kGgKC], int* srcs, const float* __restrict__ src,
                                        int K, const GgTile<TT>& tl, const uint32_t (&type)[NM],
                                        const uint8_t* const (&wrow)[NM][4],
                                        float (&acc)[NM][4][TT]) {
    const int lane = threadIdx.x & 63;
    __syncthreads();   // srcs and xs of a previous tile are consumed
    if (threadIdx.x == 0) {
#pragma unroll
        for (int t = 0; t < TT; ++t) srcs[t] = tl.src[t];
    }
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int t = 0; t < TT; ++t) acc[m][r][t] = 0.0f;
    for (int k0 = 0; k0 < K; k0 += kGgKC) {
        const int kc = min(kGgKC, K - k0);
        __syncthreads();
        gg_stage<TT>(xs, src, K, srcs, tl.nr, k0, kc);
        __syncthreads();
        const int kk = lane * 8;
        if (kk >= kc) continue;
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float w[8];
                gg_dec8<T>(type[m], wrow[m][r], k0 + kk, c_iq3xxs_grid, w);
#pragma unroll
                for (int j = 0; j < 8; ++j)
#pragma unroll
                    for (int t = 0; t < TT; ++t)
                        acc[m][r][t] = __builtin_fmaf(w[j], xs[t][kk + j], acc[m][r][t]);
            }
    }
}

// LDS tile of int8 activations: TT rows x kGgKC bytes and their per-32 scales.
template <int TT>
struct GgI8Tile {
    int q[TT][kGgKC / 4];
    float s[TT][kGgKC / 32];
};

// The int8 twin of gg_dots: xq [*, K] int8 and xsc [*, K / 32] scales; per
// 8-element fragment r = ds * dot(wq, xq) - dm * sum(xq), acc += sx * r.
template <uint32_t T, int NM, int TT>
__device__ __forceinline__ void gg_dots_i8(GgI8Tile<TT>& xt, int* srcs, const int8_t* __restrict__ xq,
                                           const float* __restrict__ xsc, int K,
                                           const GgTile<TT>& tl, const uint32_t (&type)[NM],
                                           const uint8_t* const (&wrow)[NM][4],
                                           float (&acc)[NM][4][TT]) {
    const int lane = threadIdx.x & 63;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int t = 0; t < TT; ++t) srcs[t] = tl.src[t];
    }
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int t = 0; t < TT; ++t) acc[m][r][t] = 0.0f;
    const int K32 = K / 32;
    for (int k0 = 0; k0 < K; k0 += kGgKC) {
        const int kc = min(kGgKC, K - k0);
        __syncthreads();
        for (int i = threadIdx.x; i < TT * (kGgKC / 4); i += blockDim.x) {
            const int t = i / (kGgKC / 4), c = i % (kGgKC / 4);
            int v = 0;
            if (t < tl.nr && 4 * c < kc)
                v = *reinterpret_cast<const int*>(xq + (size_t)srcs[t] * K + k0 + 4 * c);
            xt.q[t][c] = v;
        }
        for (int i = threadIdx.x; i < TT * (kGgKC / 32); i += blockDim.x) {
            const int t = i / (kGgKC / 32), c = i % (kGgKC / 32);
            xt.s[t][c] = (t < tl.nr && 32 * c < kc) ? xsc[(size_t)srcs[t] * K32 + k0 / 32 + c] : 0.0f;
        }
        __syncthreads();
        const int kk = lane * 8;
        if (kk >= kc) continue;
        int x0[TT], x1[TT], sx1[TT];
        float sx[TT];
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const int2 q = *reinterpret_cast<const int2*>(&xt.q[t][kk / 4]);
            x0[t] = q.x;
            x1[t] = q.y;
            sx[t] = xt.s[t][kk / 32];
            sx1[t] = __builtin_amdgcn_sdot4(0x01010101, q.y, __builtin_amdgcn_sdot4(0x01010101, q.x, 0, false), false);
        }
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int w0, w1;
                float ds, dm;
                gg_dec8i<T>(type[m], wrow[m][r], k0 + kk, c_iq3xxs_grid, nullptr, w0, w1, ds, dm);
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    const int si = __builtin_amdgcn_sdot4(w1, x1[t], __builtin_amdgcn_sdot4(w0, x0[t], 0, false), false);
                    float v = ds * (float)si;
                    if (T == 12 || T == 13 || (T == kGgAny && dm != 0.0f)) v = v - dm * (float)sx1[t];
                    acc[m][r][t] = __builtin_fmaf(sx[t], v, acc[m][r][t]);
                }
            }
    }
}

// ---- Streamed weights (the block types, one type per matrix set). Each wave
// owns 4 weight rows per matrix; per K chunk it loads those rows' block bytes
// with coalesced dword loads (lane l: dwords l, l + 64, ...) one chunk ahead
// into registers, parks them in a private LDS buffer and decodes from there,
// so every weight byte is one wide load and a chunk is in flight while the
// previous one is decoded. The tile's activations are staged the same way
// (shared by the four waves, one barrier per chunk).
// K per chunk: at most 3 dwords per lane per row, and 512 for 8-row tiles (LDS).
// Lane l always takes K elements 512 f + 8 l of each 512, so the sums do not
// depend on the chunk size.
constexpr int gg_kc(uint32_t t, int tt) { return (t == 8 || t == 14 || tt > 1) ? 512 : 1024; }
constexpr bool gg_streamed(uint32_t t) { return gg_bb(t) != 0; }

template <uint32_t T, int NM, int TT, bool I8>
struct GgStream {
    static constexpr int KC = gg_kc(T, TT);
    static constexpr int CB = KC / gg_be(T) * gg_bb(T);   // bytes of a row's chunk
    static constexpr int ND = CB / 4;
    static constexpr int LPR = (ND + 63) / 64;            // dword loads per lane per row
    static constexpr int XV = I8 ? TT * KC / 4 : TT * KC / 4;   // int / float4 items of x
    static constexpr int XR = (XV + kGgThreads - 1) / kGgThreads;   // per thread
    static constexpr int SR = TT * KC / 32;               // scales (I8)
    uint32_t w[2][kGgWaves][NM * 4][ND];
    uint32_t grid[T == 18 ? 256 : 1];   // the IQ3_XXS codebook
    uint32_t sgn[T == 18 ? 256 : 1];    // IQ3_XXS: byte masks of the 128 sign patterns
    float x[I8 ? 1 : 2][I8 ? 1 : TT][I8 ? 4 : KC];
    struct {
        int q[I8 ? 2 : 1][I8 ? TT : 1][I8 ? KC / 4 : 1];
        float s[I8 ? 2 : 1][I8 ? TT : 1][I8 ? KC / 32 : 1];
    } i8;
};

template <uint32_t T, int NM, int TT, bool I8>
__device__ __forceinline__ void gg_dots_stream(GgStream<T, NM, TT, I8>& L, int* srcs,
                                               const float* __restrict__ x,
                                               const int8_t* __restrict__ xq,
                                               const float* __restrict__ xsc, int K,
                                               const GgTile<TT>& tl,
                                               const uint8_t* const (&wrow)[NM][4],
                                               float (&acc)[NM][4][TT]) {
    using S = GgStream<T, NM, TT, I8>;
    constexpr int KC = S::KC, ND = S::ND, LPR = S::LPR, XR = S::XR;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tid = threadIdx.x;
    __syncthreads();   // srcs and the buffers of a previous tile are consumed
    if (tid == 0) {
#pragma unroll
        for (int t = 0; t < TT; ++t) srcs[t] = tl.src[t];
    }
    if constexpr (T == 18) {
        if (tid < 256) {
            L.grid[tid] = c_iq3xxs_grid[tid];
            // pattern e: 7 sign bits plus their parity bit, as 8 byte masks
            const uint32_t e = (uint32_t)tid >> 1;
            const uint32_t sg = e | ((uint32_t)(__builtin_popcount(e) & 1) << 7);
            L.sgn[tid] = gg_bytemask4(sg >> (4 * (tid & 1)));
        }
    }
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int t = 0; t < TT; ++t) acc[m][r][t] = 0.0f;
    __syncthreads();
    const int nch = (K + KC - 1) / KC;
    const int rowb = K / gg_be(T) * gg_bb(T);   // block bytes of a whole row
    uint32_t wr[NM * 4][LPR];
    float4 xr[XR];
    int qr[XR];
    float sr = 0.0f;
    auto load = [&](int c) {
        const int k0 = c * KC, kc = min(KC, K - k0);
        const int nd = min(ND, (rowb - c * S::CB) / 4);
#pragma unroll
        for (int i = 0; i < NM * 4; ++i)
#pragma unroll
            for (int j = 0; j < LPR; ++j) {
                const int d = j * 64 + lane;
                if (d < nd)
                    wr[i][j] = *reinterpret_cast<const uint32_t*>(wrow[i / 4][i % 4] +
                                                                  (size_t)c * S::CB + 4 * d);
            }
#pragma unroll
        for (int j = 0; j < XR; ++j) {
            const int v = tid + kGgThreads * j;
            const int t = v / (KC / 4), c4 = v % (KC / 4);
            if (v < S::XV && t < tl.nr && 4 * c4 < kc) {
                if constexpr (I8)
                    qr[j] = *reinterpret_cast<const int*>(xq + (size_t)srcs[t] * K + k0 + 4 * c4);
                else
                    xr[j] = *reinterpret_cast<const float4*>(x + (size_t)srcs[t] * K + k0 + 4 * c4);
            }
        }
        if constexpr (I8) {
            if (tid < S::SR) {
                const int t = tid / (KC / 32), c32 = tid % (KC / 32);
                sr = (t < tl.nr && 32 * c32 < kc)
                         ? xsc[(size_t)srcs[t] * (K / 32) + k0 / 32 + c32] : 0.0f;
            }
        }
    };
    auto park = [&](int b, int c) {
        const int k0 = c * KC, kc = min(KC, K - k0);
        const int nd = min(ND, (rowb - c * S::CB) / 4);
#pragma unroll
        for (int i = 0; i < NM * 4; ++i)
#pragma unroll
            for (int j = 0; j < LPR; ++j) {
                const int d = j * 64 + lane;
                if (d < nd) L.w[b][wave][i][d] = wr[i][j];
            }
#pragma unroll
        for (int j = 0; j < XR; ++j) {
            const int v = tid + kGgThreads * j;
            const int t = v / (KC / 4), c4 = v % (KC / 4);
            if (v < S::XV) {
                const bool ok = t < tl.nr && 4 * c4 < kc;
                if constexpr (I8)
                    L.i8.q[b][t][c4] = ok ? qr[j] : 0;
                else
                    *reinterpret_cast<float4*>(&L.x[b][t][4 * c4]) =
                        ok ? xr[j] : make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
        if constexpr (I8) {
            if (tid < S::SR) L.i8.s[b][tid / (KC / 32)][tid % (KC / 32)] = sr;
        }
    };
    load(0);
    park(0, 0);
    __syncthreads();
    for (int c = 0; c < nch; ++c) {
        const int b = c & 1;
        if (c + 1 < nch) load(c + 1);
        const int kc = min(KC, K - c * KC);
#pragma unroll
        for (int f = 0; f < KC / 512; ++f) {
            const int kk = f * 512 + lane * 8;
            if (kk < kc) {
                if constexpr (I8) {
                    int x0[TT], x1[TT], sx1[TT];
                    float sx[TT];
#pragma unroll
                    for (int t = 0; t < TT; ++t) {
                        const int2 q = *reinterpret_cast<const int2*>(&L.i8.q[b][t][kk / 4]);
                        x0[t] = q.x;
                        x1[t] = q.y;
                        sx[t] = L.i8.s[b][t][kk / 32];
                        sx1[t] = __builtin_amdgcn_sdot4(
                            0x01010101, q.y, __builtin_amdgcn_sdot4(0x01010101, q.x, 0, false),
                            false);
                    }
#pragma unroll
                    for (int i = 0; i < NM * 4; ++i) {
                        int w0, w1;
                        float ds, dm;
                        gg_dec8i<T, true>(T, reinterpret_cast<const uint8_t*>(L.w[b][wave][i]),
                                          kk, L.grid, L.sgn, w0, w1, ds, dm);
#pragma unroll
                        for (int t = 0; t < TT; ++t) {
                            const int si = __builtin_amdgcn_sdot4(
                                w1, x1[t], __builtin_amdgcn_sdot4(w0, x0[t], 0, false), false);
                            float v = ds * (float)si;
                            if (T == 12 || T == 13) v = v - dm * (float)sx1[t];
                            acc[i / 4][i % 4][t] = __builtin_fmaf(sx[t], v, acc[i / 4][i % 4][t]);
                        }
                    }
                } else {
                    // The integer fragment (weight = ds * wq - dm, the reference's
                    // dequantized value exactly), then
                    // acc += ds * sum(wq * x) - dm * sum(x).
                    float xv[TT][8], sx[TT];
#pragma unroll
                    for (int t = 0; t < TT; ++t) {
                        const float4 a = *reinterpret_cast<const float4*>(&L.x[b][t][kk]);
                        const float4 e = *reinterpret_cast<const float4*>(&L.x[b][t][kk + 4]);
                        xv[t][0] = a.x; xv[t][1] = a.y; xv[t][2] = a.z; xv[t][3] = a.w;
                        xv[t][4] = e.x; xv[t][5] = e.y; xv[t][6] = e.z; xv[t][7] = e.w;
                        if (T == 12 || T == 13) {
                            float v = xv[t][0];
#pragma unroll
                            for (int j = 1; j < 8; ++j) v = v + xv[t][j];
                            sx[t] = v;
                        }
                    }
#pragma unroll
                    for (int i = 0; i < NM * 4; ++i) {
                        int w0, w1;
                        float ds, dm;
                        gg_dec8i<T, true>(T, reinterpret_cast<const uint8_t*>(L.w[b][wave][i]),
                                          kk, L.grid, L.sgn, w0, w1, ds, dm);
                        float wf[8];
#pragma unroll
                        for (int j = 0; j < 8; ++j)
                            wf[j] = (float)(int8_t)((uint32_t)(j < 4 ? w0 : w1) >> (8 * (j & 3)));
#pragma unroll
                        for (int t = 0; t < TT; ++t) {
                            float v = wf[0] * xv[t][0];
#pragma unroll
                            for (int j = 1; j < 8; ++j) v = __builtin_fmaf(wf[j], xv[t][j], v);
                            float& ac = acc[i / 4][i % 4][t];
                            ac = __builtin_fmaf(ds, v, ac);
                            if (T == 12 || T == 13) ac = __builtin_fmaf(-dm, sx[t], ac);
                        }
                    }
                }
            }
        }
        if (c + 1 < nch) park(b ^ 1, c + 1);
        __syncthreads();
    }
}

// quantize_act_q8 (cuda/qgemm.cu:556-587): per 32-element block,
// sx = absmax / 127, q = round-half-even(v * (1 / sx)), 0 when sx = 0. V
// consecutive elements per thread (4 where x is 16-byte and xq 4-byte aligned),
// 32 / V lanes per block. HBM-bound: 16.8 M elements 56 -> 19 us for V 4 against 1.
template <int V>
__global__ __launch_bounds__(256) void gg_quant_q8_kernel(const float* __restrict__ x, long total,
                                                          int8_t* __restrict__ xq,
                                                          float* __restrict__ xs) {
    const long i = ((long)blockIdx.x * blockDim.x + threadIdx.x) * V;
    typedef float vec __attribute__((ext_vector_type(V)));
    vec v = 0.0f;
    if (i < total) v = *reinterpret_cast<const vec*>(x + i);   // total is a multiple of 32
    float a = fabsf(v[0]);
#pragma unroll
    for (int j = 1; j < V; ++j) a = fmaxf(a, fabsf(v[j]));
#pragma unroll
    for (int m = 16 / V; m >= 1; m >>= 1) a = fmaxf(a, __shfl_xor(a, m));
    if (i >= total) return;
    const float sx = a / 127.0f;
    const float id = sx > 0.0f ? 1.0f / sx : 0.0f;
    typedef int8_t qvec __attribute__((ext_vector_type(V)));
    qvec q;
#pragma unroll
    for (int j = 0; j < V; ++j) q[j] = (int8_t)(int)rintf(v[j] * id);
    *reinterpret_cast<qvec*>(xq + i) = q;
    if ((i & 31) == 0) xs[i / 32] = sx;
}

// gemm_q: tiles are 8 consecutive tokens (one at n = 1), one tile per
// workgroup row of the grid.
// LDS bytes of a tile's staged activations.
template <int TT, bool I8>
constexpr size_t gg_lds_bytes() {
    return I8 ? sizeof(GgI8Tile<TT>) : sizeof(float) * TT * kGgKC;
}

// I8: activations are (xq, xsc) from quantize_act_q8 instead of x (gemm_q_i8).
template <uint32_t T, int TT, bool I8>
__global__ __launch_bounds__(kGgThreads) void gg_gemv_kernel(uint32_t qtype, const float* __restrict__ x,
                                                      const int8_t* __restrict__ xq,
                                                      const float* __restrict__ xsc,
                                                      const uint8_t* __restrict__ qw,
                                                      const float* __restrict__ bias,
                                                      float* __restrict__ y, int n, int in, int out,
                                                      long row_bytes) {
    constexpr bool ST = gg_streamed(T);
    __shared__ __align__(16) char lds[ST ? sizeof(GgStream<T, 1, TT, I8>) : gg_lds_bytes<TT, I8>()];
    __shared__ int srcs[TT];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int o0 = blockIdx.x * kGgRows + wave * 4;
    const uint32_t type[1] = {qtype};
    const uint8_t* wrow[1][4];
#pragma unroll
    for (int r = 0; r < 4; ++r) wrow[0][r] = qw + (size_t)min(o0 + r, out - 1) * row_bytes;
    // token tiles: blockIdx.y, then strided by the grid's height
    for (int t0 = blockIdx.y * TT; t0 < n; t0 += gridDim.y * TT) {
        GgTile<TT> tl;
        tl.e = 0;
        tl.nr = min(TT, n - t0);
#pragma unroll
        for (int t = 0; t < TT; ++t) tl.row[t] = tl.src[t] = min(t0 + t, n - 1);
        float acc[1][4][TT];
        if constexpr (ST)
            gg_dots_stream<T, 1, TT, I8>(*reinterpret_cast<GgStream<T, 1, TT, I8>*>(lds), srcs, x,
                                         xq, xsc, in, tl, wrow, acc);
        else if constexpr (I8)
            gg_dots_i8<T, 1, TT>(*reinterpret_cast<GgI8Tile<TT>*>(lds), srcs, xq, xsc, in, tl, type,
                                 wrow, acc);
        else
            gg_dots<T, 1, TT>(reinterpret_cast<float (*)[kGgKC]>(lds), srcs, x, in, tl, type, wrow,
                              acc);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                const float v = gg_wave_sum(acc[0][r][t]);
                const int o = o0 + r;
                if (lane == 0 && t < tl.nr && o < out)
                    y[(size_t)(t0 + t) * out + o] = bias ? v + bias[o] : v;
            }
    }
}

// Tile g of the routed rows. grouped: d = [offsets E+1 | tile prefix E+1 |
// rows n*topk] from gg_group_kernel; otherwise routed row g alone.
template <int TT>
__device__ __forceinline__ bool gg_tile(int g, const int* __restrict__ ids,
                                        const int* __restrict__ d, int nk, int E, int topk,
                                        bool down, GgTile<TT>& tl) {
    if (!d) {
        // An id outside [0, E) routes nowhere: no tile (the grouping drops it
        // too, and the reduce skips its slot).
        if (g >= nk || ids[g] < 0 || ids[g] >= E) return false;
        tl.e = ids[g];
        tl.nr = 1;
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            tl.row[t] = g;
            tl.src[t] = down ? g : g / topk;
        }
        return true;
    }
    const int* off = d;
    const int* tp = d + E + 1;
    const int* rows = d + 2 * (E + 1);
    if (g >= tp[E]) return false;
    int lo = 0, hi = E;   // the expert e with tp[e] <= g < tp[e + 1]
    while (hi - lo > 1) {
        const int mid = (lo + hi) / 2;
        if (tp[mid] <= g) lo = mid;
        else hi = mid;
    }
    tl.e = lo;
    const int r0 = off[lo] + (g - tp[lo]) * TT;
    tl.nr = min(TT, off[lo + 1] - r0);
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const int r = rows[r0 + (t < tl.nr ? t : 0)];
        tl.row[t] = r;
        tl.src[t] = down ? r : r / topk;
    }
    return true;
}

struct GgMoeArgs {
    uint32_t gate_type, up_type, down_type;
    const float* x;
    const int* ids;
    const float* w;
    const uint8_t *gate_q, *up_q, *down_q;
    long gate_rb, up_rb, down_rb;
    int n, topk, H, I, E;
    float* h_act;
    float* dpart;
    const int* d;   // grouping (nullable)
    // int8 activations (moe_expert_ffn_q_i8): x as (xq, xs), h_act as (hq, hs)
    const int8_t* xq;
    const float* xs;
    const int8_t* hq;
    const float* hs;
};

// DOWN = false: phase 1 (gate/up, output rows = I features); true: phase 2.
// T: the weight type (gate and up share it in phase 1), or kGgAny.
template <bool DOWN, uint32_t T, int TT, bool I8>
__global__ __launch_bounds__(kGgThreads) void gg_moe_kernel(GgMoeArgs a) {
    constexpr bool ST = gg_streamed(T);
    __shared__ __align__(16) char lds[ST ? sizeof(GgStream<T, DOWN ? 1 : 2, TT, I8>)
                                         : gg_lds_bytes<TT, I8>()];
    __shared__ int srcs[TT];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nk = a.n * a.topk;
    GgTile<TT> tl;
    if (!gg_tile((int)blockIdx.x, a.ids, a.d, nk, a.E, a.topk, DOWN, tl)) return;
    const int out = DOWN ? a.H : a.I;
    const int o0 = blockIdx.y * kGgRows + wave * 4;
    const size_t e = (size_t)tl.e;
    if constexpr (!DOWN) {
        const uint32_t type[2] = {a.gate_type, a.up_type};
        const uint8_t* wrow[2][4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const size_t o = (size_t)min(o0 + r, out - 1);
            wrow[0][r] = a.gate_q + (e * a.I + o) * a.gate_rb;
            wrow[1][r] = a.up_q + (e * a.I + o) * a.up_rb;
        }
        float acc[2][4][TT];
        if constexpr (ST)
            gg_dots_stream<T, 2, TT, I8>(*reinterpret_cast<GgStream<T, 2, TT, I8>*>(lds), srcs, a.x,
                                         a.xq, a.xs, a.H, tl, wrow, acc);
        else if constexpr (I8)
            gg_dots_i8<T, 2, TT>(*reinterpret_cast<GgI8Tile<TT>*>(lds), srcs, a.xq, a.xs, a.H, tl,
                                 type, wrow, acc);
        else
            gg_dots<T, 2, TT>(reinterpret_cast<float (*)[kGgKC]>(lds), srcs, a.x, a.H, tl, type,
                              wrow, acc);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                const float g = gg_wave_sum(acc[0][r][t]);
                const float u = gg_wave_sum(acc[1][r][t]);
                const int o = o0 + r;
                if (lane == 0 && t < tl.nr && o < out)
                    a.h_act[(size_t)tl.row[t] * a.I + o] = gg_silu(g) * u;
            }
    } else {
        const uint32_t type[1] = {a.down_type};
        const uint8_t* wrow[1][4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const size_t o = (size_t)min(o0 + r, out - 1);
            wrow[0][r] = a.down_q + (e * a.H + o) * a.down_rb;
        }
        float acc[1][4][TT];
        if constexpr (ST)
            gg_dots_stream<T, 1, TT, I8>(*reinterpret_cast<GgStream<T, 1, TT, I8>*>(lds), srcs,
                                         a.h_act, a.hq, a.hs, a.I, tl, wrow, acc);
        else if constexpr (I8)
            gg_dots_i8<T, 1, TT>(*reinterpret_cast<GgI8Tile<TT>*>(lds), srcs, a.hq, a.hs, a.I, tl,
                                 type, wrow, acc);
        else
            gg_dots<T, 1, TT>(reinterpret_cast<float (*)[kGgKC]>(lds), srcs, a.h_act, a.I, tl, type,
                              wrow, acc);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                const float v = gg_wave_sum(acc[0][r][t]);
                const int o = o0 + r;
                if (lane == 0 && t < tl.nr && o < out) a.dpart[(size_t)tl.row[t] * a.H + o] = v;
            }
    }
}

// out[t] = ((0 + w0 y0) + w1 y1) + ... over the slots (cuda/qgemm.cu:943-955).
// Slots whose id is outside [0, E) add nothing (their dpart rows are never
// written). V outputs per thread (4: H % 4 == 0 and 16-byte aligned rows), the
// slots' ids and weights uniform per workgroup: HBM-bound; 1000 tokens x top-8
// x 6144 (221 MB) 100 -> 41 us against one output per thread.
template <int V>
__global__ __launch_bounds__(256) void gg_reduce_kernel(const float* __restrict__ dpart,
                                                        const int* __restrict__ ids,
                                                        const float* __restrict__ w, int topk, int H,
                                                        int E, float* __restrict__ out) {
    const size_t t = blockIdx.x;
    const int o = (int)(blockIdx.y * 256 + threadIdx.x) * V;
    if (o >= H) return;
    typedef float vec __attribute__((ext_vector_type(V)));
    vec acc = 0.0f;
    for (int s = 0; s < topk; ++s) {
        const int e = ids[t * topk + s];
        if (e < 0 || e >= E) continue;
        const vec v = *reinterpret_cast<const vec*>(dpart + (t * topk + s) * H + o);
        acc = acc + w[t * topk + s] * v;
    }
    *reinterpret_cast<vec*>(out + t * H + o) = acc;
}

// Groups the routed rows by expert (one workgroup): d = [offsets E+1 | tile
// prefix E+1 | rows n*topk]; rows of an expert are in any order (each row's
// result depends only on its own inputs).
__global__ __launch_bounds__(1024) void gg_group_kernel(const int* __restrict__ ids, int nk, int E,
                                                        int tile_rows, int* __restrict__ d) {
    extern __shared__ int gl[];   // cnt[E] | cursor[E]
    int* cnt = gl;
    int* cur = gl + E;
    int* off = d;
    int* tp = d + E + 1;
    int* rows = d + 2 * (E + 1);
    for (int e = threadIdx.x; e < E; e += blockDim.x) cnt[e] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < nk; i += blockDim.x) {
        const int e = ids[i];
        if (e >= 0 && e < E) atomicAdd(&cnt[e], 1);
    }
    __syncthreads();
    // Exclusive prefix sums of rows and tiles over the experts: thread i owns
    // experts [i * per, (i + 1) * per); a shuffle scan per wave, then the 16
    // wave totals.
    __shared__ int wsum[2][16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int per = (E + 1023) / 1024, e0 = min(E, tid * per), e1 = min(E, e0 + per);
    int o = 0, t = 0;
    for (int e = e0; e < e1; ++e) {
        o += cnt[e];
        t += (cnt[e] + tile_rows - 1) / tile_rows;
    }
    int so = o, st = t;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        const int a = __shfl_up(so, m), b = __shfl_up(st, m);
        if (lane >= m) {
            so += a;
            st += b;
        }
    }
    if (lane == 63) {
        wsum[0][wave] = so;
        wsum[1][wave] = st;
    }
    __syncthreads();
    int bo = so - o, bt = st - t;
    for (int w = 0; w < wave; ++w) {
        bo += wsum[0][w];
        bt += wsum[1][w];
    }
    for (int e = e0; e < e1; ++e) {
        off[e] = bo;
        tp[e] = bt;
        cur[e] = bo;
        bo += cnt[e];
        bt += (cnt[e] + tile_rows - 1) / tile_rows;
    }
    if (tid == 1023) {
        off[E] = bo;
        tp[E] = bt;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nk; i += blockDim.x) {
        const int e = ids[i];
        if (e >= 0 && e < E) rows[atomicAdd(&cur[e], 1)] = i;
    }
}

// Calls f(std::integral_constant<uint32_t, t>) for a supported type t,
// f(kGgAny constant) otherwise.
template <class F>
static void gg_by_type(uint32_t t, F&& f) {
    switch (t) {
        case 0: f(std::integral_constant<uint32_t, 0>{}); break;
        case 1: f(std::integral_constant<uint32_t, 1>{}); break;
        case 8: f(std::integral_constant<uint32_t, 8>{}); break;
        case 11: f(std::integral_constant<uint32_t, 11>{}); break;
        case 12: f(std::integral_constant<uint32_t, 12>{}); break;
        case 13: f(std::integral_constant<uint32_t, 13>{}); break;
        case 14: f(std::integral_constant<uint32_t, 14>{}); break;
        case 18: f(std::integral_constant<uint32_t, 18>{}); break;
        case 23: f(std::integral_constant<uint32_t, 23>{}); break;
        default: f(std::integral_constant<uint32_t, kGgAny>{}); break;
    }
}

// The int8-capable types (qtype_has_i8, cuda/qgemm.cu:556-567).
bool gguf_has_i8(uint32_t t) {
    return t == 8 || t == 11 || t == 12 || t == 13 || t == 14 || t == 18 || t == 23;
}

// gg_by_type over the int8-capable types (kGgAny for anything else).
template <class F>
static void gg_by_type_i8(uint32_t t, F&& f) {
    switch (t) {
        case 8: f(std::integral_constant<uint32_t, 8>{}); break;
        case 11: f(std::integral_constant<uint32_t, 11>{}); break;
        case 12: f(std::integral_constant<uint32_t, 12>{}); break;
        case 13: f(std::integral_constant<uint32_t, 13>{}); break;
        case 14: f(std::integral_constant<uint32_t, 14>{}); break;
        case 18: f(std::integral_constant<uint32_t, 18>{}); break;
        case 23: f(std::integral_constant<uint32_t, 23>{}); break;
        default: f(std::integral_constant<uint32_t, kGgAny>{}); break;
    }
}

template <bool I8, class F>
static void gg_by_type_t(uint32_t t, F&& f) {
    if constexpr (I8) gg_by_type_i8(t, f);
    else gg_by_type(t, f);
}

// The streamed kernels load weight rows as dwords and fp32 activations as
// float4: with rows or bases not aligned for that, the type is decoded by the
// runtime switch (kGgAny) with byte loads instead.
static bool gg_aligned(const void* w, long row_bytes, const void* x, int xalign) {
    return ((uintptr_t)w & 3) == 0 && (row_bytes & 3) == 0 &&
           (x == nullptr || ((uintptr_t)x & (uintptr_t)(xalign - 1)) == 0);
}

// splitmm_kernel takes whole chunks of K, output rows by 32, dword-aligned
// weight rows and 16-byte aligned fp32 activations (int8: 4).
static bool gg_sm_ok(uint32_t t, const void* w, long rb, const void* x, int xalign, int K, int out) {
    const bool type = t == 8 || t == 11 || t == 12 || t == 13 || t == 14 || t == 18 || t == 23;
    return type && K % sm_kc(t) == 0 && sm_out_ok(out) && gg_aligned(w, rb, x, xalign);
}

// f(constant) for a type gg_sm_ok accepts.
template <class F>
static int gg_sm_type(uint32_t t, F&& f) {
    switch (t) {
        case 8: return f(std::integral_constant<uint32_t, 8>{});
        case 11: return f(std::integral_constant<uint32_t, 11>{});
        case 12: return f(std::integral_constant<uint32_t, 12>{});
        case 13: return f(std::integral_constant<uint32_t, 13>{});
        case 14: return f(std::integral_constant<uint32_t, 14>{});
        case 18: return f(std::integral_constant<uint32_t, 18>{});
        default: return f(std::integral_constant<uint32_t, 23>{});
    }
}

template <bool I8>
static int gg_gemm(uint32_t qtype, const float* x, const int8_t* xq, const float* xsc,
                   const uint8_t* qw, const float* bias, float* y, int n, int in, int out,
                   long row_bytes, hipStream_t s) {
    // Every n: 6144 -> 2048 Q8_0, fp32 rows, us at n = 1 / 8 / 64 / 1000: 12 / 17 / 28 / 235 against
    // 20 / 43 / 118 / 1815 of gg_gemv_kernel (int8 rows: 9 / 11 / 15 / 105 against 19 / 32 / 70 / 920).
    if (gg_sm_ok(qtype, qw, row_bytes, I8 ? (const void*)xq : (const void*)x, I8 ? 4 : 16, in, out)) {
        SmArgs a{};
        a.x = x; a.xq = xq; a.xs = xsc; a.w0 = qw; a.rb0 = row_bytes; a.bias = bias; a.y = y;
        a.K = in; a.out = out; a.n = n;
        return gg_sm_type(qtype, [&](auto tc) { return sm_dense<decltype(tc)::value>(I8, a, s); });
    }
    const int tt = n == 1 ? 1 : 8;
    const dim3 grid((unsigned)((out + kGgRows - 1) / kGgRows),
                    (unsigned)std::min((n + tt - 1) / tt, 65535));
    const bool al = gg_aligned(qw, row_bytes, I8 ? (const void*)xq : (const void*)x, I8 ? 4 : 16);
    gg_by_type_t<I8>(al ? qtype : kGgAny, [&](auto tc) {
        constexpr uint32_t T = decltype(tc)::value;
        if (n == 1)
            hipLaunchKernelGGL((gg_gemv_kernel<T, 1, I8>), grid, dim3(kGgThreads), 0, s, qtype, x, xq,
                               xsc, qw, bias, y, n, in, out, row_bytes);
        else
            hipLaunchKernelGGL((gg_gemv_kernel<T, 8, I8>), grid, dim3(kGgThreads), 0, s, qtype, x, xq,
                               xsc, qw, bias, y, n, in, out, row_bytes);
    });
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

int launch_gg_gemm(uint32_t qtype, const float* x, const uint8_t* qw, const float* bias, float* y,
                   int n, int in, int out, long row_bytes, hipStream_t s) {
    return gg_gemm<false>(qtype, x, nullptr, nullptr, qw, bias, y, n, in, out, row_bytes, s);
}

int launch_gg_gemm_i8(uint32_t qtype, const int8_t* xq, const float* xs, const uint8_t* qw,
                      const float* bias, float* y, int n, int in, int out, long row_bytes,
                      hipStream_t s) {
    return gg_gemm<true>(qtype, nullptr, xq, xs, qw, bias, y, n, in, out, row_bytes, s);
}

int launch_gg_quant_q8(const float* x, long total, int8_t* xq, float* xs, hipStream_t s) {
    if (((uintptr_t)x & 15) == 0 && ((uintptr_t)xq & 3) == 0)
        hipLaunchKernelGGL(gg_quant_q8_kernel<4>, dim3((unsigned)((total + 1023) / 1024)), dim3(256), 0, s, x,
                           total, xq, xs);
    else
        hipLaunchKernelGGL(gg_quant_q8_kernel<1>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, x,
                           total, xq, xs);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

// I8: h_act is quantized into (hq, hs) between the phases.
template <int TT, bool I8>
static int gg_moe_phases(uint32_t gt, uint32_t ut, uint32_t dt, const GgMoeArgs& a, unsigned tiles,
                         hipStream_t s) {
    const dim3 g1(tiles, (unsigned)((a.I + kGgRows - 1) / kGgRows));
    const bool al1 = gg_aligned(a.gate_q, a.gate_rb, I8 ? (const void*)a.xq : (const void*)a.x,
                                I8 ? 4 : 16) &&
                     gg_aligned(a.up_q, a.up_rb, nullptr, 1);
    const bool al2 = gg_aligned(a.down_q, a.down_rb,
                                I8 ? (const void*)a.hq : (const void*)a.h_act, I8 ? 4 : 16);
    if (gt == ut && al1)
        gg_by_type_t<I8>(gt, [&](auto tc) {
            hipLaunchKernelGGL((gg_moe_kernel<false, decltype(tc)::value, TT, I8>), g1, dim3(kGgThreads),
                               0, s, a);
        });
    else
        hipLaunchKernelGGL((gg_moe_kernel<false, kGgAny, TT, I8>), g1, dim3(kGgThreads), 0, s, a);
    if (hipGetLastError() != hipSuccess) return -4;
    if constexpr (I8) {
        if (launch_gg_quant_q8(a.h_act, (long)a.n * a.topk * a.I, const_cast<int8_t*>(a.hq),
                               const_cast<float*>(a.hs), s))
            return -4;
    }
    const dim3 g2(tiles, (unsigned)((a.H + kGgRows - 1) / kGgRows));
    gg_by_type_t<I8>(al2 ? dt : kGgAny, [&](auto tc) {
        hipLaunchKernelGGL((gg_moe_kernel<true, decltype(tc)::value, TT, I8>), g2, dim3(kGgThreads), 0, s,
                           a);
    });
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

static int gg_reduce(const GgMoeArgs& a, float* out, hipStream_t s) {
    const bool v4 = a.H % 4 == 0 && (((uintptr_t)a.dpart | (uintptr_t)out) & 15) == 0;
    const int per = v4 ? 1024 : 256;
    const dim3 grid((unsigned)a.n, (unsigned)((a.H + per - 1) / per));
    if (v4)
        hipLaunchKernelGGL(gg_reduce_kernel<4>, grid, dim3(256), 0, s, a.dpart, a.ids, a.w, a.topk, a.H, a.E, out);
    else
        hipLaunchKernelGGL(gg_reduce_kernel<1>, grid, dim3(256), 0, s, a.dpart, a.ids, a.w, a.topk, a.H, a.E, out);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

// Rows per tile of splitmm_kernel for this call, 0 where the kernels of this
// file take it: types, shapes or alignments splitmm does not cover (and gate
// and up of different types), or too little work for its 64-row workgroups.
// The choice among tiles depends on the rows per expert (nk / E), which the
// host knows only on average. Measured on the 6144 x 2048 x 256 layer, top-8,
// IQ3_XXS / IQ4_XS (us for tiles of 4 / 8 / 16 / 32 / 64 rows, and before):
//   fp32  n = 16: 601 / 704 / 836 / - / - (791); 64: 1240 / 1168 / 1382 / - /
//         1962 (2303); 128: - / 1705 / 1631 / 1636 / 2155 (4202); 256: - / 2590 /
//         2249 / 1895 / 2713 (8815); 1000: - / 8001 / 5304 / 3575 / 3942 (27440)
//   int8  n = 16: 504 / 518 / 593 / - / - (650); 64: 970 / 855 / 983 / - / 1257
//         (1681); 256: - / 1861 / 1378 / 1437 / 1665 (2705); 512: - / 3134 / 2142 /
//         1877 / 1889; 1000: - / 5310 / 3544 / 2636 / 2406 (3837)
// With the rows on a few hot experts (Zipf 1.1) or narrow experts the larger
// tile wins earlier (int8 n = 256: 907 / 705 / 671 for 16 / 32 / 64). The
// 64-row tile has fewer, larger steps and 256 registers full: int8 takes it
// from 16 rows per expert, fp32 only where every expert has several (64), Q8_0
// with fp32 rows never (1000: 4122 against 6492). The K-quants decode more per
// tile: 16 rows up to 16 per expert (Q4_K, Q4_K, Q6_K, n = 256: 3176 / 3581,
// 1000: 8517 / 6539), and the types with a scale per 16 K take the one-wave
// sums of the larger tiles only up to K 4096, where their rounding error is not
// above the vector kernels'. int8 calls below
// 2048 routed rows stay on the small tiles, whose sums do not depend on the
// tile: grouped and ungrouped calls agree bit for bit there.
// Narrow layers of few experts have few of the large workgroups (128 features x
// tile), so fp32 rows take 16-row tiles where gate/up has less than 64 of them
// (1024 x 512 x 8, top-2, n = 24 / 120, IQ4_XS: 25 / 30 us against 52 / 54, vector kernels
// 46 / 108; the limit could be twice that on some layers and not on others: 6144 x 256 x
// 64, top-8, n = 120: 231 against 176), and int8 rows 32 instead of 64 below one
// per CU (2048 x 512 x 32, top-4, n = 600: 105 against 122, before these kernels 106;
// with 856 of them, 2048 x 1024 x 64, top-8: 289 against 278).
// Too little work: the vector kernels' 16-row workgroups win at n = 1 of that
// layer with IQ types (71 against 77 us) and on small layers (2048 x 512,
// top-4, n = 1: 17 against 26 us, n = 16: 72 against 41). They are also
// faster, but further from 64 bits (block error at n = 16 1.83e-7 against 1.64e-7), and
// not taken, for fp32 IQ rows at width 256 ungrouped or about one to an expert
// (6144 x 256 x 256, top-8, n = 16: 187 against 232, n = 20: 233 against 231).
template <bool I8>
static int gg_sm_tile(const GgMoeArgs& a, bool grouped) {
    const uint32_t gt = a.gate_type, dt = a.down_type;
    const int nk = a.n * a.topk, E = a.E;
    if (gt != a.up_type ||
        !gg_sm_ok(gt, a.gate_q, a.gate_rb, I8 ? (const void*)a.xq : (const void*)a.x, I8 ? 4 : 16, a.H, a.I) ||
        !gg_aligned(a.up_q, a.up_rb, nullptr, 1) ||
        !gg_sm_ok(dt, a.down_q, a.down_rb, I8 ? (const void*)a.hq : (const void*)a.h_act, I8 ? 4 : 16, a.I, a.H))
        return 0;
    auto kquant = [](uint32_t t) { return t >= 11 && t <= 14; };
    const bool iq = gt == 18 || gt == 23, kq = kquant(gt) || kquant(dt);
    const long work = (long)nk * (a.I / 32) * (a.H / 256);
    if (nk <= E && work < (iq ? 24576 : 2048)) return 0;
    if (!grouped || nk <= E) return 4;
    if (nk <= 4 * E) return 8;
    if (I8 && nk < 2048) return 16;
    const bool large = sm_large_tile(gt, I8) && sm_large_tile(dt, I8);
    if (kq) {
        const bool long16 = (sm_g16(gt) && a.H > 4096) || (sm_g16(dt) && a.I > 4096);
        return nk <= 16 * E || long16 ? 16 : kSmMidTile;
    }
    // gate/up workgroups for tiles of t rows, the last of each expert half full
    auto wgs = [&](int t) { return (long)(nk / t + E / 2) * ((a.I + 127) / 128); };
    if (!I8 && wgs(kSmMidTile) < 64) return 16;
    if (!large || nk <= (I8 ? 16 : 64) * E || (I8 && wgs(kSmLargeTile) < 256)) return kSmMidTile;
    return kSmLargeTile;
}

// Gate/up and down on splitmm_kernel; d: the grouping in tiles of `tile` rows.
template <bool I8>
static int gg_sm_phases(const GgMoeArgs& a, const int* d, int tile, unsigned tiles, hipStream_t s) {
    SmArgs m{};
    m.x = a.x; m.xq = a.xq; m.xs = a.xs;
    m.w0 = a.gate_q; m.rb0 = a.gate_rb;
    m.w1 = a.up_q; m.rb1 = a.up_rb;
    m.y = a.h_act;
    m.K = a.H; m.out = a.I; m.n = a.n; m.E = a.E; m.topk = a.topk;
    m.ids = a.ids; m.d = d;
    int rc = gg_sm_type(a.gate_type, [&](auto tc) {
        return sm_moe<decltype(tc)::value>(false, I8, tile, m, tiles, s);
    });
    if (rc) return rc;
    if constexpr (I8) {
        if (launch_gg_quant_q8(a.h_act, (long)a.n * a.topk * a.I, const_cast<int8_t*>(a.hq),
                               const_cast<float*>(a.hs), s))
            return -4;
    }
    m.x = a.h_act; m.xq = a.hq; m.xs = a.hs;
    m.w0 = m.w1 = a.down_q; m.rb0 = m.rb1 = a.down_rb;
    m.y = a.dpart;
    m.K = a.I; m.out = a.H;
    return gg_sm_type(a.down_type, [&](auto tc) {
        return sm_moe<decltype(tc)::value>(true, I8, tile, m, tiles, s);
    });
}

template <bool I8>
static int gg_moe(GgMoeArgs a, float* out, int* dispatch, hipStream_t s) {
    const uint32_t gt = a.gate_type, ut = a.up_type, dt = a.down_type;
    const int E = a.E, nk = a.n * a.topk;
    const int* ids = a.ids;
    if (const int tile = gg_sm_tile<I8>(a, dispatch != nullptr)) {
        unsigned tiles = (unsigned)nk;
        if (dispatch) {
            hipLaunchKernelGGL(gg_group_kernel, dim3(1), dim3(1024), (size_t)2 * E * 4, s, ids, nk, E, tile,
                               dispatch);
            if (hipGetLastError() != hipSuccess) return -4;
            tiles = (unsigned)std::min(nk, (nk + tile - 1) / tile + E);
        }
        const int rc = gg_sm_phases<I8>(a, dispatch, tile, tiles, s);
        return rc ? rc : gg_reduce(a, out, s);
    }
    // Rows per tile: about the rows an expert holds (decode: one or a few). With
    // one row per tile, grouping changes nothing but the order of the tiles, so
    // the routed rows are taken as they come (an exact grid, no counting pass).
    const int tt = !dispatch || nk <= E ? 1 : nk <= 4 * E ? 4 : 8;
    if (tt == 1) {
        dispatch = nullptr;
        a.d = nullptr;
    }
    unsigned tiles = (unsigned)nk;
    if (dispatch) {
        hipLaunchKernelGGL(gg_group_kernel, dim3(1), dim3(1024), (size_t)2 * E * 4, s, ids, nk, E,
                           tt, dispatch);
        if (hipGetLastError() != hipSuccess) return -4;
        tiles = (unsigned)((nk + tt - 1) / tt + E);
    }
    const int rc = tt == 1 ? gg_moe_phases<1, I8>(gt, ut, dt, a, tiles, s)
                 : tt == 4 ? gg_moe_phases<4, I8>(gt, ut, dt, a, tiles, s)
                           : gg_moe_phases<8, I8>(gt, ut, dt, a, tiles, s);
    return rc ? rc : gg_reduce(a, out, s);
}

int launch_gg_moe(uint32_t gt, uint32_t ut, uint32_t dt, const float* x, const int* ids,
                  const float* w, const uint8_t* gq, const uint8_t* uq, const uint8_t* dq, int n,
                  int topk, int H, int I, int E, long grb, long urb, long drb, float* h_act,
                  float* dpart, float* out, int* dispatch, hipStream_t s) {
    GgMoeArgs a{gt, ut, dt, x, ids, w, gq, uq, dq, grb, urb, drb, n, topk, H, I, E, h_act, dpart,
                dispatch, nullptr, nullptr, nullptr, nullptr};
    return gg_moe<false>(a, out, dispatch, s);
}

int launch_gg_moe_i8(uint32_t gt, uint32_t ut, uint32_t dt, const int8_t* xq, const float* xs,
                     const int* ids, const float* w, const uint8_t* gq, const uint8_t* uq,
                     const uint8_t* dq, int n, int topk, int H, int I, int E, long grb, long urb,
                     long drb, float* h_act, int8_t* hq, float* hs, float* dpart, float* out,
                     int* dispatch, hipStream_t s) {
    GgMoeArgs a{gt, ut, dt, nullptr, ids, w, gq, uq, dq, grb, urb, drb, n, topk, H, I, E, h_act,
                dpart, dispatch, xq, xs, hq, hs};
    return gg_moe<true>(a, out, dispatch, s);
}

}  // namespace glmmoe
