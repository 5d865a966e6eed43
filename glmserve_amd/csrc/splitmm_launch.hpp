// Launch shapes of splitmm_kernel, instantiated per weight format (one file
// each, so that they compile side by side).
#pragma once

#include "splitmm.hpp"

namespace glmmoe {

// MoE launches: the small tiles (4, 8, 16 tokens) split K over the workgroup's
// four waves, the others (32, 64) its weight rows.
template <uint32_t T, int MODE, bool I8, int RW, int KW, int NB, int NT, int KX>
static int sm_go(const SmArgs& a, unsigned gx, hipStream_t s) {
    constexpr int rows = (MODE == kSmGateUp ? 32 : 32 * NB) * RW;
    hipLaunchKernelGGL((splitmm_kernel<T, MODE, I8, RW, KW, NB, NT, KX>),
                       dim3(gx, (unsigned)((a.out + rows - 1) / rows)), dim3(64 * RW * KW), 0, s, a);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

// K staged at a time for tiles of nt tokens; less where a row's chunk is wide, so
// that two 4-wave workgroups' LDS fits a CU (all but the 8- and 16-token expert tiles
// of Q6_K with fp32 rows: 84 and 85 KiB). The linears' 8-wave workgroups of 16 and 32
// fp32 rows (86 to 155 KiB) have a CU to themselves, and those of Q6_K with 4 fp32 or
// 32 int8 rows (83 KiB).
constexpr int sm_kx(uint32_t t, int nt) {
    const int k = nt <= 8 ? 128 : 64;
    return t == 12 || t == 13 || t == 14 ? k / 2 : k;
}

// The tiles of 4 to 16 and the 32-token ones of the IQ types, Q8_0 and Q3_K keep
// everything in registers. Spilled to scratch, in registers: 32-token tiles of Q4_K
// (fp32 14), Q5_K (fp32 43, int8 15) and Q6_K (fp32 17, int8 40), 64-token tiles up
// to 3 with int8 rows, 7 to 17 with fp32; faster than the smaller tiles all the same
// where gg_sm_tile takes them.
// -2: a tile that no call of this type takes (sm_large_tile).
template <uint32_t T, int MODE, bool I8>
static int sm_moe_mode(int tile, const SmArgs& a, unsigned tiles, hipStream_t s) {
    if (tile == 4) return sm_go<T, MODE, I8, 1, 4, 2, 4, sm_kx(T, 4)>(a, tiles, s);
    if (tile == 8) return sm_go<T, MODE, I8, 1, 4, 2, 8, sm_kx(T, 8)>(a, tiles, s);
    if (tile == 16) return sm_go<T, MODE, I8, 1, 4, 2, 16, sm_kx(T, 16)>(a, tiles, s);
    if (tile == kSmMidTile)
        return sm_go<T, MODE, I8, 4, 1, 2, 32, I8 || T == 8 ? 128 : T == 14 ? 32 : 64>(a, tiles, s);
    if constexpr (sm_large_tile(T, I8)) {
        if (tile == kSmLargeTile) return sm_go<T, MODE, I8, 4, 1, 2, 64, I8 ? 128 : sm_kx(T, 64)>(a, tiles, s);
    }
    return -2;
}

template <uint32_t T>
int sm_moe(bool down, bool i8, int tile, const SmArgs& a, unsigned tiles, hipStream_t s) {
    if (i8)
        return down ? sm_moe_mode<T, kSmDown, true>(tile, a, tiles, s)
                    : sm_moe_mode<T, kSmGateUp, true>(tile, a, tiles, s);
    return down ? sm_moe_mode<T, kSmDown, false>(tile, a, tiles, s)
                : sm_moe_mode<T, kSmGateUp, false>(tile, a, tiles, s);
}

// One matrix. Up to 32 tokens per tile a workgroup takes 32 output rows and
// splits K over 8 waves, so that few outputs still spread over the chip. Where
// 64-token x 256-row tiles make at least 192 workgroups they take half the
// time: each weight is decoded for 64 tokens and each activation split once
// for 256 rows (Q8_0, 6144 outputs of K 2048, fp32 rows: 1000 tokens 140
// against 253 us; below, 203 tokens 111 against 67). Not for the types with a
// scale per 16 K: twice the pieces to add, whose one-wave sum has more rounding
// error than the vector kernels' (9.7e-8 against 9.4e-8).
template <uint32_t T, bool I8>
static int sm_dense_i(const SmArgs& a, hipStream_t s) {
    auto tiles = [&](int t) { return (unsigned)((a.n + t - 1) / t); };
    if constexpr (!sm_g16(T)) {
        if ((long)tiles(64) * ((a.out + 255) / 256) >= 192)
            return sm_go<T, kSmDense, I8, 4, 1, 2, 64, I8 ? 128 : sm_kx(T, 64)>(a, tiles(64), s);
    }
    if (a.n <= 4) return sm_go<T, kSmDense, I8, 1, 8, 1, 4, sm_kx(T, 4)>(a, tiles(4), s);
    if (a.n <= 16) return sm_go<T, kSmDense, I8, 1, 8, 1, 16, sm_kx(T, 16)>(a, tiles(16), s);
    return sm_go<T, kSmDense, I8, 1, 8, 1, 32, sm_kx(T, 32)>(a, tiles(32), s);
}

template <uint32_t T>
int sm_dense(bool i8, const SmArgs& a, hipStream_t s) {
    if constexpr (T != kSmW4 && T != kSmFp8) {
        if (i8) return sm_dense_i<T, true>(a, s);
    }
    return sm_dense_i<T, false>(a, s);
}

}  // namespace glmmoe
