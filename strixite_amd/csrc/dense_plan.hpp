// Which kernel a dense BF16 projection (experts.hip, dense_projection) takes: host arithmetic on its sizes alone.
#pragma once

#include <algorithm>
#include <cstdint>

namespace strix::kernels::dnp {

// - Tiles: exact_tile.hip's 16-row tiles, K split over a block's waves: the shortest walk of K, and the codes converted once
//   for 16 tokens, so its time grows with outputs x K (in half rounds of the chip past kRound). Its loads take 16 rows at
//   once, which share cache sets where a row's bytes are a power of two: 1.2 to 1.4 of the time there, from K 1024.
// - Stream: the expert stream kernel over 16 tokens x 32 rows a wave: a wave walks K alone, flat up to kRound outputs and by
//   rounds beyond. The better one only where K is short and a power of two (Q8 g128, N 4096 at 127 tokens, us, stream /
//   tiles: K 1024 13 / 15, 1536 18 / 17, 2048 22 / 35, 2560 31 / 28).
// - Gemm: the LDS-tiled GEMM of 64 tokens x 256 rows: a longer walk of K, flat up to kGemmFlat outputs.
enum class Dense { Tiles, Stream, Gemm };

constexpr int64_t kRound = 524288, kGemmFlat = 5115000, kStreamK = 2048, kGemmMinTokens = 64, kGemmMinTokensF32 = 128;

// us a 1024 of K (and at no K: g0, s0, t0) on MI355X; sm, tm: what a full 16-token tile adds to one token's; tpow: the tiles'
// factor at a power of two. Fitted to 2500 timings of each kernel (M 1 .. 1500, N 512 .. 131072, K 512 .. 5120): the choice is
// 1.002 of the best kernel's time on average, 1.25 at worst. By a line on M N alone (tiles up to 400000 outputs, the GEMM from
// there) it was 1.17 on average, and calls that the stream kernel had served before were up to 2 x slower. us, stream / tiles
// / GEMM: Q4 g128, N 4096, K 2048 at 100 tokens 18.3 / 21.2 / 28.4, N 32768 at 1 15.2 / 17.2 / 27.4; Q8 g128, N 4096, K 2048
// at 100 21.2 / 31.5 / 34.7, N 32768 at 1 19 / 31 / 38; Q4 g64, N 4096, K 1024 at 127 14.4 / 18.5 / 19.2; Q4 g128, N 4096,
// K 3072 at 127 27 / 23 / 42, at 200 48 / 38 / 41.
struct Cost {
    double g0, gk, s0, sk, sm, t0, tk, tp, tm, tpow;
};
constexpr Cost kCosts[2][2] = {  // [Q8][G >= 128]
    {{5.9, 13.4, 1.4, 14.7, 1.6, 3.4, 1.7, 11.2, 2.2, 1.26}, {3.8, 14.9, 6.5, 5.4, 1.7, 3.5, 1.8, 3.8, 1.5, 1.44}},
    {{4.2, 17.5, 0.9, 17.6, 1.9, 3.1, 2.2, 13.6, 2.7, 1.22}, {6.6, 21.2, 4.3, 11.4, 1.2, 3.2, 3.4, 9.4, 2.0, 1.42}},
};

// gemm_ok: the GEMM takes the shape (its K steps and groups a row). It is the least exact of the three (its sums carry Q4's
// code offset of 128 along all of K), so FP32 outputs, whose rounding does not hide that, take it from 128 tokens only.
inline Dense plan(int bits, int64_t G, int64_t M, int64_t N, int64_t K, bool out_f32, bool gemm_ok) {
    // the stream kernel and the GEMM address their tensors by 32-bit offsets
    constexpr int64_t kLimit = 1ll << 31;
    if (N * K * bits / 8 >= kLimit || N * (K / G) * 2 >= kLimit || M * K * 2 >= kLimit || M * N * (out_f32 ? 4 : 2) >= kLimit)
        return Dense::Tiles;
    const int64_t padded = (M + 15) / 16 * 16 * N;
    const bool pow2 = (K & (K - 1)) == 0, s = pow2 && K <= kStreamK;
    if (G < 64) {
        // us, stream / tiles: Q4 K 512, N 3072 at 100 tokens 12.0 / 14.4, at 500 23 / 40, at 2000 72 / 141, N 32768 at 1 10.5 /
        // 15.3; K 1024, N 4096 at 128 29 / 32, at 2000 394 / 457; K 2048, N 131072 at 1 179 / 194, Q8, N 1088 at 823 115 / 105; K
        // 3072, N 4096 at 700 440 / 405; K 1408 (Q8), N 10464 at 560 412 / 275; few outputs: K 512, N 512 at 500 12.0 / 11.4, K
        // 1024, N 1024 at 300 29 / 25
        return s && K <= (bits == 8 ? 1024 : kStreamK) && padded > (K <= 512 ? 280000 : 400000) ? Dense::Stream : Dense::Tiles;
    }
    const Cost &c = kCosts[bits == 8][G >= 128];
    const double k = (double)K / 1024, m = (double)std::min<int64_t>(M, 16) / 16, u = (double)padded / kRound;
    const int64_t rounds = (padded + kRound - 1) / kRound, halves = (2 * padded + kRound - 1) / kRound;
    const double gemm = (c.g0 + c.gk * k) * std::max(1.0, (double)((M + 63) / 64 * 64 * N) / kGemmFlat);
    const double stream = c.s0 + k * (c.sk + c.sm * m) * (1 + 0.92 * (double)(rounds - 1));
    const double filled = padded <= kRound ? u : 0.55 * (double)halves;
    const double tiles = c.t0 + k * (pow2 && K >= 1024 ? c.tpow : 1.0) * (c.tk + (c.tp + c.tm * m) * filled);
    const bool g = gemm_ok && M >= (out_f32 ? kGemmMinTokensF32 : kGemmMinTokens);
    if (g && gemm <= tiles && (!s || gemm <= stream)) return Dense::Gemm;
    return s && stream < tiles ? Dense::Stream : Dense::Tiles;
}

}  // namespace strix::kernels::dnp
