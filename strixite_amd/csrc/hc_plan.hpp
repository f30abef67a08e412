// Which kernel of the hyper-connection mix (hc.hip) a call takes: host arithmetic on its sizes alone.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace strix::kernels::hcp {

// ---- down ------------------------------------------------------------------------------------------------------------
// The kernels (us on MI355X at d 2560, r 320, Q4 g64):
// - lane dots up to this many BF16 tokens: 4.3 at 1 token, 6.1 at 4, 10.2 at 16, 19 at 40, 27 at 64, in proportion;
// - split-K tiles above, as long as their blocks are at most the CUs (16 tokens x 16 rows a block 18 us flat, 16 x 32 24,
//   32 x 32 36, 32 x 64 50): a block's time is its K walk, whatever the grid;
// - then the staged tiles, flat in T until their blocks pass the CUs.
// FP32 streams (three MFMA rows or products a value), and streams too wide for the split-K tiles' LDS: the cheaper of lane
// dots and staged tiles (dots_beat_tiles).
// Before: vector rows 5.6 / 12 / 24 / 35 / 45, 146 at 255 tokens (FP32 43 at 16, 426 at 255), staged tiles 104 from 256.
constexpr int64_t kDownDotTokens = 32;
constexpr size_t kDownSplitLds = 160 * 1024 - 1024;
constexpr int64_t kStageK = 128, kStageRows = 192, kStageTok = 32;  // the staged tiles: k a stage, rows and tokens a block

enum class Down { Dots, Split, Tiles };

// A split-K block: TT 16-token tiles x RT 16-row tiles, NW waves
struct Split {
    int TT, RT, NW;
};
constexpr Split kSplits[4] = {{1, 1, 16}, {1, 2, 16}, {2, 2, 8}, {2, 4, 8}};

inline int64_t split_blocks(const Split &s, int64_t T, int64_t R) {
    return ((R + 16 * s.RT - 1) / (16 * s.RT)) * ((T + 16 * s.TT - 1) / (16 * s.TT));
}
// codes a K step of the split-K tiles
inline int split_step(int64_t d, int64_t G) { return G >= 64 && d % 64 == 0 ? 64 : 32; }
// groups a wave's K range can touch
inline uint32_t split_groups(const Split &s, int64_t d, int64_t G) {
    const int64_t sp = split_step(d, G), pw = s.NW / 4, steps = (d / sp + pw - 1) / pw;
    return (uint32_t)((steps * sp + G - 1) / G + 1);
}
// the waves' scales and mins, then their sums
inline size_t split_lds(const Split &s, int64_t d, int64_t G) {
    return std::max((size_t)s.NW * s.TT * (s.RT + 1) * 64 * 16, (size_t)s.NW * split_groups(s, d, G) * 16 * s.RT * 4);
}

inline int64_t tile_blocks(int64_t T, int64_t R) {
    return ((R + kStageRows - 1) / kStageRows) * ((T + kStageTok - 1) / kStageTok);
}

// The lane dots' time is in proportion to tokens x rows x (d + 530) (the reductions at a row's end cost as much as 530 more
// codes), FP32 Q8 x 1.5; the staged tiles' to the stages of K times the rounds their blocks take on the CUs (one a CU).
// kTileUnits: what d's worth of stages costs in units of the dots' (0.323e-6 us), the dots' 1.5 taken out. Measured on
// MI355X, us, dots / tiles:
// - FP32, d 2560, Q4 g64: r 320, 400 tokens 134 / 172, r 384, 439 tokens 171 / 174, r 768, 256 tokens 203 / 168, r 1020,
//   300 tokens 296 / 175; d 1024, r 320, 439 tokens 75 / 69; Q8, r 384, 256 and 439 tokens 155 and 239 / 182;
// - BF16, r 320, 1000 tokens: Q4 g32 d 5120 511 / 155, Q4 g64 d 10240 945 / 292, Q8 g32 d 5120 525 / 295.
inline bool dots_beat_tiles(int bits, bool f32, int64_t T, int64_t R, int64_t d, int64_t cus) {
    constexpr int64_t kTileUnits[2][2] = {{94000, 178000}, {200000, 147000}};  // [f32][Q8]
    return T * R * (d + 530) < (tile_blocks(T, R) + cus - 1) / cus * d * kTileUnits[f32][bits == 8];
}

struct DownPlan {
    Down kernel;
    int split;   // of kSplits
    int halves;  // staged tiles: K in halves, a wave group each
};

// K in halves fills a CU that has one block (BF16 streams, Q4: the stages of FP32 and of Q8 fill the LDS with one). Where
// the blocks pass the CUs, two blocks of one half share a CU and do the same without the totals' exchange, except with
// groups of 32, whose four rescales a stage leave a group of waves more to hide. Measured on MI355X at d 2560, two halves /
// one, us: Q4 g64, r 320, 2000 tokens (126 blocks) 81 / 104, r 384, 4000 (375) 164 / 153, r 768, 2000 (315) 166 / 154, 6000
// 333 / 305; g128, r 768, 2000 140 / 132; g32, r 384, 4000 165 / 172, r 768, 6000 332 / 338.
inline int tile_halves(int bits, bool f32, int64_t G, int64_t T, int64_t R, int64_t cus) {
    return !f32 && bits == 4 && (G == 32 || tile_blocks(T, R) <= cus) ? 2 : 1;
}

inline DownPlan plan_down(int bits, bool f32, int64_t G, int64_t T, int64_t R, int64_t d, int64_t cus) {
    const bool stages = d % kStageK == 0;  // the staged tiles take the shape
    if (!f32) {
        if (T <= kDownDotTokens) return {Down::Dots, 0, 1};
        int v = 0;  // the first whose blocks are at most the CUs
        while (v < 3 && split_blocks(kSplits[v], T, R) > cus) ++v;
        const bool fits = split_lds(kSplits[v], d, G) <= kDownSplitLds;
        if (fits && (!stages || split_blocks(kSplits[v], T, R) <= cus)) return {Down::Split, v, 1};
        if (fits) return {Down::Tiles, 0, tile_halves(bits, f32, G, T, R, cus)};
        // a stream too wide for the scales' LDS space
    }
    if (stages && !dots_beat_tiles(bits, f32, T, R, d, cus)) return {Down::Tiles, 0, tile_halves(bits, f32, G, T, R, cus)};
    return {Down::Dots, 0, 1};
}

// ---- up --------------------------------------------------------------------------------------------------------------
// LDS of a block's MT 16-token tiles of h: three bf16 pieces and the group sums
inline size_t up_lds(int MT, int64_t r, int64_t G) {
    const int64_t ngr4 = (r / G + 3) / 4 * 4;
    return (size_t)(3 * 16 * MT * (r / 2 + 4) + ngr4 * 16 * MT) * 4;
}

struct UpPlan {
    bool small;  // 16-token tiles of 4 waves a block (else 32-token tiles of 8 waves)
    bool two;    // the variant of two blocks a CU
};

// 16-token tiles of 4 waves a block up to 16 tokens, 32-token tiles of 8 waves above (the h tile shared by more
// columns); 32-token tiles of h fit the LDS up to r = 768.
// Two blocks a CU, at half the registers and a ring of two chunks: where there are more blocks than CUs and the LDS holds
// two tiles of h (r about 410); Q8 only beside short rows and BF16 streams (its ring is twice the registers). Measured on
// MI355X, d 2560, g 64, 2000 tokens, two / one, us: Q4 r 320 83 / 91, r 384 93 / 95, r 448 119 / 117, r 768 177 / 158, FP32
// streams r 320 78 / 88, r 768 182 / 164; Q8 r 64 49 / 53, r 128 61 / 61, r 320 101 / 99, r 448 163 / 122, FP32 105 / 103.
inline UpPlan plan_up(int bits, bool f32, int64_t T, int64_t d, int64_t r, int64_t G, int64_t cus) {
    const bool small = T <= 16 || r > 768;
    const int64_t MT = small ? 1 : 2, waves = small ? 4 : 8;
    const int64_t blocks = (d / 16 + waves - 1) / waves * ((T + 16 * MT - 1) / (16 * MT));
    const bool pays = bits == 4 || (!f32 && r <= 128);
    return {small, !small && blocks > cus && pays && 2 * up_lds(2, r, G) <= 160 * 1024};
}

}  // namespace strix::kernels::hcp
