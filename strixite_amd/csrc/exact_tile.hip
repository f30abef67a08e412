// Exact-weight projections on 16-row tiles: y = x . dequant(W)^T with x in FP32 or BF16 and W in Q4, Q5 or Q8, FP32
// accumulation (strixite kernels/linear_q4.hpp:23-58, moe_grouped.hpp:3-16, :93-104, linear_q8.hpp:13-14). It serves the
// FP32 activation mode and the Q5 experts (calls too small for it: a wave an output element, lanes_take), and the dense BF16
// projections that dense_plan.hpp sends here.
//
// A tile is the 16 A rows of v_mfma_f32_16x16x32_bf16 against RT tiles of 16 weight rows, the B columns. BF16: a row each
// of 16 slots of one expert (or tokens). FP32: x = hi + mid + lo, the top 16 bits of x, of the rest and of the rest of
// that (24 significant bits, exact), and the pieces of one row are three A rows, so a tile holds five rows and the
// matrix cores do one product where three passes over the weights' fragments would (at decode sizes a bucket rarely has
// more than five slots; 40 tokens: 276 experts, 1.4 slots each); an output is the sum of its three rows. A non-finite x
// makes its row NaN.
// Weights enter as integer codes exact in bf16 (Q4: 16 + n, Q5: 32 + n, Q8: c - 128) and each quantization group's
// product D is rescaled on the FP32 accumulator: w . x = s D' + m' sum(x), with D' and m' for the codes about the middle of
// their range (D' = D - EXTRA sum(x), m' = m + MID s). The error is relative to what the sums pass through, not to the
// result: D's running sum carries the offset (up to 31 or 63 times sum |x| a group), and D' and m' sum(x) cancel where a
// group's codes lie at one end of their range. Measured against 64 bits (2-norm, FP32, Q4 g128, K 3072): 1.3e-7
// with activations and weights of mean zero, 1.2e-6 with activations of mean and deviation 1, 2.6e-7 with codes 0 .. 2 and no
// min. sum(x) comes from one more MFMA, against ones.
//
// What bounds it: grouped, the weight stream beside ~80 vector instructions a wave per 32 k x 64 weight rows (the split
// and the codes' conversion); dense, latency, so K is split over the block's waves (8 from 32 steps, 4 from 8) and their
// parts meet in LDS in wave order. The split depends on K and the format only, so a per-slot call gives the grouped
// call's bits.
// Measured on MI355X: 40 tokens, H 3072, I 512, 512 experts top-10, Q4 g128, FP32 activations, one wave an output element
// before: gate_up 651 -> 179 us, down 897 -> 91 us (with the pieces as three MFMAs on one A tile: 201, 123; two weight tiles a
// wave instead of four: 222, 117), and with the scales through LDS (tile_dot) 34 us less for the two.
#include "common.hpp"
#include "exact_frag.hpp"
#include "exact_tile.hpp"
#include "route_small.hpp"

#include <algorithm>
#include <type_traits>

namespace strix::kernels::xt {
namespace {

using namespace strix::dev;
constexpr int kWave = 64;
constexpr int kMaxWaves = 8;  // waves a block

// The RT weight tiles' rows: a uniform first row each, and the lane's row in it (clamped at the last one for SwiGLU's
// ragged ends)
template <int RT> struct Rows {
    __amdgpu_buffer_rsrc_t q[RT], s[RT], m[RT];
    uint32_t j[RT];
};

// columns c0 + 16 t of an expert: SwiGLU takes gate tiles 0 .. RT / 2 - 1 and the matching up tiles; a tile past the
// columns reads the first one's rows (never stored)
template <int FMT, bool SWI, int RT>
__device__ __forceinline__ Rows<RT> tile_rows(const Args &a, int64_t expert, int64_t c0) {
    const int j = threadIdx.x % 16;
    const int64_t row_bytes = FMT == 8 ? a.K : FMT == 4 ? a.K / 2 : a.K / 2 + a.K / 8, groups = a.K / a.G;
    Rows<RT> r;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        int64_t c = c0 + 16 * (SWI ? t % (RT / 2) : t);
        if (c >= a.ncol) c = 0;
        const int64_t last = a.ncol - 1 - c;
        r.j[t] = j < last ? j : (uint32_t)last;
        const int64_t row = expert * a.N + c + (SWI && t >= RT / 2 ? a.ncol : 0);
        auto res = [](const void *p, int64_t bytes) {
            return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
        };
        const int64_t n = last < 15 ? last + 1 : 16;  // the tile's rows
        r.q[t] = res(a.q + row * row_bytes, n * row_bytes);
        r.s[t] = res(a.scale + row * groups, n * groups * 2);
        r.m[t] = res(a.minv + row * groups, n * groups * 2);
    }
    return r;
}

// LDS between the lanes of one wave
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// acc[t] = the tile's sums over K steps [s0, s1): lane (g, j) holds rows 4 g .. 4 g + 3 against weight row j of tile t.
// xp: the activation row of MFMA row lane % 16 (any row for an unused one: rows do not mix, and nobody reads its sums).
// sm: the wave's own LDS for the scales and mins of kWindow groups, [group][row] pairs. (Loaded as 2 bytes a row and step
// they were half of a step's loads, each a cache line a row for 2 bytes of it: per-slot gate_up of 80 slots, H 2560, I 1024,
// Q4 g32, FP32 303 us, now 124; 32 slots of Q5 g64, BF16, H 3072, I 1024 105, now 66; FP32 gate_up and down of 40 tokens at H
// 3072, I 512, Q4 g128 with the rest of their sublayer 320, now 286.)
constexpr int kWindow = 16;
template <int RT> constexpr int scale_words() { return kWindow * 16 * RT; }
template <int FMT, int SP, typename TX, int RT>
__device__ __forceinline__ void tile_dot(const Args &a, const Rows<RT> &rw, const TX *xp, int s0, int s1,
                                         uint32_t *sm, float4v (&acc)[RT]) {
    using F = Fmt<FMT, SP>;
    const int g = threadIdx.x % kWave / 16;
    const uint32_t row_bytes = (uint32_t)(FMT == 8 ? a.K : FMT == 4 ? a.K / 2 : a.K / 2 + a.K / 8);
    const uint32_t groups = (uint32_t)(a.K / a.G), G = (uint32_t)a.G;
    struct Buf {
        Codes c[RT];
        Act8<TX> x[F::NT];
    };
    auto fetch = [&](int s, Buf &b) {
        const uint32_t k = (uint32_t)s * SP + g * F::CPL;
#pragma unroll
        for (int t = 0; t < RT; ++t) load_codes<FMT, SP>(rw.q[t], rw.j[t] * row_bytes, (uint32_t)a.K, k, b.c[t]);
#pragma unroll
        for (int u = 0; u < F::NT; ++u) {
            b.x[u].load(xp + k + 8 * u);
        }
    };
    // the scales and mins of groups [w0, w0 + kWindow) that the wave's steps reach: consecutive lanes read consecutive groups of
    // a row. Rows past a tile's last one read zeros (their sums are not stored).
    uint32_t w0 = 0, w1 = 0;
    const uint32_t g_end = s1 > s0 ? ((uint32_t)s1 * SP - 1) / G + 1 : 0;
    auto stage = [&](uint32_t first) {
        w0 = first, w1 = first + kWindow;
        const uint32_t n = (w1 < g_end ? w1 : g_end) - w0;
        const int sh = n > 8 ? 4 : n > 4 ? 3 : n > 2 ? 2 : n > 1 ? 1 : 0;
        wave_sync();  // what the space held has been read
        for (uint32_t i0 = 0; i0 < 16u << sh; i0 += kWave) {
            // (lanes past the 16 rows and groups past the last repeat or read what nobody takes)
            const uint32_t i = i0 + threadIdx.x % kWave, row = (i >> sh) % 16, gi = i & ((1u << sh) - 1);
            const uint32_t o = (row * groups + w0 + gi) * 2;
            uint16_t sv[RT], mv[RT];
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                sv[t] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rw.s[t], o, 0, 0);
                mv[t] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rw.m[t], o, 0, 0);
            }
#pragma unroll
            for (int t = 0; t < RT; ++t) sm[gi * 16 * RT + 16 * t + row] = sv[t] | (uint32_t)mv[t] << 16;
        }
        wave_sync();
    };
    auto step = [&](Buf &b, int s, int next) {
        const Frag ones{{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u}};
        float4v d[RT], dx = {0, 0, 0, 0};  // dx: the activations' own sums
#pragma unroll
        for (int t = 0; t < RT; ++t) d[t] = float4v{0, 0, 0, 0};
#pragma unroll
        for (int u = 0; u < F::NT; ++u) {
            const Frag xf = b.x[u].frag(threadIdx.x % 16);
#pragma unroll
            for (int t = 0; t < RT; ++t) d[t] = mfma_bf16(xf, code_frag<FMT>(b.c[t], u), d[t]);
            dx = mfma_bf16(xf, ones, dx);
            __builtin_amdgcn_sched_barrier(0);  // a group of codes is decoded just before its MFMAs (registers)
        }
        float sc[RT], mp[RT];
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            const uint32_t w = sm[((uint32_t)s * SP / G - w0) * 16 * RT + 16 * t + threadIdx.x % 16];
            sc[t] = __uint_as_float(w << 16);
            mp[t] = fmaf(F::MID, sc[t], __uint_as_float(w & 0xFFFF0000u));
        }
        if (next < s1) fetch(next, b);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                const float n = F::EXTRA != 0.f ? fmaf(-F::EXTRA, dx[i], d[t][i]) : d[t][i];
                acc[t][i] = fmaf(sc[t], n, fmaf(mp[t], dx[i], acc[t][i]));
            }
    };
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t] = float4v{0, 0, 0, 0};
    Buf b0, b1;
    if (s0 < s1) fetch(s0, b0);
    if (s0 + 1 < s1) fetch(s0 + 1, b1);
    for (int s = s0; s < s1; s += 2) {
        if (((uint32_t)s + 1) * SP / G >= w1) stage((uint32_t)s * SP / G);  // (the first pair: w1 is 0)
        step(b0, s, s + 2);
        if (s + 1 < s1) step(b1, s + 1, s + 3);
    }
    wave_sync();  // the scales are read: the space is the caller's again
}

__device__ __forceinline__ void store(const Args &a, bool f32, int64_t row, int64_t col, float v) {
    if (f32) static_cast<float *>(a.y)[row * a.ldy + col] = v;
    else static_cast<uint16_t *>(a.y)[row * a.ldy + col] = f32_to_bf16(v);
}

__device__ __forceinline__ void report(uint32_t *err, int32_t id, int64_t slot) {
    if (atomicCAS(&err[0], 0u, 1u) == 0u) err[1] = (uint32_t)id, err[2] = (uint32_t)slot;
}

// MFMA row r's sum over the parts of ks waves (wave order), column j of tile t
template <int RT>
__device__ __forceinline__ float row_sum(const float4v (*red)[RT][kWave], int w0, int ks, int t, int r, int j) {
    auto at = [&](int w) { return reinterpret_cast<const float *>(&red[w][t][r / 4 * 16 + j])[r % 4]; };
    float v = at(w0);
    for (int w = 1; w < ks; ++w) v += at(w0 + w);
    return v;
}
// tile row r: the sum of its MFMA rows
template <typename TX, int RT>
__device__ __forceinline__ float tile_sum(const float4v (*red)[RT][kWave], int w0, int ks, int t, int r, int j) {
    const float v = row_sum<RT>(red, w0, ks, t, r, j);
    if constexpr (std::is_same_v<TX, float>)
        return v + (row_sum<RT>(red, w0, ks, t, r + 5, j) + row_sum<RT>(red, w0, ks, t, r + 10, j));
    return v;
}

// Block (tile, column block): ks waves split K (ks = 1: each of the block's waves takes a column block of its own). A
// grouped tile record holds up to 16 slots: FP32 takes them five at a time (the weights again from L1 / L2).
template <int FMT, int SP, bool SWI, typename TX, int RT>
__global__ void __launch_bounds__(kMaxWaves *kWave)
    exact_tile_kernel(Args a, int mode, bool y_f32, int tiles_bound, int cbs, int bpt, int ks) {
    static_assert(!SWI || RT % 2 == 0, "SwiGLU: gate and up tiles");
    constexpr int TC = SWI ? RT / 2 : RT, TR = tile_rows_of<TX>();  // column tiles; rows a tile
    __shared__ float4v red[kMaxWaves][RT][kWave];
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int g = lane / 16, j = lane % 16, nw = (int)(blockDim.x / kWave);
    const int tile = (int)(blockIdx.x / (uint32_t)bpt), cb = (int)(blockIdx.x % (uint32_t)bpt) * (nw / ks) + (ks > 1 ? 0 : wave);
    int64_t expert = 0;
    int rows, rec = 0;  // the record's rows; lane j: its row j as an output row
    bool nan = false;
    if (mode == GROUPED) {
        if (tile >= a.ws[0] || tile >= tiles_bound) return;  // whole block, before any barrier
        const int32_t *p = a.ws + route::Layout{a.S, a.E, 0, 0, 0}.t16_rec() + route::kRec16 * (int64_t)tile;
        const int32_t b = __builtin_amdgcn_readfirstlane(p[0]);
        nan = b < 0 || b >= a.E;
        expert = nan ? 0 : b;
        rows = __builtin_amdgcn_readfirstlane(p[2]);
        rec = p[4 + j];
    } else if (mode == PERSLOT) {
        const int32_t id = __builtin_amdgcn_readfirstlane(a.ids[tile]);
        nan = id < 0 || id >= a.E;
        expert = nan ? 0 : id;
        rows = 1, rec = tile;
        if (nan && blockIdx.x % (uint32_t)bpt == 0 && threadIdx.x == 0) report(a.err, id, tile);
    } else {
        rows = (int)(a.S - (int64_t)tile * TR < TR ? a.S - (int64_t)tile * TR : TR);
        rec = tile * TR + j;
    }
    const int64_t c0 = (int64_t)cb * 16 * TC;
    if (cb >= cbs) return;  // ks = 1 only (its waves meet no barrier)
    const int spans = (int)(a.K / SP), part = ks > 1 ? wave : 0;
    const Rows<RT> rw = tile_rows<FMT, SWI, RT>(a, expert, c0);
    for (int r0 = 0; r0 < rows; r0 += TR) {
        const int n = rows - r0 < TR ? rows - r0 : TR;
        const int xi = std::is_same_v<TX, float> ? (j < 15 ? j % 5 : 15) : j;  // the tile row of MFMA row j
        const int my = __shfl(rec, r0 + (xi < n ? xi : 0), kWave);
        const TX *xp = static_cast<const TX *>(a.x) + (int64_t)((uint32_t)my / (uint32_t)a.A) * a.K;
        float4v acc[RT];
        tile_dot<FMT, SP, TX, RT>(a, rw, xp, spans * part / ks, spans * (part + 1) / ks,
                                  reinterpret_cast<uint32_t *>(red[wave]), acc);  // the scales where its sums will go
#pragma unroll
        for (int t = 0; t < RT; ++t) red[wave][t][lane] = acc[t];
        if (ks > 1) __syncthreads();
        else wave_sync();
        // ks > 1: wave t finishes column tile t; else each wave its own. Lane (g, j): rows g, g + 4, ... of column j
        for (int r = 0; r < n; r += 4) {
            const int row = __shfl(rec, r0 + (r + g < n ? r + g : 0), kWave);
#pragma unroll
            for (int t = 0; t < TC; ++t) {
                const int64_t col = c0 + 16 * t + j;
                if ((ks > 1 && t != wave) || r + g >= n || col >= a.ncol) continue;
                const int w0 = ks > 1 ? 0 : wave;
                float v = tile_sum<TX, RT>(red, w0, ks, t, r + g, j);
                if constexpr (SWI) v = silu(v) * tile_sum<TX, RT>(red, w0, ks, RT / 2 + t, r + g, j);
                store(a, y_f32, row, col, nan ? qnan() : v);
            }
        }
        if (ks > 1 && r0 + TR < rows) __syncthreads();  // red is read before the next rows' parts
    }
}

// Block (token, 16 output columns): ks waves split K of a slot, sg slots at a time (kCombineWaves waves at most), each as
// exact_tile_kernel's one-row tile (MFMA rows 0, 5 and 10 of an FP32 slot, row 0 of a BF16 one), the slots' dots summed with
// the coefficients in slot order. What bounds it: latency, a round of K's walk for every sg slots. Measured on MI355X, H
// 3072, I 512, 10 slots a token, Q4 g128, FP32: 11 us at 1 token, 21 at 4 (a slot a round 44 and 47, a wave an output 20 and
// 67).
constexpr int kCombineWaves = 16;
template <int FMT, int SP, typename TX>
__global__ void __launch_bounds__(kCombineWaves *kWave)
    exact_perslot_combine_kernel(Args a, const float *coef, bool y_f32, int cbs, int ks, int sg) {
    constexpr bool F32 = std::is_same_v<TX, float>;
    __shared__ float red[2][kCombineWaves][kWave];  // lane (g, j), g < 3: MFMA row 5 g of column j
    __shared__ uint32_t sm[kCombineWaves][scale_words<1>()];
    __shared__ float cf[kWave];
    __shared__ int32_t sid[kWave];
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int g = lane / 16, j = lane % 16, sub = wave / ks, part = wave % ks, A = (int)a.A;
    const int64_t m = blockIdx.x / (uint32_t)cbs, c0 = (int64_t)(blockIdx.x % (uint32_t)cbs) * 16;
    if ((int)threadIdx.x < A) {  // A is at most 64: the first wave
        sid[threadIdx.x] = a.ids[m * A + threadIdx.x];
        cf[threadIdx.x] = coef[m * A + threadIdx.x];
    }
    const int spans = (int)(a.K / SP);
    float out = 0.f;
    bool bad = false;
    for (int s0 = 0, round = 0; s0 < A; s0 += sg, ++round) {
        float(&rb)[kCombineWaves][kWave] = red[round & 1];  // two buffers: one barrier a round
        if (s0 + sub < A) {
            const int64_t slot = m * A + s0 + sub;
            const int32_t id = __builtin_amdgcn_readfirstlane(a.ids[slot]);
            float4v acc[1];
            tile_dot<FMT, SP, TX, 1>(a, tile_rows<FMT, false, 1>(a, id < 0 || id >= a.E ? 0 : id, c0),
                                     static_cast<const TX *>(a.x) + slot * a.K, spans * part / ks, spans * (part + 1) / ks,
                                     sm[wave], acc);
            rb[wave][lane] = g == 0 ? acc[0][0] : g == 1 ? acc[0][1] : acc[0][2];
        }
        __syncthreads();
        if (threadIdx.x >= 16) continue;
        for (int s = 0; s < sg && s0 + s < A; ++s) {
            auto row_sum = [&](int i) {  // the parts in wave order
                float v = rb[s * ks][i];
                for (int w = 1; w < ks; ++w) v += rb[s * ks + w][i];
                return v;
            };
            float v = row_sum(j);
            if constexpr (F32) v += row_sum(16 + j) + row_sum(32 + j);
            out = fmaf(cf[s0 + s], v, out);
            const int32_t id = sid[s0 + s];
            const bool nan = id < 0 || id >= a.E;
            if (nan && !bad && c0 == 0 && threadIdx.x == 0) report(a.err, id, m * A + s0 + s);  // the token's first
            bad = bad || nan;
        }
    }
    if (threadIdx.x < 16 && c0 + j < a.ncol) store(a, y_f32, m, c0 + j, bad ? qnan() : out);
}

// One token: block (16 output columns), a wave a slot over all of K; the slots' dots meet in LDS. What bounds it: latency
// (the rows of eight to eleven experts, one round of loads a K step). A launch and the partials' round trip less than
// down and combine apart: measured on MI355X, H 2048, I 512, 8 slots, Q8: 7.0 + 4.4 -> 7.6 us; H 2560, I 640, 11 slots,
// Q4: 9.4 + 4.4 -> 8.1.
template <int FMT, int SP>
__global__ void __launch_bounds__(kOneTokenSlots *kWave)
    one_token_down_kernel(Args a, const float *coef, const uint16_t *resid, uint16_t *out) {
    __shared__ float dots[kOneTokenSlots][16], cf[kOneTokenSlots];
    __shared__ int bad[kOneTokenSlots];
    __shared__ uint32_t sm[kOneTokenSlots][scale_words<1>()];
    const int lane = threadIdx.x % kWave, slot = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int64_t c0 = (int64_t)blockIdx.x * 16;
    const int32_t id = __builtin_amdgcn_readfirstlane(a.ids[slot]);
    const bool nan = id < 0 || id >= a.E;
    const float c = coef[slot];
    const uint16_t xr = out != nullptr && threadIdx.x < 16 ? resid[c0 + threadIdx.x] : (uint16_t)0;
    float4v acc[1];
    tile_dot<FMT, SP, uint16_t, 1>(a, tile_rows<FMT, false, 1>(a, nan ? 0 : id, c0),
                                   static_cast<const uint16_t *>(a.x) + (int64_t)slot * a.K, 0, (int)(a.K / SP), sm[slot], acc);
    if (lane < 16) dots[slot][lane] = acc[0][0];  // MFMA row 0
    if (lane == 0) cf[slot] = c, bad[slot] = nan;
    __syncthreads();
    const int j = threadIdx.x;
    if (j >= 16) return;
    float v = 0.f;
    bool b = false;
    for (int s = 0; s < (int)a.A; ++s) v = fmaf(cf[s], dots[s][j], v), b = b || bad[s];
    const uint16_t y = f32_to_bf16(b ? qnan() : v);
    static_cast<uint16_t *>(a.y)[c0 + j] = y;
    if (out != nullptr) out[c0 + j] = f32_to_bf16(bf16_to_f32(xr) + bf16_to_f32(y));
}

// ---- small calls: a wave an output element ------------------------------------------------------------------------------
// Lane l takes the row's 32-code chunks l, l + 64, ...: acc = s (x . codes) + m sum(x) a chunk, FP32 with fmaf, the codes
// about the middle of their range as in the tiles, then a butterfly over the lanes. Every load of a row is in flight at once,
// so a call whose outputs do not fill the chip costs one round trip, where a tile's waves walk K two steps at a time; a row's
// codes are converted once an output, so its time grows with the outputs from there (lanes_take).
template <int FMT> struct ChunkCodes {
    static constexpr int W = FMT == 5 ? 4 : FMT;
    uint32_t w[W], hi;
    // chunk c of the row at p (FMT 5: low plane [K / 2], then bit 4 of code k at bit k % 8 of byte k / 8)
    __device__ __forceinline__ void load(const uint8_t *p, int64_t K, int64_t c) {
#pragma unroll
        for (int i = 0; i < W / 4; ++i) {
            const uint4 u = *reinterpret_cast<const uint4 *>(p + c * (4 * W) + 16 * i);
            w[4 * i] = u.x, w[4 * i + 1] = u.y, w[4 * i + 2] = u.z, w[4 * i + 3] = u.w;
        }
        if constexpr (FMT == 5) hi = *reinterpret_cast<const uint32_t *>(p + K / 2 + c * 4);
    }
    // code i about the middle of its range, as a signed field: its top bit turned over
    __device__ __forceinline__ void centre() {
        if constexpr (FMT == 5) hi = ~hi;
        else
#pragma unroll
            for (int i = 0; i < W; ++i) w[i] ^= FMT == 8 ? 0x80808080u : 0x88888888u;
    }
    __device__ __forceinline__ float code(int i) const {
        constexpr int bits = FMT == 8 ? 8 : 4, per = 32 / bits;
        const uint32_t v = w[i / per];
        const int at = bits * (i % per);
        if constexpr (FMT == 5)  // n - 16: the low plane's four bits, and -16 where bit 4 is clear
            return (float)((int32_t)((v >> at) & 15u) | ((int32_t)(hi << (31 - i)) >> 31) * 16);
        else return (float)((int32_t)(v << (32 - bits - at)) >> (32 - bits));
    }
};

// the dot of an activation row with a weight row, in every lane
template <int FMT, typename TX> __device__ __forceinline__ float lane_dot(const Args &a, const TX *xr, int64_t wrow) {
    const int64_t row_bytes = FMT == 8 ? a.K : FMT == 4 ? a.K / 2 : a.K / 2 + a.K / 8, groups = a.K / a.G;
    float acc = 0.f;
    for (int64_t c = threadIdx.x % kWave; c < a.K / 32; c += kWave) {
        ChunkCodes<FMT> cc;
        cc.load(a.q + wrow * row_bytes, a.K, c);
        cc.centre();
        const int64_t gi = wrow * groups + c * 32 / a.G;
        const float s = bf16_to_f32(a.scale[gi]), m = fmaf(Fmt<FMT, 32>::MID, s, bf16_to_f32(a.minv[gi]));
        float dot[4], xs[4];  // eight codes each: short chains of roundings
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            float v[8];
            if constexpr (std::is_same_v<TX, float>) {
                const float4 u = *reinterpret_cast<const float4 *>(xr + c * 32 + 8 * p),
                             w = *reinterpret_cast<const float4 *>(xr + c * 32 + 8 * p + 4);
                v[0] = u.x, v[1] = u.y, v[2] = u.z, v[3] = u.w, v[4] = w.x, v[5] = w.y, v[6] = w.z, v[7] = w.w;
            } else {
                const uint4 u = *reinterpret_cast<const uint4 *>(xr + c * 32 + 8 * p);
                const uint32_t d[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = __uint_as_float(i % 2 ? d[i / 2] & 0xffff0000u : d[i / 2] << 16);
            }
            dot[p] = v[0] * cc.code(8 * p), xs[p] = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
#pragma unroll
            for (int i = 1; i < 8; ++i) dot[p] = fmaf(v[i], cc.code(8 * p + i), dot[p]);
        }
        acc = fmaf(s, (dot[0] + dot[1]) + (dot[2] + dot[3]), fmaf(m, (xs[0] + xs[1]) + (xs[2] + xs[3]), acc));
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, kWave);
    return acc;
}

constexpr int kLaneBlock = 256;

// output row r of a grouped workspace is position r: its bucket by bisection of the offsets
template <int FMT, bool SWI, typename TX>
__global__ void __launch_bounds__(kLaneBlock) lane_rows_kernel(Args a, int mode, bool y_f32) {
    const uint32_t item = blockIdx.x * (kLaneBlock / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if (item >= (uint32_t)(a.S * a.ncol)) return;  // whole wave; no barrier in this kernel (lanes_take: few outputs)
    const uint32_t r = item / (uint32_t)a.ncol, j = item % (uint32_t)a.ncol;
    uint32_t row = r;  // DENSE: A is 1
    int32_t expert = 0;
    if (mode == GROUPED) {
        int32_t lo = 0, hi = (int32_t)a.E;  // buckets 0 .. E (E: invalid ids)
        while (lo < hi) {
            const int32_t mid = (lo + hi + 1) / 2;
            if (a.ws[4 + mid] <= (int32_t)r) lo = mid;
            else hi = mid - 1;
        }
        row = (uint32_t)a.ws[route::Layout{a.S, a.E, 0, 0, 0}.slots() + r], expert = lo;
    } else if (mode == PERSLOT) {
        expert = a.ids[r];
        if ((expert < 0 || expert >= a.E) && j == 0 && threadIdx.x % kWave == 0) report(a.err, expert, r);
    }
    const bool nan = expert < 0 || expert >= a.E;
    const int64_t w0 = (nan ? 0 : expert) * a.N + j;
    const TX *xr = static_cast<const TX *>(a.x) + (int64_t)(row / (uint32_t)a.A) * a.K;
    float v = lane_dot<FMT, TX>(a, xr, w0);
    if constexpr (SWI) v = silu(v) * lane_dot<FMT, TX>(a, xr, w0 + a.ncol);
    if (threadIdx.x % kWave == 0) store(a, y_f32, row, j, nan ? qnan() : v);
}

template <int FMT, typename TX>
__global__ void __launch_bounds__(kLaneBlock) lane_perslot_combine_kernel(Args a, const float *coef, bool y_f32) {
    const uint32_t item = blockIdx.x * (kLaneBlock / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if (item >= (uint32_t)(a.S * a.ncol)) return;  // whole wave; no barrier in this kernel
    const int64_t m = item / (uint32_t)a.ncol, n = item % (uint32_t)a.ncol;
    float out = 0.f;
    bool bad = false;
    for (int64_t slot = m * a.A; slot < (m + 1) * a.A; ++slot) {
        const int32_t id = a.ids[slot];
        const bool nan = id < 0 || id >= a.E;
        if (nan && n == 0 && threadIdx.x % kWave == 0) report(a.err, id, slot);
        bad = bad || nan;
        out = fmaf(coef[slot], lane_dot<FMT, TX>(a, static_cast<const TX *>(a.x) + slot * a.K, (nan ? 0 : id) * a.N + n), out);
    }
    if (threadIdx.x % kWave == 0) store(a, y_f32, m, n, bad ? qnan() : out);
}

// waves that split K: by the K steps alone (the bits of a dot follow from it)
int split_of(int64_t spans) { return spans >= 32 ? 8 : spans >= 8 ? 4 : 1; }

// the K step of a format and group size: the 16-byte load's span unless the group is smaller
template <typename F> void by_format(int fmt, int64_t G, F &&f) {
    using std::integral_constant;
    if (fmt == 4) {
        if (G == 128) f(integral_constant<int, 4>{}, integral_constant<int, 128>{});
        else if (G == 64) f(integral_constant<int, 4>{}, integral_constant<int, 64>{});
        else f(integral_constant<int, 4>{}, integral_constant<int, 32>{});
    } else if (fmt == 5) {
        if (G == 128) f(integral_constant<int, 5>{}, integral_constant<int, 128>{});
        else if (G == 64) f(integral_constant<int, 5>{}, integral_constant<int, 64>{});
        else f(integral_constant<int, 5>{}, integral_constant<int, 32>{});
    } else {
        if (G >= 64) f(integral_constant<int, 8>{}, integral_constant<int, 64>{});
        else f(integral_constant<int, 8>{}, integral_constant<int, 32>{});
    }
}

// Whether a call is small enough for a wave an output element (dots: outputs, SwiGLU's twice; BF16: Q5 only, the dense BF16
// calls' tiles being faster at every size). That form's time grows with dots x (K + 1400), 0.55 of that with BF16 activations,
// the tiles' with the K steps a wave walks (about 0.25 us each, 0.55 where eight waves split K), from about one start each; over
// 900 calls of 1 to 80 slots the line's choice is 1.016 of the better form's time on average. Measured on MI355X, wave / tiles,
// us: dense FP32, Q4 g128, N 1024, K 3072 at 4 tokens 9.9 / 12.2, at 8 16 / 13.6; N 4096, K 4096 at 1 11 / 13, at 2 19 / 14; Q8
// g64, N 640, K 5120 at 12 24 / 28; FP32 gate_up of 4 slots, H 2048, I 512, Q8 8.1 / 12.4, of 16 23 / 22; per-slot down of 7
// slots, K 128, N 3072, Q4 g32 12.7 / 6.1. And Q5 in groups under 128 with BF16 rows, long K, a slot an expert at most: the tiles
// then read the second plane 2 bytes a row and step for one row in 16 (K 2048, gate_up of 44 slots, I 1024 48 / 71; K 4096,
// I 768, 16 slots 1.21 of the wave's). By the slots' count and the shape alone, so that a per-slot call and a grouped one take
// the same form (the same bits). Error against 64 bits (2-norm, FP32): 0.9e-7 to 1.1e-7, the tiles 0.6e-7 to 1.3e-7.
bool lanes_take(int fmt, Act act, int64_t K, int64_t G, int64_t E, int64_t slots, int64_t dots) {
    if ((act != Act::F32 && fmt != 5) || dots >= 1 << 24) return false;
    if (act != Act::F32 && G < 128 && K >= 2048 && slots <= E) return true;
    const int64_t span = fmt == 8 ? std::min<int64_t>(G, 64) : G, spans = K / span, ks = split_of(spans);
    const double walk = (double)((spans + ks - 1) / ks) * (ks == 8 ? 55 : 25) * (G == 32 ? 0.8 : 1.0);
    return (double)dots * (double)(K + 1400) * (act == Act::F32 ? 1.0 : 0.55) < 1e5 * (15 + walk);
}
template <typename F> void by_lanes(int fmt, Act act, F &&f) {
    using std::integral_constant;
    auto by_act = [&](auto fc) {
        if (act == Act::F32) f(fc, float{});
        else f(fc, uint16_t{});
    };
    if (fmt == 5) by_act(integral_constant<int, 5>{});
    else if (fmt == 4) f(integral_constant<int, 4>{}, float{});  // BF16: Q5 only (lanes_take)
    else f(integral_constant<int, 8>{}, float{});
}

}  // namespace

void project(int fmt, Mode mode, bool swiglu, Act x_act, Act y_act, const Args &a, hipStream_t stream) {
    if (lanes_take(fmt, x_act, a.K, a.G, a.E, a.S, a.S * a.ncol * (swiglu ? 2 : 1))) {
        const unsigned blocks = (unsigned)((a.S * a.ncol + kLaneBlock / kWave - 1) / (kLaneBlock / kWave));
        return by_lanes(fmt, x_act, [&](auto fc, auto tx) {
            auto k = swiglu ? lane_rows_kernel<decltype(fc)::value, true, decltype(tx)>
                            : lane_rows_kernel<decltype(fc)::value, false, decltype(tx)>;
            k<<<blocks, kLaneBlock, 0, stream>>>(a, (int)mode, y_act == Act::F32);
        });
    }
    const int64_t tr = x_act == Act::F32 ? tile_rows_of<float>() : tile_rows_of<uint16_t>();
    const int64_t tiles = mode == GROUPED ? std::min(a.S, a.S / 16 + a.E + 2) : mode == DENSE ? (a.S + tr - 1) / tr : a.S;
    by_format(fmt, a.G, [&](auto fc, auto sc) {
        constexpr int FMT = decltype(fc)::value, SP = decltype(sc)::value;
        const int ks = split_of(a.K / SP), nw = ks > 1 ? ks : 4;
        auto go = [&](auto swc, auto tx, auto rtc) {
            constexpr bool SWI = decltype(swc)::value;
            constexpr int RT = decltype(rtc)::value, TC = SWI ? RT / 2 : RT;
            const int64_t cbs = (a.ncol + 16 * TC - 1) / (16 * TC), bpt = ks > 1 ? cbs : (cbs + nw - 1) / nw;
            STRIX_CHECK(tiles * bpt < (1ll << 31) && a.S < (1ll << 31), "exact projection: ", a.S, " x ", a.ncol,
                        " outputs, too many");
            exact_tile_kernel<FMT, SP, SWI, decltype(tx), RT>
                <<<(unsigned)(tiles * bpt), nw * kWave, 0, stream>>>(a, (int)mode, y_act == Act::F32, (int)tiles, (int)cbs,
                                                                     (int)bpt, ks);
        };
        auto by_rt = [&](auto swc, auto tx) {
            // four weight tiles a wave share the activations' pieces; two where four would leave most CUs without a block
            const int64_t tc4 = decltype(swc)::value ? 2 : 4;
            if (tiles * ((a.ncol + 16 * tc4 - 1) / (16 * tc4)) / (ks > 1 ? 1 : 4) < 2 * device_cus())
                go(swc, tx, std::integral_constant<int, 2>{});
            else go(swc, tx, std::integral_constant<int, 4>{});
        };
        auto by_x = [&](auto swc) {
            if (x_act == Act::F32) by_rt(swc, float{});
            else by_rt(swc, uint16_t{});
        };
        if (swiglu) by_x(std::true_type{});
        else by_x(std::false_type{});
    });
}

void perslot_combine(int fmt, Act act, const Args &a, const float *coef, hipStream_t stream) {
    if (lanes_take(fmt, act, a.K, a.G, a.E, a.S * a.A, a.S * a.A * a.ncol)) {  // as the grouped down of the same slots
        const unsigned blocks = (unsigned)((a.S * a.ncol + kLaneBlock / kWave - 1) / (kLaneBlock / kWave));
        return by_lanes(fmt, act, [&](auto fc, auto tx) {
            lane_perslot_combine_kernel<decltype(fc)::value, decltype(tx)>
                <<<blocks, kLaneBlock, 0, stream>>>(a, coef, act == Act::F32);
        });
    }
    const int64_t cbs = (a.ncol + 15) / 16;
    STRIX_CHECK(a.A >= 1 && a.A <= kWave && a.S * cbs < (1ll << 31), "exact per-slot combine: ", a.S, " tokens of ", a.A,
                " slots, ", a.ncol, " columns");
    by_format(fmt, a.G, [&](auto fc, auto sc) {
        constexpr int FMT = decltype(fc)::value, SP = decltype(sc)::value;
        // slots at a time: all that a block's waves hold while the blocks leave CUs idle, then four waves' worth (their rounds
        // overlap other blocks'; us, all / four waves: 10 slots, H 3072, I 512, Q4 g128 at 1 token 10.9 / 13.3, 3 24 / 21, 10 56
        // / 41; 4 slots, H 4096, I 512, Q4 g64 at 2 12.4 / 11.7, 6 28 / 22, 40 170 / 110)
        const int ks = split_of(a.K / SP), waves = a.S * cbs > 2 * device_cus() ? 4 : kCombineWaves;
        const int sg = (int)std::max<int64_t>(1, std::min<int64_t>(a.A, waves / ks));
        auto go = [&](auto tx) {
            exact_perslot_combine_kernel<FMT, SP, decltype(tx)>
                <<<(unsigned)(a.S * cbs), ks * sg * kWave, 0, stream>>>(a, coef, act == Act::F32, (int)cbs, ks, sg);
        };
        if (act == Act::F32) go(float{});
        else go(uint16_t{});
    });
}

void one_token_down(int fmt, const Args &a, const float *coef, const uint16_t *resid, uint16_t *out, hipStream_t stream) {
    STRIX_CHECK((fmt == 4 || fmt == 8) && a.A >= 1 && a.A <= kOneTokenSlots && a.ncol % 16 == 0, "one-token down: Q", fmt,
                ", ", a.A, " slots, ", a.ncol, " columns");
    by_format(fmt, a.G, [&](auto fc, auto sc) {
        constexpr int FMT = decltype(fc)::value, SP = decltype(sc)::value;
        if constexpr (FMT != 5)
            one_token_down_kernel<FMT, SP><<<(unsigned)(a.ncol / 16), (unsigned)a.A * kWave, 0, stream>>>(a, coef, resid, out);
    });
}

}  // namespace strix::kernels::xt
