// MFMA fragments of exact products (exact_tile.hip, hc.hip): quantized codes as small integers exact in bf16, FP32
// activations as three bf16 pieces that sum to them exactly.
#pragma once

#include "common.hpp"

#include <type_traits>

namespace strix::kernels::xt {

using namespace strix::dev;

// A K step covers SP codes of a row (one quantization group at most): 4 lane groups x CPL codes
template <int FMT, int SP> struct Fmt {
    static constexpr int W = FMT == 8 ? 8 : 4;       // bits a code in the first plane
    static constexpr int CPL = SP / 4, LB = CPL * W / 8, NT = CPL / 8;
    // a code enters as EXTRA + (n - MID), MID the middle of its range
    static constexpr float MID = FMT == 4 ? 8.f : FMT == 5 ? 16.f : 128.f, EXTRA = FMT == 4 ? 24.f : FMT == 5 ? 48.f : 0.f;
    static_assert(LB == 16 || LB == 8 || LB == 4, "bytes a lane loads a step");
};

struct Codes {
    uint32_t w[4], hi;
};

// row: byte offset of the lane's row from the tile's first (a uniform buffer resource: no 64-bit lane addresses)
template <int FMT, int SP>
__device__ __forceinline__ void load_codes(__amdgpu_buffer_rsrc_t rq, uint32_t row, uint32_t K, uint32_t k, Codes &c) {
    using F = Fmt<FMT, SP>;
    const uint32_t p = row + k * F::W / 8;
    if constexpr (F::LB == 16) {
        typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
        const u32x4v u = __builtin_amdgcn_raw_buffer_load_b128(rq, p, 0, 0);
        c.w[0] = u.x, c.w[1] = u.y, c.w[2] = u.z, c.w[3] = u.w;
    } else if constexpr (F::LB == 8) {
        typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));
        const u32x2v u = __builtin_amdgcn_raw_buffer_load_b64(rq, p, 0, 0);
        c.w[0] = u.x, c.w[1] = u.y;
    } else {
        c.w[0] = __builtin_amdgcn_raw_buffer_load_b32(rq, p, 0, 0);
    }
    if constexpr (FMT == 5) {  // bit 4 of the codes: code k at bit k % 8 of byte k / 8 of the row's second plane
        const uint32_t h = row + K / 2 + k / 8;
        if constexpr (F::CPL == 32) c.hi = __builtin_amdgcn_raw_buffer_load_b32(rq, h, 0, 0);
        else if constexpr (F::CPL == 16) c.hi = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rq, h, 0, 0);
        else c.hi = (uint8_t)__builtin_amdgcn_raw_buffer_load_b8(rq, h, 0, 0);
    }
}

// bits 0, 2, 4, 6 of e to bit 6 of the bytes 0 .. 3
__device__ __forceinline__ uint32_t spread_bits(uint32_t e) {
    e &= 0x55u;
    return ((e << 6) | (e << 12) | (e << 18) | (e << 24)) & 0x40404040u;
}

// codes 8 u .. 8 u + 7 of the lane as bf16 (OFF + code) in the paired k order k0 k2 k4 k6 k1 k3 k5 k7
template <int FMT> __device__ __forceinline__ Frag code_frag(const Codes &c, int u) {
    if constexpr (FMT == 8) {
        const uint32_t a = c.w[2 * u] ^ 0x80808080u, b = c.w[2 * u + 1] ^ 0x80808080u;  // c - 128, signed
        auto sb = [](uint32_t w, int i) { return (float)(int8_t)(uint8_t)(w >> (8 * i)); };
        return Frag{{hi16_pair(sb(a, 0), sb(a, 2)), hi16_pair(sb(b, 0), sb(b, 2)), hi16_pair(sb(a, 1), sb(a, 3)),
                     hi16_pair(sb(b, 1), sb(b, 3))}};
    } else {
        const uint32_t w = c.w[u];
        uint32_t t, v, top;
        if constexpr (FMT == 4) {  // 0x4180 | n << 3 = 16 + n
            t = ((w << 3) & 0x78787878u) | 0x80808080u, v = ((w >> 1) & 0x78787878u) | 0x80808080u, top = 0x41414141u;
        } else {  // 0x4200 | n << 2 = 32 + n
            const uint32_t h = c.hi >> (8 * u);
            t = ((w << 2) & 0x3C3C3C3Cu) | spread_bits(h), v = ((w >> 2) & 0x3C3C3C3Cu) | spread_bits(h >> 1);
            top = 0x42424242u;
        }
        return Frag{{__builtin_amdgcn_perm(top, t, 0x04010400u), __builtin_amdgcn_perm(top, t, 0x04030402u),
                     __builtin_amdgcn_perm(top, v, 0x04010400u), __builtin_amdgcn_perm(top, v, 0x04030402u)}};
    }
}

// Activation rows of the MFMA: BF16 rows are themselves (16 a tile). An FP32 row is three MFMA rows, one per bf16 piece,
// so a tile holds five: MFMA row r is piece r / 5 of the tile's row r % 5 (row 15 unused), and an output is the sum of
// its three rows'.
template <typename TX> constexpr int tile_rows_of() { return std::is_same_v<TX, float> ? 5 : 16; }

// 8 activations of MFMA row j as bf16 in the paired order
template <typename TX> struct Act8;
template <> struct Act8<float> {
    float4 a, b;
    __device__ __forceinline__ void load(const float *p) {
        a = *reinterpret_cast<const float4 *>(p), b = *reinterpret_cast<const float4 *>(p + 4);
    }
    // piece j / 5: the top 16 bits of x, of the rest, of the rest of that (exact: 24 significant bits)
    __device__ __forceinline__ Frag frag(int j) const {
        const uint32_t m1 = j >= 5 ? 0xFFFF0000u : 0u, m2 = j >= 10 ? 0xFFFF0000u : 0u;
        float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[i] -= __uint_as_float(__float_as_uint(v[i]) & m1);
            v[i] -= __uint_as_float(__float_as_uint(v[i]) & m2);
        }
        return Frag{{hi16_pair(v[0], v[2]), hi16_pair(v[4], v[6]), hi16_pair(v[1], v[3]), hi16_pair(v[5], v[7])}};
    }
};
template <> struct Act8<uint16_t> {
    uint4 a;
    __device__ __forceinline__ void load(const uint16_t *p) { a = *reinterpret_cast<const uint4 *>(p); }
    __device__ __forceinline__ Frag frag(int) const {
        return Frag{{__builtin_amdgcn_perm(a.y, a.x, 0x05040100u), __builtin_amdgcn_perm(a.w, a.z, 0x05040100u),
                     __builtin_amdgcn_perm(a.y, a.x, 0x07060302u), __builtin_amdgcn_perm(a.w, a.z, 0x07060302u)}};
    }
};

}  // namespace strix::kernels::xt
