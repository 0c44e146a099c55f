// bgl_mfma_a.h -- weights as fp16 matrix-core operands: the raw loads of 32 rows (two 16-row blocks) of a
// 64-row tile, the lane exchange into the operand layout and the exact decode, shared by the dense GEMM
// (bgl_mfma.hip, where the layouts and the numerics are described) and the routed gather
// (bgl_moe_m.hip).
#pragma once
#include "bgl_gemv_impl.h"

typedef _Float16 mf_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 mf_h2 __attribute__((ext_vector_type(2)));
typedef float mf_f4 __attribute__((ext_vector_type(4)));
typedef unsigned int mf_u4 __attribute__((ext_vector_type(4)));
typedef unsigned int mf_u2 __attribute__((ext_vector_type(2)));

#define MF_RBW 2             // 16-row blocks per wave
#define MF_RSRC_W3 0x00020000   // buffer resource word 3 on gfx9: 32-bit data format, raw addressing

// ==================================================================================== weights
// Raw A-fragment words of one K-step for one lane (row 16*rb + lane%16, slot q = lane/16).
template <int FMT, int NB> struct ARaw { uint32_t w[1]; };
template <int NB> struct ARaw<BGL_Q8G64, NB> { uint32_t w[2]; };
template <int NB> struct ARaw<BGL_QNG64, NB> {
    static constexpr int H8 = (NB >> 3) & 1, H4 = (NB >> 2) & 1, H2 = (NB >> 1) & 1, H1 = NB & 1;
    uint32_t w[2 * H8 + H4 + H2 + H1 > 0 ? 2 * H8 + H4 + H2 + H1 : 1];
};

template <int FMT> constexpr int ksteps_per_unit() { return FMT == BGL_QNG64 ? 4 : 2; }
// quantization groups per unit: two for the fp16-pair (Q4G32H) and float2 (qNg64) scale words
template <int FMT> constexpr int groups_per_unit() { return FMT == BGL_Q4G32H || FMT == BGL_QNG64 ? 2 : 1; }
// bytes of scale data per row and unit in the device layout
template <int FMT> constexpr int scale_bytes() { return FMT == BGL_QNG64 ? 8 : 4; }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t mf_rsrc(const void *p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, MF_RSRC_W3);
}

// Code planes of a format: byte codes (q8g64; qNg64 with n >= 8), nibbles (int4; qNg64 bit 2 of
// n), crumbs and single bits (qNg64).
template <int FMT, int NB> struct Planes {
    static constexpr int P8 = FMT == BGL_Q8G64 ? 1 : FMT == BGL_QNG64 ? (NB >> 3) & 1 : 0;
    static constexpr int P4 = FMT == BGL_Q4G64 || FMT == BGL_Q4G32H || FMT == BGL_Q4G64A || FMT == BGL_MXFP4 ? 1 : FMT == BGL_QNG64 ? (NB >> 2) & 1 : 0;
    static constexpr int P2 = FMT == BGL_QNG64 ? (NB >> 1) & 1 : 0;
    static constexpr int P1 = FMT == BGL_QNG64 ? NB & 1 : 0;
    static constexpr int PX = P2 | P1;
    static constexpr int WORDS = 8 * P8 + 4 * P4 + 4 * PX;            // per lane and K-step pair
};

// Raw words of one K-step pair (s, s+1) for a wave's two 16-row blocks, as loaded.
//  - byte codes and nibbles are read a whole 16-byte chunk row per lane (one buffer_load_dwordx4
//    covers 32 rows of two chunks: lanes 32..63 take the second), so each quarter-wave reads 256
//    contiguous bytes; the MFMA operand layout (4 lanes per row) is rebuilt with lane swaps;
//  - crumbs and bits (2/n and 1/n of a qNg64 tensor's bytes): one chunk row of each covers the pair, so
//    one load brings both -- lanes < 32 the crumbs, lanes >= 32 the bits of the same 32 rows -- and lane
//    swaps hand a row's words to its four lanes.  (As the operand's own dwords they took 8 loads per
//    pair: 28672 x 4096 n = 7 at 8 columns 60 -> 48 us, n = 10 at 16 52 -> 47; the mixed gather 202 -> 167.)
template <int FMT, int NB> struct PRaw {
    using P = Planes<FMT, NB>;
    uint32_t w8[P::P8 ? 8 : 1];      // byte codes: K-step j of the pair in words 4j..4j+3
    uint32_t w4[P::P4 ? 4 : 1];      // nibbles: lanes < 32 K-step s, lanes >= 32 K-step s+1
    uint32_t wx[P::PX ? 4 : 1];      // crumb / bit chunk row
};

// Per-lane byte offsets within a tile's chunk, fixed for the kernel: the chunk-row reads (rows
// 16*rb0 + lane%32 of chunk lane/32), and the same rows without the chunk.
struct AOff { uint32_t op, row; };

__device__ __forceinline__ AOff a_offsets(int rb0, int lane) {
    AOff o;
    o.row = (uint32_t)(16 * rb0 + (lane & 31)) * 16u;
    o.op = (uint32_t)(lane >> 5) * 1024u + o.row;
    return o;
}

// Loads K-steps s, s+1 (s even, already clamped into the tensor) of the wave's rows; tchunk is the
// first chunk of the wave's tile.
template <int FMT, int NB>
__device__ __forceinline__ void ld_pair(PRaw<FMT, NB> &p, __amdgpu_buffer_rsrc_t rs, const AOff &o, uint32_t tchunk, int s) {
    using P = Planes<FMT, NB>;
    // both are wave-uniform; said so explicitly, so every offset below is a scalar operand (a value
    // the compiler cannot prove uniform would wrap each load in a loop over the lanes' values)
    tchunk = __builtin_amdgcn_readfirstlane(tchunk);
    s = __builtin_amdgcn_readfirstlane(s);
    if constexpr (FMT == BGL_Q8G64) {                    // K-step s is chunks 2s, 2s+1
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const mf_u4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, o.op, (tchunk + 2u * (s + j)) * 1024u, 0);
            p.w8[4 * j] = v[0]; p.w8[4 * j + 1] = v[1]; p.w8[4 * j + 2] = v[2]; p.w8[4 * j + 3] = v[3];
        }
    } else if constexpr (FMT == BGL_QNG64) {
        constexpr int K4 = 8 * P::P8, K2 = K4 + 4 * P::P4, K1 = K2 + 2 * P::P2;
        const uint32_t u = (uint32_t)s >> 2, j0 = (uint32_t)s & 3, c0 = tchunk + u * NB;
        if constexpr (P::P8) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const mf_u4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, o.op, (c0 + 2 * (j0 + j)) * 1024u, 0);
                p.w8[4 * j] = v[0]; p.w8[4 * j + 1] = v[1]; p.w8[4 * j + 2] = v[2]; p.w8[4 * j + 3] = v[3];
            }
        }
        if constexpr (P::P4) {
            const mf_u4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, o.op, (c0 + K4 + j0) * 1024u, 0);
            p.w4[0] = v[0]; p.w4[1] = v[1]; p.w4[2] = v[2]; p.w4[3] = v[3];
        }
        if constexpr (P::PX) {
            // crumbs: chunk K2 + half of the unit; bits: chunk K1 (= K2 + 2 beside crumbs)
            const uint32_t h = j0 >> 1;
            const uint32_t off = P::P2 && P::P1 ? o.op + (o.op - o.row) * (1u - h) : o.row;
            const mf_u4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, off, (c0 + (P::P2 ? K2 + h : K1)) * 1024u, 0);
            p.wx[0] = v[0]; p.wx[1] = v[1]; p.wx[2] = v[2]; p.wx[3] = v[3];
        }
    } else {                                             // int4: K-step s is chunk s
        const mf_u4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, o.op, (tchunk + (uint32_t)s) * 1024u, 0);
        p.w4[0] = v[0]; p.w4[1] = v[1]; p.w4[2] = v[2]; p.w4[3] = v[3];
    }
}

// Operand words of both K-steps and row blocks from a loaded pair.  Nibble chunks: a 4x4 transpose
// of (quarter-wave, word) -- quarter-wave 2j+rb holds rows 16rb..+15 of K-step j -- puts word q of
// row 16rb + r into lane (r, q), register 2j+rb.  Byte chunks: quarter-wave 2c+rb holds chunk c of
// rows 16rb..+15; swapping odd with even quarter-waves puts bytes 8q..8q+7 of the row (chunk q/2,
// words 2(q%2), +1) into lane (r, q), registers (2rb, 2rb+1).  Crumb and bit chunks: every word of a
// row's chunk goes to its four lanes; the crumb operand of K-step j is word 2j + q/2, the bit operand
// word 2h + j.  h: which half of its 128-value unit the pair is (qNg64).
template <int FMT, int NB>
__device__ __forceinline__ void exch(const PRaw<FMT, NB> &p, ARaw<FMT, NB> (&a)[2][MF_RBW], int h) {
    using P = Planes<FMT, NB>;
    int i = 0;
    if constexpr (P::P8) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const auto e = __builtin_amdgcn_permlane16_swap(p.w8[4 * j], p.w8[4 * j + 2], false, false);
            const auto f = __builtin_amdgcn_permlane16_swap(p.w8[4 * j + 1], p.w8[4 * j + 3], false, false);
            a[j][0].w[i] = e[0]; a[j][0].w[i + 1] = f[0];
            a[j][1].w[i] = e[1]; a[j][1].w[i + 1] = f[1];
        }
        i += 2;
    }
    if constexpr (P::P4) {
        const auto x = __builtin_amdgcn_permlane32_swap(p.w4[0], p.w4[2], false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(p.w4[1], p.w4[3], false, false);
        const auto c = __builtin_amdgcn_permlane16_swap(x[0], y[0], false, false);
        const auto d = __builtin_amdgcn_permlane16_swap(x[1], y[1], false, false);
        a[0][0].w[i] = c[0]; a[0][1].w[i] = c[1]; a[1][0].w[i] = d[0]; a[1][1].w[i] = d[1];
        i += 1;
    }
    if constexpr (P::PX) {
        // lanes >= 32 hold the bits (beside crumbs) or the same rows again
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int w = 0; w < 4; w++) {
            lo[w] = hi[w] = p.wx[w];
            if constexpr (P::P2 && P::P1) {
                const auto t = __builtin_amdgcn_permlane32_swap(p.wx[w], p.wx[w], false, false);
                lo[w] = t[0]; hi[w] = t[1];
            }
        }
        if constexpr (P::P2) {
            const uint32_t up = (threadIdx.x & 32) ? 0xffffffffu : 0u;   // q / 2 (masks: a select of array elements may go through memory)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint32_t w = (lo[2 * j + 1] & up) | (lo[2 * j] & ~up);
                const auto t = __builtin_amdgcn_permlane16_swap(w, w, false, false);
                a[j][0].w[i] = t[0]; a[j][1].w[i] = t[1];
            }
            i += 1;
        }
        if constexpr (P::P1) {
            const uint32_t hm = 0u - (uint32_t)h;
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const uint32_t w = (hi[2 + j] & hm) | (hi[j] & ~hm);
                const auto t = __builtin_amdgcn_permlane16_swap(w, w, false, false);
                a[j][0].w[i] = t[0]; a[j][1].w[i] = t[1];
            }
        }
    }
}

// Two floats as halves to nearest, in one v_cvt_pk_f16_f32: the lo parts (the hi parts go toward zero).
__device__ __forceinline__ mf_h2 mf_cvt_rn(float a, float b) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    const f2 v = {a, b};
    return __builtin_convertvector(v, mf_h2);
}

// Whether three of some byte's bits are set (scalar work).  Lanes 8g..8g+7 hold a 64-value group, 8 values
// each: bgl_x_level1 wants 22 small ones (or 33 small and zero ones), so at least three of them hold one.
__device__ __forceinline__ bool mf_three_lanes(uint64_t m) {
    m -= (m >> 1) & 0x5555555555555555ull;
    m = (m & 0x3333333333333333ull) + ((m >> 2) & 0x3333333333333333ull);
    m = (m + (m >> 4)) & 0x0F0F0F0F0F0F0F0Full;
    return ((m + 0x7D7D7D7D7D7D7D7Dull) & 0x8080808080808080ull) != 0;
}

__device__ __forceinline__ uint32_t sub_h2(uint32_t p, _Float16 c) {
    mf_h2 v = __builtin_bit_cast(mf_h2, p);
    const mf_h2 cc = {c, c};
    v = v + cc;                                          // exact: both operands and the result are fp16 integers
    return __builtin_bit_cast(uint32_t, v);
}

// (a & m) | o in one v_and_or_b32.  gfx9's three-operand encoding takes no literal constant and
// reads at most one scalar register, so m comes in a scalar register and o in a vector register.
__device__ __forceinline__ uint32_t and_or(uint32_t a, uint32_t m, uint32_t o) {
    uint32_t r;
    asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(m), "v"(o));
    return r;
}

// Codes of the lane's 8 elements as halves in the order {0,2,1,3,4,6,5,7}.
template <int FMT, int NB>
__device__ __forceinline__ mf_h8 dec_a(const ARaw<FMT, NB> &a, int q) {
    constexpr uint32_t MAG = 0x64006400u;                // fp16 1024.0 in both halves
    uint32_t p02, p13, p46, p57;
    _Float16 off;
    if constexpr (FMT == BGL_Q8G64) {
        const uint32_t x0 = a.w[0] ^ 0x80808080u, x1 = a.w[1] ^ 0x80808080u;   // u = code + 128
        p02 = and_or(x0, 0x00FF00FFu, MAG); p13 = and_or(x0 >> 8, 0x00FF00FFu, MAG);
        p46 = and_or(x1, 0x00FF00FFu, MAG); p57 = and_or(x1 >> 8, 0x00FF00FFu, MAG);
        off = (_Float16)-1152.0f;
    } else if constexpr (FMT == BGL_QNG64) {
        constexpr int H8 = ARaw<FMT, NB>::H8, H4 = ARaw<FMT, NB>::H4, H2 = ARaw<FMT, NB>::H2, H1 = ARaw<FMT, NB>::H1;
        constexpr int SH4 = 8 * H8, SH2 = SH4 + 4 * H4, SH1 = SH2 + 2 * H2;
        uint32_t u02 = 0, u13 = 0, u46 = 0, u57 = 0;
        int i = 0;
        if constexpr (H8) {
            const uint32_t x0 = a.w[i] ^ 0x80808080u, x1 = a.w[i + 1] ^ 0x80808080u;
            u02 = x0 & 0x00FF00FFu; u13 = (x0 >> 8) & 0x00FF00FFu;
            u46 = x1 & 0x00FF00FFu; u57 = (x1 >> 8) & 0x00FF00FFu;
            i += 2;
        }
        if constexpr (H4) {
            const uint32_t w = a.w[i++];
            u02 |= (w & 0x000F000Fu) << SH4; u13 |= ((w >> 8) & 0x000F000Fu) << SH4;
            u46 |= ((w >> 4) & 0x000F000Fu) << SH4; u57 |= ((w >> 12) & 0x000F000Fu) << SH4;
        }
        if constexpr (H2) {
            const uint32_t w = a.w[i++] >> (4 * (q & 1));   // crumbs 2(q%2) (elements 0..3) and +1 (4..7)
            u02 |= (w & 0x00030003u) << SH2; u13 |= ((w >> 8) & 0x00030003u) << SH2;
            u46 |= ((w >> 2) & 0x00030003u) << SH2; u57 |= ((w >> 10) & 0x00030003u) << SH2;
        }
        if constexpr (H1) {
            const uint32_t w = a.w[i++] >> (2 * q);          // bits 2q (elements 0..3) and 2q+1 (4..7)
            u02 |= (w & 0x00010001u) << SH1; u13 |= ((w >> 8) & 0x00010001u) << SH1;
            u46 |= ((w >> 1) & 0x00010001u) << SH1; u57 |= ((w >> 9) & 0x00010001u) << SH1;
        }
        p02 = u02 | MAG; p13 = u13 | MAG; p46 = u46 | MAG; p57 = u57 | MAG;
        off = (_Float16)(-(1024.0f + (float)(1 << (NB - 1))));
    } else {
        const uint32_t w = a.w[0];
        p02 = and_or(w, 0x000F000Fu, MAG); p13 = and_or(w >> 8, 0x000F000Fu, MAG);
        p46 = and_or(w >> 4, 0x000F000Fu, MAG); p57 = and_or(w >> 12, 0x000F000Fu, MAG);
        off = (_Float16)-1032.0f;
    }
    mf_u4 r = {sub_h2(p02, off), sub_h2(p13, off), sub_h2(p46, off), sub_h2(p57, off)};
    return __builtin_bit_cast(mf_h8, r);
}
