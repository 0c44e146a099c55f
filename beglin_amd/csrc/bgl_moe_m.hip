// bgl_moe_m.hip -- the routed gather on the fp16 matrix cores (moe_ffn_batched, qwen_infer.c:5238-5350), for
// calls of several tokens.
//
// k_moe_x digitises every token in every tile's workgroup and multiplies three digits per value and token
// on the vector ALUs: at 64 tokens of the DeepSeek-V2-Lite layer that is what bounds it (gate+up 282 us,
// down 195 us for 470 and 240 MB).  Here a call's rows are split once into fp16 hi + lo (k_moe_frag;
// bgl_mfma.hip has the numerics: exact weights, activations to 2^-21 of themselves or 2^-38 of the row's
// maximum; rows of a wide range once more, with what that leaves over) and a workgroup multiplies 16 tokens at
// a time:
//
//   workgroup = one 64-row tile of one expert (gate and up rows together), 4 waves = 2 row halves x 2 K
//   slices.  A wave streams its 32 rows' weights straight from HBM (a pair of K-steps ahead, or two for
//   int4), decodes them once per 16 tokens and multiplies them by the tokens' fragments, read from the
//   L2: the rows of a segment lie anywhere, a lane reads 16 bytes of its own token's row.  Nothing is
//   staged and nothing synchronises until the slices' sums meet in LDS at the end.
//
// The weights are the MFMA's B operand, so a lane's sums lie in one weight row: its scale is one dword,
// loaded with the weights, and the store writes consecutive rows.  qNg64 n > 10 codes are not exact in
// fp16 as one number: the low byte and 256 times the rest are two operands (n = 11..15).  Affine int4
// takes codes minus 8 and adds (b + 8 s) * sum(x), the sum from two more products with ones.
// (DeepSeek-V2-Lite mixed layer at 64 / 8 tokens: 548 -> 242, 179 -> 154 us; affine int4 at 16 218 -> 125.)
//
// What bounds it: the weights' arrival at 12 waves per CU (mixed layer at 64 tokens: 3.0 TB/s over all seven
// launches).  3 waves per SIMD leave 168 registers, where 4 of the widest formats' gate+up spill; at 4 waves
// (128 registers) 89 did.  2 x 4 slices at 4 waves: 272 us at 64 tokens, 161 at 8, affine int4 at 16 123; 2 x 2
// at 4 waves 278, 167, 117; 2 x 2 at 3 waves 249, 149, 116.  (8 waves a workgroup fit a CU at 3 per SIMD only
// once.)  Sending the first weights out before the token's row number is known changed nothing (272, 162, 124).
#include <string.h>

#include "bgl_internal.h"
#include "bgl_mfma_a.h"

#define MM_COLS 16               // tokens per pass over the weights
#define MM_KS 2                  // K slices (waves) per row half
#define MM_WAVES (2 * MM_KS)

// ------------------------------------------------------------------ activation fragments
// One workgroup per row: x' = x * 2^(14-e) (e: exponent of the row's largest finite |x|) as hi = fp16(x')
// toward zero and lo = fp16(x' - hi) to nearest, in [row][K/32][hi: 32 halves | lo: 32 halves], eight values as
// {0,2,1,3,4,6,5,7}; xe[row] = {e - 14, bit 0: the row holds NaN or +-Inf (as 0 here)}.
// A row of a wide range (a 64-value group with as many elements below 2^(e-14) as bgl_x_level1 asks for: the
// parts then hold less than exact digits under that group's own exponent would) also gets the parts of what
// hi and lo leave over, times 2^MM_RES_BITS, res further on, and bit 1 in xe[row].y.
#define MM_RES_BITS 22
struct MoeFrag {
    const float *x[2];
    uint4 *fr[2];
    int2 *xe[2];
    int K[2], rows0;             // rows [0, rows0) belong to set 0
    size_t res;                  // from a row's parts to its leftover's, in uint4
};
// hi + lo of the scaled pair v0, v1; the leftover (exact, below 2^-8) in v0, v1
__device__ __forceinline__ void mm_parts2(float &v0, float &v1, uint32_t &h, uint32_t &l) {
    const mf_h2 hh = __builtin_bit_cast(mf_h2, __builtin_amdgcn_cvt_pkrtz(v0, v1));
    v0 -= (float)hh[0]; v1 -= (float)hh[1];
    const mf_h2 ll = mf_cvt_rn(v0, v1);
    v0 -= (float)ll[0]; v1 -= (float)ll[1];
    h = __builtin_bit_cast(uint32_t, hh);
    l = __builtin_bit_cast(uint32_t, ll);
}

__global__ __launch_bounds__(256) void k_moe_frag(MoeFrag F) {
    __shared__ uint32_t red[4];
    const int b = blockIdx.x, st = b >= F.rows0, row = st ? b - F.rows0 : b, K = F.K[st];
    const float *x = F.x[st] + (size_t)row * K;
    typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
    const int n8 = K / 8;
    uint32_t mb = 0u, nf = 0u, lo = 0x7fffffffu;
    f4u a[2], c[2];                                       // the first two slots stay in registers
    for (int i = threadIdx.x, j = 0; i < n8; i += 256, j++) {
        const f4u v = *reinterpret_cast<const f4u *>(x + 8 * i), w = *reinterpret_cast<const f4u *>(x + 8 * i + 4);
        if (j == 0) { a[0] = v; c[0] = w; }
        if (j == 1) { a[1] = v; c[1] = w; }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint32_t p = __float_as_uint(v[k]) & 0x7fffffffu, q = __float_as_uint(w[k]) & 0x7fffffffu;
            mb = max(mb, max(p < 0x7f800000u ? p : 0u, q < 0x7f800000u ? q : 0u));
            nf |= (p >= 0x7f800000u || q >= 0x7f800000u) ? 1u : 0u;
            lo = min(lo, min(p, q));
        }
    }
    mb = wave_max_u32(mb);
    nf = __any(nf) ? 1u : 0u;
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mb | (nf << 31);
    __syncthreads();
    mb = 0u; nf = 0u;
#pragma unroll
    for (int k = 0; k < 4; k++) { mb = max(mb, red[k] & 0x7fffffffu); nf |= red[k] >> 31; }
    int e = 0;
    const float mx = __uint_as_float(mb);
    if (mx > 0.0f) frexpf(mx, &e);
    const int sh = mx > 0.0f ? 14 - e : 0;
    uint4 *fr = F.fr[st] + (size_t)row * n8 * 2;
    auto slot = [&](int i, int j, float (&v8)[8]) {       // in the parts' order
        f4u v, w;
        if (j < 2) { v = j ? a[1] : a[0]; w = j ? c[1] : c[0]; }
        else { v = *reinterpret_cast<const f4u *>(x + 8 * i); w = *reinterpret_cast<const f4u *>(x + 8 * i + 4); }
        const float t[8] = {v.x, v.z, v.y, v.w, w.x, w.z, w.y, w.w};
#pragma unroll
        for (int k = 0; k < 8; k++) v8[k] = isfinite(t[k]) ? t[k] : 0.0f;
    };
    for (int i = threadIdx.x, j = 0; i < n8; i += 256, j++) {
        float v8[8];
        slot(i, j, v8);
        uint32_t H[4], Lo[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            float v0 = ldexpf(v8[2 * k], sh), v1 = ldexpf(v8[2 * k + 1], sh);
            mm_parts2(v0, v1, H[k], Lo[k]);
        }
        uint4 *d = fr + (i >> 2) * 8 + (i & 3);
        d[0] = make_uint4(H[0], H[1], H[2], H[3]);
        d[4] = make_uint4(Lo[0], Lo[1], Lo[2], Lo[3]);
    }
    bool wide = false;
    const float thr = ldexpf(1.0f, e - 14);
    const uint64_t low = __ballot(__uint_as_float(lo) < thr);
    if (low && mf_three_lanes(low))                       // (a group's 8 slots are 8 lanes, all of them or none in the row)
        for (int i = threadIdx.x, j = 0; i < n8; i += 256, j++) {
            float v8[8];
            slot(i, j, v8);
            int n = 0;                                    // small + 256 * large
#pragma unroll
            for (int k = 0; k < 8; k++) n += fabsf(v8[k]) >= thr ? 256 : v8[k] != 0.0f ? 1 : 0;
            n += dpp_i<0xB1>(n);
            n += dpp_i<0x4E>(n);
            n += dpp_i<0x141>(n);
            wide = wide || bgl_x_level1(n & 255, n >> 8);
        }
    wide = __syncthreads_or(wide);
    if (threadIdx.x == 0) F.xe[st][row] = make_int2(-sh, (int)(nf | (wide ? 2u : 0u)));
    if (!wide) return;
    fr += F.res;
    for (int i = threadIdx.x, j = 0; i < n8; i += 256, j++) {
        float v8[8];
        slot(i, j, v8);
        uint32_t H[4], Lo[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            float v0 = ldexpf(v8[2 * k], sh), v1 = ldexpf(v8[2 * k + 1], sh);
            mm_parts2(v0, v1, H[k], Lo[k]);
            v0 = ldexpf(v0, MM_RES_BITS); v1 = ldexpf(v1, MM_RES_BITS);
            mm_parts2(v0, v1, H[k], Lo[k]);
        }
        uint4 *d = fr + (i >> 2) * 8 + (i & 3);
        d[0] = make_uint4(H[0], H[1], H[2], H[3]);
        d[4] = make_uint4(Lo[0], Lo[1], Lo[2], Lo[3]);
    }
}

// ------------------------------------------------------------------ weights
// The operands of one K-step and row block: W of them (two for qNg64 n > 10, summed into one result).
template <int FMT, int NB> constexpr int mm_parts() { return FMT == BGL_QNG64 && NB > 10 ? 2 : 1; }

template <int FMT, int NB>
__device__ __forceinline__ void mm_decode(const ARaw<FMT, NB> &a, int q, mf_h8 (&w)[mm_parts<FMT, NB>()]) {
    if constexpr (mm_parts<FMT, NB>() == 2) {
        constexpr uint32_t MAG = 0x64006400u;
        constexpr int H4 = ARaw<FMT, NB>::H4, H2 = ARaw<FMT, NB>::H2, H1 = ARaw<FMT, NB>::H1;
        constexpr int SH2 = 4 * H4, SH1 = SH2 + 2 * H2;   // bit offsets above the low byte
        const uint32_t x0 = a.w[0] ^ 0x80808080u, x1 = a.w[1] ^ 0x80808080u;
        const mf_u4 lo = {sub_h2(and_or(x0, 0x00FF00FFu, MAG), (_Float16)-1024.0f), sub_h2(and_or(x0 >> 8, 0x00FF00FFu, MAG), (_Float16)-1024.0f),
                          sub_h2(and_or(x1, 0x00FF00FFu, MAG), (_Float16)-1024.0f), sub_h2(and_or(x1 >> 8, 0x00FF00FFu, MAG), (_Float16)-1024.0f)};
        w[0] = __builtin_bit_cast(mf_h8, lo);
        uint32_t u02 = 0, u13 = 0, u46 = 0, u57 = 0;
        int i = 2;
        if constexpr (H4) {
            const uint32_t v = a.w[i++];
            u02 |= v & 0x000F000Fu; u13 |= (v >> 8) & 0x000F000Fu; u46 |= (v >> 4) & 0x000F000Fu; u57 |= (v >> 12) & 0x000F000Fu;
        }
        if constexpr (H2) {
            const uint32_t v = a.w[i++] >> (4 * (q & 1));
            u02 |= (v & 0x00030003u) << SH2; u13 |= ((v >> 8) & 0x00030003u) << SH2;
            u46 |= ((v >> 2) & 0x00030003u) << SH2; u57 |= ((v >> 10) & 0x00030003u) << SH2;
        }
        if constexpr (H1) {
            const uint32_t v = a.w[i++] >> (2 * q);
            u02 |= (v & 0x00010001u) << SH1; u13 |= ((v >> 8) & 0x00010001u) << SH1;
            u46 |= ((v >> 1) & 0x00010001u) << SH1; u57 |= ((v >> 9) & 0x00010001u) << SH1;
        }
        // 256 * (u - 2^(n-9)): halves 1024 + u, minus, times 256 (all exact)
        const _Float16 off = (_Float16)(-(1024.0f + (float)(1 << (NB - 9))));
        const mf_h2 m = {(_Float16)256.0f, (_Float16)256.0f};
        auto up = [&](uint32_t u) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(mf_h2, sub_h2(u | MAG, off)) * m); };
        const mf_u4 hi = {up(u02), up(u13), up(u46), up(u57)};
        w[1] = __builtin_bit_cast(mf_h8, hi);
    } else if constexpr (FMT == BGL_MXFP4) {
        // the doubled E2M1 values 0, 1, 2, 3, 4, 6, 8, 12 have fp16 bytes 00, 3C, 40, 42, 44, 46, 48, 4A over
        // a zero low byte; the code's fourth bit is the sign
        auto hb = [&](uint32_t c) {                       // four codes (one per byte) -> four high bytes
            return __builtin_amdgcn_perm(0x4A484644u, 0x42403C00u, c & 0x07070707u) | ((c << 4) & 0x80808080u);
        };
        const uint32_t l = hb(a.w[0] & 0x0F0F0F0Fu), h = hb((a.w[0] >> 4) & 0x0F0F0F0Fu);
        const mf_u4 r = {(l << 8) & 0xFF00FF00u, l & 0xFF00FF00u, (h << 8) & 0xFF00FF00u, h & 0xFF00FF00u};
        w[0] = __builtin_bit_cast(mf_h8, r);
    } else {
        w[0] = dec_a<FMT, NB>(a, q);
    }
}

// the lane's row's scales of pair p (64 values): s[j] of K-step j; affine: also the bias b + 8 s
struct MmScale { uint32_t s, b; };
template <int FMT>
__device__ __forceinline__ MmScale mm_scale_ld(__amdgpu_buffer_rsrc_t rs, __amdgpu_buffer_rsrc_t rb, uint32_t row4, int U, int tile, int p) {
    MmScale r;
    r.b = 0u;
    if constexpr (FMT == BGL_QNG64) r.s = __builtin_amdgcn_raw_buffer_load_b32(rs, 2 * row4 + 4u * (p & 1), ((uint32_t)tile * U + (p >> 1)) * 512u, 0);
    else r.s = __builtin_amdgcn_raw_buffer_load_b32(rs, row4, ((uint32_t)tile * U + p) * 256u, 0);
    if constexpr (FMT == BGL_Q4G64A) r.b = __builtin_amdgcn_raw_buffer_load_b32(rb, row4, ((uint32_t)tile * U + p) * 256u, 0);
    return r;
}
template <int FMT> __device__ __forceinline__ float mm_scale(const MmScale &m, int j) {
    if constexpr (FMT == BGL_Q4G32H) return __half2float(__ushort_as_half((unsigned short)(m.s >> (16 * j))));
    else if constexpr (FMT == BGL_MXFP4) return mx_scale((m.s >> (8 * j)) & 255u);
    else return __uint_as_float(m.s);
}

// ------------------------------------------------------------------ one tile
template <int FMT, int NB, bool GLU>
__device__ __forceinline__ void moe_m_tile(const MoeTask &Mt, const BglDevTensor &Ta, const BglDevTensor &Tb, int tile, int s0, int s1,
                                           float *red) {
    constexpr int NM = GLU ? 2 : 1, PARTS = mm_parts<FMT, NB>();
    constexpr int RES = MM_KS * NM * 1024;                        // red: the sums, then those of the leftover
    constexpr int RD = Planes<FMT, NB>::WORDS <= 4 ? 2 : 1;       // K-step pairs of weights in flight
    constexpr bool PERSTEP = FMT == BGL_Q4G32H || FMT == BGL_MXFP4;   // a scale per K-step (32 values), else per pair
    constexpr bool AFF = FMT == BGL_Q4G64A;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, q = lane >> 4;
    const int rh = wave & 1, ks = wave >> 1;
    const int K = Ta.K, NP = K >> 6, U = Ta.nunits;
    const int per = (NP + MM_KS - 1) / MM_KS, p0 = min(ks * per, NP), p1 = min(p0 + per, NP);
    __amdgpu_buffer_rsrc_t rw[NM], rs[NM], rbias[NM];
#pragma unroll
    for (int m = 0; m < NM; m++) {
        const BglDevTensor &T = m ? Tb : Ta;
        rw[m] = mf_rsrc(T.w, (uint32_t)Ta.ntiles * Ta.cpr * 1024u);
        rs[m] = mf_rsrc(T.s0, (uint32_t)Ta.ntiles * U * 64u * scale_bytes<FMT>());
        rbias[m] = mf_rsrc(AFF ? (const void *)T.s1 : T.s0, (uint32_t)Ta.ntiles * U * 256u);
    }
    const AOff ao = a_offsets(2 * rh, lane);
    const uint32_t tchunk = (uint32_t)tile * Ta.cpr;
    const uint32_t row4 = (32u * rh + (lane & 15)) * 4u;          // scale byte offset of row block 0's row

    for (int c0 = s0, level = 0; c0 < s1;) {                      // level 1: rows of a wide range once more, with their leftover's parts
        // the lane's token (A operand row lane % 16; past the segment: its last one, not stored)
        const int sp = min(c0 + (lane & 15), s1 - 1);
        const int xrow = Mt.cols ? Mt.cols[sp] : sp;
        const BGL_GLOBAL bgl_u32x4 *xp = (const BGL_GLOBAL bgl_u32x4 *)(Mt.xfr) + (size_t)xrow * (K >> 2) + q + (level ? Mt.xres : 0);
        struct XF { mf_h8 h[2], l[2]; };
        auto load_x = [&](XF &f, int p) {
            const int pc = min(p, NP - 1);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                f.h[j] = __builtin_bit_cast(mf_h8, (bgl_u32x4)xp[(2 * pc + j) * 8]);
                f.l[j] = __builtin_bit_cast(mf_h8, (bgl_u32x4)xp[(2 * pc + j) * 8 + 4]);
            }
        };
        struct WP { PRaw<FMT, NB> w[NM]; MmScale s[NM][2]; };
        auto load_w = [&](WP &r, int m, int p) {
            const int pc = __builtin_amdgcn_readfirstlane(min(p, NP - 1));
            ld_pair<FMT, NB>(r.w[m], rw[m], ao, tchunk, 2 * pc);
#pragma unroll
            for (int b = 0; b < 2; b++) r.s[m][b] = mm_scale_ld<FMT>(rs[m], rbias[m], row4 + 64u * b, U, tile, pc);
        };
        mf_f4 acc[NM][2];
#pragma unroll
        for (int m = 0; m < NM; m++) { acc[m][0] = mf_f4{0, 0, 0, 0}; acc[m][1] = mf_f4{0, 0, 0, 0}; }
        WP ring[RD];
        XF xf[2];
        load_x(xf[0], p0);
#pragma unroll
        for (int d = 0; d < RD; d++)
#pragma unroll
            for (int m = 0; m < NM; m++) load_w(ring[d], m, p0 + d);
        // step p: the next pair's fragments go out before the next weights, so waiting for them (loads
        // complete in order) waits for no weights but the ones that step needs too
        auto step = [&](WP &r, const XF &x, XF &xn, int p) {
            load_x(xn, p + 1);
            mf_f4 sx = {0, 0, 0, 0};
            if constexpr (AFF) {
                const mf_u4 one = {0x3C003C00u, 0x3C003C00u, 0x3C003C00u, 0x3C003C00u};
                const mf_h8 ones = __builtin_bit_cast(mf_h8, one);
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    sx = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.h[j], ones, sx, 0, 0, 0);
                    sx = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.l[j], ones, sx, 0, 0, 0);
                }
            }
#pragma unroll
            for (int m = 0; m < NM; m++) {
                ARaw<FMT, NB> a[2][MF_RBW];
                exch<FMT, NB>(r.w[m], a, p & 1);
                const MmScale sc[2] = {r.s[m][0], r.s[m][1]};
                load_w(r, m, p + RD);
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    mf_f4 cg = {0, 0, 0, 0};
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        if (PERSTEP) cg = mf_f4{0, 0, 0, 0};
                        mf_h8 w[PARTS];
                        mm_decode<FMT, NB>(a[j][b], q, w);
#pragma unroll
                        for (int i = PARTS - 1; i >= 0; i--) {
                            cg = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.h[j], w[i], cg, 0, 0, 0);
                            cg = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.l[j], w[i], cg, 0, 0, 0);
                        }
                        if (PERSTEP) {
                            const float s = mm_scale<FMT>(sc[b], j);
#pragma unroll
                            for (int v = 0; v < 4; v++) acc[m][b][v] = __fmaf_rn(cg[v], s, acc[m][b][v]);
                        }
                    }
                    if (!PERSTEP) {
                        const float s = mm_scale<FMT>(sc[b], 0);
#pragma unroll
                        for (int v = 0; v < 4; v++) acc[m][b][v] = __fmaf_rn(cg[v], s, acc[m][b][v]);
                        if constexpr (AFF) {
                            const float bb = __fmaf_rn(8.0f, s, __uint_as_float(sc[b].b));
#pragma unroll
                            for (int v = 0; v < 4; v++) acc[m][b][v] = __fmaf_rn(sx[v], bb, acc[m][b][v]);
                        }
                    }
                }
            }
        };
        int p = p0;
        for (; p + 2 <= p1; p += 2) {
            step(ring[0], xf[0], xf[1], p);
            step(ring[RD - 1], xf[1], xf[0], p + 1);
        }
        if (p < p1) step(ring[0], xf[0], xf[1], p);

        // the slices' sums through LDS: [slice][matrix][row half][row block][v][lane]; the tokens' exponents
        // and flags (lane % 16) on their way meanwhile
        const int sq = min(c0 + (lane & 15), s1 - 1), xr = Mt.cols ? Mt.cols[sq] : sq;
        const int2 xq = Mt.xe[xr];
        float *my = red + (level ? RES : 0) + (size_t)ks * (NM * 1024) + rh * 512 + lane;
#pragma unroll
        for (int m = 0; m < NM; m++)
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int v = 0; v < 4; v++) my[m * 1024 + b * 256 + v * 64] = acc[m][b][v];
        __syncthreads();
        if (!level && __any(xq.y & 2)) {                          // uniform over the workgroup: the same 16 tokens
            level = 1;
            continue;
        }
        for (int o = threadIdx.x; o < 1024; o += MM_WAVES * 64) {
            const int tk = __builtin_amdgcn_readfirstlane(o >> 6), r = o & 63, n = tile * BGL_TILE + r, s = c0 + tk;
            if (s >= s1 || n >= Ta.N) continue;
            const float *src = red + (r >> 5) * 512 + ((r >> 4) & 1) * 256 + (tk & 3) * 64 + 16 * (tk >> 2) + (r & 15);
            const int row = __builtin_amdgcn_readlane(xr, tk);
            const int ex = __builtin_amdgcn_readlane(xq.x, tk), fl = __builtin_amdgcn_readlane(xq.y, tk);
            float val[NM];
#pragma unroll
            for (int m = 0; m < NM; m++) {
                float t = 0.0f;
#pragma unroll
                for (int k = 0; k < MM_KS; k++) t += src[(k * NM + m) * 1024];
                t = ldexpf(t, ex);
                if (fl & 2) {
                    float u = 0.0f;
#pragma unroll
                    for (int k = 0; k < MM_KS; k++) u += src[RES + (k * NM + m) * 1024];
                    t += ldexpf(u, ex - MM_RES_BITS);
                }
                if (fl & 1) {                                     // NaN, +-Inf: their products one at a time
                    const float *x = Mt.a.xf + (size_t)row * K;
#pragma unroll 1
                    for (int k = 0; k < K; k++)
                        if (!isfinite(x[k])) t += (m ? w_at_t<FMT, NB>(Tb, n, k) : w_at_t<FMT, NB>(Ta, n, k)) * x[k];
                }
                val[m] = t;
            }
            const float out = GLU ? (val[0] / (1.0f + expf(-val[0]))) * val[NM - 1] : val[0];
            Mt.y[(size_t)(Mt.ymap ? Mt.ymap[s] : s) * Mt.ystride + n] = out;
        }
        __syncthreads();
        level = 0;
        c0 += MM_COLS;
    }
}

// an expert's record through the constant address space (scalar loads, wave-uniform addresses)
__device__ __forceinline__ BglDevTensor mm_tensor(const BglDevTensor *p) {
    int w[sizeof(BglDevTensor) / 4];
    ucint q = uni(reinterpret_cast<const int *>(p));
#pragma unroll
    for (int i = 0; i < (int)(sizeof(BglDevTensor) / 4); i++) w[i] = q[i];
    BglDevTensor t;
    __builtin_memcpy(&t, w, sizeof t);
    return t;
}

// (down: 3 waves per SIMD at most, else the compiler gives up registers for a fourth: 4 tokens of the mixed
// layer 30.5 -> 37.8 us)
template <bool GLU>
__global__ __launch_bounds__(MM_WAVES * 64) __attribute__((amdgpu_waves_per_eu(3, GLU ? 8 : 3))) void k_moe_m(MoePair P) {
    __shared__ float red[2 * MM_KS * (GLU ? 2 : 1) * 1024];
    const int second = (int)blockIdx.x >= P.nb0, b = second ? (int)blockIdx.x - P.nb0 : (int)blockIdx.x;
    MoeTask Mt = P.t[0];
    if (second) Mt = P.t[1];
    const int e = b / Mt.tpe, tile = b - e * Mt.tpe;
    int s0, s1;
    if (Mt.off) { s0 = uni(Mt.off)[e]; s1 = uni(Mt.off)[e + 1]; }
    else { s0 = e * Mt.seg; s1 = min(s0 + Mt.seg, Mt.ncols); }    // one tensor, its columns in segments
    if (s0 >= s1) return;
    const BglDevTensor Ta = Mt.ta ? mm_tensor(Mt.ta + e) : Mt.da, Tb = GLU ? (Mt.tb ? mm_tensor(Mt.tb + e) : Mt.db) : Ta;
    if (tile >= Ta.ntiles) return;
#define MM_GO(F_, N_) moe_m_tile<F_, N_, GLU>(Mt, Ta, Tb, tile, s0, s1, red)
    switch (Ta.fmt) {
    case BGL_Q4G64: MM_GO(BGL_Q4G64, 0); break;
    case BGL_Q4G32H: MM_GO(BGL_Q4G32H, 0); break;
    case BGL_Q8G64: MM_GO(BGL_Q8G64, 0); break;
    case BGL_Q4G64A: MM_GO(BGL_Q4G64A, 0); break;
    case BGL_MXFP4: MM_GO(BGL_MXFP4, 0); break;
    case BGL_QNG64:
        switch (Ta.bits) {
        case 2: MM_GO(BGL_QNG64, 2); break;
        case 3: MM_GO(BGL_QNG64, 3); break;
        case 4: MM_GO(BGL_QNG64, 4); break;
        case 5: MM_GO(BGL_QNG64, 5); break;
        case 6: MM_GO(BGL_QNG64, 6); break;
        case 7: MM_GO(BGL_QNG64, 7); break;
        case 8: MM_GO(BGL_QNG64, 8); break;
        case 9: MM_GO(BGL_QNG64, 9); break;
        case 10: MM_GO(BGL_QNG64, 10); break;
        case 11: MM_GO(BGL_QNG64, 11); break;
        case 12: MM_GO(BGL_QNG64, 12); break;
        case 13: MM_GO(BGL_QNG64, 13); break;
        case 14: MM_GO(BGL_QNG64, 14); break;
        case 15: MM_GO(BGL_QNG64, 15); break;
        }
        break;
    }
#undef MM_GO
}

// ------------------------------------------------------------------ host side
bool bgl_moe_m_tensor(const BglDevTensor &T) {
    const bool f = T.fmt == BGL_Q4G64 || T.fmt == BGL_Q4G32H || T.fmt == BGL_Q8G64 || T.fmt == BGL_Q4G64A || T.fmt == BGL_MXFP4 ||
                   (T.fmt == BGL_QNG64 && T.bits >= 2 && T.bits <= 15);
    return f && (size_t)T.ntiles * T.cpr * 1024 < (1ull << 31) && (size_t)T.ntiles * T.nunits * 512 < (1ull << 31);
}

size_t bgl_moe_frag_bytes(long rows, int K) { return (size_t)rows * K * 4; }

void bgl_launch_moe_frag(const float *x0, int K0, int rows0, void *fr0, void *xe0, const float *x1, int K1, int rows1, void *fr1,
                         void *xe1, size_t res, hipStream_t st) {
    MoeFrag F;
    F.x[0] = x0; F.x[1] = x1;
    F.fr[0] = (uint4 *)fr0; F.fr[1] = (uint4 *)fr1;
    F.xe[0] = (int2 *)xe0; F.xe[1] = (int2 *)xe1;
    F.K[0] = K0; F.K[1] = K1;
    F.rows0 = rows0;
    F.res = res / 16;
    hipLaunchKernelGGL(k_moe_frag, dim3(rows0 + rows1), dim3(256), 0, st, F);
}

// The tasks' xfr / xe / xres hold their rows' fragments; b null: one task.  Both are SwiGLU launches or neither.
int bgl_launch_moe_m(const MoeTask &a, const MoeTask *b, hipStream_t st) {
    if (b && a.swiglu != b->swiglu) return -1;
    MoePair P;
    memset(&P, 0, sizeof P);
    P.t[0] = a;
    P.t[1] = b ? *b : a;
    P.nb0 = a.E * a.tpe;
    const dim3 g(P.nb0 + (b ? b->E * b->tpe : 0)), bl(MM_WAVES * 64);
    if (a.swiglu) hipLaunchKernelGGL((k_moe_m<true>), g, bl, 0, st, P);
    else hipLaunchKernelGGL((k_moe_m<false>), g, bl, 0, st, P);
    return 0;
}
