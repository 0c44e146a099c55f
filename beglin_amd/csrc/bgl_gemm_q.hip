// bgl_gemm_q.hip -- W4A8 products of many columns (and of 2..16 over many rows) on the matrix cores
// (gemm_qXg64_sdot_mt, q4gemv.h:779-791; gemm_q4g256sf_sdot_mt, q4gemv_g256.h:366-383; q4g64, q8g64,
// g256sf, plain g256): up to 64 columns per launch, every (row, column) folded by the wave that owns it.
//
// The reference's sum is sequential: acc += ((isum * wscale) * ascale) over the groups in order, each
// step rounded to fp32 (g256sf: ((comb * wsuper) * (1/63)) * ascale).  Bit-identical outputs leave
// four vector instructions per output and group (convert, two products, one sum) -- that, not the
// integer products, bounds these launches: 28672 x 4096 at 64 columns is 117 M folds, 14 us of every
// SIMD, against 4 us of v_mfma_i32 and 13 us of weight bytes (measured: 27 us; 4 launches of
// k_gemv_qm, 16 columns each, took 216).  So little else may cost vector instructions per output:
//   - a wave owns a whole tile of rows x columns and walks K in group order with the sums in
//     registers (no terms through LDS, no second pass);
//   - the weights are the MFMA's B operand, so a lane's outputs all lie in ONE weight row (the lane's)
//     and 4 or 16 columns: the weight scale is one register, loaded with the weights; the activation
//     scales of the lane's columns are 16-byte LDS broadcasts;
//   - int4 codes are used as 16 * (code - 8), which is two bit operations per four codes, and the
//     activation scales are staged as their sixteenth: every rounding step scales by 16 exactly, as
//     long as the weight scales stay far from the ends of fp32 (checked; else the tile is done again
//     with the integer sums shifted back).
//
// Tiles: 32 rows x 32 columns through v_mfma_i32_32x32x32_i8, where a lane's 16-byte weight load (one
// chunk = 32 int4 codes of its row) is exactly its operand of the two products of a 64-value group,
// with no lane exchange; a workgroup is the 64 rows of one device tile x up to 64 columns.  Launches
// with too few such tiles take 16 x 16 tiles through v_mfma_i32_16x16x64_i8 (8-byte loads), a
// workgroup being 16 rows x up to 64 columns.
//
// The codes are quantized once per launch by k_act_q_tiles (k_act_w4a8's arithmetic, optionally with
// the MLP block's SwiGLU) straight into the operand order: per 64-value group and 32 columns, [part]
// [lane][16 bytes] with lane = 32 h + column % 32 holding values 32 h + 16 part .. + 15 -- or, for the
// 32-row int4 tiles, dwords part, part + 2, .. of its 32 values (those the low / high nibbles of its
// chunk multiply).  Its scales are [group][column], a sixteenth for int4 (exact: a scale is at least
// 1e-8 / 127).  The codes are read from the L2 (M x K bytes) and the weights from HBM through one
// register ring per wave, 8 or 16 groups deep: with the weights left out the same launch takes 26 us
// of its 31 under the tracer, without the folds 30, so what is left is the latency of two waves per
// SIMD.  (Tried: a producer wave filling an LDS ring of weights, one barrier per 4-8 groups, 51 us;
// 3 waves per SIMD, spilled; the scales staged through registers, spilled.)
#include <string.h>

#include <algorithm>

#include "bgl_gemv_q.h"
#include "bgl_internal.h"

#define HIPCHK(expr)                                                                             \
    do {                                                                                         \
        hipError_t e_ = (expr);                                                                  \
        if (e_ != hipSuccess) return bgl_fail(BGL_E_HIP, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

#define GQ_COLS 64            // columns per launch
#define GQ_LDS_MAX (150 * 1024)   // the launch's activation scales: K/group x columns floats

// fp32 rows of the caller: 16-byte accesses that assume no more than a float's alignment
typedef float gq_f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned int gq_u4 __attribute__((ext_vector_type(4)));
typedef unsigned int gq_u2 __attribute__((ext_vector_type(2)));
typedef int gq_i4 __attribute__((ext_vector_type(4)));
typedef int gq_i16 __attribute__((ext_vector_type(16)));

struct GemmQLaunch {
    GemvTask t[BGL_MAX_TASKS];     // blk0 in workgroups
    int ntasks;
    const uint8_t *xt;             // codes in operand order, [K/64][CB32][2][64][16]
    const float *as;               // activation scales [K/gq][GQ_COLS], rows in fours
    int cb32;                      // 32-column blocks of the launch
    int m0, mcols;                 // columns [m0, m0 + mcols) of y
};

// ------------------------------------------------------------------ activations in operand order
// One wave per column and 256 values (lane l: values 4l..4l+3): q4_quant_act_i8 / _g256 bit for bit
// (k_act_w4a8's comment has the non-finite cases), GQ = 64 or 256.  u != null: the column is
// h = silu(x) * u, also written to h.
template <int GQ>
__global__ __launch_bounds__(256) void k_act_q_tiles(const float *__restrict__ x, int M, int K, int cb32, int split, float am, uint8_t *__restrict__ xt,
                                                     float *__restrict__ as, const float *__restrict__ u, float *__restrict__ h) {
    const int NP = (K + 255) / 256;
    const int wid = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6), lane = threadIdx.x & 63;
    if (wid >= M * NP) return;
    const int m = wid / NP, p = wid % NP, k = 256 * p + 4 * lane;
    const bool in = k < K;                                       // K % 64 == 0: whole 16-lane rows are in or out
    const size_t o = (size_t)m * K + (in ? k : 0);
    const gq_f4u xv = *reinterpret_cast<const gq_f4u *>(x + o);
    float4 v = make_float4(xv.x, xv.y, xv.z, xv.w);
    if (u) {
        const gq_f4u uv = *reinterpret_cast<const gq_f4u *>(u + o);
        auto sw = [](float g, float w) {
            const float e = (float)exp(-(double)g);
            return __fmul_rn(__fdiv_rn(g, __fadd_rn(1.0f, e)), w);
        };
        v = make_float4(sw(v.x, uv.x), sw(v.y, uv.y), sw(v.z, uv.z), sw(v.w, uv.w));
        if (in) *reinterpret_cast<gq_f4u *>(h + o) = gq_f4u{v.x, v.y, v.z, v.w};
    }
    uint32_t mb = umax(umax(abs_bits(v.x), abs_bits(v.y)), umax(abs_bits(v.z), abs_bits(v.w)));
    if (GQ == 256) {
        mb = in ? mb : 0u;
        mb = wave_max_u32(mb);
    } else {
        mb = umax(mb, dpp_u<0xB1>(mb));
        mb = umax(mb, dpp_u<0x4E>(mb));
        mb = umax(mb, dpp_u<0x141>(mb));
        mb = umax(mb, dpp_u<0x140>(mb));                         // the 16-lane row's maximum
    }
    const bool nf = mb >= 0x7f800000u;
    const float sc = __fdiv_rn(__uint_as_float(umax(mb, __float_as_uint(1e-8f))), 127.0f), inv = __fdiv_rn(1.0f, sc);
    if (!in) return;
    const uint32_t w = quant_byte(v.x, inv, nf) | (quant_byte(v.y, inv, nf) << 8) | (quant_byte(v.z, inv, nf) << 16) |
                       (quant_byte(v.w, inv, nf) << 24);
    const int g = k >> 6, l = lane & 15;                          // 64-value group, dword within it
    const int part = split ? l & 1 : (l >> 2) & 1, dw = split ? (l >> 1) & 3 : l & 3;
    const size_t at = ((size_t)(g * cb32 + (m >> 5)) * 2 + part) * 1024 + (size_t)(32 * (l >> 3) + (m & 31)) * 16 + 4 * dw;
    *reinterpret_cast<uint32_t *>(xt + at) = w;
    if (GQ == 256 ? lane == 0 : l == 0) as[(size_t)(GQ == 256 ? p : g) * GQ_COLS + m] = __fmul_rn(sc, am);
}

// ------------------------------------------------------------------ the product
template <int FMT> struct GqFmt {
    static constexpr int SG = FMT == BGL_Q4G256SF ? 4 : 1;        // 64-value sub-groups per unit
    static constexpr int BYTES = FMT == BGL_Q8G64 ? 64 : 32;      // bytes per row and sub-group
    static constexpr bool X16 = FMT != BGL_Q8G64;                 // integer sums come 16x
};

// 16 * (code - 8) of a dword's low and high nibbles (q4g64 stores unsigned codes, g256sf signed ones)
template <int FMT> __device__ __forceinline__ int gq_lo(uint32_t w) {
    return (int)(FMT == BGL_Q4G256SF ? (w << 4) & 0xF0F0F0F0u : ((w << 4) & 0xF0F0F0F0u) ^ 0x80808080u);
}
template <int FMT> __device__ __forceinline__ int gq_hi(uint32_t w) {
    return (int)(FMT == BGL_Q4G256SF ? w & 0xF0F0F0F0u : (w & 0xF0F0F0F0u) ^ 0x80808080u);
}

// A wave's raw weight operand of one sub-group: 32-row tiles take 16 bytes per lane (int4: chunk
// l / 32; int8: chunks 2 (l / 32) and + 1), 16-row tiles 8 (int4) or 16 (int8).
template <int FMT, int R> struct GqRaw { uint32_t w[GqFmt<FMT>::BYTES * R / 256]; };

// off: the sub-group's first chunk (uniform bytes); lane: the lane's byte offset within its chunks
template <int FMT, int R>
__device__ __forceinline__ void gq_load(GqRaw<FMT, R> &a, __amdgpu_buffer_rsrc_t rw, uint32_t lane, uint32_t off) {
    if constexpr (FMT != BGL_Q8G64 && R == 16) {
        const gq_u2 v = __builtin_amdgcn_raw_buffer_load_b64(rw, lane, off, 0);
        a.w[0] = v[0]; a.w[1] = v[1];
    } else {
#pragma unroll
        for (int i = 0; i < (int)sizeof(a.w) / 16; i++) {
            const gq_u4 v = __builtin_amdgcn_raw_buffer_load_b128(rw, lane + 1024u * i, off, 0);
            a.w[4 * i] = v[0]; a.w[4 * i + 1] = v[1]; a.w[4 * i + 2] = v[2]; a.w[4 * i + 3] = v[3];
        }
    }
}

// a wave's code operand of one sub-group: 32 columns 32 bytes per lane, 16 columns 16
template <int R> struct GqCol { uint32_t w[R == 32 ? 8 : 4]; };

template <int FMT, int R> struct GqSum;
template <int FMT> struct GqSum<FMT, 32> {
    static constexpr int V = 16;
    typedef gq_i16 T;
    static __device__ __forceinline__ T dot(const GqRaw<FMT, 32> &a, const GqCol<32> &x) {
        gq_i4 b0, b1, x0, x1;
        x0 = gq_i4{(int)x.w[0], (int)x.w[1], (int)x.w[2], (int)x.w[3]};
        x1 = gq_i4{(int)x.w[4], (int)x.w[5], (int)x.w[6], (int)x.w[7]};
        if constexpr (FMT == BGL_Q8G64) {
            b0 = gq_i4{(int)a.w[0], (int)a.w[1], (int)a.w[2], (int)a.w[3]};
            b1 = gq_i4{(int)a.w[4], (int)a.w[5], (int)a.w[6], (int)a.w[7]};
        } else {                                                  // dword j: values 8j..8j+3 low, 8j+4..8j+7 high
            b0 = gq_i4{gq_lo<FMT>(a.w[0]), gq_lo<FMT>(a.w[1]), gq_lo<FMT>(a.w[2]), gq_lo<FMT>(a.w[3])};
            b1 = gq_i4{gq_hi<FMT>(a.w[0]), gq_hi<FMT>(a.w[1]), gq_hi<FMT>(a.w[2]), gq_hi<FMT>(a.w[3])};
        }
        T d = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        d = __builtin_amdgcn_mfma_i32_32x32x32_i8(x0, b0, d, 0, 0, 0);
        return __builtin_amdgcn_mfma_i32_32x32x32_i8(x1, b1, d, 0, 0, 0);
    }
};
template <int FMT> struct GqSum<FMT, 16> {
    static constexpr int V = 4;
    typedef gq_i4 T;
    static __device__ __forceinline__ T dot(const GqRaw<FMT, 16> &a, const GqCol<16> &x) {
        gq_i4 b;
        if constexpr (FMT == BGL_Q8G64) b = gq_i4{(int)a.w[0], (int)a.w[1], (int)a.w[2], (int)a.w[3]};
        else b = gq_i4{gq_lo<FMT>(a.w[0]), gq_hi<FMT>(a.w[0]), gq_lo<FMT>(a.w[1]), gq_hi<FMT>(a.w[1])};
        return __builtin_amdgcn_mfma_i32_16x16x64_i8(gq_i4{(int)x.w[0], (int)x.w[1], (int)x.w[2], (int)x.w[3]}, b,
                                                     T{0, 0, 0, 0}, 0, 0, 0);
    }
};

#define GQ_AS GQ_COLS         // activation scales: columns of a unit's row
__device__ __forceinline__ __amdgpu_buffer_rsrc_t gq_rsrc(const void *p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
}

// R: rows (and columns) of a wave's tile.  Workgroup: R == 32: 2 row halves x column blocks of one
// 64-row tile; R == 16: one 16-row block x column blocks.  Every load is a buffer load with a constant
// lane offset and a scalar unit offset (no vector instruction), clamped into the tensor.
template <int FMT, int R>
__global__ __launch_bounds__(256, 2) void k_gemm_q(GemmQLaunch L) {
    extern __shared__ __align__(16) unsigned char lds[];
    using F = GqFmt<FMT>;
    using S = GqSum<FMT, R>;
    constexpr int V = S::V;
    // units in flight per wave, weights and codes alike: loads complete in order, so a code load waits
    // for every older weight load
    constexpr int D = F::SG == 4 ? (R == 32 ? 2 : 4) : FMT == BGL_Q8G64 && R == 32 ? 4 : R == 32 ? 8 : 16;
    float *sa = reinterpret_cast<float *>(lds);
    const int b = blockIdx.x;
    int ti = 0;
#pragma unroll
    for (int i = 1; i < BGL_MAX_TASKS; i++) if (i < L.ntasks && b >= L.t[i].blk0) ti = i;
    GemvTask task = L.t[0];
#pragma unroll
    for (int i = 1; i < BGL_MAX_TASKS; i++) if (i == ti) task = L.t[i];
    const BglDevTensor &T = task.T;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int lb = b - task.blk0;
    // the wave's tile: row block rb of the 64-row tile, column block cb
    const int tile = R == 32 ? lb : lb >> 2, rb = R == 32 ? wave & 1 : lb & 3, cb = R == 32 ? wave >> 1 : wave;
    const int row = R * rb + lane % R, q = lane / R;              // the lane's row of the tile, its k part
    const int U = T.nunits, last = U - 1;
    constexpr uint32_t UB = F::SG * F::BYTES / 16 * 1024u;        // bytes of a unit's chunks in the tile
    constexpr uint32_t SB = F::SG == 4 ? 512u : 256u;             // bytes of a unit's scales in the tile
    const uint32_t XB = F::SG * L.cb32 * 2048u;                   // bytes of a unit's codes
    const __amdgpu_buffer_rsrc_t rw = gq_rsrc(T.w + (size_t)tile * T.cpr * 1024, (uint32_t)T.cpr * 1024u);
    const __amdgpu_buffer_rsrc_t rs = gq_rsrc((const uint8_t *)T.s0 + (size_t)tile * U * SB, (uint32_t)U * SB);
    const __amdgpu_buffer_rsrc_t rx = gq_rsrc(L.xt, (uint32_t)U * XB);
    const uint32_t woff = FMT == BGL_Q8G64 ? (R == 32 ? 2u * q : (uint32_t)q) * 1024u + row * 16u
                        : R == 32 ? q * 1024u + row * 16u : (uint32_t)(q >> 1) * 1024u + row * 16u + 8u * (q & 1);
    const uint32_t soff = row * (F::SG == 4 ? 8u : 4u);
    // codes: 32 columns: parts 0 and 1 of the lane's record; 16 columns: the record of values 16 q .. + 15
    const uint32_t xoff = R == 32 ? cb * 2048u + lane * 16u
                                  : (cb >> 1) * 2048u + (q & 1) * 1024u + (32u * (q >> 1) + 16u * (cb & 1) + lane % 16) * 16u;
    struct Unit { GqRaw<FMT, R> a[F::SG]; GqCol<R> x[F::SG]; float s; uint32_t sub; };
    auto load_w = [&](Unit &un, int u) {
#pragma unroll
        for (int s = 0; s < F::SG; s++) gq_load<FMT, R>(un.a[s], rw, woff, u * UB + s * (UB / F::SG));
        if constexpr (F::SG == 4) {
            const gq_u2 w = __builtin_amdgcn_raw_buffer_load_b64(rs, soff, u * SB, 0);
            un.s = __uint_as_float(w[0]);
            un.sub = w[1];
        } else {
            un.s = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, soff, u * SB, 0));
        }
    };
    auto load_x = [&](GqCol<R> (&x)[F::SG], int u) {
#pragma unroll
        for (int s = 0; s < F::SG; s++)
#pragma unroll
            for (int i = 0; i < (R == 32 ? 2 : 1); i++) {
                const gq_u4 v = __builtin_amdgcn_raw_buffer_load_b128(rx, xoff + 1024u * i, u * XB + s * (XB / F::SG), 0);
                x[s].w[4 * i] = v[0]; x[s].w[4 * i + 1] = v[1]; x[s].w[4 * i + 2] = v[2]; x[s].w[4 * i + 3] = v[3];
            }
    };
    // the launch's activation scales, all of them, straight into LDS; unit u in row u + 1, row 0 belongs
    // to the zero sums before the first unit
    for (int i = wave; i < (U + 3) / 4; i += (int)(blockDim.x >> 6))
        __builtin_amdgcn_global_load_lds((const BGL_GLOBAL void *)(L.as + 4 * GQ_AS * i + 4 * lane),
                                         (__attribute__((address_space(3))) void *)(sa + GQ_AS + 4 * GQ_AS * i), 16, 0, 0);
    if (threadIdx.x < GQ_AS) sa[threadIdx.x] = 0.0f;
    Unit ring[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
        const int u = __builtin_amdgcn_readfirstlane(min(d, last));
        load_w(ring[d], u);
        load_x(ring[d].x, u);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

    float acc[V];
#pragma unroll
    for (int v = 0; v < V; v++) acc[v] = 0.0f;
    const float *sp = sa + R * cb + 4 * q;                        // the lane's columns: 8 k + 4 q + 0..3 (32) or 4 q + 0..3 (16)
    typedef typename S::T Sum;
    auto dots = [&](const Unit &un, const GqCol<R> (&x)[F::SG]) -> Sum {
        if constexpr (F::SG == 4) {
            const Sum d0 = S::dot(un.a[0], x[0]), d1 = S::dot(un.a[1], x[1]), d2 = S::dot(un.a[2], x[2]), d3 = S::dot(un.a[3], x[3]);
            const int s0 = un.sub & 255, s1 = (un.sub >> 8) & 255, s2 = (un.sub >> 16) & 255, s3 = un.sub >> 24;
            Sum d;
#pragma unroll
            for (int v = 0; v < V; v++)                           // |16 isum| <= 2^20, sub < 2^8
                d[v] = __mul24(d0[v], s0) + __mul24(d1[v], s1) + __mul24(d2[v], s2) + __mul24(d3[v], s3);
            return d;
        } else {
            return S::dot(un.a[0], x[0]);
        }
    };
    // the unit's fp32 terms; the staged activation scales are a sixteenth for 16x sums
    struct As { float a[V]; };
    auto read_as = [&](const float *p) -> As {
        As r;
#pragma unroll
        for (int k = 0; k < V / 4; k++) {
            const float4 a4 = *reinterpret_cast<const float4 *>(p + 8 * k);
            r.a[4 * k] = a4.x; r.a[4 * k + 1] = a4.y; r.a[4 * k + 2] = a4.z; r.a[4 * k + 3] = a4.w;
        }
        return r;
    };
    auto fold = [&](const Sum &d, float ws, const As &as) {
#pragma unroll
        for (int v = 0; v < V; v++) {
            float t = __fmul_rn((float)d[v], ws);
            if constexpr (F::SG == 4) t = __fmul_rn(t, T.gmul);
            acc[v] = __fadd_rn(acc[v], __fmul_rn(t, as.a[v]));
        }
    };
    uint32_t wlo = 0xffffffffu, whi = 0u;                         // range of the |scale| bits seen (zeros left out of wlo)
    // a unit's products run while the unit before it is folded; before the first, the sums are zeros
    Sum dp;
#pragma unroll
    for (int v = 0; v < V; v++) dp[v] = 0;
    float wp = 0.0f;
    As ap = read_as(sp);                                          // read a unit ahead of its use
    auto one = [&](Unit &un, int u, const float *asn) {
        const Sum dn = dots(un, un.x);
        const int un1 = __builtin_amdgcn_readfirstlane(min(u + D, last));
        const As an = read_as(asn);
        load_x(un.x, un1);
        fold(dp, wp, ap);
        ap = an;
        if constexpr (F::X16) {
            const uint32_t wb = abs_bits(un.s);
            wlo = min(wlo, wb - 1u);
            whi = max(whi, wb);
        }
        dp = dn;
        wp = un.s;
        load_w(un, un1);
        __builtin_amdgcn_sched_barrier(0);
    };
    int u = 0;
    for (; u + D <= U; u += D) {
#pragma unroll
        for (int d = 0; d < D; d++) one(ring[d], u + d, sp + (d + 1) * GQ_AS);
        sp += D * GQ_AS;
    }
#pragma unroll
    for (int d = 0; d < D; d++)
        if (u + d < U) one(ring[d], u + d, sp + (d + 1) * GQ_AS);
    fold(dp, wp, ap);
    if constexpr (F::X16) {
        // scales of 2^90 and more, or below 2^-90: 16x a term may leave fp32's range (or its subnormal
        // rounding) where the term itself does not: once more with the sums shifted back
        if (__any(wlo < __float_as_uint(0x1p-90f) - 1u || whi >= __float_as_uint(0x1p90f))) {
#pragma unroll
            for (int v = 0; v < V; v++) acc[v] = 0.0f;
            sp = sa + GQ_AS + R * cb + 4 * q;
#pragma unroll 1
            for (int w = 0; w < U; w++) {
                Unit un;
                load_w(un, w);
                load_x(un.x, w);
                const Sum d = dots(un, un.x);
#pragma unroll
                for (int k = 0; k < V / 4; k++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        float t = __fmul_rn((float)(d[4 * k + v] >> 4), un.s);
                        if constexpr (F::SG == 4) t = __fmul_rn(t, T.gmul);
                        acc[4 * k + v] = __fadd_rn(acc[4 * k + v], __fmul_rn(t, 16.0f * sp[w * GQ_AS + 8 * k + v]));
                    }
            }
        }
    }

    const int n = tile * BGL_TILE + row;
    if (n >= T.N) return;
    const float bb = task.bias ? task.bias[n] : 0.0f;
#pragma unroll
    for (int v = 0; v < V; v++) {
        const int m = R * cb + 4 * q + 8 * (v / 4) + v % 4;
        if (m < L.mcols) task.y[(size_t)(L.m0 + m) * task.ystride + n] = __fadd_rn(bb, acc[v]);
    }
}

// ------------------------------------------------------------------ host side
static size_t gq_lds(int units) { return (size_t)(1 + (units + 3) / 4 * 4) * GQ_AS * 4; }   // the activation scales

// The calls that go here.  More than 16 columns: all that fit (k_gemv_qm's launches hold 16 columns and
// take every unit's terms through LDS; the Llama-8B q4g64 MLP block at 64 columns 548 -> 68 us).
// Fewer: where the tiles fill the chip -- 16384 rows --, or the terms of K do not fit k_gemv_qm's LDS
// and the dot4 kernel would run.  Measured, us, before / here, 8 columns unless said:
//   q4g64   28672 x 4096 42.4 / 23.9 (2 columns 34.0 / 23.3)  17920 x 1536 28.9 / 13.4 (4: 12.0 / 12.7)
//           16384 x 2048, 6: 27.1 / 11.2 (4: 10.8 / 11.3)     4096 x 14336 43.3 / 27.3 (4: 23.3 / 27.2)
//           1536 x 8960 13.6 / 18.7 (16: 24.2 / 19.0)         4096 x 4096 10.3 / 12.8
//   g256sf  28672 x 4096 41.8 / 21.0 (2: 26.7 / 20.6)         17920 x 1536 12.1 / 12.7 (16: 18.3 / 13.1)
//           4096 x 14336 15.0 / 18.5
//   q8g64   28672 x 4096 41.2 / 30.4 (4: 31.1 / 30.5)         17920 x 1536 26.5 / 12.1
// More than 16 columns over few rows, 17 / 64 columns (the rows do not matter up to 3072: a wave walks K
// alone): 64 rows q4g64 K = 512 8.4 / 7.3 and 22.7 / 7.6, 4096 16.0 / 11.4 and 39.0 / 12.2, 14336 53.4 / 25.1
// and 172.7 / 29.1; g256sf 512 8.3 / 7.5 and 22.7 / 7.5, 14336 23.7 / 18.4 and 62.4 / 23.2; q8g64 512 7.9 / 7.5
// and 21.3 / 7.6, 14336 49.7 / 23.7 and 161.1 / 26.9.
bool gemm_q_ok(bgl_ctx *c, const BglDevTensor *Ts, int n, int M) {
    if (c->no_qmfma || M < 2) return false;
    const int fmt = Ts[0].fmt, K = Ts[0].K;
    long rows = 0;
    for (int i = 0; i < n; i++) {
        if (Ts[i].fmt != BGL_Q4G64 && Ts[i].fmt != BGL_Q8G64 && Ts[i].fmt != BGL_Q4G256SF) return false;
        if ((size_t)Ts[i].cpr * 1024 >= (1u << 31)) return false;   // a tile is addressed through 32-bit offsets
        rows += 64l * Ts[i].ntiles;
    }
    if (gq_lds(Ts[0].nunits) > GQ_LDS_MAX) return false;
    if (M > 16) return true;
    if (rows >= 16384) return rows * K >= 64l << 20 || (M >= 5 && (fmt != BGL_Q4G256SF || M > 8));
    return M >= 5 && bgl_gemv_qm_lds(fmt, K, M, 1, true) > 64 * 1024 && (M > 8 || rows * K >= 32l << 20);
}

template <int FMT>
static void gq_launch(const GemmQLaunch &L, int R, int blocks, size_t lds, hipStream_t st) {
    if (R == 32) hipLaunchKernelGGL((k_gemm_q<FMT, 32>), dim3(blocks), dim3(128 * L.cb32), lds, st, L);
    else hipLaunchKernelGGL((k_gemm_q<FMT, 16>), dim3(blocks), dim3(64 * ((L.mcols + 15) / 16)), lds, st, L);
}

// y[m][n] = bias[n] + the W4A8 product for n tensors sharing x (same kind and K), M columns in launches
// of up to 64.  u / h (one tensor): the columns are h = silu(x) * u, written to h.
int run_gemm_q(bgl_ctx *c, int n, const BglDevTensor *Ts, const float *x_dev, const float *u, float *h, int M,
               const float *const *bias, float *const *y) {
    const int K = Ts[0].K, fmt = Ts[0].fmt, gq = fmt == BGL_Q4G256SF ? 256 : 64;
    const int mc0 = std::min(M, GQ_COLS), cbm = (mc0 + 31) / 32;
    // The codes and scales lie in the partials' buffer, which no call leaves anything in: operands that
    // bgl_prep_act_dev left stay.  The same call at fewer columns prepares its own, possibly in a capture.
    const size_t xb = (size_t)32 * cbm * K, sb = (size_t)GQ_COLS * ((K / gq + 3) / 4 * 4) * 4;   // (xb: a multiple of 2048)
    if (dbuf_reserve(c, c->part, xb + sb, false)) return bgl_last_code();
    const size_t few = std::min(M, 16);
    if (!c->fixed_base && act_reserve_fewer(c, few * K, few * (K / gq) * 4, few * (K / 64) * 4)) return bgl_last_code();
    uint8_t *const xt = (uint8_t *)c->part.p;
    float *const as = (float *)(xt + xb);
    for (int m0 = 0; m0 < M; m0 += GQ_COLS) {
        const int mc = std::min(GQ_COLS, M - m0);
        GemmQLaunch L;
        memset(&L, 0, sizeof L);
        L.cb32 = (mc + 31) / 32;
        L.xt = xt;
        L.as = as;
        L.m0 = m0;
        L.mcols = mc;
        L.ntasks = n;
        long tiles = 0;
        for (int i = 0; i < n; i++) tiles += Ts[i].ntiles;
        // 32 x 32 tiles once there is more than one for every second SIMD.  (K = 4096, 64 columns, 16- and
        // 32-row tiles, us: 4096 rows 13.7 / 21.4, 8192 18.7 / 22.1 -- g256sf 17.6 / 17.6 --, 12288 25.7 /
        // 22.9, 28672 49.4 / 29.7; 24 columns: 12288 15.8 / 19.4, 17920 23.0 / 23.5, 28672 31.8 / 24.5.)
        const int R = tiles * 2 * L.cb32 > 512 ? 32 : 16;
        const int split = R == 32 && fmt != BGL_Q8G64;
        const float am = fmt == BGL_Q8G64 ? 1.0f : 0.0625f;
        const size_t xo = (size_t)m0 * K;
        const unsigned pb = (unsigned)(((long)mc * ((K + 255) / 256) + 3) / 4);
        int tok = prof_begin(c, 0);
        if (gq == 256)
            hipLaunchKernelGGL((k_act_q_tiles<256>), dim3(pb), dim3(256), 0, c->stream, x_dev + xo, mc, K, L.cb32, split, am,
                               xt, as, u ? u + xo : nullptr, h ? h + xo : nullptr);
        else
            hipLaunchKernelGGL((k_act_q_tiles<64>), dim3(pb), dim3(256), 0, c->stream, x_dev + xo, mc, K, L.cb32, split, am,
                               xt, as, u ? u + xo : nullptr, h ? h + xo : nullptr);
        prof_end(c, tok);
        HIPCHK(hipGetLastError());
        int blocks = 0;
        for (int i = 0; i < n; i++) {
            GemvTask &t = L.t[i];
            t.T = Ts[i];
            t.y = y[i];
            t.bias = bias ? bias[i] : nullptr;
            t.ystride = Ts[i].N;
            t.blk0 = blocks;
            blocks += Ts[i].ntiles * (R == 32 ? 1 : 4);
        }
        const size_t lds = gq_lds(Ts[0].nunits);
        tok = prof_begin(c, 1);
        switch (fmt) {
        case BGL_Q4G64: gq_launch<BGL_Q4G64>(L, R, blocks, lds, c->stream); break;
        case BGL_Q8G64: gq_launch<BGL_Q8G64>(L, R, blocks, lds, c->stream); break;
        default: gq_launch<BGL_Q4G256SF>(L, R, blocks, lds, c->stream); break;
        }
        prof_end(c, tok);
        HIPCHK(hipGetLastError());
    }
    return 0;
}
