// bgl_mfma.hip -- batched GEMM for M >= 2 activation rows on the gfx950 fp16 matrix cores
// (the M-column case of gemm_qXg64_mt / qng64_matmul_f32, q4gemv.h:761-769, qng64_dense.c:70-79).
//
// Numerics.  Weight codes are exact in fp16 (int4 and int8 codes, qNg64 codes for n <= 10), so
// the decode is exact.  Each activation column is scaled by a power of two so its largest
// magnitude lies in [2^13, 2^14), then split as hi = fp16(x') and lo = fp16(x' - hi), hi rounded
// toward zero (x' - hi is exact in fp32) and lo to nearest: hi + lo holds x' to 2^-22 of itself.  v_mfma_f32_16x16x32_f16 multiplies exactly and
// accumulates in fp32; each quantization group's partial sum is folded with its fp32 scale (one
// FMA per output per group) and the column factor 2^-(14-e) is applied at the end.
// The fp16 parts end at 2^-24, 2^-38 of the column's maximum over the split.  At 2..15 columns, which the
// exact digits of the dot4 kernels held to 2^-23 of each 64-group's own maximum (2^-46 in groups of many
// small elements), a column with such a group below 2^-14 of its maximum is multiplied a second time by
// what the parts leave over (mf_wide, mf_leftover), so it is held to 2^-60.  (One test and the branch:
// 28672 x 4096 at 5 columns 23.4 -> 23.8 us, 4096 x 4096 at 5 and 15 11.1 -> 11.4 and 12.0 -> 12.3; a call
// with such a column takes up to twice as long.)
//
// Layout.  A (weights, 16 rows x 32 k per instruction): lane l holds row l%16 and the 8 elements
// 8*(l/16)..+7 of the 32-element K-step -- with the device's 16-byte chunk layout that is one
// dword (int4) or two (int8) per lane and row block, and a wave's load covers 256 contiguous
// bytes.  The int4 nibble order (byte i: element i low, element 4+i high) decodes into halves in
// the order {0,2,1,3,4,6,5,7}; the activation fragments are stored in that same order, since the
// MFMA only needs A and B to agree element for element.  B (activations, 32 k x 16 columns):
// lane l holds column l%16, elements 8*(l/16)..+7.  D: lane l holds column l%16, rows
// 4*(l/16)..+3 of the 16-row block.
//
// Work split.  A workgroup owns 4 consecutive 64-row weight tiles (256 rows) over one K range (a
// split) and has KW K-slices of 8 waves; in a slice two waves share a tile (two 16-row blocks
// each).  The split's activation fragments and the 4 tiles' scales are staged in LDS once (up to
// 152 KB, which bounds the split's length), then each wave streams its own weights with no further
// barrier: a register ring keeps the next K-steps' loads in flight.  Splits are sized so the grid
// fills the chip; k_mfma_reduce adds their fp32 partials in split order (deterministic; no
// atomics).  All tensors of a group (same format and K, one activation) run in one launch and one
// reduce.  (A reduce inside the GEMM by the last workgroup of each row group -- an agent-scope
// ticket -- measured slower: the cache write-back and the serial tail cost more than the launch.)
//
// Memory access.  Weights are read a whole 16-byte chunk row per lane (buffer_load_dwordx4: each
// quarter-wave reads 256 contiguous bytes) and the operand layout above -- four lanes per row -- is
// rebuilt with v_permlane16/32_swap; the per-lane part of every address is fixed for the kernel and
// the per-step part is a scalar offset, so the loads cost no vector ALU work.  Offsets are clamped
// into the tensors, so no load is conditional (a conditional load makes the compiler wait for
// every load in flight), and steps past K meet zero fragments.
//
// Schedule.  The fold is software-pipelined: a group's MFMA sums are folded while the next group's
// MFMAs run, so the vector ALUs and the matrix cores overlap.
//
// Output.  The sums leave through LDS (the stage is free by then): stored straight from the MFMA
// layout, each store instruction would write 4 bytes to each of 16 output rows, and the partials
// of a 14336 x 4096 tensor at M = 32 took 3.8 us to write that way; staged, every lane writes 16
// consecutive bytes and each wave 1 KB runs (2 us faster per such launch).
#include <string.h>

#include <algorithm>

#include "bgl_internal.h"
#include "bgl_mfma_a.h"

#define HIPCHK(expr)                                                                             \
    do {                                                                                         \
        hipError_t e_ = (expr);                                                                  \
        if (e_ != hipSuccess) return bgl_fail(BGL_E_HIP, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

#define MF_TILES 4           // 64-row weight tiles per workgroup (they share the staged activations)
#define MF_WAVES (MF_TILES * 4 / MF_RBW)
#define MF_KSTEP_PAD 16      // split length granularity in K-steps (every ring depth divides it)
#define MF_MAXCT 4           // column tiles (16 columns each) per launch: up to 64 columns
#define MF_MAXN 10           // qNg64 widths whose codes are exact in fp16 via the 1024+u trick

struct MfmaTask {
    BglDevTensor T;
    const float *bias;       // [N] or null
    float *y;                // y[m][n] at y + m*ystride + n
    float *part;             // K-split partials [S][M][N] (S > 1)
    int ystride;
    int wg0;                 // first workgroup of this task in the launch
    int wgr;                 // workgroups along the rows (groups of 4 tiles)
    int kps;                 // K-steps per split, a multiple of MF_KSTEP_PAD
};

struct MfmaLaunch {
    MfmaTask t[BGL_MAX_TASKS];
    int ntasks;
    int M;                   // valid columns (<= 16*CT)
    const float *x;          // activations x[m][k], M rows of K floats
    int residual;            // columns of a wide range get a second product (one column tile only)
};

// ==================================================================================== GEMM kernel
// Task of this workgroup: the last task whose first workgroup is <= blockIdx.x (uniform).
__device__ __forceinline__ int mf_task(const MfmaLaunch &L) {
    int ti = 0;
#pragma unroll
    for (int i = 1; i < BGL_MAX_TASKS; i++)
        if (i < L.ntasks && (int)blockIdx.x >= L.t[i].wg0) ti = i;
    return ti;
}

// Raw A words per K-step and row block.
template <int FMT, int NB> constexpr int a_words() {
    return FMT == BGL_Q8G64 ? 2 : FMT == BGL_QNG64 ? 2 * ((NB >> 3) & 1) + ((NB >> 2) & 1) + ((NB >> 1) & 1) + (NB & 1) : 1;
}
// K-steps of weights a wave keeps in flight: a ring of depth/2 K-step pairs, Planes::WORDS
// registers each.
// (qNg64: the lane swaps of its planes want registers too; deeper rings, or this one beside 3 and 4 column
// tiles, spilled: n = 4 at 16 columns 28672 x 4096 58.0 us with 16, 30.5 with 8)
template <int FMT, int NB, int CT> constexpr int ring_depth() {
    constexpr int W = Planes<FMT, NB>::WORDS;
    return FMT == BGL_QNG64 ? (W <= 8 && CT <= 2 ? 8 : 4) : W <= 4 ? 16 : W <= 8 ? 8 : 4;
}
// LDS bytes per staged K-step: activation fragments (CT x hi/lo x 1 KB, + 16 B of row padding) +
// the 4 tiles' scale words in the device layout (512 B for every format).
constexpr int mf_step_lds(int CT) { return CT * 2048 + 16 + 512; }
// K-steps one workgroup stages (its split's whole K range): as many as fit 152 KB, a multiple of
// 16 (every ring depth divides it).
constexpr int mf_kps_max(int CT) { return (155648 / mf_step_lds(CT)) / 16 * 16; }

// Sum of code * scale * x over the non-finite x[k], k in [k0, k1), for weight row n (the rare path
// of a column that holds NaN or +-Inf).
template <int FMT, int NB>
__device__ __forceinline__ float mf_nonfinite(const BglDevTensor &T, int n, const float *x, int k0, int k1) {
    float acc = 0.0f;
#pragma unroll 1
    for (int k = k0; k < k1; k++) {
        const float v = x[k];
        if (!isfinite(v)) acc += w_at_t<FMT, NB>(T, n, k) * v;
    }
    return acc;
}

// What the two fp16 parts of x * 2^sh leave over (exact; below 2^-8, as x * 2^sh is below 2^14): scaled by
// 2^MF_RES_BITS, a second product's column.
#define MF_RES_BITS 22
__device__ __forceinline__ float mf_leftover(float x, int sh) {
    const float v = ldexpf(x, sh);
    const mf_h2 h = __builtin_bit_cast(mf_h2, __builtin_amdgcn_cvt_pkrtz(v, 0.0f));
    const float r = v - (float)h[0];
    const mf_h2 l = mf_cvt_rn(r, 0.0f);
    return r - (float)l[0];
}

// Whether a wave's column (its slots in v, of which those below n are real; low: the lanes that hold a small one,
// e: the exponent of the column's largest magnitude) has a 64-value group with as many small elements as
// bgl_x_level1 asks for, small being below 2^(e-14).  In the other groups at most 21 elements lie that low
// and at least as many above, so the digits, 2^-23 of their largest, were no finer than the fp16 parts.
template <int SPL>
__device__ __forceinline__ bool mf_wide(const float4 (&v)[SPL][2], uint64_t low, int n, int e) {
    const float thr = ldexpf(1.0f, e - 14);
    if (!low || !mf_three_lanes(low)) return false;                // (ordinary columns: one value in 5000 lies there)
    const int lane = threadIdx.x & 63;
    bool wide = false;
#pragma unroll
    for (int j = 0; j < SPL; j++) {
        const bool in = lane + 64 * j < n;
        int c = 0;                                                 // small + 256 * large of the lane's 8, then of its group's 64
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float4 q = v[j][h];
            auto one = [&](float x) { return fabsf(x) >= thr ? 256 : x != 0.0f ? 1 : 0; };
            c += one(q.x) + one(q.y) + one(q.z) + one(q.w);
        }
        c += dpp_i<0xB1>(c);
        c += dpp_i<0x4E>(c);
        c += dpp_i<0x141>(c);
        wide = wide || (in && bgl_x_level1(c & 255, c >> 8));
    }
    return __any(wide);
}

template <int FMT, int NB, int CT, int KW>
__global__ __launch_bounds__(MF_WAVES * KW * 64) void k_gemm_mfma(MfmaLaunch L) {
    constexpr int NT = MF_WAVES * KW * 64;
    constexpr int KPM = mf_kps_max(CT);                             // staged K-steps (max)
    constexpr int SPU = ksteps_per_unit<FMT>();
    constexpr int GPU = groups_per_unit<FMT>();
    constexpr int SCW = scale_bytes<FMT>();
    constexpr int SPG = SPU / GPU;                                 // K-steps per scale group
    constexpr int BST = CT * 2 * 64;                               // activation uint4 per K-step
    constexpr int XS = BST + 1;                                    // their row stride in the stage
    constexpr int UMAX = KPM / SPU;                                // staged units (max)
    constexpr int SUT = 64 * SCW / 16;                             // scale uint4 per tile and unit
    // ring depth: halved with two slices (each wave runs half the split, and 16 waves share the
    // registers); at least 4 so that a unit's groups keep their parity pattern
    constexpr int D = KW == 1 || ring_depth<FMT, NB, CT>() == 4 ? ring_depth<FMT, NB, CT>() : ring_depth<FMT, NB, CT>() / 2;
    static_assert(KPM % D == 0 && KPM % SPU == 0 && D % SPU == 0, "staged range must hold whole rings and units");
    __shared__ uint4 xs[KPM * XS];                                 // [step][CT][hi/lo][64 lanes], rows XS apart
    __shared__ uint4 ss[MF_TILES * UMAX * SUT];                    // [tile][unit][64 rows] scale words

    __shared__ int cex[16 * MF_MAXCT];                             // per column: the exponent of its sums,
    __shared__ int cnf[16 * MF_MAXCT];                             // whether it holds NaN or +-Inf in the split,
    __shared__ int cwd[CT == 1 ? 16 : 1];                          // whether its range is wide (one column tile)
    int level = 0;
second_product:                                                    // level 1: added to what level 0 stored
    int tid = threadIdx.x;
    if constexpr (CT == 1) asm("" : "+v"(tid));                    // (opaque: no address kept in registers for it)
    const int ti = mf_task(L);
    const MfmaTask &tk = L.t[ti];
    const BglDevTensor &T = tk.T;
    // the wave index is uniform: in a scalar register, every offset derived from it is scalar too
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, q = lane >> 4;
    const int kw = wave / MF_WAVES, w8 = wave % MF_WAVES;          // K-slice, wave within the slice
    const int wt = w8 / (4 / MF_RBW), rbase = (w8 % (4 / MF_RBW)) * MF_RBW;   // tile in the group, first row block
    const int local = (int)blockIdx.x - tk.wg0;
    const int split = local / tk.wgr, tg = local % tk.wgr;
    const int tile0 = tg * MF_TILES, tile = tile0 + wt;
    const int KS = T.K >> 5;
    const int s0 = split * tk.kps, ns = min(tk.kps, KS - s0);      // this split: K-steps [s0, s0 + ns)
    const int nrings = (ns + D - 1) / D;                           // whole rings (steps past ns are zeros)
    const int nsr = nrings * D;
    const int u0 = s0 / SPU, nu = nsr / SPU;
    // slice kw runs rings [r0, r1) of the split
    const int rsplit = (nrings + KW - 1) / KW;
    const int ls0 = min(kw * rsplit, nrings) * D, ls1 = min((kw + 1) * rsplit, nrings) * D;

    const __amdgpu_buffer_rsrc_t rw = mf_rsrc(T.w, (uint32_t)T.ntiles * T.cpr * 1024u);
    const __amdgpu_buffer_rsrc_t rx = mf_rsrc(L.x, (uint32_t)L.M * (uint32_t)T.K * 4u);
    const __amdgpu_buffer_rsrc_t rsc = mf_rsrc(T.s0, (uint32_t)T.ntiles * T.nunits * 64 * SCW);

    // ---- activations of the split: each wave loads 8-element slots of its columns ----
    // Column m belongs to wave m % NW; lane l takes slots l, l+64, ... (slot g = K elements
    // 8g..8g+7 of the split).  Loads are unconditional (clamped) and issued before the weights, so
    // the conversion below waits for them alone.
    constexpr int NW = MF_WAVES * KW;                              // waves
    constexpr int CPW = (16 * CT + NW - 1) / NW;                   // columns per wave
    constexpr int SPL = KPM / 16;                                  // slots per lane (4 per K-step)
    float4 xv[CPW][SPL][2];
#pragma unroll
    for (int ci = 0; ci < CPW; ci++)
#pragma unroll
        for (int j = 0; j < SPL; j++) {
            const int m = ci * NW + wave, g = lane + 64 * j;
            const bool ok = m < L.M && g < 4 * ns;
            const uint32_t off = ((uint32_t)(ok ? m : 0) * (uint32_t)T.K + (uint32_t)s0 * 32u + 8u * (uint32_t)(ok ? g : 0)) * 4u;
            const mf_u4 a = __builtin_amdgcn_raw_buffer_load_b128(rx, off, 0, 0);
            const mf_u4 b = __builtin_amdgcn_raw_buffer_load_b128(rx, off + 16u, 0, 0);
            xv[ci][j][0] = make_float4(__uint_as_float(a[0]), __uint_as_float(a[1]), __uint_as_float(a[2]), __uint_as_float(a[3]));
            xv[ci][j][1] = make_float4(__uint_as_float(b[0]), __uint_as_float(b[1]), __uint_as_float(b[2]), __uint_as_float(b[3]));
        }

    // ---- the 4 tiles' scales of the split: loaded now (a fixed count per thread, clamped), put
    // into LDS after the conversion below, so that nothing waits for them before the weights are
    // requested ----
    // (up to 32 columns, where that is one per thread; other shapes stage them here, before the
    // weights, as holding them through the conversion made the compiler spill in their main loops)
    constexpr int SLT = (MF_TILES * UMAX * SUT + NT - 1) / NT;     // scale uint4 per thread (max)
    constexpr bool EARLY = SLT == 1 && CT <= 2;
    const int nsu = nu * SUT;                                      // scale uint4 per tile in this split
    auto scale_ld = [&](int e) -> mf_u4 {
        e = min(e, MF_TILES * nsu - 1);                            // clamped: every load is real
        const int st = e / nsu, rem = e % nsu, uu = rem / SUT;
        const int tc = min(tile0 + st, T.ntiles - 1), uc = min(u0 + uu, T.nunits - 1);
        return __builtin_amdgcn_raw_buffer_load_b128(rsc, ((uint32_t)tc * T.nunits + uc) * (64 * SCW) + (uint32_t)(rem % SUT) * 16u, 0, 0);
    };
    auto scale_st = [&](int e, const mf_u4 &g) {
        const int st = e / nsu, rem = e % nsu, uu = rem / SUT;
        ss[(st * UMAX + uu) * SUT + rem % SUT] = uu * SPU < ns ? make_uint4(g[0], g[1], g[2], g[3]) : make_uint4(0, 0, 0, 0);
    };
    mf_u4 sreg;
    if constexpr (EARLY) sreg = scale_ld(tid);
    else
        for (int e = tid; e < MF_TILES * nsu; e += NT) scale_st(e, scale_ld(e));

    // ---- the weight ring: local K-step s lives in slot (s - ls0) % D until it is computed ----
    const int tile_c = min(tile, T.ntiles - 1);                    // waves past the tensor read a real tile
    const uint32_t tchunk = (uint32_t)tile_c * T.cpr;
    const AOff ao = a_offsets(rbase, lane);
    PRaw<FMT, NB> ring[D / 2];
    auto load_w = [&](PRaw<FMT, NB> &slot, int s) {             // local K-steps s, s+1 (s even)
        const int sc = min(s0 + s, KS - 2);                        // past the split: reread, multiplied by zeros
        ld_pair<FMT, NB>(slot, rw, ao, tchunk, sc);
    };
    // the activation and scale loads go out first: the conversion below waits for them by the
    // in-order load counter, which would also wait for any weight load issued before them
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 0; d < D / 2; d++) load_w(ring[d], ls0 + 2 * d);

    // ---- activation fragments: each column is scaled by a power of two so its largest magnitude
    // over the split lies in [2^13, 2^14), then split into hi = fp16(x') and lo = fp16(x' - hi) in
    // the MFMA operand order; the split's column factor 2^(e-14) is applied to its partial sums ----
    // Non-finite values (NaN, +-Inf) enter the fragments as 0 and flag the column; the store adds
    // their products code * scale * x one element at a time (IEEE propagation, as the reference's
    // fp32-product sums).
    int xe[CPW];                                                   // one column tile: the columns' exponents, and the
    uint64_t xlow[CPW];                                            // lanes with small values, for what follows the barrier
#pragma unroll
    for (int ci = 0; ci < CPW; ci++) {
        const int m = ci * NW + wave;
        if (m >= 16 * CT) break;                                   // uniform
        // the column's largest |x| bits over the split; Inf / NaN bits exceed every finite value's, so
        // only then (rare) are they zeroed and the maximum taken again
        uint32_t mb = 0u;
        uint32_t lo = 0x7fffffffu;                                 // one column tile: the lane's smallest |x| bits
#pragma unroll
        for (int j = 0; j < SPL; j++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float4 v = xv[ci][j][h];
                const uint32_t a = __float_as_uint(v.x) & 0x7fffffffu, b = __float_as_uint(v.y) & 0x7fffffffu;
                const uint32_t c = __float_as_uint(v.z) & 0x7fffffffu, d = __float_as_uint(v.w) & 0x7fffffffu;
                const uint32_t t = max(max(a, b), max(c, d));
                mb = m < L.M && lane + 64 * j < 4 * ns ? max(mb, t) : mb;
                // (slots past the split are copies of the column's first)
                if constexpr (CT == 1) lo = min(min(min(a, b), min(c, d)), lo);
            }
        mb = wave_max_u32(mb);
        if (lane == 0) cnf[m] = 0;
        if (mb >= 0x7f800000u) {                                   // uniform: Inf or NaN in this column's split
            mb = 0u;
#pragma unroll
            for (int j = 0; j < SPL; j++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    float4 &v = xv[ci][j][h];
                    const bool in = m < L.M && lane + 64 * j < 4 * ns;
                    auto screen = [&](float &e) {
                        const uint32_t ab = __float_as_uint(e) & 0x7fffffffu;
                        const bool bad = ab >= 0x7f800000u;
                        e = bad ? 0.0f : e;
                        mb = (!bad && in && ab > mb) ? ab : mb;
                    };
                    screen(v.x); screen(v.y); screen(v.z); screen(v.w);
                }
            mb = wave_max_u32(mb);
            if (lane == 0) cnf[m] = level ? 0 : 1;                 // (their products are added once)
        }
        const float mx = __uint_as_float(mb);
        int e = 0;
        if (mx > 0.0f) frexpf(mx, &e);                             // mx in [2^(e-1), 2^e)
        // x' = x * 2^(14-e), applied to each value (the factor alone leaves fp32's range for
        // e < -113, columns whose largest |x| is below 2^-114); the sums are unscaled by 2^(e-14)
        int sh = mx > 0.0f ? 14 - e : 0;
        if (lane == 0) cex[m] = -sh;
        bool use = m < L.M;
        if constexpr (CT == 1) {
            if (level) {                                           // the split's leftover in place of the column
#pragma unroll
                for (int j = 0; j < SPL; j++)
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        float4 &v = xv[ci][j][h];
                        v = make_float4(mf_leftover(v.x, sh), mf_leftover(v.y, sh), mf_leftover(v.z, sh), mf_leftover(v.w, sh));
                    }
                if (lane == 0) cex[m] = -sh - MF_RES_BITS;
                sh = MF_RES_BITS;
                use = use && cwd[m];                               // (this wave wrote it)
            }
            xe[ci] = __builtin_amdgcn_readfirstlane(e);
            xlow[ci] = __ballot(__uint_as_float(lo) < ldexpf(1.0f, e - 14));
        }
        const int ct = m >> 4, ml = m & 15;
#pragma unroll
        for (int j = 0; j < SPL; j++) {
            const int g = lane + 64 * j;
            if (g >= 4 * nsr) break;
            const bool ok = (CT == 1 ? use : m < L.M) && g < 4 * ns;
            const float4 a = xv[ci][j][0], b = xv[ci][j][1];
            const float v8[8] = {a.x, a.z, a.y, a.w, b.x, b.z, b.y, b.w};   // element order {0,2,1,3,4,6,5,7}
            // hi = fp16(x') rounded toward zero, two at a time; x' - hi is exact in fp32 (hi is x'
            // cut to 11 bits); lo = fp16 of that, to nearest (toward zero its error would not cancel:
            // 1.6e-7 of the product, see the numerics above)
            uint32_t H[4], Lo[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float v0 = ldexpf(v8[2 * k], sh), v1 = ldexpf(v8[2 * k + 1], sh);   // power-of-two scaling: exact
                const mf_h2 hh = __builtin_bit_cast(mf_h2, __builtin_amdgcn_cvt_pkrtz(v0, v1));
                const float r0 = v0 - (float)hh[0], r1 = v1 - (float)hh[1];
                const uint32_t hw = __builtin_bit_cast(uint32_t, hh);
                const uint32_t lw = __builtin_bit_cast(uint32_t, mf_cvt_rn(r0, r1));
                H[k] = ok ? hw : 0u;                               // K-steps past the split: zero fragments
                Lo[k] = ok ? lw : 0u;
            }
            // step rows are XS = BST + 1 uint4 apart: the lanes of one store hold 16 steps of one
            // column, which then fall on 16 different bank groups instead of one
            uint4 *d = xs + (g >> 2) * XS + ct * 128 + ml + 16 * (g & 3);
            d[0] = make_uint4(H[0], H[1], H[2], H[3]);
            d[64] = make_uint4(Lo[0], Lo[1], Lo[2], Lo[3]);
        }
    }
    // the scales, into LDS (scale units past the split are zeroed)
    if constexpr (EARLY)
        if (tid < MF_TILES * nsu) scale_st(tid, sreg);
    __syncthreads();
    // (after the barrier, while the weights are on their way: nothing waits for it before the end)
    if constexpr (CT == 1)
        if (L.residual && !level) {
#pragma unroll
            for (int ci = 0; ci < CPW; ci++) {
                const int m = ci * NW + wave;
                const bool wide = m < L.M && mf_wide<SPL>(xv[ci], xlow[ci], 4 * ns, xe[ci]);
                if (lane == 0) cwd[m] = wide;
            }
        }

    mf_f4 acc[MF_RBW][CT];
#pragma unroll
    for (int r = 0; r < MF_RBW; r++)
#pragma unroll
        for (int c = 0; c < CT; c++) acc[r][c] = mf_f4{0, 0, 0, 0};

    // Scale words of this lane's 4 rows (16*(rbase+rb) + 4q .. +3) for staged unit u: one uint4
    // (4 rows x one fp32, or x an fp16 pair), or for qNg64 the two groups' float2s split into one
    // mf_f4 per group.
    struct SW { uint4 w; mf_f4 g0, g1; };
    auto scale_words = [&](int u, int rb) -> SW {
        const int row = 16 * (rbase + rb) + 4 * q;
        const uint4 *base = ss + (wt * UMAX + u) * SUT;
        SW r;
        if constexpr (SCW == 8) {
            const uint4 a = base[row >> 1], b = base[(row >> 1) + 1];
            r.g0 = mf_f4{__uint_as_float(a.x), __uint_as_float(a.z), __uint_as_float(b.x), __uint_as_float(b.z)};
            r.g1 = mf_f4{__uint_as_float(a.y), __uint_as_float(a.w), __uint_as_float(b.y), __uint_as_float(b.w)};
        } else {
            r.w = base[row >> 2];
        }
        return r;
    };
    auto scale_of = [&](const SW &r, int g) -> mf_f4 {
        if constexpr (FMT == BGL_Q4G32H) {                         // fp16 pairs: group g is half g of each word
            const uint32_t sh = 16 * g;
            return mf_f4{__half2float(__ushort_as_half((unsigned short)(r.w.x >> sh))),
                         __half2float(__ushort_as_half((unsigned short)(r.w.y >> sh))),
                         __half2float(__ushort_as_half((unsigned short)(r.w.z >> sh))),
                         __half2float(__ushort_as_half((unsigned short)(r.w.w >> sh)))};
        } else if constexpr (FMT == BGL_QNG64) {
            return g == 0 ? r.g0 : r.g1;
        } else {
            return mf_f4{__uint_as_float(r.w.x), __uint_as_float(r.w.y), __uint_as_float(r.w.z), __uint_as_float(r.w.w)};
        }
    };
    // Activation fragments of local step s (clamped into the staged range).
    struct BF { mf_h8 h[CT], l[CT]; };
    auto load_b = [&](int s) -> BF {
        const uint4 *p = xs + min(s, nsr - 1) * XS + lane;
        BF r;
#pragma unroll
        for (int c = 0; c < CT; c++) {
            r.h[c] = __builtin_bit_cast(mf_h8, p[c * 128]);
            r.l[c] = __builtin_bit_cast(mf_h8, p[c * 128 + 64]);
        }
        return r;
    };

    // ---- main loop: no barriers; each wave streams its own weights D K-steps ahead, and the next
    // step's fragments and the unit's scales are read from LDS a step ahead of their use.  The
    // fold is software-pipelined: a group's MFMA sums (cg[g % 2]) are folded into acc while the
    // next group's MFMAs run, so the matrix cores and the vector ALUs work at the same time ----
    static_assert((D / SPG) % 2 == 0, "group parity must repeat every ring");
    mf_f4 cg[2][MF_RBW][CT], scp[MF_RBW];
#pragma unroll
    for (int r = 0; r < MF_RBW; r++) {
        scp[r] = mf_f4{0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < CT; c++) { cg[0][r][c] = mf_f4{0, 0, 0, 0}; cg[1][r][c] = mf_f4{0, 0, 0, 0}; }
    }
    auto fold = [&](const mf_f4 (&g)[MF_RBW][CT]) {
#pragma unroll
        for (int rb = 0; rb < MF_RBW; rb++)
#pragma unroll
            for (int c = 0; c < CT; c++)
#pragma unroll
                for (int v = 0; v < 4; v++) acc[rb][c][v] = __fmaf_rn(g[rb][c][v], scp[rb][v], acc[rb][c][v]);
    };
    BF bnext;
    if constexpr (KW == 1) bnext = load_b(ls0);
    for (int sb = ls0; sb < ls1; sb += D) {
        SW swd[MF_RBW];
        ARaw<FMT, NB> apair[2][MF_RBW];
#pragma unroll
        for (int d = 0; d < D; d++) {
            const int s = sb + d, par = (d / SPG) & 1;
            if (d % SPU == 0) {
#pragma unroll
                for (int rb = 0; rb < MF_RBW; rb++) swd[rb] = scale_words(s / SPU, rb);
            }
            // one slice (2 waves per SIMD) reads the next step's fragments ahead; two slices read
            // them in place (the other waves cover the LDS latency, and the registers are needed)
            BF bc;
            if constexpr (KW == 1) { bc = bnext; bnext = load_b(s + 1); }
            else bc = load_b(s);
            if (d % 2 == 0) {                                       // a new K-step pair: exchange, refill the slot
                exch<FMT, NB>(ring[d / 2], apair, ((s0 + s) >> 1) & 1);
                load_w(ring[d / 2], s + D);                         // unconditional, clamped
            }
            mf_h8 A[MF_RBW];
#pragma unroll
            for (int r = 0; r < MF_RBW; r++) A[r] = dec_a<FMT, NB>(apair[d % 2][r], q);
            const bool gstart = d % SPG == 0;                       // first K-step of a scale group
#pragma unroll
            for (int h = 0; h < 2; h++)                             // all hi products, then the lo ones
#pragma unroll
                for (int c = 0; c < CT; c++)
#pragma unroll
                    for (int r = 0; r < MF_RBW; r++)
                        cg[par][r][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            A[r], h ? bc.l[c] : bc.h[c], gstart && !h ? mf_f4{0, 0, 0, 0} : cg[par][r][c], 0, 0, 0);
            if (gstart) fold(cg[par ^ 1]);                          // the previous group, while these run
            if ((d + 1) % SPG == 0) {                                // group complete: its scales for the next fold
                const int g = (d % SPU) / SPG;
#pragma unroll
                for (int rb = 0; rb < MF_RBW; rb++) scp[rb] = scale_of(swd[rb], g);
            }
        }
    }
    fold(cg[((D / SPG) - 1) & 1]);                                  // the last group

    // ---- outputs through LDS: a lane's sums lie on rows 16 apart per column (stored directly, each
    // store instruction would touch 16 output rows), so every wave puts its sums into
    // ob[slice][column][256 rows of the workgroup] and the stores below write runs of consecutive
    // rows, 16 bytes per lane.  Row index nl of column m sits at nl ^ 4*(m % 16) (a swizzle of whole
    // float4s that spreads a wave's writes over the banks).  The K-slices' sums are added there,
    // slice 0 + slice 1 ----
    constexpr int OBR = MF_TILES * BGL_TILE;                        // rows per workgroup
    static_assert(KW * 16 * CT * OBR * 4 <= (int)sizeof(xs), "output staging must fit the stage");
    __syncthreads();                                                // every wave is done with the staged data
    float *ob = reinterpret_cast<float *>(xs);
#pragma unroll
    for (int rb = 0; rb < MF_RBW; rb++)
#pragma unroll
        for (int c = 0; c < CT; c++) {
            // the lane's 4 sums of column m are rows nl..nl+3: one 16-byte write
            const int m = 16 * c + (lane & 15), nl = wt * BGL_TILE + 16 * (rbase + rb) + 4 * q;
            *reinterpret_cast<float4 *>(ob + (kw * 16 * CT + m) * OBR + (nl ^ ((m & 15) << 2))) =
                make_float4(acc[rb][c][0], acc[rb][c][1], acc[rb][c][2], acc[rb][c][3]);
        }
    __syncthreads();

    const int S = (KS + tk.kps - 1) / tk.kps;
    const int nb = tile0 * BGL_TILE;                                // first row of the workgroup
    if constexpr (CT == 1)
        if (level) {                                               // onto what this thread stored
            for (int i = tid; i < 16 * (OBR / 4); i += NT) {
                const int m = i / (OBR / 4), nl = (i % (OBR / 4)) * 4, n = nb + nl;
                if (m >= L.M || !cwd[m]) continue;
                const float *a = ob + m * OBR + (nl ^ ((m & 15) << 2));
                float *dst = (S > 1 ? tk.part + ((size_t)split * L.M + m) * T.N : tk.y + (size_t)m * tk.ystride) + n;
                for (int e = 0; e < 4; e++)
                    if (n + e < T.N) dst[e] += ldexpf(KW == 2 ? a[e] + a[16 * OBR + e] : a[e], cex[m]);
            }
            return;
        }
    for (int i = tid; i < 16 * CT * (OBR / 4); i += NT) {
        const int m = i / (OBR / 4), nl = (i % (OBR / 4)) * 4, n = nb + nl;
        if (m >= L.M || n >= T.N) continue;
        const int sw = nl ^ ((m & 15) << 2);
        const float4 a = *reinterpret_cast<const float4 *>(ob + m * OBR + sw);
        float o[4] = {a.x, a.y, a.z, a.w};
        if constexpr (KW == 2) {
            const float4 b = *reinterpret_cast<const float4 *>(ob + (16 * CT + m) * OBR + sw);
            o[0] += b.x; o[1] += b.y; o[2] += b.z; o[3] += b.w;
        }
        const int ce = cex[m];
        float *dst = (S > 1 ? tk.part + ((size_t)split * L.M + m) * T.N : tk.y + (size_t)m * tk.ystride) + n;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            o[e] = ldexpf(o[e], ce);
            if (n + e < T.N) {
                if (cnf[m]) o[e] += mf_nonfinite<FMT, NB>(T, n + e, L.x + (size_t)m * T.K, 32 * s0, min(32 * (s0 + ns), T.K));
                if (S == 1 && tk.bias) o[e] += tk.bias[n + e];
            }
        }
        if (n + 3 < T.N && ((uintptr_t)dst & 15) == 0) {
            *reinterpret_cast<float4 *>(dst) = make_float4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < T.N) dst[e] = o[e];
        }
    }
    if constexpr (CT == 1)
        if (L.residual) {
            int wide = 0;
#pragma unroll
            for (int m = 0; m < 16; m++) wide |= cwd[m];
            if (wide) {                                            // uniform
                level = 1;
                __syncthreads();                                   // the stage is read out
                goto second_product;
            }
        }
}

// ==================================================================================== K-split reduce
// y[m][n] = bias[n] + sum_s part[s][m][n], s in order, for every task of a launch with S > 1.  A
// thread owns 4 consecutive n of one m and keeps MF_RED_BATCH partials in flight.
// SwiGLU pair mode (glu_h set; tasks 0 and 1 are gate and up of one shape): a thread forms both
// tasks' values at its (m, n) -- the split sums as above, or y as the GEMM stored it when the task
// did not split -- and stores h = silu(g) * u (k_swiglu's arithmetic: exp in double, rounded once)
// instead of g and u.
#define MF_RED_BATCH 8
struct MfmaReduceTask {
    const float *part;
    const float *bias;
    float *y;
    int N, S, ystride, q0;   // q0: first quad of this task in the grid
};
struct MfmaReduce {
    MfmaReduceTask t[BGL_MAX_TASKS];
    int ntasks, M, nquads;
    float *glu_h;            // SwiGLU pair mode: h [M][glu_stride]
    int glu_stride;
};

// bias[n] + sum_s part[s][m][n] for the 4 values n.. of row m, s in order
__device__ __forceinline__ void mf_red_quad(const MfmaReduceTask &t, int M, int m, int n, float (&a)[4]) {
    const size_t plane = (size_t)M * t.N;
    const float *p = t.part + (size_t)m * t.N + n;
    const bool vec = (t.N & 3) == 0;
#pragma unroll
    for (int e = 0; e < 4; e++) a[e] = 0.0f;
    for (int s0 = 0; s0 < t.S; s0 += MF_RED_BATCH) {               // a batch of partials in flight, added in order
        float v[MF_RED_BATCH][4];
#pragma unroll
        for (int i = 0; i < MF_RED_BATCH; i++) {
            const int s = s0 + i;
            if (s >= t.S) break;
            if (vec) {
                const float4 f = *reinterpret_cast<const float4 *>(p + s * plane);
                v[i][0] = f.x; v[i][1] = f.y; v[i][2] = f.z; v[i][3] = f.w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) v[i][e] = n + e < t.N ? p[s * plane + e] : 0.0f;
            }
        }
#pragma unroll
        for (int i = 0; i < MF_RED_BATCH; i++) {
            if (s0 + i >= t.S) break;
#pragma unroll
            for (int e = 0; e < 4; e++) a[e] = s0 + i == 0 ? v[i][e] : a[e] + v[i][e];
        }
    }
#pragma unroll
    for (int e = 0; e < 4; e++) a[e] = (t.bias && n + e < t.N ? t.bias[n + e] : 0.0f) + a[e];
}

__global__ __launch_bounds__(256) void k_mfma_reduce(MfmaReduce R) {
    const int qd = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (qd >= R.nquads) return;
    if (R.glu_h) {
        const MfmaReduceTask &tg = R.t[0], &tu = R.t[1];
        const int nq = (tg.N + 3) >> 2, m = qd / nq, n = 4 * (qd % nq);
        float g[4], u[4];
        if (tg.S > 1) mf_red_quad(tg, R.M, m, n, g);
        else {
#pragma unroll
            for (int e = 0; e < 4; e++) g[e] = n + e < tg.N ? tg.y[(size_t)m * tg.ystride + n + e] : 0.0f;
        }
        if (tu.S > 1) mf_red_quad(tu, R.M, m, n, u);
        else {
#pragma unroll
            for (int e = 0; e < 4; e++) u[e] = n + e < tu.N ? tu.y[(size_t)m * tu.ystride + n + e] : 0.0f;
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (n + e >= tg.N) break;
            const float ex = (float)exp(-(double)g[e]);
            R.glu_h[(size_t)m * R.glu_stride + n + e] = (g[e] / (1.0f + ex)) * u[e];
        }
        return;
    }
    int ti = 0;
#pragma unroll
    for (int i = 1; i < BGL_MAX_TASKS; i++)
        if (i < R.ntasks && qd >= R.t[i].q0) ti = i;
    const MfmaReduceTask &t = R.t[ti];
    const int nq = (t.N + 3) >> 2, lq = qd - t.q0;
    const int m = lq / nq, n = 4 * (lq % nq);
    float a[4];
    mf_red_quad(t, R.M, m, n, a);
#pragma unroll
    for (int e = 0; e < 4; e++) {
        if (n + e >= t.N) break;
        t.y[(size_t)m * t.ystride + n + e] = a[e];
    }
}

// ==================================================================================== host side
bool bgl_mfma_ok(int fmt, int bits) {
    if (fmt == BGL_Q4G64 || fmt == BGL_Q4G32H || fmt == BGL_Q8G64) return true;
    return fmt == BGL_QNG64 && bits >= 2 && bits <= MF_MAXN;
}

// Two K-slices (16 waves, <= 128 VGPRs) where that instance compiles without private memory --
// which instances fit depends on the register allocator, so it is read from the code object --
// else one slice (8 waves, <= 256 VGPRs), unless that one needs even more private memory.
template <int FMT, int NB, int CT>
static void launch_ct(const MfmaLaunch &L, dim3 grid, hipStream_t st) {
    static int kw2 = -1;
    if (kw2 < 0) {
        hipFuncAttributes a2, a1;
        const bool ok2 = hipFuncGetAttributes(&a2, reinterpret_cast<const void *>(&k_gemm_mfma<FMT, NB, CT, 2>)) == hipSuccess;
        const bool ok1 = hipFuncGetAttributes(&a1, reinterpret_cast<const void *>(&k_gemm_mfma<FMT, NB, CT, 1>)) == hipSuccess;
        // two slices unless they need more than a few spilled registers and one slice needs less
        kw2 = ok2 && (a2.localSizeBytes <= 32 || !ok1 || a2.localSizeBytes <= a1.localSizeBytes);
    }
    if (kw2) hipLaunchKernelGGL((k_gemm_mfma<FMT, NB, CT, 2>), grid, dim3(MF_WAVES * 2 * 64), 0, st, L);
    else hipLaunchKernelGGL((k_gemm_mfma<FMT, NB, CT, 1>), grid, dim3(MF_WAVES * 64), 0, st, L);
}

template <int FMT, int NB>
static int launch_fmt(const MfmaLaunch &L, int CT, dim3 grid, hipStream_t st) {
    switch (CT) {
    case 1: launch_ct<FMT, NB, 1>(L, grid, st); return 0;
    case 2: launch_ct<FMT, NB, 2>(L, grid, st); return 0;
    case 3: launch_ct<FMT, NB, 3>(L, grid, st); return 0;
    case 4: launch_ct<FMT, NB, 4>(L, grid, st); return 0;
    default: return -1;
    }
}

static int launch_any(const MfmaLaunch &L, int fmt, int bits, int CT, dim3 grid, hipStream_t st) {
    switch (fmt) {
    case BGL_Q4G64: return launch_fmt<BGL_Q4G64, 0>(L, CT, grid, st);
    case BGL_Q4G32H: return launch_fmt<BGL_Q4G32H, 0>(L, CT, grid, st);
    case BGL_Q8G64: return launch_fmt<BGL_Q8G64, 0>(L, CT, grid, st);
    case BGL_QNG64:
        switch (bits) {
        case 2: return launch_fmt<BGL_QNG64, 2>(L, CT, grid, st);
        case 3: return launch_fmt<BGL_QNG64, 3>(L, CT, grid, st);
        case 4: return launch_fmt<BGL_QNG64, 4>(L, CT, grid, st);
        case 5: return launch_fmt<BGL_QNG64, 5>(L, CT, grid, st);
        case 6: return launch_fmt<BGL_QNG64, 6>(L, CT, grid, st);
        case 7: return launch_fmt<BGL_QNG64, 7>(L, CT, grid, st);
        case 8: return launch_fmt<BGL_QNG64, 8>(L, CT, grid, st);
        case 9: return launch_fmt<BGL_QNG64, 9>(L, CT, grid, st);
        case 10: return launch_fmt<BGL_QNG64, 10>(L, CT, grid, st);
        default: return -1;
        }
    default: return -1;
    }
}

static double mf_weight_bytes(const BglDevTensor &T) {
    const double per = T.fmt == BGL_Q8G64 ? 1.0625 : T.fmt == BGL_QNG64 ? T.bits / 8.0 + 0.0625 : 0.5625;
    return per * T.N * T.K;
}

// A split's K range must fit the workgroup's LDS (kpm steps); beyond that, split K until
// the grid has ~min_blocks workgroups while the partials (written and read back once
// each) stay under mf_pcap x the weight bytes (1 by default: at 0.5 the 4096 x 4096
// qNg64 n=5 tensors of a 32-column launch ran 64 workgroups, 19.3 us, against 128 and
// 15.0 us; finer splits than 16 K-steps measured no faster).
static int mf_splits(const bgl_ctx *c, const BglDevTensor &T, int Mc, int &kps) {
    const int CT = (Mc + 15) / 16, KS = T.K / 32, wgr = (T.ntiles + MF_TILES - 1) / MF_TILES;
    const int kpm = CT == 1 ? mf_kps_max(1) : CT == 2 ? mf_kps_max(2) : CT == 3 ? mf_kps_max(3) : mf_kps_max(4);
    const int smin = (KS + kpm - 1) / kpm;
    int S = (c->min_blocks + wgr - 1) / wgr;
    const int capS = (int)(c->mf_pcap * mf_weight_bytes(T) / (8.0 * Mc * T.N));
    if (S > capS) S = capS;
    if (S < smin) S = smin;
    if (S < 1) S = 1;
    kps = (KS + S - 1) / S;
    kps = (kps + MF_KSTEP_PAD - 1) / MF_KSTEP_PAD * MF_KSTEP_PAD;
    if (kps > kpm) kps = kpm;
    return (KS + kps - 1) / kps;
}

// The K-split partials (floats) of a launch of Mc columns.
static size_t mf_partials(const bgl_ctx *c, int n, const BglDevTensor *Ts, int Mc) {
    size_t fl = 0;
    for (int i = 0; i < n; i++) {
        int kps;
        const int S = mf_splits(c, Ts[i], Mc, kps);
        if (S > 1) fl += (size_t)S * Mc * Ts[i].N;
    }
    return fl;
}

// Scratch for the same call at fewer columns, which a caller may capture once this one has run: the
// partials do not grow strictly with the columns (this bounds them), and one column over a long K takes
// the digits of k_act_x24.  Operands that bgl_prep_act_dev left in the digits' buffers move with them.
static int mf_reserve_fewer(bgl_ctx *c, int n, const BglDevTensor *Ts, int M) {
    const int Mc = std::min(M, 16 * MF_MAXCT), CT = (Mc + 15) / 16;
    const int kpm = CT == 1 ? mf_kps_max(1) : CT == 2 ? mf_kps_max(2) : CT == 3 ? mf_kps_max(3) : mf_kps_max(4);
    const size_t ng = Ts[0].K / 64;
    double fl = 0.0;
    for (int i = 0; i < n; i++) {
        const int wgr = (Ts[i].ntiles + MF_TILES - 1) / MF_TILES, smin = (Ts[i].K / 32 + kpm - 1) / kpm;
        const double most = std::min((double)((c->min_blocks + wgr - 1) / wgr) * Mc * Ts[i].N, c->mf_pcap * mf_weight_bytes(Ts[i]) / 8.0);
        fl += std::max(most, smin > 1 ? (double)smin * Mc * Ts[i].N : 0.0);
    }
    const size_t pb = (size_t)fl * 4;
    const bool dig = !gemv_x_fuses(c, Ts[0].K) || Ts[0].K > BGL_GEMV_X_FUSE_MAX_K;
    if (c->part.bytes < pb) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        HIPCHK(hipStreamIsCapturing(c->stream, &cs));
        if (cs != hipStreamCaptureStatusNone) return 0;            // this call may still have all that it needs
        if (dbuf_reserve(c, c->part, pb, false)) return bgl_last_code();
    }
    return dig ? act_reserve_fewer(c, 2 * ng * 192, 2 * ng * 4, 4 * ng * 16) : 0;
}

// From 2 columns.  The dot4 kernels multiply three digits per value and column (k_gemv: 4 or 8 columns
// a launch), the matrix cores take 16 columns for the price of one; a wave's weights are the same.
// Measured, us, dot4 / here: q4g64 28672 x 4096 at 2 / 5 / 15 columns 40.2 / 28.9, 73.1 / 29.4, 153 /
// 32.5; 4096 x 4096 14.3 / 12.3, 19.7 / 12.4, 35.8 / 13.0; 1536 x 1536 13.6 / 11.3, 17.5 / 11.7, 31.8 /
// 12.4; q8g64 28672 x 4096 at 2 columns 41.1 / 34.9; qNg64 n = 6, 10 at 2: 54.5 / 38.8, 56.8 / 47.7.
// n = 3 at 2 / 4: 49.4 / 34.9, 52.2 / 35.3.  Against 64 bits the N(0, 1) products err by 1.6e-7 here, 2.9e-7
// there.
// Below 16 columns the dot4 kernels also keep what they alone can run: tensors of 2 GiB and more, and
// no-alloc calls whose K-split partials do not fit the fixed array.
bool mfma_takes(const bgl_ctx *c, int n, const BglDevTensor *Ts, int M) {
    if (c->no_mfma || M < 2) return false;
    for (int i = 0; i < n; i++)
        if (!bgl_mfma_ok(Ts[i].fmt, Ts[i].bits)) return false;
    if (M >= 16) return true;
    for (int i = 0; i < n; i++)
        if ((double)Ts[i].ntiles * Ts[i].cpr * 1024.0 >= 2147483648.0) return false;
    if (c->fixed_base && c->fixed_used + mf_partials(c, n, Ts, M) * 4 + 256 > c->fixed_cap) return false;
    return true;
}


// y[m][n] = bias[n] + sum_k W[n][k] x[m][k] for the n tensors of a group sharing x (same format,
// width and K), M >= 1 columns (mfma_takes says which calls come here).  Columns go in launches of up to
// 64: one fragment prep, one GEMM over every tensor, and one reduce when any tensor splits K.
int run_gemm_mfma(bgl_ctx *c, int n, const BglDevTensor *Ts, const float *x_dev, int M, const float *const *bias,
                  float *const *y, const int *ystride, float *glu_h) {
    const int K = Ts[0].K;
    if (glu_h && (n != 2 || Ts[1].N != Ts[0].N))
        return bgl_fail(BGL_E_ARG, "MFMA path: the SwiGLU pair needs two tensors of one shape");
    if (K % 64) return bgl_fail(BGL_E_ARG, "MFMA path: in=%d %% 64 != 0", K);
    if (n < 1 || n > BGL_MAX_TASKS) return bgl_fail(BGL_E_ARG, "MFMA path: %d tensors in a group (1..%d)", n, BGL_MAX_TASKS);
    for (int i = 0; i < n; i++) {
        if (!bgl_mfma_ok(Ts[i].fmt, Ts[i].bits)) return bgl_fail(BGL_E_UNSUPPORTED, "MFMA path: kind %d", Ts[i].fmt);
        if (Ts[i].fmt != Ts[0].fmt || Ts[i].bits != Ts[0].bits || Ts[i].K != K)
            return bgl_fail(BGL_E_ARG, "MFMA path: a group shares kind, bits and in");
        const double wb = (double)Ts[i].ntiles * Ts[i].cpr * 1024.0;
        if (wb >= 2147483648.0) return bgl_fail(BGL_E_UNSUPPORTED, "MFMA path: tensor %d holds >= 2 GiB (32-bit buffer offsets)", i);
    }
    if (!c->fixed_base) {
        const int rc = mf_reserve_fewer(c, n, Ts, M);
        if (rc) return rc;
    }
    // The chunks run in stream order, so each reuses the same K-split partials.  In a no-alloc call
    // the fixed array is handed out by a bump pointer: rewind it to this mark before every chunk,
    // so the first (largest) chunk's reservation bounds the whole call.
    const size_t fixed_mark = c->fixed_used;
    for (int m0 = 0; m0 < M; m0 += 16 * MF_MAXCT) {
        const int Mc = M - m0 < 16 * MF_MAXCT ? M - m0 : 16 * MF_MAXCT;
        if (c->fixed_base) c->fixed_used = fixed_mark;
        const int CT = (Mc + 15) / 16;
        MfmaLaunch L;
        memset(&L, 0, sizeof L);
        L.ntasks = n; L.M = Mc; L.residual = M < 16; L.x = x_dev + (size_t)m0 * K;
        int wgs = 0;
        size_t poff[BGL_MAX_TASKS], pfl = 0;              // partial offsets (floats) in the shared buffer
        int S_[BGL_MAX_TASKS];
        for (int i = 0; i < n; i++) {
            const BglDevTensor &T = Ts[i];
            const int wgr = (T.ntiles + MF_TILES - 1) / MF_TILES;
            int kps;
            const int S = mf_splits(c, T, Mc, kps);
            S_[i] = S;
            MfmaTask &t = L.t[i];
            t.T = T; t.bias = bias ? bias[i] : nullptr;
            t.ystride = ystride ? ystride[i] : T.N;
            t.y = y[i] + (size_t)m0 * t.ystride;
            t.wg0 = wgs; t.wgr = wgr; t.kps = kps;
            wgs += wgr * S;
            poff[i] = pfl;
            if (S > 1) pfl += (size_t)S * Mc * T.N;
        }
        MfmaReduce R;
        memset(&R, 0, sizeof R);
        R.M = Mc;
        if (pfl) {
            if (dbuf_reserve(c, c->part, pfl * 4, false)) return bgl_last_code();
            int nq = 0;
            for (int i = 0; i < n; i++) {
                if (S_[i] == 1) continue;
                MfmaTask &t = L.t[i];
                t.part = (float *)c->part.p + poff[i];
                MfmaReduceTask &rt = R.t[R.ntasks++];
                rt.part = t.part; rt.bias = t.bias; rt.y = t.y; rt.N = t.T.N; rt.S = S_[i]; rt.ystride = t.ystride;
                rt.q0 = nq;
                nq += Mc * ((t.T.N + 3) / 4);
            }
            R.nquads = nq;
        }
        if (glu_h) {                    // SwiGLU pair: both tasks, split or not, one quad grid
            for (int i = 0; i < 2; i++) {
                const MfmaTask &t = L.t[i];
                MfmaReduceTask &rt = R.t[i];
                rt.part = S_[i] > 1 ? t.part : nullptr; rt.bias = t.bias; rt.y = t.y;
                rt.N = t.T.N; rt.S = S_[i]; rt.ystride = t.ystride; rt.q0 = 0;
            }
            R.ntasks = 2;
            R.glu_h = glu_h + (size_t)m0 * Ts[0].N;
            R.glu_stride = Ts[0].N;
            R.nquads = Mc * ((Ts[0].N + 3) / 4);
        }
        int tok = prof_begin(c, 1);
        if (launch_any(L, Ts[0].fmt, Ts[0].bits, CT, dim3(wgs), c->stream)) return bgl_fail(BGL_E_UNSUPPORTED, "MFMA path: format");
        prof_end(c, tok);
        HIPCHK(hipGetLastError());
        if (R.ntasks) {
            tok = prof_begin(c, 2);
            hipLaunchKernelGGL(k_mfma_reduce, dim3((R.nquads + 255) / 256), dim3(256), 0, c->stream, R);
            prof_end(c, tok);
            HIPCHK(hipGetLastError());
        }
    }
    return 0;
}
