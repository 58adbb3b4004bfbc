// ut_gemm.hip -- QTensor::matmul (undertow-quant/src/qtensor.rs:281-319) on
// gfx950 for more rows than the skinny GEMVs take: digit planes of the
// activations and the matrix-core product (ut_gemm_core.h).
#include "ut_gemm.h"

#include <cmath>

#include "ut_gemm_core.h"

namespace ut {

// ------------------------------------------------------- digit planes ---
size_t planes_bytes(int64_t M, int64_t K) {
    return (((size_t)M * 4 + 255) & ~size_t(255)) + (size_t)M * 3 * planes_pitch(K);
}
DigitPlanes planes_view(void *base, int64_t M, int64_t K) {
    DigitPlanes d;
    d.exps = (int32_t *)base;
    d.p = (int8_t *)base + (((size_t)M * 4 + 255) & ~size_t(255));
    d.kp = planes_pitch(K);
    return d;
}

// A row's values: f32, bf16 (widened), or silu(g) * u of an MLP's two halves
// (undertow-quant/src/lib.rs:121; model.rs:241-247).
struct RowF32 {
    const float *x;
    int64_t ld;
    __device__ __forceinline__ float at(int64_t m, int64_t k) const { return x[m * ld + k]; }
    __device__ __forceinline__ void at4(int64_t m, int64_t k, float (&v)[4]) const {
        const float4 f = ld_global<float4>(x + m * ld + k);
        v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
    }
    bool vec() const { return ((uintptr_t)x & 15) == 0 && ld % 4 == 0; }
};
struct RowBf16 {
    const uint16_t *x;
    int64_t ld;
    __device__ __forceinline__ float at(int64_t m, int64_t k) const {
        return __uint_as_float((uint32_t)x[m * ld + k] << 16);
    }
    __device__ __forceinline__ void at4(int64_t m, int64_t k, float (&v)[4]) const {
        const uint2 u = ld_global<uint2>(x + m * ld + k);
        v[0] = __uint_as_float(u.x << 16); v[1] = __uint_as_float(u.x & 0xffff0000u);
        v[2] = __uint_as_float(u.y << 16); v[3] = __uint_as_float(u.y & 0xffff0000u);
    }
    bool vec() const { return ((uintptr_t)x & 7) == 0 && ld % 4 == 0; }
};
struct RowSilu {
    const float *g, *u;
    int64_t ld;
    static __device__ __forceinline__ float h(float g, float u) {
        return __fmul_rn(g / (1.0f + expf(-g)), u);
    }
    __device__ __forceinline__ float at(int64_t m, int64_t k) const {
        return h(g[m * ld + k], u[m * ld + k]);
    }
    __device__ __forceinline__ void at4(int64_t m, int64_t k, float (&v)[4]) const {
        const float4 a = ld_global<float4>(g + m * ld + k), b = ld_global<float4>(u + m * ld + k);
        v[0] = h(a.x, b.x); v[1] = h(a.y, b.y); v[2] = h(a.z, b.z); v[3] = h(a.w, b.w);
    }
    bool vec() const { return (((uintptr_t)g | (uintptr_t)u) & 15) == 0 && ld % 4 == 0; }
};

// One workgroup per row: max|x|, exponent, then four columns a time into
// one word per plane.  The first kPlaneRegs * 1024 columns stay in
// registers between the two passes.  Bound by the row's read: one round
// trip (512 rows of 16,384 columns: 33.5 MB in, 25 MB out).
constexpr int kPlaneRegs = 8;
template <typename Row, bool VEC>
__global__ __launch_bounds__(256) void k_planes(Row row, int64_t K, int8_t *__restrict__ pl,
                                                int64_t kp, int32_t *__restrict__ exps) {
    __shared__ uint32_t red[4];
    const int64_t m = blockIdx.x;
    const int tid = threadIdx.x;
    float v[kPlaneRegs][4];
    auto load = [&](int64_t c, float (&o)[4]) {
        if (VEC && c + 4 <= K) {
            row.at4(m, c, o);
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) o[j] = c + j < K ? row.at(m, c + j) : 0.0f;
        }
    };
    uint32_t mx = 0;
#pragma unroll
    for (int i = 0; i < kPlaneRegs; i++) {
        const int64_t c = 4 * (tid + 256 * (int64_t)i);
        if (c < kp) load(c, v[i]);
    }
#pragma unroll
    for (int i = 0; i < kPlaneRegs; i++)
        if (4 * (tid + 256 * (int64_t)i) < kp)
#pragma unroll
            for (int j = 0; j < 4; j++) mx = max(mx, __float_as_uint(fabsf(v[i][j])));
    for (int64_t c = 4 * (tid + 256 * (int64_t)kPlaneRegs); c < K; c += 1024) {
        float t[4];
        load(c, t);
#pragma unroll
        for (int j = 0; j < 4; j++) mx = max(mx, __float_as_uint(fabsf(t[j])));
    }
    mx = block_reduce(mx, [](uint32_t a, uint32_t b) { return a > b ? a : b; }, red);
    // non-finite rows (|x| bits >= +inf) produce NaN outputs downstream
    const bool bad = mx >= 0x7f800000u;
    int E = 0;
    if (!bad && mx != 0) (void)frexpf(__uint_as_float(mx), &E);
    const int sh = bad ? INT32_MIN : 22 - E;
    if (tid == 0) exps[m] = bad ? INT32_MIN : E - 22;
    auto put = [&](int64_t c, const float (&o)[4]) {
        uint32_t w[3];
        digit_words<UT_FMT_INT8>(o, 4, sh, w);
#pragma unroll
        for (int p = 0; p < 3; p++) *(uint32_t *)(pl + (m * 3 + p) * kp + c) = bad ? 0u : w[p];
    };
#pragma unroll
    for (int i = 0; i < kPlaneRegs; i++) {
        const int64_t c = 4 * (tid + 256 * (int64_t)i);
        if (c < kp) put(c, v[i]);
    }
    for (int64_t c = 4 * (tid + 256 * (int64_t)kPlaneRegs); c < kp; c += 1024) {
        float t[4];
        load(c, t);
        put(c, t);
    }
}

template <typename Row>
static int32_t planes_t(ut_ctx *ctx, const char *name, const Row &row, int64_t M, int64_t K,
                        const DigitPlanes &pl) {
    if (M <= 0) return UT_OK;
    int tok = timing_begin(ctx, name);
    if (row.vec())
        hipLaunchKernelGGL((k_planes<Row, true>), dim3((unsigned)M), dim3(256), 0, ctx->stream, row,
                           K, pl.p, pl.kp, pl.exps);
    else
        hipLaunchKernelGGL((k_planes<Row, false>), dim3((unsigned)M), dim3(256), 0, ctx->stream, row,
                           K, pl.p, pl.kp, pl.exps);
    timing_end(ctx, tok);
    return launch_check(ctx, "k_planes");
}
int32_t launch_planes(ut_ctx *ctx, const float *x, int64_t ldx, int64_t M, int64_t K,
                      const DigitPlanes &pl) {
    return planes_t(ctx, "planes", RowF32{x, ldx}, M, K, pl);
}
int32_t launch_planes(ut_ctx *ctx, const uint16_t *x, int64_t ldx, int64_t M, int64_t K,
                      const DigitPlanes &pl) {
    return planes_t(ctx, "planes", RowBf16{x, ldx}, M, K, pl);
}
int32_t launch_silu_planes(ut_ctx *ctx, const float *g, const float *u, int64_t M, int64_t I,
                           const DigitPlanes &pl) {
    return planes_t(ctx, "silu_planes", RowSilu{g, u, I}, M, I, pl);
}

// --------------------------------------------------------------- GEMM ---
// One or two weights of one format and width against the same rows.
struct GemmWeight {
    const uint8_t *w, *end;
    const float *scales;
    int64_t O;  // weight rows
    float *out;
    int64_t ldo;
};
struct GemmArgs {
    GemmWeight w[2];
    int64_t row_bytes;  // from one weight row to the next (all of them read)
    int to0;            // weight tiles of w[0]; the launch's others are w[1]'s
    const int8_t *pl;
    int64_t kp;
    const int32_t *exps;
    int64_t M;
    int accumulate;
    // units = weight tiles x K splits; a unit's activation tiles run on one XCD
    int to, tm, ks;
    int64_t kslice;
    int64_t *part;  // ks > 1: totals [ks][M][O], w[1]'s rows after w[0]'s
};

// A wave's finished tile: rows o0 .. of weight wi, activation rows m0 ..
template <int FMT, int TO, int TM>
__device__ __forceinline__ void gemm_store(const GemmArgs &a, int wi,
                                           const ut_i32x4 (&acc)[TO][TM][3], int64_t o0, int64_t m0,
                                           int z) {
    const GemmWeight &W = a.w[wi];
    const int64_t po0 = wi ? a.w[0].O : 0, OT = a.w[0].O + a.w[1].O;
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int t = 0; t < TO; t++) {
        const int64_t o = o0 + 16 * t + 4 * q;
#pragma unroll
        for (int n = 0; n < TM; n++) {
            const int64_t m = m0 + 16 * n + r;
            if (m >= a.M || o >= W.O) continue;
            int64_t S[4];
#pragma unroll
            for (int i = 0; i < 4; i++) S[i] = gemm_total(acc[t][n], i);
            if (a.ks > 1) {
                int64_t *p = a.part + ((int64_t)z * a.M + m) * OT + po0 + o;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (o + i < W.O) p[i] = S[i];
                continue;
            }
            const int32_t e = gemm_exp<FMT>(a.exps[m]);
            float *po = W.out + m * W.ldo + o;
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (o + i < W.O) {
                    const float v = int_total_to_f32(S[i], e, ld_global_f32(W.scales + o + i));
                    po[i] = a.accumulate ? __fadd_rn(po[i], v) : v;
                }
        }
    }
}

// Up to kGlMinRows rows, and any number of rows of unaligned weights.  The
// weights' read bounds the few rows (int8 7168 x 16384 from memory: 16 rows
// 47 us, 2.5 TB/s; the four-row GEMV passes took 118 us), the unaligned loads
// the others (200 rows of 1003 x 1537: 29 us).
constexpr int kGemmTO = 4;
template <int FMT, int TM, bool UNAL>
__global__ __launch_bounds__(kGemmThreads, 2) void k_gemm(GemmArgs a) {
    __shared__ uint4 lds[gemm_lds_uint4<TM>()];
    // consecutive workgroups go to the 8 XCDs in turn: the activation tiles
    // of one weight tile are given to one XCD, so its L2 serves the weights
    // to all but the first of them
    const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
    const int unit = (j / a.tm) * 8 + xcd, mt = j % a.tm;
    if (unit >= a.to * a.ks) return;
    const int ut = unit % a.to, z = unit / a.to, wi = ut >= a.to0, ot = wi ? ut - a.to0 : ut;
    const GemmWeight &W = a.w[wi];
    const int tid = threadIdx.x, r = tid & 15;
    const int64_t o0 = (int64_t)ot * (64 * kGemmTO) + (tid >> 6) * (16 * kGemmTO);
    const int64_t m0 = (int64_t)mt * (16 * TM);
    GemmRows<kGemmTO> rows;
#pragma unroll
    for (int t = 0; t < kGemmTO; t++) {
        const int64_t o = o0 + 16 * t + r;
        rows.row[t] = W.w + (o < W.O ? o : W.O - 1) * a.row_bytes;
    }
    rows.end = W.end;
    const int8_t *src[gemm_stage_n<TM>()];
#pragma unroll
    for (int i = 0; i < gemm_stage_n<TM>(); i++) {
        const GemmChunk c = gemm_chunk(tid + i * kGemmThreads);
        const int64_t m = m0 + c.m < a.M ? m0 + c.m : a.M - 1;
        src[i] = a.pl + (m * 3 + (c.p < 3 ? c.p : 0)) * a.kp + c.off;
    }
    const int64_t kb = z * a.kslice, ke = kb + a.kslice < a.kp ? kb + a.kslice : a.kp;
    ut_i32x4 acc[kGemmTO][TM][3];
    gemm_tile<FMT, kGemmTO, TM, UNAL>(rows, a.row_bytes, kb, ke, src, lds, acc);
    gemm_store<FMT, kGemmTO, TM>(a, wi, acc, o0, m0, z);
}

// More than kGlMinRows rows of 16-byte aligned weights: 128 weight rows x 64
// activation rows per workgroup, two workgroups per CU.  Bound by the matrix
// cores (from registers alone the instruction reaches 3.55 POP/s on random
// data; a large int8 library product 2.1): 512 rows of int8 7168 x 16384
// 285 us with the direct tile, 197 us with eight waves of 2 x 2 tiles;
// 129280 x 7168 1,982 -> 1,545; int4 18432 x 7168 260 -> 226 (without the
// digitising).  256 x 64 tiles, one workgroup per CU: 217 / 1,724 / 265;
// stages of 64 columns, three workgroups: 257 / 1,796 / 269.  At 32 rows and
// fewer the launch is bound by the weights' read, which the direct tile keeps
// more of in flight (129280 x 7168 at 16 rows 183 against 234 us); at 64 this
// one leads (7168 x 16384 67 -> 61 us, 18432 x 7168 72 -> 63).
constexpr int64_t kGlMinRows = 32;
//
// LONG (slices of more than kGlLong stages): four waves of 4 x 2 tiles, which
// read 10 fragments for 24 matrix instructions instead of 8 for 12, each
// half stage's beside the matrix instructions of the half before (PIPE): a
// wave's reads otherwise stand before its products.  Counters: matrix cores
// 51% busy over 129280 x 7168 and 41% over 7168 x 16384, 29% of the wave
// cycles waiting, no LDS bank conflicts.  512 rows of 129280 x 7168
// 1,472 -> 1,375 us (2.07 POP/s), 18432 x 7168 251 -> 227, int4 234 -> 212,
// 7168 x 16384 214 -> 204 and at 64 rows 65.1 -> 63.1, with the digitising.
// The short slices' eight waves fill the pipeline sooner: 509 rows of
// 24576 x 1536 92.3 us, 94.7 with LONG; 200 of int4 7168 x 2048 27.9 / 29.4.
// Four buffers of 64-column stages, three in flight, copy half lines of 128
// bytes: 243 us at 7168 x 16384 and 1,637 at 129280 x 7168, with PIPE reads
// 250 and 1,686.
constexpr int kGlTM = 2, kGlWM = 2;
constexpr int kGlRows = 128;  // weight rows per workgroup
constexpr int64_t kGlLong = 16;
template <bool LONG> constexpr int gl_to() { return LONG ? 4 : 2; }
template <bool LONG> constexpr int gl_threads() { return 64 * kGlRows / (16 * gl_to<LONG>()) * kGlWM; }
template <int FMT, bool LONG>
__global__ __launch_bounds__(gl_threads<LONG>(), 2) void k_gemm_lds(GemmArgs a) {
    constexpr int TO = gl_to<LONG>(), WO = kGlRows / (16 * TO);
    using L = GemmLds<FMT, TO, kGlTM, WO, kGlWM>;
    __shared__ L s0, s1;
    const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
    const int unit = (j / a.tm) * 8 + xcd, mt = j % a.tm;
    if (unit >= a.to * a.ks) return;
    const int ut = unit % a.to, z = unit / a.to, wi = ut >= a.to0, ot = wi ? ut - a.to0 : ut;
    const GemmWeight &W = a.w[wi];
    const int wave = threadIdx.x >> 6;
    const int64_t ob = (int64_t)ot * L::kARows, mb = (int64_t)mt * (16 * kGlTM * kGlWM);
    GemmSrc<FMT, TO, kGlTM, WO, kGlWM> src;
    gemm_src<FMT, TO, kGlTM, WO, kGlWM>(
        src,
        [&](int row) { return W.w + (ob + row < W.O ? ob + row : W.O - 1) * a.row_bytes; },
        [&](int m, int p) { return a.pl + ((mb + m < a.M ? mb + m : a.M - 1) * 3 + p) * a.kp; });
    const int64_t kb = z * a.kslice, ke = kb + a.kslice < a.kp ? kb + a.kslice : a.kp;
    ut_i32x4 acc[TO][kGlTM][3];
    gemm_tile_lds<LONG, FMT, TO, kGlTM, WO, kGlWM>(src, a.row_bytes, kb, ke, s0, s1, acc);
    gemm_store<FMT, TO, kGlTM>(a, wi, acc, ob + (wave % WO) * (16 * TO),
                               mb + (wave / WO) * (16 * kGlTM), z);
}

// The K splits' totals summed and scaled (exact integers: any order).
template <int FMT>
__global__ __launch_bounds__(256) void k_gemm_sum(GemmArgs a) {
    const int64_t OT = a.w[0].O + a.w[1].O, i = (int64_t)blockIdx.x * 256 + threadIdx.x, n = a.M * OT;
    if (i >= n) return;
    const int64_t m = i / OT, x = i - m * OT;
    const int wi = x >= a.w[0].O;
    const int64_t o = wi ? x - a.w[0].O : x;
    const GemmWeight &W = a.w[wi];
    int64_t S = 0;
#pragma unroll 8
    for (int z = 0; z < a.ks; z++) S += a.part[z * n + i];
    const float v = int_total_to_f32(S, gemm_exp<FMT>(a.exps[m]), W.scales[o]);
    float *po = W.out + m * W.ldo + o;
    *po = a.accumulate ? __fadd_rn(*po, v) : v;
}

bool gemm_ok(const ut_qtensor *w, int64_t M) {
    // 65,536 columns: the planes' int32 sums (K x 128 x 128) cannot overflow
    return M >= kGemmMinRows && (w->fmt == UT_FMT_INT8 || w->fmt == UT_FMT_INT4) &&
           w->in_dim >= 1 && w->in_dim <= 65536;
}

bool gemm_pair_ok(const ut_qtensor *w, const ut_qtensor *w2, int64_t M) {
    return gemm_ok(w, M) && gemm_ok(w2, M) && w->fmt == w2->fmt && w->in_dim == w2->in_dim &&
           w->row_bytes == w2->row_bytes &&
           ((((uintptr_t)w->payload ^ (uintptr_t)w2->payload) & 15) == 0);
}

int32_t launch_gemm(ut_ctx *ctx, const ut_qtensor *w, const DigitPlanes &x, int64_t M, float *out,
                    int64_t ldo, int accumulate, const ut_qtensor *w2, float *out2, int64_t ldo2) {
    if (w2 && !gemm_pair_ok(w, w2, M)) {
        set_error(ctx, "gemm: the two weights must share format, width and alignment");
        return UT_ERR_ARG;
    }
    GemmArgs a{};
    auto weight = [](const ut_qtensor *t, float *o, int64_t ld) {
        const uint8_t *p = (const uint8_t *)t->payload;
        return GemmWeight{p, p + t->out_dim * t->row_bytes, t->scales, t->out_dim, o, ld};
    };
    a.row_bytes = w->row_bytes;
    a.kp = x.kp;
    a.accumulate = accumulate;
    const bool unal = ((uintptr_t)w->payload & 15) != 0 || w->row_bytes % 16 != 0;
    const int64_t cap = 1 << 16;  // rows per launch: grids stay within 2^32 threads
    const int64_t O2 = w2 ? w2->out_dim : 0, OT = w->out_dim + O2;
    for (int64_t s0 = 0; s0 < M; s0 += cap) {
        a.M = M - s0 < cap ? M - s0 : cap;
        a.pl = x.p + s0 * 3 * x.kp;
        a.exps = x.exps + s0;
        a.w[0] = weight(w, out + s0 * ldo, ldo);
        if (w2) a.w[1] = weight(w2, out2 + s0 * ldo2, ldo2);
        const bool big = !unal && a.M > kGlMinRows;
        const int tmr = big ? kGlTM * kGlWM : a.M <= 16 ? 1 : 2;
        const int tor = big ? kGlRows : 64 * kGemmTO;
        a.to0 = (int)((w->out_dim + tor - 1) / tor);
        a.to = a.to0 + (int)((O2 + tor - 1) / tor);
        a.tm = (int)((a.M + 16 * tmr - 1) / (16 * tmr));
        // split K until the launch has two workgroups per CU, at least two
        // steps each, partials within their buffer, and not beyond where a
        // split's partials (16 bytes a total written and read, at 4 MB a us)
        // cost more than it takes off the steps (0.8 us each, unaligned rows
        // 2.5): the sum of both is least at sqrt(steps * step / split)
        // splits.  37 rows of int4 2048 x 7168 31.0 -> 22.6 us (28 splits were
        // 17 MB of partials beside an 8 MB weight), 77 rows of int8 1536 x 7168
        // 31.1 -> 25.1, 128 of 576 x 7168 32.1 -> 25.9; 0.3 and 2 us a step:
        // 22.9 / 28.7, 27.6 / 29.9, 25.6 / 28.0; 200 unaligned rows of
        // 1003 x 1537 29.3 us at 2.5, 31.9 at 0.8.
        int64_t ks = (2 * ctx->multiprocessors) / ((int64_t)a.to * a.tm);
        const int64_t steps = a.kp / kGemmStep;
        if (ks > steps / 2) ks = steps / 2;
        const double split_us = (double)a.M * (double)OT * 16.0 / 4.0e6;
        const int64_t best = (int64_t)(sqrt((double)steps * (unal ? 2.5 : 0.8) / split_us) + 0.5);
        if (ks > best) ks = best;
        while (ks > 1 && ks * a.M * OT * 8 > kSplitKPartBytes) ks--;
        // (a first call under capture has no buffer for the partials)
        if (ks < 1 || (!ctx->splitk && ks > 1 && stream_capturing(ctx))) ks = 1;
        a.kslice = (steps + ks - 1) / ks * kGemmStep;
        a.ks = (int)((a.kp + a.kslice - 1) / a.kslice);
        if (a.ks > 1) UT_TRY(splitk_buffer(ctx, &a.part));
        const int64_t units = (int64_t)a.to * a.ks;
        const dim3 grid((unsigned)((units + 7) / 8 * 8 * a.tm));
        int tok = timing_begin(ctx, "gemm");
#define UT_GM(F, T, U) hipLaunchKernelGGL((k_gemm<F, T, U>), grid, dim3(kGemmThreads), 0, ctx->stream, a)
#define UT_GMT(F, U)                    \
    do {                                \
        if (tmr == 1) UT_GM(F, 1, U);   \
        else UT_GM(F, 2, U);            \
    } while (0)
        if (big) {
            const bool lng = a.kslice > kGlLong * kGemmStep;
#define UT_GL(F, LG) hipLaunchKernelGGL((k_gemm_lds<F, LG>), grid, dim3(gl_threads<LG>()), 0, ctx->stream, a)
            if (w->fmt == UT_FMT_INT8) {
                if (lng) UT_GL(UT_FMT_INT8, true);
                else UT_GL(UT_FMT_INT8, false);
            } else {
                if (lng) UT_GL(UT_FMT_INT4, true);
                else UT_GL(UT_FMT_INT4, false);
            }
#undef UT_GL
        } else if (w->fmt == UT_FMT_INT8) {
            if (unal) UT_GMT(UT_FMT_INT8, true);
            else UT_GMT(UT_FMT_INT8, false);
        } else {
            if (unal) UT_GMT(UT_FMT_INT4, true);
            else UT_GMT(UT_FMT_INT4, false);
        }
#undef UT_GMT
#undef UT_GM
        UT_TRY(launch_check(ctx, "k_gemm"));
        if (a.ks > 1) {
            const dim3 sg((unsigned)((a.M * OT + 255) / 256));
            if (w->fmt == UT_FMT_INT8)
                hipLaunchKernelGGL(k_gemm_sum<UT_FMT_INT8>, sg, dim3(256), 0, ctx->stream, a);
            else
                hipLaunchKernelGGL(k_gemm_sum<UT_FMT_INT4>, sg, dim3(256), 0, ctx->stream, a);
            UT_TRY(launch_check(ctx, "k_gemm_sum"));
        }
        timing_end(ctx, tok);
    }
    return UT_OK;
}

}  // namespace ut
