// ut_gemm_f32.hip -- f32 weights against more activation rows than the f32
// GEMVs take (undertow-quant/src/qtensor.rs:281-319 over a prompt's rows).
// Both kernels add each output's products in the order of the GEMV that one
// to four rows take, so a row's value does not depend on how many rows
// share the call; that rules the f32 matrix cores out, whose order is fixed.
#include "ut_gemm.h"

#include "ut_gemv_core.h"

namespace ut {

// ------------------------------------------------ k_gemv's f32 order ---
// A K slice of k_gemv adds, for each of 16 lanes s, the columns 64 t + 4 s
// + [0, 4) in t order, the 16 lane sums by a butterfly (xor 8, 4, 2, 1), and
// the slices' values in slice order.  Here a thread holds 4 x 4 outputs and
// runs the lanes' chains one after another, adding each to its butterfly
// partner as soon as both are there (at most three sums wait), so the
// products of 64 rows x 64 outputs share their operands through LDS.
constexpr int kF32Tile = 64;
struct F32Args {
    const float *w, *x;
    int64_t O, K, M, ldx;
    float *out;
    int64_t ldo;
    int accumulate;
    int ks;
    int64_t kslice;
    float *part;  // ks > 1: [ks][M][O]
};

template <int T> struct F32Tiles {
    float x[kF32Tile][64 * T + 4], w[kF32Tile][64 * T + 4];
};
struct F32Acc {
    float v[4][4];
};
template <int T>
__device__ __forceinline__ F32Acc f32_chain(const F32Tiles<T> &l, int ty, int tx, int s) {
    F32Acc a;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) a.v[i][j] = 0.0f;
#pragma unroll
    for (int t = 0; t < T; t++) {
        float4 xv[4], wv[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            xv[i] = *(const float4 *)&l.x[ty + 16 * i][64 * t + 4 * s];
            wv[i] = *(const float4 *)&l.w[tx + 16 * i][64 * t + 4 * s];
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float c = a.v[i][j];
                c = __builtin_fmaf(wv[j].x, xv[i].x, c);
                c = __builtin_fmaf(wv[j].y, xv[i].y, c);
                c = __builtin_fmaf(wv[j].z, xv[i].z, c);
                c = __builtin_fmaf(wv[j].w, xv[i].w, c);
                a.v[i][j] = c;
            }
    }
    return a;
}
__device__ __forceinline__ void f32_add(F32Acc &a, const F32Acc &b) {
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) a.v[i][j] = __fadd_rn(a.v[i][j], b.v[i][j]);
}
// The 16 lanes' butterfly: after xor 8 the value of lane s is a[s] + a[s^8],
// and so on (f32 addition commutes, so a butterfly's lanes all hold the same
// value).  Lanes 0..7 in bit-reversed order meet their partners of xor 4, 2
// and 1 as a binary counter carries.  A loop, not an unrolled tree: its
// reads would be hoisted past the register file.
template <int T> __device__ __forceinline__ F32Acc f32_tree(const F32Tiles<T> &l, int ty, int tx) {
    F32Acc b, s4, s2, s1;
#pragma unroll 1
    for (int u = 0; u < 8; u++) {
        const int s = ((u & 1) << 2) | (u & 2) | (u >> 2);
        b = f32_chain<T>(l, ty, tx, s);
        f32_add(b, f32_chain<T>(l, ty, tx, s + 8));
        if (!(u & 1)) {
            s4 = b;
            continue;
        }
        f32_add(b, s4);
        if (!(u & 2)) {
            s2 = b;
            continue;
        }
        f32_add(b, s2);
        if (!(u & 4)) s1 = b;
        else f32_add(b, s1);
    }
    return b;
}

// 64 rows x 64 outputs x one slice of up to 64 T columns.  Bound by the
// vector unit (the FMAs and 15 additions per 64 T columns) beside its LDS
// reads: 512 rows of 256 x 7168 with the sum 61 us (24 us of FMAs at the
// unit's rate) against 1,339 us in four-row passes.
template <int T>
__global__ __launch_bounds__(256) void k_gemm_f32(F32Args a, int to) {
    __shared__ __attribute__((aligned(16))) F32Tiles<T> l;
    const int64_t o0 = (int64_t)(blockIdx.x % to) * kF32Tile, m0 = (int64_t)(blockIdx.x / to) * kF32Tile;
    const int z = blockIdx.y, tid = threadIdx.x;
    const int64_t kb = z * a.kslice, ke = kb + a.kslice < a.K ? kb + a.kslice : a.K;
    for (int i = tid; i < kF32Tile * 16 * T; i += 256) {
        const int r = i / (16 * T), c = 4 * (i - r * 16 * T);
        const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        *(float4 *)&l.x[r][c] = m0 + r < a.M && kb + c < ke ? ld_global<float4>(a.x + (m0 + r) * a.ldx + kb + c) : zero;
        *(float4 *)&l.w[r][c] = o0 + r < a.O && kb + c < ke ? ld_global<float4>(a.w + (o0 + r) * a.K + kb + c) : zero;
    }
    __syncthreads();
    const int tx = tid & 15, ty = tid >> 4;
    const F32Acc v = f32_tree<T>(l, ty, tx);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t m = m0 + ty + 16 * i, o = o0 + tx + 16 * j;
            if (m >= a.M || o >= a.O) continue;
            if (a.ks > 1) {
                a.part[((int64_t)z * a.M + m) * a.O + o] = v.v[i][j];
            } else {
                float *p = a.out + m * a.ldo + o;
                *p = a.accumulate ? __fadd_rn(*p, v.v[i][j]) : v.v[i][j];
            }
        }
}

__global__ __launch_bounds__(256) void k_gemm_f32_sum(F32Args a) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, n = a.M * a.O;
    if (i >= n) return;
    const int64_t m = i / a.O, o = i - m * a.O;
    float v = a.part[i];
#pragma unroll 8
    for (int z = 1; z < a.ks; z++) v = __fadd_rn(v, a.part[z * n + i]);
    float *p = a.out + m * a.ldo + o;
    *p = a.accumulate ? __fadd_rn(*p, v) : v;
}

// The fewest rows whose product of whole 64-row tiles beats the GEMV's
// four-row passes.  A tile takes about 3 us per 64 columns of its slice
// however few of its rows are there; a pass takes 3.5 us, with split K 6 and
// more and a second launch.
// Split K, slices of up to 128 columns in one wave of workgroups (two per
// CU): from five rows on (256 x 7168 18.7 us in passes, 16.2 so, 512 x 4096
// 21.7 / 14.9, 1024 x 1024 14.4 / 13.4); in more (1024 x 7168 at six 28.8 /
// 30.1, at nine 43.6 / 29.9) from nine.  Longer slices in one wave (one per
// CU) also from five: up to eight rows the passes lead on a stream that the
// host keeps full (512 x 260 12.5 against 15.3), the product in calls made one
// after another from Python (16.6 / 15.2: two launches, not four); in two
// waves (3000 x 1500 at nine 28.1 / 30.5) from thirteen, in more (2048 x 7168
// at twelve 50.4 / 77.7, at seventeen 82 / 78) from seventeen.
// Unsplit: 64 x 64 at five 7.0 / 6.2; two steps from nine (1000 x 128 at eight
// 7.6 / 9.8, at nine 10.4 / 9.9), three from thirteen (256 x 192 at twelve
// 11.6 / 13.0, at thirteen 14.6 / 13.0), four from fourteen (256 x 252 at
// thirteen 15.6 / 16.0, at sixteen 17.2 / 16.2), and where their tiles (one
// per CU) are more than one wave, 25 (20000 x 256 at 20 rows 26.7 / 32.4).
static int64_t gemm_f32_min_rows(int64_t O, int ks, int64_t kslice) {
    const int64_t tiles = (O + kF32Tile - 1) / kF32Tile, steps = (kslice + 63) / 64;
    if (ks > 1 && steps <= 2) return tiles * ks <= 512 ? kGemmMinRows : 9;
    if (ks > 1) return tiles * ks <= 256 ? kGemmMinRows : tiles * ks <= 512 ? 13 : 17;
    if (steps <= 2) return steps == 1 ? kGemmMinRows : 9;
    return tiles > 256 ? 25 : steps == 3 ? 13 : 14;
}

bool gemm_f32_ok(const ut_qtensor *w, const float *x, int64_t M) {
    if (w->fmt != UT_FMT_F32 || M < kGemmMinRows || w->in_dim % 4 != 0 ||
        (((uintptr_t)w->payload | (uintptr_t)x) & 15) != 0)
        return false;
    int ks;
    int64_t kslice;
    gemv_f32_split(w->out_dim, w->in_dim, &ks, &kslice);
    return M >= gemm_f32_min_rows(w->out_dim, ks, kslice) && kslice <= 256 &&
           (ks == 1 || (int64_t)ks * w->out_dim * kF32Tile * 4 <= kSplitKPartBytes);
}

int32_t launch_gemm_f32(ut_ctx *ctx, const ut_qtensor *w, const float *x, int64_t M, float *out,
                        int64_t ldo, int accumulate) {
    F32Args a{};
    a.w = (const float *)w->payload;
    a.O = w->out_dim;
    a.K = w->in_dim;
    a.ldx = w->in_dim;
    a.ldo = ldo;
    a.accumulate = accumulate;
    gemv_f32_split(a.O, a.K, &a.ks, &a.kslice);
    int64_t chunk = 1 << 16;
    if (a.ks > 1) {
        int64_t *part = nullptr;
        UT_TRY(splitk_buffer(ctx, &part));
        a.part = (float *)part;
        const int64_t fit = kSplitKPartBytes / ((int64_t)a.ks * a.O * 4) / kF32Tile * kF32Tile;
        if (fit < chunk) chunk = fit;
    }
    const int to = (int)((a.O + kF32Tile - 1) / kF32Tile), T = (int)((a.kslice + 63) / 64);
    for (int64_t m0 = 0; m0 < M; m0 += chunk) {
        a.M = M - m0 < chunk ? M - m0 : chunk;
        a.x = x + m0 * a.ldx;
        a.out = out + m0 * ldo;
        const dim3 grid((unsigned)((a.M + kF32Tile - 1) / kF32Tile * to), (unsigned)a.ks);
        int tok = timing_begin(ctx, "gemm_f32");
        switch (T) {
        case 1: hipLaunchKernelGGL(k_gemm_f32<1>, grid, dim3(256), 0, ctx->stream, a, to); break;
        case 2: hipLaunchKernelGGL(k_gemm_f32<2>, grid, dim3(256), 0, ctx->stream, a, to); break;
        case 3: hipLaunchKernelGGL(k_gemm_f32<3>, grid, dim3(256), 0, ctx->stream, a, to); break;
        default: hipLaunchKernelGGL(k_gemm_f32<4>, grid, dim3(256), 0, ctx->stream, a, to); break;
        }
        UT_TRY(launch_check(ctx, "k_gemm_f32"));
        if (a.ks > 1) {
            hipLaunchKernelGGL(k_gemm_f32_sum, dim3((unsigned)((a.M * a.O + 255) / 256)), dim3(256),
                               0, ctx->stream, a);
            UT_TRY(launch_check(ctx, "k_gemm_f32_sum"));
        }
        timing_end(ctx, tok);
    }
    return UT_OK;
}

// ------------------------------------------- k_rowdot_f32's order ---
// The router gate over a prompt: k_rowdot_f32's chains (thread t: columns
// 4 t + 1024 j in j order), wave sums and wave order, with a workgroup's EPW
// weight rows held in registers while up to kRowsPerWG activation rows pass
// (the next row's loads in flight).  Bound by x's passes through L2 (O / EPW
// of them); few weight or activation rows take fewer rows per workgroup, so
// that their loads' round trips run side by side (48 rows of 8 x 256: 12.8 us
// at 16 rows a workgroup, 2.7 at one).
constexpr int kRowsPerWG = 16;
template <int NJ, int EPW>
__global__ __launch_bounds__(256) void k_rowdot_f32_rows(const float *__restrict__ w, int64_t K,
                                                         const float *__restrict__ x, int64_t M,
                                                         float *__restrict__ out, int64_t ldo,
                                                         int64_t O, int per) {
    __shared__ float red[kRowsPerWG][EPW][4];
    const int tid = threadIdx.x;
    const int64_t o0 = (int64_t)blockIdx.x * EPW, m0 = (int64_t)blockIdx.y * per;
    const int rows = (int)(M - m0 < per ? M - m0 : per);
    float4 wv[EPW][NJ], xv[NJ], xn[NJ];
    auto ld = [&](const float *p, float4 (&v)[NJ]) {
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int64_t c = 4 * tid + 1024 * j;
            v[j] = c < K ? ld_global<float4>(p + c) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    };
    ld(x + m0 * K, xv);
#pragma unroll
    for (int e = 0; e < EPW; e++) ld(w + (o0 + e < O ? o0 + e : O - 1) * K, wv[e]);
    for (int r = 0; r < rows; r++) {
        if (r + 1 < rows) ld(x + (m0 + r + 1) * K, xn);
#pragma unroll
        for (int e = 0; e < EPW; e++) {
            float a = 0.0f;
#pragma unroll
            for (int j = 0; j < NJ; j++)
                if (4 * tid + 1024 * j < K) {
                    a = __builtin_fmaf(wv[e][j].x, xv[j].x, a);
                    a = __builtin_fmaf(wv[e][j].y, xv[j].y, a);
                    a = __builtin_fmaf(wv[e][j].z, xv[j].z, a);
                    a = __builtin_fmaf(wv[e][j].w, xv[j].w, a);
                }
            a = wave_reduce_dpp(a, [](float p, float q) { return p + q; });
            if ((tid & 63) == 0) red[r][e][tid >> 6] = a;
        }
#pragma unroll
        for (int j = 0; j < NJ; j++) xv[j] = xn[j];
    }
    __syncthreads();
    if (tid < EPW * rows) {
        const int r = tid / EPW, e = tid - r * EPW;
        if (o0 + e < O)
            out[(m0 + r) * ldo + o0 + e] =
                ((red[r][e][0] + red[r][e][1]) + red[r][e][2]) + red[r][e][3];
    }
}

int32_t launch_rowdot_f32_rows(ut_ctx *ctx, const ut_qtensor *w, const float *x, int64_t M,
                               float *out, int64_t ldo) {
    if (!rowdot_f32_ok(w, 1) || ((uintptr_t)x & 15) != 0) {
        set_error(ctx, "rowdot_f32_rows: unsupported shape or alignment");
        return UT_ERR_ARG;
    }
    constexpr int EPW = 4;
    const int64_t K = w->in_dim, O = w->out_dim;
    const int nj = (int)((K + 1023) / 1024);
    const int64_t og = (O + EPW - 1) / EPW, want = M * og / (2 * ctx->multiprocessors);
    const int per = (int)(want < 1 ? 1 : want > kRowsPerWG ? kRowsPerWG : want);
    const dim3 grid((unsigned)og, (unsigned)((M + per - 1) / per));
    int tok = timing_begin(ctx, "rowdot_f32_rows");
    const float *wp = (const float *)w->payload;
#define UT_RR(NJ) \
    hipLaunchKernelGGL((k_rowdot_f32_rows<NJ, EPW>), grid, dim3(256), 0, ctx->stream, wp, K, x, M, out, ldo, O, per)
    if (nj <= 1) UT_RR(1);
    else if (nj <= 2) UT_RR(2);
    else if (nj <= 4) UT_RR(4);
    else if (nj <= 7) UT_RR(7);
    else UT_RR(8);
#undef UT_RR
    timing_end(ctx, tok);
    return launch_check(ctx, "k_rowdot_f32_rows");
}

}  // namespace ut
