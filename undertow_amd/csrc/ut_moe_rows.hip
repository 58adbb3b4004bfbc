// ut_moe_rows.hip -- the routed experts of a prompt's rows (moe_forward,
// adapters/undertow-deepseek-moe/src/model.rs:210-281) as grouped products:
// the (row, choice) pairs are sorted by expert on the device, every expert's
// rows are one matrix-core tile (or several), and its weights are read once
// for all of them.
//
//   k_moe_group        pairs -> per-expert lists and the tile list
//   k_planes           x rows -> digit planes (ut_gemm.hip)
//   k_moe_rows_gate_up gate and up tiles, h = silu(g) * u per pair
//   k_planes           h rows -> digit planes
//   k_moe_rows_down    down tiles, d per pair
//   k_moe_rows_combine choices summed in router order
#include "ut_moe_rows.h"

#include "ut_gemm_core.h"

namespace ut {

constexpr int kTileRows = 32;  // rows of an expert per tile (two 16-row operands)
struct MoeTile {
    int32_t expert, pos, n;  // rows pos .. pos + n of the sorted pairs
};

bool moe_rows_ok(int fmt, int64_t M, int64_t E, int64_t H, int64_t I) {
    return M >= kGemmMinRows && (fmt == UT_FMT_INT8 || fmt == UT_FMT_INT4) &&
           moe_shape_ok(fmt, H, I) && E <= kMoeRowsMaxExperts && H <= 65536 && I <= 65536;
}

namespace {
struct RowsLayout {
    size_t total = 0, tiles = 0, count = 0, list = 0, pos = 0, xp = 0, h = 0, hp = 0, d = 0;
    int64_t max_tiles = 0;
};
RowsLayout rows_layout(int64_t M, int64_t k, int64_t E, int64_t H, int64_t I, bool planes) {
    RowsLayout L;
    const int64_t n = M * k;
    auto take = [&](size_t b) { size_t o = L.total; L.total += (b + 255) & ~size_t(255); return o; };
    // every expert's last tile may be partial
    L.max_tiles = n / kTileRows + (n < E ? n : E);
    L.tiles = take((size_t)L.max_tiles * sizeof(MoeTile));
    L.count = take(4);
    L.list = take((size_t)n * 4);
    L.pos = take((size_t)n * 4);
    L.xp = take(planes ? planes_bytes(M, H) : 0);
    L.h = take((size_t)n * I * 4);
    L.hp = take(planes_bytes(n, I));
    L.d = take((size_t)n * H * 4);
    return L;
}
}  // namespace

size_t moe_rows_bytes(int64_t M, int64_t k, int64_t E, int64_t H, int64_t I, bool planes) {
    return rows_layout(M, k, E, H, I, planes).total;
}

// One workgroup: counts the pairs of each expert, lays the experts out one
// after another and lists their tiles, then scatters the pairs.  The order
// of an expert's pairs is whatever the LDS atomics give; no result depends
// on it.  Invalid ids (out of range or not loaded) set the sticky error flag
// and get position -1, as make_plan.
__global__ __launch_bounds__(1024) void k_moe_group(const int32_t *__restrict__ ids, int n, int E,
                                                    const uint8_t *const *__restrict__ gate_tbl,
                                                    int32_t *__restrict__ list,
                                                    int32_t *__restrict__ pos,
                                                    MoeTile *__restrict__ tiles,
                                                    int32_t *__restrict__ ntiles,
                                                    int32_t *__restrict__ err_flag) {
    __shared__ int cnt[kMoeRowsMaxExperts];
    __shared__ int wsum[16][2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int e = tid; e < E; e += 1024) cnt[e] = 0;
    __syncthreads();
    for (int i = tid; i < n; i += 1024) {
        const int e = ids[i];
        if (e >= 0 && e < E && gate_tbl[e]) atomicAdd(&cnt[e], 1);
        else if (e != -1 && err_flag) *err_flag = 1;
    }
    __syncthreads();
    // exclusive scans of the counts and of the tiles: four experts per thread
    int c[4], p0 = 0, t0 = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        c[j] = 4 * tid + j < E ? cnt[4 * tid + j] : 0;
        p0 += c[j];
        t0 += (c[j] + kTileRows - 1) / kTileRows;
    }
    int ps = p0, ts = t0;
    for (int o = 1; o < 64; o <<= 1) {
        const int a = __shfl_up(ps, o, 64), b = __shfl_up(ts, o, 64);
        if (lane >= o) { ps += a; ts += b; }
    }
    if (lane == 63) { wsum[wave][0] = ps; wsum[wave][1] = ts; }
    __syncthreads();
    int pb = ps - p0, tb = ts - t0;
    for (int w = 0; w < wave; w++) { pb += wsum[w][0]; tb += wsum[w][1]; }
    if (tid == 1023) *ntiles = tb + t0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int e = 4 * tid + j;
        if (e < E) {
            cnt[e] = pb;  // the expert's next free position
            for (int r = 0; r < c[j]; r += kTileRows) {
                const int left = c[j] - r;
                tiles[tb++] = MoeTile{e, pb + r, left < kTileRows ? left : kTileRows};
            }
            pb += c[j];
        }
    }
    __syncthreads();
    for (int i = tid; i < n; i += 1024) {
        const int e = ids[i];
        int p = -1;
        if (e >= 0 && e < E && gate_tbl[e]) {
            p = atomicAdd(&cnt[e], 1);
            list[p] = i;
        }
        pos[i] = p;
    }
}

struct MoeRowsArgs {
    ExpertPtrs tbl;
    const MoeTile *tiles;
    const int32_t *ntiles, *list;
    int k;
    int64_t H, I, row_h, row_i;  // row_h / row_i: payload bytes of a row of H / I columns
    const int8_t *pl;            // the launch's input planes
    int64_t kp;
    const int32_t *exps;
    float *out;                  // gate/up: h [pairs][I]; down: d [pairs][H]
};

// The staging chunks' sources for a tile's rows (rowof: tile row -> plane
// row; rows past the tile repeat its last).
template <int TM, typename F>
__device__ __forceinline__ void rows_src(const MoeRowsArgs &a, int n, F &&rowof,
                                         const int8_t *(&src)[gemm_stage_n<TM>()]) {
#pragma unroll
    for (int i = 0; i < gemm_stage_n<TM>(); i++) {
        const GemmChunk c = gemm_chunk(threadIdx.x + i * kGemmThreads);
        const int64_t m = rowof(c.m < n ? c.m : n - 1);
        src[i] = a.pl + (m * 3 + (c.p < 3 ? c.p : 0)) * a.kp + c.off;
    }
}

// Gate and up of 128 h rows against a tile's rows: wave w's four weight
// tiles are gate and up rows of the same 32 h rows, so silu(g) * u is formed
// from one lane's accumulators.
template <int FMT, int TM>
__device__ __forceinline__ void rows_gate_up(const MoeRowsArgs &a, const MoeTile &t, int rt,
                                             uint4 *lds) {
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;
    const int64_t h0 = (int64_t)rt * 128 + (tid >> 6) * 32;
    GemmRows<4> rows;
    rows.end = nullptr;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int64_t h = h0 + 16 * (i & 1) + r;
        rows.row[i] = (i < 2 ? a.tbl.gate_w : a.tbl.up_w)[t.expert] + (h < a.I ? h : a.I - 1) * a.row_h;
    }
    const int8_t *src[gemm_stage_n<TM>()];
    rows_src<TM>(a, t.n, [&](int m) { return (int64_t)(a.list[t.pos + m] / a.k); }, src);
    ut_i32x4 acc[4][TM][3];
    gemm_tile<FMT, 4, TM, false>(rows, a.row_h, 0, a.kp, src, lds, acc);
    const float *gs = a.tbl.gate_s[t.expert], *us = a.tbl.up_s[t.expert];
#pragma unroll
    for (int n = 0; n < TM; n++) {
        const int m = 16 * n + r;
        if (m >= t.n) continue;
        const int32_t e = gemm_exp<FMT>(a.exps[a.list[t.pos + m] / a.k]);
        float *ho = a.out + (int64_t)(t.pos + m) * a.I;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int64_t h = h0 + 16 * i + 4 * q;
            if (h >= a.I) continue;  // I % 16 == 0: four columns or none
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float g = int_total_to_f32(gemm_total(acc[i][n], j), e, ld_global_f32(gs + h + j));
                const float u = int_total_to_f32(gemm_total(acc[i + 2][n], j), e, ld_global_f32(us + h + j));
                // silu(g) * u (undertow-quant/src/lib.rs:121; model.rs:241-247)
                v[j] = __fmul_rn(g / (1.0f + expf(-g)), u);
            }
            *(float4 *)(ho + h) = make_float4(v[0], v[1], v[2], v[3]);
        }
    }
}

template <int FMT, int TM>
__device__ __forceinline__ void rows_down(const MoeRowsArgs &a, const MoeTile &t, int rt, uint4 *lds) {
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;
    const int64_t o0 = (int64_t)rt * 256 + (tid >> 6) * 64;
    GemmRows<4> rows;
    rows.end = nullptr;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int64_t o = o0 + 16 * i + r;
        rows.row[i] = a.tbl.down_w[t.expert] + (o < a.H ? o : a.H - 1) * a.row_i;
    }
    const int8_t *src[gemm_stage_n<TM>()];
    rows_src<TM>(a, t.n, [&](int m) { return (int64_t)(t.pos + m); }, src);
    ut_i32x4 acc[4][TM][3];
    gemm_tile<FMT, 4, TM, false>(rows, a.row_i, 0, a.kp, src, lds, acc);
    const float *ds = a.tbl.down_s[t.expert];
#pragma unroll
    for (int n = 0; n < TM; n++) {
        const int m = 16 * n + r;
        if (m >= t.n) continue;
        const int32_t e = gemm_exp<FMT>(a.exps[t.pos + m]);
        float *po = a.out + (int64_t)(t.pos + m) * a.H;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t o = o0 + 16 * i + 4 * q;
            if (o >= a.H) continue;  // H % 16 == 0
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; j++)
                v[j] = int_total_to_f32(gemm_total(acc[i][n], j), e, ld_global_f32(ds + o + j));
            *(float4 *)(po + o) = make_float4(v[0], v[1], v[2], v[3]);
        }
    }
}

// Grid: tiles x weight-row tiles, row tiles fastest, so a launch's
// consecutive workgroups stream one expert's matrix.  A tile of up to 16
// rows takes one 16-row operand, one of 17..32 two: at a prompt's 8 to 32
// rows per expert the weights are read once and at most half of the matrix
// work is padding.
template <int FMT, bool DOWN>
__global__ __launch_bounds__(kGemmThreads, 2) void k_moe_rows(MoeRowsArgs a, int nrt) {
    __shared__ uint4 lds[gemm_lds_uint4<2>()];
    const int ti = blockIdx.x / nrt, rt = blockIdx.x - ti * nrt;
    if (ti >= *a.ntiles) return;
    const MoeTile t = a.tiles[ti];
    if constexpr (DOWN) {
        if (t.n <= 16) rows_down<FMT, 1>(a, t, rt, lds);
        else rows_down<FMT, 2>(a, t, rt, lds);
    } else {
        if (t.n <= 16) rows_gate_up<FMT, 1>(a, t, rt, lds);
        else rows_gate_up<FMT, 2>(a, t, rt, lds);
    }
}

// Four columns of one row: the choices in router order (zero, then += w*d
// per choice), then the shared expert's row, then the residual.
__global__ __launch_bounds__(256) void k_moe_rows_combine(const int32_t *__restrict__ pos,
                                                          const float *__restrict__ weights,
                                                          const float *__restrict__ d, int k,
                                                          int64_t H,
                                                          const float *__restrict__ shared,
                                                          float *__restrict__ out, int64_t ldo,
                                                          int accumulate) {
    const int64_t m = blockIdx.y, c = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
    if (c >= H) return;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 8
    for (int j = 0; j < k; j++) {
        const int p = pos[m * k + j];
        if (p < 0) continue;
        const float w = weights[m * k + j];
        const float4 v = ld_global<float4>(d + (int64_t)p * H + c);
        acc[0] = __fadd_rn(acc[0], __fmul_rn(w, v.x));
        acc[1] = __fadd_rn(acc[1], __fmul_rn(w, v.y));
        acc[2] = __fadd_rn(acc[2], __fmul_rn(w, v.z));
        acc[3] = __fadd_rn(acc[3], __fmul_rn(w, v.w));
    }
    float *po = out + m * ldo + c;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (shared) acc[j] = __fadd_rn(acc[j], shared[m * H + c + j]);
        po[j] = accumulate ? __fadd_rn(po[j], acc[j]) : acc[j];
    }
}

int32_t launch_moe_rows(ut_ctx *ctx, const MoeRows &c, void *scratch) {
    // (a prompt's last call may hold fewer rows than moe_rows_ok asks)
    if (c.M < 1 || !moe_rows_ok(c.fmt, kGemmMinRows, c.E, c.H, c.I) || c.M > moe_rows_chunk(c.k) || c.k < 1) {
        set_error(ctx, "moe_rows: %lld rows of format %d not supported", (long long)c.M, c.fmt);
        return UT_ERR_ARG;
    }
    const RowsLayout L = rows_layout(c.M, c.k, c.E, c.H, c.I, !c.planes);
    char *b = (char *)scratch;
    const int64_t n = c.M * c.k;
    MoeRowsArgs a{};
    a.tbl = c.tbl;
    a.tiles = (const MoeTile *)(b + L.tiles);
    a.ntiles = (const int32_t *)(b + L.count);
    a.list = (const int32_t *)(b + L.list);
    a.k = c.k;
    a.H = c.H;
    a.I = c.I;
    a.row_h = payload_bytes(c.fmt, 1, c.H);
    a.row_i = payload_bytes(c.fmt, 1, c.I);
    int32_t *pos = (int32_t *)(b + L.pos);
    float *h = (float *)(b + L.h), *d = (float *)(b + L.d);
    int tok = timing_begin(ctx, "moe_group");
    hipLaunchKernelGGL(k_moe_group, dim3(1), dim3(1024), 0, ctx->stream, c.ids, (int)n, (int)c.E,
                       c.tbl.gate_w, (int32_t *)(b + L.list), pos, (MoeTile *)(b + L.tiles),
                       (int32_t *)(b + L.count), c.err_flag);
    timing_end(ctx, tok);
    UT_TRY(launch_check(ctx, "k_moe_group"));
    DigitPlanes xp;
    if (c.planes) xp = *c.planes;
    else {
        xp = planes_view(b + L.xp, c.M, c.H);
        if (c.xh) UT_TRY(launch_planes(ctx, c.xh, c.H, c.M, c.H, xp));
        else UT_TRY(launch_planes(ctx, c.x, c.H, c.M, c.H, xp));
    }
    auto launch = [&](const char *name, const DigitPlanes &pl, float *out, int64_t rows, int per,
                      bool down) -> int32_t {
        a.pl = pl.p;
        a.kp = pl.kp;
        a.exps = pl.exps;
        a.out = out;
        const int nrt = (int)((rows + per - 1) / per);
        const dim3 grid((unsigned)(L.max_tiles * nrt));
        int tk = timing_begin(ctx, name);
        if (c.fmt == UT_FMT_INT4) {
            if (down) hipLaunchKernelGGL((k_moe_rows<UT_FMT_INT4, true>), grid, dim3(kGemmThreads), 0, ctx->stream, a, nrt);
            else hipLaunchKernelGGL((k_moe_rows<UT_FMT_INT4, false>), grid, dim3(kGemmThreads), 0, ctx->stream, a, nrt);
        } else {
            if (down) hipLaunchKernelGGL((k_moe_rows<UT_FMT_INT8, true>), grid, dim3(kGemmThreads), 0, ctx->stream, a, nrt);
            else hipLaunchKernelGGL((k_moe_rows<UT_FMT_INT8, false>), grid, dim3(kGemmThreads), 0, ctx->stream, a, nrt);
        }
        timing_end(ctx, tk);
        return launch_check(ctx, name);
    };
    UT_TRY(launch("moe_rows_gate_up", xp, h, c.I, 128, false));
    const DigitPlanes hp = planes_view(b + L.hp, n, c.I);
    UT_TRY(launch_planes(ctx, h, c.I, n, c.I, hp));
    UT_TRY(launch("moe_rows_down", hp, d, c.H, 256, true));
    tok = timing_begin(ctx, "moe_rows_combine");
    hipLaunchKernelGGL(k_moe_rows_combine, dim3((unsigned)((c.H / 4 + 255) / 256), (unsigned)c.M),
                       dim3(256), 0, ctx->stream, pos, c.weights, d, c.k, c.H, c.shared, c.out,
                       c.ldo, c.accumulate);
    timing_end(ctx, tok);
    return launch_check(ctx, "k_moe_rows_combine");
}

}  // namespace ut
