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

// The fewest rows: up to five (int4) or seven (int8) most choices name
// different experts, and the four-row passes' launches are the shorter ones
// (config 2's block: 5 rows 315 against 328 us, 7 rows 426 against 433, 8
// rows 489 against 461; int4 5 rows 200 against 205, 6 rows 242 against 228).
constexpr int64_t kMoeRowsMinI8 = 8, kMoeRowsMinI4 = 6;

bool moe_rows_ok(int fmt, int64_t M, int64_t E, int64_t H, int64_t I) {
    return M >= (fmt == UT_FMT_INT8 ? kMoeRowsMinI8 : kMoeRowsMinI4) &&
           (fmt == UT_FMT_INT8 || fmt == UT_FMT_INT4) && moe_shape_ok(fmt, H, I) && E <= kMoeRowsMaxExperts && H <= 65536 && I <= 65536;
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

// Weight tiles of 16 rows per wave.  Four workgroups
// of 128 weight rows per CU (int4; 40 KB of LDS each): config 2's int4 block
// at 500 rows 1,315 us with direct weight loads, 1,239 so; at 64 rows 725 ->
// 669, at 5 rows 235 -> 205.  256-row workgroups, two per CU: 1,279 / 660 /
// 224; stages of 64 columns: 1,564 / 817 / 270.  Up to 64 rows the weights'
// read bounds it (222 experts, 4.9 GB, at 64 rows); at 500 the read (0.83 ms)
// and the padded tiles' matrix work (23 of 32 rows on average) together do.
constexpr int kMrTO = 2;
constexpr int kMrRows = 64 * kMrTO;

// A workgroup's tile: weight rows wrow(row of the tile) against a tile's
// activation rows arow(m) (rows past the tile repeat its last).
template <int FMT, int TM, typename W, typename A>
__device__ __forceinline__ void rows_tile(const MoeRowsArgs &a, int n, int64_t len, W &&wrow,
                                          A &&arow, void *s0, void *s1, ut_i32x4 (&acc)[kMrTO][TM][3]) {
    using L = GemmLds<FMT, kMrTO, TM, 4, 1>;
    GemmSrc<FMT, kMrTO, TM, 4, 1> src;
    gemm_src<FMT, kMrTO, TM, 4, 1>(src, wrow, [&](int m, int p) {
        return a.pl + (arow(m < n ? m : n - 1) * 3 + p) * a.kp;
    });
    gemm_tile_lds<false, FMT, kMrTO, TM, 4, 1>(src, len, 0, a.kp, *(L *)s0, *(L *)s1, acc);
}

// Gate and up of kMrRows / 2 h rows against a tile's rows: a wave's weight
// tiles are gate rows and up rows of the same h rows, so silu(g) * u is
// formed from one lane's accumulators.
template <int FMT, int TM>
__device__ __forceinline__ void rows_gate_up(const MoeRowsArgs &a, const MoeTile &t, int rt,
                                             void *s0, void *s1) {
    constexpr int G = kMrTO / 2;  // gate tiles of a wave
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4, wave = threadIdx.x >> 6;
    const int64_t hb = (int64_t)rt * (kMrRows / 2), h0 = hb + wave * (16 * G);
    const uint8_t *gw = a.tbl.gate_w[t.expert], *uw = a.tbl.up_w[t.expert];
    ut_i32x4 acc[kMrTO][TM][3];
    rows_tile<FMT, TM>(
        a, t.n, a.row_h,
        [&](int row) {
            const int x = row / 16, i = x % kMrTO;  // tile of the workgroup, of its wave
            const int64_t h = hb + (x / kMrTO * G + i % G) * 16 + row % 16;
            return (i < G ? gw : uw) + (h < a.I ? h : a.I - 1) * a.row_h;
        },
        [&](int m) { return (int64_t)(a.list[t.pos + m] / a.k); }, s0, s1, acc);
    const float *gs = a.tbl.gate_s[t.expert], *us = a.tbl.up_s[t.expert];
#pragma unroll
    for (int n = 0; n < TM; n++) {
        const int m = 16 * n + r;
        if (m >= t.n) continue;
        const int32_t e = gemm_exp<FMT>(a.exps[a.list[t.pos + m] / a.k]);
        float *ho = a.out + (int64_t)(t.pos + m) * a.I;
#pragma unroll
        for (int i = 0; i < G; i++) {
            const int64_t h = h0 + 16 * i + 4 * q;
            if (h >= a.I) continue;  // I % 16 == 0: four columns or none
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float g = int_total_to_f32(gemm_total(acc[i][n], j), e, ld_global_f32(gs + h + j));
                const float u = int_total_to_f32(gemm_total(acc[i + G][n], j), e, ld_global_f32(us + h + j));
                // silu(g) * u (undertow-quant/src/lib.rs:121; model.rs:241-247)
                v[j] = __fmul_rn(g / (1.0f + expf(-g)), u);
            }
            *(float4 *)(ho + h) = make_float4(v[0], v[1], v[2], v[3]);
        }
    }
}

template <int FMT, int TM>
__device__ __forceinline__ void rows_down(const MoeRowsArgs &a, const MoeTile &t, int rt, void *s0,
                                          void *s1) {
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4, wave = threadIdx.x >> 6;
    const int64_t ob = (int64_t)rt * kMrRows, o0 = ob + wave * (16 * kMrTO);
    const uint8_t *dw = a.tbl.down_w[t.expert];
    ut_i32x4 acc[kMrTO][TM][3];
    rows_tile<FMT, TM>(
        a, t.n, a.row_i,
        [&](int row) { return dw + (ob + row < a.H ? ob + row : a.H - 1) * a.row_i; },
        [&](int m) { return (int64_t)(t.pos + m); }, s0, s1, acc);
    const float *ds = a.tbl.down_s[t.expert];
#pragma unroll
    for (int n = 0; n < TM; n++) {
        const int m = 16 * n + r;
        if (m >= t.n) continue;
        const int32_t e = gemm_exp<FMT>(a.exps[t.pos + m]);
        float *po = a.out + (int64_t)(t.pos + m) * a.H;
#pragma unroll
        for (int i = 0; i < kMrTO; i++) {
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
__global__ __launch_bounds__(kGemmThreads, FMT == UT_FMT_INT4 ? 4 : 2) void k_moe_rows(MoeRowsArgs a, int nrt) {
    // two objects: the compiler then knows which one a copy in flight fills
    __shared__ GemmLds<FMT, kMrTO, 2, 4, 1> s0, s1;
    const int ti = blockIdx.x / nrt, rt = blockIdx.x - ti * nrt;
    if (ti >= *a.ntiles) return;
    const MoeTile t = a.tiles[ti];
    if constexpr (DOWN) {
        if (t.n <= 16) rows_down<FMT, 1>(a, t, rt, &s0, &s1);
        else rows_down<FMT, 2>(a, t, rt, &s0, &s1);
    } else {
        if (t.n <= 16) rows_gate_up<FMT, 1>(a, t, rt, &s0, &s1);
        else rows_gate_up<FMT, 2>(a, t, rt, &s0, &s1);
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
    if (c.M < 1 || !moe_rows_ok(c.fmt, kMoeRowsMinI8, c.E, c.H, c.I) || c.M > moe_rows_chunk(c.k) || c.k < 1) {
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
    UT_TRY(launch("moe_rows_gate_up", xp, h, c.I, kMrRows / 2, false));
    const DigitPlanes hp = planes_view(b + L.hp, n, c.I);
    UT_TRY(launch_planes(ctx, h, c.I, n, c.I, hp));
    UT_TRY(launch("moe_rows_down", hp, d, c.H, kMrRows, true));
    tok = timing_begin(ctx, "moe_rows_combine");
    hipLaunchKernelGGL(k_moe_rows_combine, dim3((unsigned)((c.H / 4 + 255) / 256), (unsigned)c.M),
                       dim3(256), 0, ctx->stream, pos, c.weights, d, c.k, c.H, c.shared, c.out,
                       c.ldo, c.accumulate);
    timing_end(ctx, tok);
    return launch_check(ctx, "k_moe_rows_combine");
}

}  // namespace ut
