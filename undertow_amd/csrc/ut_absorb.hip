// ut_absorb.hip -- the absorbed halves of kv_b (adapters/undertow-deepseek-moe/
// src/attention.rs:202-245) over a prompt's rows, on the f32 matrix cores.
//
// v_mfma_f32_16x16x4_f32 adds its four products to the accumulator one after
// another, each with one rounding (checked against fmaf chains on the card),
// so a chain of them is the FMA chain a lane of the vector kernels runs.
// Codes are exact in f32, operands keep all their bits.
//
// Operand layout of the instruction: lane l holds row / column l % 16 and
// product l / 16 of the four.  For 16 consecutive products (four
// instructions) lane group g so needs products g, 4 + g, 8 + g, 12 + g.
// f32 rows are loaded 16 bytes a lane (products 4g .. 4g + 3) and transposed
// among the four lane groups by permlane swaps; int8 codes are transposed
// when they are staged: one LDS word holds a lane's four codes.
#include "ut_gemv_core.h"
#include "ut_ops.h"

namespace ut {

typedef float ab_f32x4 __attribute__((ext_vector_type(4)));
constexpr int kAbRows = 64;  // rows per workgroup: 16 per wave

// Products 4g + i of lane group g in v[i] -> products 4i + g.
__device__ __forceinline__ void ab_transpose(float (&v)[4]) {
    auto swap32 = [](float &a, float &b) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        a = __uint_as_float(r[0]);
        b = __uint_as_float(r[1]);
    };
    auto swap16 = [](float &a, float &b) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        a = __uint_as_float(r[0]);
        b = __uint_as_float(r[1]);
    };
    swap32(v[0], v[2]);
    swap32(v[1], v[3]);
    swap16(v[0], v[1]);
    swap16(v[2], v[3]);
}
__device__ __forceinline__ float ab_code(uint32_t w, int s) {
    return (float)(int8_t)(w >> (8 * s));
}
// 4 x 4 byte transpose: byte c of out[r] = byte r of in[c].
__device__ __forceinline__ void ab_bytes4x4(const uint32_t (&in)[4], uint32_t (&out)[4]) {
    const uint32_t a = __builtin_amdgcn_perm(in[1], in[0], 0x05010400u);  // 0.0 1.0 0.1 1.1
    const uint32_t b = __builtin_amdgcn_perm(in[1], in[0], 0x07030602u);  // 0.2 1.2 0.3 1.3
    const uint32_t c = __builtin_amdgcn_perm(in[3], in[2], 0x05010400u);
    const uint32_t d = __builtin_amdgcn_perm(in[3], in[2], 0x07030602u);
    out[0] = __builtin_amdgcn_perm(c, a, 0x05040100u);
    out[1] = __builtin_amdgcn_perm(c, a, 0x07060302u);
    out[2] = __builtin_amdgcn_perm(d, b, 0x05040100u);
    out[3] = __builtin_amdgcn_perm(d, b, 0x07060302u);
}

// q_abs[r, h] = sum_d (q[r, h, d] * scale[d]) code[d] over 128 nope rows d,
// latent width 512: one head and 64 rows per workgroup, a wave 16 rows x 512
// columns.  The vector kernel rounds each product before adding it; here
// that rounding is gone.  Bound by the f32 matrix rate (157 TFLOP/s) beside
// the q_abs write: 509 rows x 128 heads 382 us with the vector kernel, 140 so
// (55 us of products, 133 MB written).
constexpr int kAbqCols = 512, kAbqPitch = kAbqCols + 16;  // words; +16: no bank conflicts
__global__ __launch_bounds__(256, 2) void k_absorb_q_rows(const uint8_t *__restrict__ w,
                                                          const float *__restrict__ scales,
                                                          int64_t row_bytes,
                                                          const float *__restrict__ q, int64_t rows,
                                                          int64_t heads, int64_t rope, int64_t kvh,
                                                          float *__restrict__ qabs,
                                                          float *__restrict__ qrope, int64_t pos_base,
                                                          const float2 *__restrict__ table) {
    constexpr int D = 128, CH = D / 16;
    __shared__ uint32_t sw[CH * 4 * kAbqPitch];  // [chunk][group][column]: rows 16c + g + 4s
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, g = lane >> 4;
    const int64_t h = blockIdx.x, r0 = (int64_t)blockIdx.y * kAbRows;
    const int64_t qh = D + rope;
    const uint8_t *wh = w + h * kvh * row_bytes;
    for (int i = tid; i < CH * 4 * (kAbqCols / 4); i += 256) {
        const int c4 = i % (kAbqCols / 4), cg = i / (kAbqCols / 4), d = cg / 4 * 16 + cg % 4;
        uint32_t in[4], out[4];
#pragma unroll
        for (int s = 0; s < 4; s++) in[s] = *(const uint32_t *)(wh + (d + 4 * s) * row_bytes + 4 * c4);
        ab_bytes4x4(in, out);
        *(uint4 *)&sw[cg * kAbqPitch + 4 * c4] = make_uint4(out[0], out[1], out[2], out[3]);
    }
    const int64_t ra = r0 + wave * 16 + n, rc = ra < rows ? ra : rows - 1;
    const float *qr = q + (rc * heads + h) * qh;
    const float *sc = scales + h * kvh;
    ab_f32x4 acc[32];
#pragma unroll
    for (int t = 0; t < 32; t++) acc[t] = ab_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    __syncthreads();
    for (int c = 0; c < CH; c++) {
        const float4 x = ld_global<float4>(qr + 16 * c + 4 * g), y = ld_global<float4>(sc + 16 * c + 4 * g);
        float f[4] = {__fmul_rn(x.x, y.x), __fmul_rn(x.y, y.y), __fmul_rn(x.z, y.z), __fmul_rn(x.w, y.w)};
        ab_transpose(f);
#pragma unroll
        for (int t = 0; t < 32; t++) {
            const uint32_t cw = sw[(c * 4 + g) * kAbqPitch + 16 * t + n];
#pragma unroll
            for (int s = 0; s < 4; s++)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[s], ab_code(cw, s), acc[t], 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int64_t r = r0 + wave * 16 + 4 * g + i;
        if (r >= rows) continue;
        float *o = qabs + (r * heads + h) * kAbqCols + n;
#pragma unroll
        for (int t = 0; t < 32; t++) o[16 * t] = acc[t][i];
    }
    // q_rope = rope_interleave(q[nope:], pos_base + r) (attention.rs:106-118,156-166)
    const int64_t half = rope / 2;
    for (int64_t i = tid; i < kAbRows * rope; i += 256) {
        const int64_t r = r0 + i / rope, jj = i % rope;
        if (r >= rows) continue;
        const float *in = q + (r * heads + h) * qh + D;
        const int64_t j = jj < half ? jj : jj - half;
        const float a = in[2 * j], b = in[2 * j + 1];
        const float2 cs = table[(pos_base + r) * half + j];
        qrope[(r * heads + h) * rope + jj] =
            jj < half ? __fsub_rn(__fmul_rn(a, cs.x), __fmul_rn(b, cs.y))
                      : __fadd_rn(__fmul_rn(b, cs.x), __fmul_rn(a, cs.y));
    }
}

bool absorb_q_rows_ok(const ut_qtensor *kv_b, const float *q, int64_t rows, int64_t nope,
                      int64_t rope, int64_t vh, int64_t pos_base) {
    // 16-byte loads of each head's query and scales: rows of 128 + rope and
    // 128 + vh floats.  Contexts of up to 128 positions keep the vector
    // kernel's rounding, so a short prompt's rows equal its decode steps' bit
    // for bit
    return kv_b->fmt == UT_FMT_INT8 && kv_b->in_dim == kAbqCols && nope == 128 && rows > 16 &&
           pos_base + rows > 128 && rope % 4 == 0 && vh % 4 == 0 && kv_b->row_bytes % 4 == 0 &&
           ((uintptr_t)kv_b->payload & 3) == 0 && (((uintptr_t)q | (uintptr_t)kv_b->scales) & 15) == 0;
}

int32_t launch_absorb_q_rows(ut_ctx *ctx, const ut_qtensor *kv_b, const float *q, int64_t rows,
                             int64_t heads, int64_t rope, int64_t vh, float *qabs, float *qrope,
                             int64_t pos_base, const float2 *table) {
    int tok = timing_begin(ctx, "absorb_q_rows");
    hipLaunchKernelGGL(k_absorb_q_rows,
                       dim3((unsigned)heads, (unsigned)((rows + kAbRows - 1) / kAbRows)), dim3(256), 0,
                       ctx->stream, (const uint8_t *)kv_b->payload, kv_b->scales, kv_b->row_bytes, q,
                       rows, heads, rope, 128 + vh, qabs, qrope, pos_base, table);
    timing_end(ctx, tok);
    return launch_check(ctx, "k_absorb_q_rows");
}

// ctx[r, h, j] = scale * (clat[r, h] . code[h, j]) with k_absorb_v_i8's sums
// bit for bit: its lane k's chain over columns 16k .. 16k + 15 is four
// instructions on a zero accumulator, and the butterfly over 32 lanes (xor
// 16, 8, 4, 2, 1) adds the chunks k and k + 16, taken in bit-reversed order
// of k, as a binary counter carries (f32 addition commutes).  A wave takes
// 16 rows x 128 outputs j.  509 rows x 128 heads: 562 us with k_absorb_v_i8,
// 148 so (55 us of products, 133 MB read).
constexpr int kAbvJ = 128, kAbvPitch = kAbvJ + 16;
__global__ __launch_bounds__(256, 2) void k_absorb_v_rows(const uint8_t *__restrict__ w,
                                                          const float *__restrict__ scales,
                                                          int64_t row_bytes,
                                                          const float *__restrict__ clat,
                                                          int64_t rows, int64_t heads, int64_t nope,
                                                          int64_t vh, float *__restrict__ out) {
    constexpr int L = 512, CH = L / 16, T = kAbvJ / 16;
    __shared__ uint32_t sw[CH * 4 * kAbvPitch];  // [chunk][group][j]: columns 16c + g + 4s
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = lane & 15, g = lane >> 4;
    const int64_t h = blockIdx.x, r0 = (int64_t)blockIdx.y * kAbRows, j0 = (int64_t)blockIdx.z * kAbvJ;
    const int64_t row0 = h * (nope + vh) + nope;
    for (int i = tid; i < kAbvJ * CH; i += 256) {
        const int c = i % CH, j = i / CH;
        const int64_t jr = j0 + j < vh ? j0 + j : vh - 1;
        const uint4 v = *(const uint4 *)(w + (row0 + jr) * row_bytes + 16 * c);
        const uint32_t in[4] = {v.x, v.y, v.z, v.w};  // columns 4s .. 4s + 3
        uint32_t o[4];
        ab_bytes4x4(in, o);
#pragma unroll
        for (int q = 0; q < 4; q++) sw[(c * 4 + q) * kAbvPitch + j] = o[q];
    }
    const int64_t ra = r0 + wave * 16 + n, rc = ra < rows ? ra : rows - 1;
    const float *xr = clat + (rc * heads + h) * L;
    __syncthreads();
    ab_f32x4 b[T], s8[T], s4[T], s2[T], s1[T];
    auto chunk = [&](int c, ab_f32x4 (&o)[T]) {
        const float4 x = ld_global<float4>(xr + 16 * c + 4 * g);
        float f[4] = {x.x, x.y, x.z, x.w};
        ab_transpose(f);
#pragma unroll
        for (int t = 0; t < T; t++) {
            const uint32_t cw = sw[(c * 4 + g) * kAbvPitch + 16 * t + n];
            ab_f32x4 a{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < 4; s++)
                a = __builtin_amdgcn_mfma_f32_16x16x4f32(f[s], ab_code(cw, s), a, 0, 0, 0);
            o[t] = a;
        }
    };
    auto add = [](ab_f32x4 (&a)[T], const ab_f32x4 (&o)[T]) {
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) a[t][i] = __fadd_rn(a[t][i], o[t][i]);
    };
    auto set = [](ab_f32x4 (&a)[T], const ab_f32x4 (&o)[T]) {
#pragma unroll
        for (int t = 0; t < T; t++) a[t] = o[t];
    };
#pragma unroll 1
    for (int u = 0; u < 16; u++) {
        const int k = ((u & 1) << 3) | ((u & 2) << 1) | ((u & 4) >> 1) | (u >> 3);
        chunk(k, b);
        {
            ab_f32x4 p[T];
            chunk(k + 16, p);
            add(b, p);
        }
        if (!(u & 1)) { set(s8, b); continue; }
        add(b, s8);
        if (!(u & 2)) { set(s4, b); continue; }
        add(b, s4);
        if (!(u & 4)) { set(s2, b); continue; }
        add(b, s2);
        if (!(u & 8)) set(s1, b);
        else add(b, s1);
    }
#pragma unroll
    for (int t = 0; t < T; t++) {
        const int64_t j = j0 + 16 * t + n;
        if (j >= vh) continue;
        const float sc = ld_global_f32(scales + row0 + j);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t r = r0 + wave * 16 + 4 * g + i;
            if (r < rows) out[r * heads * vh + h * vh + j] = __fmul_rn(b[t][i], sc);
        }
    }
}

bool absorb_v_rows_ok(const ut_qtensor *kv_b, const float *clat, int64_t rows) {
    return absorb_v_max_ok(kv_b) && rows > 16 && ((uintptr_t)clat & 15) == 0;
}

int32_t launch_absorb_v_rows(ut_ctx *ctx, const ut_qtensor *kv_b, const float *clat, int64_t rows,
                             int64_t heads, int64_t nope, int64_t vh, float *out) {
    int tok = timing_begin(ctx, "absorb_v_rows");
    hipLaunchKernelGGL(k_absorb_v_rows,
                       dim3((unsigned)heads, (unsigned)((rows + kAbRows - 1) / kAbRows),
                            (unsigned)((vh + kAbvJ - 1) / kAbvJ)),
                       dim3(256), 0, ctx->stream, (const uint8_t *)kv_b->payload, kv_b->scales,
                       kv_b->row_bytes, clat, rows, heads, nope, vh, out);
    timing_end(ctx, tok);
    return launch_check(ctx, "k_absorb_v_rows");
}

}  // namespace ut
