// ut_gemm.h -- quantized matrix products over more rows than the skinny
// GEMVs take (prompts): internal interface of ut_gemm.hip.
#pragma once

#include "ut_internal.h"

namespace ut {

// A batch of activation rows as base-256 digit planes: plane p of row m is
// the kp bytes at p + (m*3 + p)*kp, zero past K (kp: K rounded up to 128),
// exps[m] the row's exponent (XDigits).
struct DigitPlanes {
    int8_t *p = nullptr;
    int64_t kp = 0;
    int32_t *exps = nullptr;
};
inline int64_t planes_pitch(int64_t K) { return (K + 127) / 128 * 128; }
size_t planes_bytes(int64_t M, int64_t K);
DigitPlanes planes_view(void *base, int64_t M, int64_t K);
// Digitises x [M, K] (row stride ldx), f32 or bf16.
int32_t launch_planes(ut_ctx *ctx, const float *x, int64_t ldx, int64_t M, int64_t K,
                      const DigitPlanes &pl);
int32_t launch_planes(ut_ctx *ctx, const uint16_t *x, int64_t ldx, int64_t M, int64_t K,
                      const DigitPlanes &pl);
// Digitises h = silu(g) * u of M rows [M, I].
int32_t launch_silu_planes(ut_ctx *ctx, const float *g, const float *u, int64_t M, int64_t I,
                           const DigitPlanes &pl);
// A batch's base-256 digits are the GEMM's planes where rows need no padding.
inline bool xdigits_planes(const XDigits &xd, int64_t K, DigitPlanes *pl) {
    if (!xd.dig8 || planes_pitch(K) != K || ((uintptr_t)xd.dig8 & 15)) return false;
    pl->p = (int8_t *)xd.dig8;
    pl->kp = K;
    pl->exps = xd.exps;
    return true;
}

// The fewest rows that take the matrix-core GEMM; four-row GEMV passes over
// the weight are slower from the second pass on (five rows, GEMV passes
// against GEMM: int8 7168 x 16384 63.7 -> 43.9 us, 576 x 7168 25.0 -> 18.8,
// 256 x 256 13.4 -> 9.8, int4 7168 x 2048 21.9 -> 12.9).
constexpr int64_t kGemmMinRows = 5;
bool gemm_ok(const ut_qtensor *w, int64_t M);
// out[m, o] (+)= x[m] . w[o] for M digitised rows; the values are the
// GEMVs', bit for bit.
// (w2: a second weight of the same format and width, gemm_pair_ok, into out2
// in the same launch.)
bool gemm_pair_ok(const ut_qtensor *w, const ut_qtensor *w2, int64_t M);
int32_t launch_gemm(ut_ctx *ctx, const ut_qtensor *w, const DigitPlanes &x, int64_t M, float *out,
                    int64_t ldo, int accumulate, const ut_qtensor *w2 = nullptr,
                    float *out2 = nullptr, int64_t ldo2 = 0);

// f32 weights (ut_gemm_f32.hip), each output's products added in the order
// of the GEMV that fewer rows take.  gemv_f32_split: that GEMV's K split, of
// the weight's shape alone.
void gemv_f32_split(int64_t O, int64_t K, int *ks, int64_t *kslice);
bool gemm_f32_ok(const ut_qtensor *w, const float *x, int64_t M);
int32_t launch_gemm_f32(ut_ctx *ctx, const ut_qtensor *w, const float *x, int64_t M, float *out,
                        int64_t ldo, int accumulate);
// launch_rowdot_f32 over any number of rows x [M, K].
int32_t launch_rowdot_f32_rows(ut_ctx *ctx, const ut_qtensor *w, const float *x, int64_t M,
                               float *out, int64_t ldo);

}  // namespace ut
