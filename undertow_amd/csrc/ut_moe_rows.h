// ut_moe_rows.h -- the routed-expert block over more rows than one pass of
// the skinny expert kernels takes (prompts): internal interface of
// ut_moe_rows.hip.
#pragma once

#include "ut_gemm.h"
#include "ut_moe.h"

namespace ut {

// Rows per call of the grouped expert products: 8,192 (row, choice) pairs,
// which bounds their scratch (375 MB at 1,024 rows of hidden 7168, inter
// 2048, top 8).
inline int64_t moe_rows_chunk(int64_t k) { return k >= 128 ? 64 : 8192 / (k > 0 ? k : 1); }
constexpr int64_t kMoeRowsMaxExperts = 4096;
// Whether M rows of experts of this format and shape take the grouped path.
bool moe_rows_ok(int fmt, int64_t M, int64_t E, int64_t H, int64_t I);
// Device bytes for M (<= moe_rows_chunk) rows; planes: with the rows' digit
// planes (false: the caller has them).
size_t moe_rows_bytes(int64_t M, int64_t k, int64_t E, int64_t H, int64_t I, bool planes);

struct MoeRows {
    int fmt = UT_FMT_INT4;
    ExpertPtrs tbl;
    int64_t E = 0, H = 0, I = 0, M = 0;
    int k = 1;
    const int32_t *ids = nullptr;    // [M, k]
    const float *weights = nullptr;  // [M, k]
    const float *x = nullptr;        // [M, H], or
    const uint16_t *xh = nullptr;    // bf16 in place of x, or
    const DigitPlanes *planes = nullptr;  // digitised already
    const float *shared = nullptr;   // [M, H] added after the choices
    float *out = nullptr;            // [M, ldo]
    int64_t ldo = 0;
    int accumulate = 0;
    int32_t *err_flag = nullptr;
};
// out[m] (+)= sum_c weights[m, c] * expert(ids[m, c])(x[m]), choices in
// order (then + shared[m]); the values are moe_pass's, bit for bit.
int32_t launch_moe_rows(ut_ctx *ctx, const MoeRows &c, void *scratch);

}  // namespace ut
