// ut_gemm_core.h -- the tile of the matrix-core product of quantized weights
// with digitised activation rows.
//
// A row of the product is S = sum_k x~[k] q[k] over the activation's integer
// form x~ (ut_internal.h), which three balanced base-256 digits hold: the
// tile multiplies the weight codes with the three digit planes on
// v_mfma_i32_16x16x64_i8 and adds S = a0 + 256 a1 + 65536 a2 in 64 bits, so
// the totals are the GEMVs' whatever the tile or the K split.
//
// A workgroup of four waves takes 64*TO weight rows (TO tiles of 16 per
// wave) against 16*TM activation rows.  The weights go from memory straight
// to the registers of the one wave that uses them (each lane a 16-byte
// piece of one row); only the digit planes, which all four waves read, go
// through LDS: at TO = 4 each digit fragment read feeds four matrix
// instructions, so LDS runs at half the matrix cores' time.  Both are
// fetched a step of 128 columns ahead; the barrier waits for LDS only, so the
// loads stay in flight across it.  LDS rows of 128 bytes keep
// their 16-byte chunks XOR-swizzled by the row's low three bits: eight lanes
// that read one chunk of eight rows read eight different slots of the 256
// bytes that the 64 banks hold.
#pragma once

#include "ut_gemv_mfma.h"

namespace ut {

constexpr int kGemmThreads = 256;
constexpr int kGemmStep = 128;  // columns per step (two matrix instructions deep)
template <int TM> __host__ __device__ constexpr int gemm_lds_uint4() {
    return 2 * TM * 48 * (kGemmStep / 16);  // two buffers of 48 TM plane rows
}
template <int TM> constexpr int gemm_stage_n() { return (TM * 48 * 8 + kGemmThreads - 1) / kGemmThreads; }

// Where a lane's weights come from: row bases (this lane's row of each
// tile), and for rows that are not 16-byte aligned the payload's end.
template <int TO> struct GemmRows {
    const uint8_t *row[TO];
    const uint8_t *end;
};

// 16 bytes at p + off of a weight row of `len` bytes.  Aligned rows clamp a
// chunk past the row to its last one (its columns meet zero digits); others
// read the chunk unaligned, or byte by byte where it would leave the payload.
template <bool UNAL>
__device__ __forceinline__ uint4 gemm_ld16(const uint8_t *p, int64_t off, int64_t len,
                                           const uint8_t *end) {
    if constexpr (!UNAL) return ld_global<uint4>(p + (off < len ? off : len - 16));
    uint4 v = make_uint4(0, 0, 0, 0);
    if (off >= len) return v;
    const uint8_t *q = p + off;
    if (q + 16 <= end) {
        typedef unsigned int u32x4u __attribute__((ext_vector_type(4), aligned(1)));
        const u32x4u t = *(const __attribute__((address_space(1))) u32x4u *)q;
        return make_uint4(t.x, t.y, t.z, t.w);
    }
    uint32_t w[4] = {0, 0, 0, 0};
    const int n = (int)(end - q);
    for (int i = 0; i < n; i++) w[i >> 2] |= (uint32_t)q[i] << (8 * (i & 3));
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// One step's weights of TO tiles: int8 two 16-byte pieces per row (columns
// 64s + 16q of the step for matrix instruction s and lane quarter q), int4
// one (columns 32q + 16s).
template <int FMT, int TO> struct GemmA {
    static constexpr int NP = FMT == UT_FMT_INT8 ? 2 : 1;
    uint4 v[TO][NP];
};
template <int FMT, int TO, bool UNAL>
__device__ __forceinline__ void gemm_load_a(GemmA<FMT, TO> &a, const GemmRows<TO> &r, int64_t col,
                                            int64_t len, int q) {
#pragma unroll
    for (int t = 0; t < TO; t++)
#pragma unroll
        for (int i = 0; i < GemmA<FMT, TO>::NP; i++) {
            const int64_t off = FMT == UT_FMT_INT8 ? col + 64 * i + 16 * q : col / 2 + 16 * q;
            a.v[t][i] = gemm_ld16<UNAL>(r.row[t], off, len, r.end);
        }
}
// 16 int4 codes as bytes, times 16 (a nibble in the byte's high half is its
// own sign extension), which the epilogue's exponent takes back.
__device__ __forceinline__ ut_i32x4 gemm_i4_codes(uint32_t u0, uint32_t u1) {
    ut_i32x4 f;
    const uint32_t u[2] = {u0, u1};
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const uint32_t lo = (u[j] << 4) & 0xF0F0F0F0u, hi = u[j] & 0xF0F0F0F0u;
        f[2 * j] = (int)__builtin_amdgcn_perm(hi, lo, 0x05010400u);
        f[2 * j + 1] = (int)__builtin_amdgcn_perm(hi, lo, 0x07030602u);
    }
    return f;
}
// The A operand of matrix instruction s: 16 codes per lane.
template <int FMT, int TO>
__device__ __forceinline__ ut_i32x4 gemm_frag_a(const GemmA<FMT, TO> &a, int t, int s) {
    ut_i32x4 f;
    if constexpr (FMT == UT_FMT_INT8) {
        const uint4 v = a.v[t][s];
        f[0] = (int)v.x; f[1] = (int)v.y; f[2] = (int)v.z; f[3] = (int)v.w;
    } else {
        const uint4 v = a.v[t][0];
        f = s ? gemm_i4_codes(v.z, v.w) : gemm_i4_codes(v.x, v.y);
    }
    return f;
}
template <int FMT> __device__ __forceinline__ int32_t gemm_exp(int32_t e) {
    return FMT == UT_FMT_INT4 && e != INT32_MIN ? e - 4 : e;
}

// acc[t][n][p] = tile over columns [kb, ke) (kb a multiple of 128, columns
// past K zero in the planes).  src[i]: the digit bytes of this thread's
// staging chunk i at column 0 (its chunk offset included).  Two steps are held
// in registers, one in flight while the other computes.  Four measured no
// better at 5 to 64 rows (int8 7168 x 16384 at 5 rows 44.2 against 43.7 us)
// and worse at 512 (int4 18432 x 7168 272 against 260 us).
template <int FMT, int TO, int TM, bool UNAL>
__device__ __forceinline__ void gemm_tile(const GemmRows<TO> &rows, int64_t len, int64_t kb,
                                          int64_t ke, const int8_t *const (&src)[gemm_stage_n<TM>()],
                                          uint4 *lds, ut_i32x4 (&acc)[TO][TM][3]) {
    constexpr int D = 2;  // (the LDS buffer of a step is its slot's parity)
    constexpr int NB = gemm_stage_n<TM>(), CH = TM * 48 * 8;
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int t = 0; t < TO; t++)
#pragma unroll
        for (int n = 0; n < TM; n++)
#pragma unroll
            for (int p = 0; p < 3; p++) acc[t][n][p] = ut_i32x4{0, 0, 0, 0};
    GemmA<FMT, TO> a[D];
    uint4 b[D][NB];
    const int n = (int)((ke - kb + kGemmStep - 1) / kGemmStep);
    auto load = [&](int d, int i) {
        const int64_t k = kb + (int64_t)i * kGemmStep;
#pragma unroll
        for (int j = 0; j < NB; j++)
            if (tid + j * kGemmThreads < CH) b[d][j] = ld_global<uint4>(src[j] + k);
        gemm_load_a<FMT, TO, UNAL>(a[d], rows, k, len, q);
    };
    auto store_b = [&](int d, int buf) {
#pragma unroll
        for (int j = 0; j < NB; j++)
            if (tid + j * kGemmThreads < CH) lds[buf * CH + tid + j * kGemmThreads] = b[d][j];
    };
    auto compute = [&](const GemmA<FMT, TO> &av, const uint4 *buf) {
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const int chunk = (FMT == UT_FMT_INT8 ? 4 * s + q : 2 * q + s) ^ (r & 7);
            ut_i32x4 f[TO];
#pragma unroll
            for (int t = 0; t < TO; t++) f[t] = gemm_frag_a<FMT, TO>(av, t, s);
#pragma unroll
            for (int m = 0; m < TM; m++)
#pragma unroll
                for (int p = 0; p < 3; p++) {
                    const uint4 v = buf[((m * 3 + p) * 16 + r) * 8 + chunk];
                    const ut_i32x4 w{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
#pragma unroll
                    for (int t = 0; t < TO; t++)
                        acc[t][m][p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f[t], w, acc[t][m][p], 0, 0, 0);
                }
        }
    };
    // LDS-only barrier: the loads of later steps stay in flight across it
    auto barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
#pragma unroll
    for (int d = 0; d < D; d++)
        if (d < n) load(d, d);
    store_b(0, 0);
    barrier();
    for (int base = 0; base < n; base += D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            const int i = base + d;
            if (i < n) {
                compute(a[d], lds + (d & 1) * CH);
                if (i + 1 < n) store_b((d + 1) % D, (d + 1) & 1);
                if (i + D < n) load(d, i + D);
                barrier();
            }
        }
    }
}

// ------------------------------------------------ tile through LDS ---
// The same tile with the weights through LDS too, for launches that the
// matrix cores bound: a lane's direct weight load takes 16 bytes of its own
// row, so each 16 lanes touch 16 cache lines, and at 512 rows those lookups
// held the direct tile at a quarter of the matrix rate.  Here both operands
// are copied by global_load_lds (no registers) in stages of 128 columns, one
// in flight while one is computed on, and WO x WM waves share them: each
// wave TO tiles of 16 weight rows against 16 TM activation rows.  LDS has
// 64 banks: a staged row's 16-byte chunks are XOR-swizzled so that the 16
// rows a lane group reads take 16 different slots of 256 bytes.
template <int FMT, int TO, int TM, int WO, int WM> struct GemmLds {
    static constexpr int S = kGemmStep;
    static constexpr int kThreads = 64 * WO * WM;
    static constexpr int kARows = 16 * TO * WO, kBRows = 48 * TM * WM;
    static constexpr int kAC = FMT == UT_FMT_INT8 ? S / 16 : S / 32, kBC = S / 16;  // chunks of a row
    static constexpr int kA = kARows * kAC, kB = kBRows * kBC;  // chunks of a stage
    static constexpr int kNA = kA / kThreads, kNB = (kB + kThreads - 1) / kThreads;
    static_assert(kA % kThreads == 0 && kB % 64 == 0, "whole copies; a last one of whole waves");
    uint4 a[kA], b[kB];
};
// Chunk c of a row of C chunks sits at slot c ^ gemm_swz<C>(row).
template <int C> __device__ __forceinline__ int gemm_swz(int row) {
    static_assert(C == 4 || C == 8, "rows of 64 or 128 bytes");
    return (row / (16 / C)) & (C - 1);
}

// This thread's copy sources at column 0 (row pointers are the caller's);
// aoff: the A chunk's byte offset in its row's step.
template <int FMT, int TO, int TM, int WO, int WM> struct GemmSrc {
    using L = GemmLds<FMT, TO, TM, WO, WM>;
    const uint8_t *a[L::kNA];
    const int8_t *b[L::kNB];
    int aoff;
};
template <int FMT, int TO, int TM, int WO, int WM, typename ARow, typename BRow>
__device__ __forceinline__ void gemm_src(GemmSrc<FMT, TO, TM, WO, WM> &s, ARow &&arow,
                                         BRow &&brow) {
    using L = GemmLds<FMT, TO, TM, WO, WM>;
    const int tid = threadIdx.x;
#pragma unroll
    for (int i = 0; i < L::kNA; i++) {
        const int c = tid + i * L::kThreads, row = c / L::kAC, ph = c % L::kAC;
        s.a[i] = arow(row);
        // a copy covers a multiple of 16 rows, so every copy's chunk offset
        // is the same
        if (i == 0) s.aoff = (ph ^ gemm_swz<L::kAC>(row)) * 16;
    }
#pragma unroll
    for (int i = 0; i < L::kNB; i++) {
        const int t = tid + i * L::kThreads, c = t < L::kB ? t : 0;
        const int row = c / L::kBC, n = row / 48, x = row - 48 * n;
        s.b[i] = brow(16 * n + (x & 15), x >> 4) + ((c % L::kBC) ^ gemm_swz<L::kBC>(row)) * 16;
    }
}

// This wave's copies landed, then the workgroup's barrier.  (The builtin and
// not inline asm: the compiler then knows that the stage has landed, and
// does not wait for the next stage's copies before reading it.)
__device__ __forceinline__ void gemm_wait_copies() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(7 << 4);  // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// PIPE: a stage's second half is multiplied after the next stage's first half
// has been read, so a wave's LDS reads run beside its matrix instructions
// instead of before them (twice the fragments in registers).
template <bool PIPE, int FMT, int TO, int TM, int WO, int WM>
__device__ __forceinline__ void gemm_tile_lds(const GemmSrc<FMT, TO, TM, WO, WM> &src, int64_t len,
                                              int64_t kb, int64_t ke, GemmLds<FMT, TO, TM, WO, WM> &s0,
                                              GemmLds<FMT, TO, TM, WO, WM> &s1,
                                              ut_i32x4 (&acc)[TO][TM][3]) {
    constexpr int S = kGemmStep;
    using L = GemmLds<FMT, TO, TM, WO, WM>;
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4, wave = tid >> 6;
    const int wo = wave % WO, wm = wave / WO;
#pragma unroll
    for (int t = 0; t < TO; t++)
#pragma unroll
        for (int n = 0; n < TM; n++)
#pragma unroll
            for (int p = 0; p < 3; p++) acc[t][n][p] = ut_i32x4{0, 0, 0, 0};
    const int w64 = __builtin_amdgcn_readfirstlane(wave) * 64;
    const int n = (int)((ke - kb) / S);  // K slices are whole 128-column steps
    // (past the last stage: the last one again, into a buffer nothing reads)
    auto copy = [&](L &s, int i) {
        const int64_t k = kb + (int64_t)(i < n ? i : n - 1) * S;
        // columns past K meet zero digits: any in-bounds weight chunk will do
        int64_t off = (FMT == UT_FMT_INT8 ? k : k / 2) + src.aoff;
        off = off < len ? off : len - 16;
#pragma unroll
        for (int j = 0; j < L::kNA; j++)
            __builtin_amdgcn_global_load_lds(
                (const void *)(src.a[j] + off),
                (__attribute__((address_space(3))) void *)(s.a + j * L::kThreads + w64), 16, 0, 0);
#pragma unroll
        for (int j = 0; j < L::kNB; j++)
            if (L::kB % L::kThreads == 0 || j * L::kThreads + w64 < L::kB)
                __builtin_amdgcn_global_load_lds(
                    (const void *)(src.b[j] + k),
                    (__attribute__((address_space(3))) void *)(s.b + j * L::kThreads + w64), 16, 0, 0);
    };
    // the operands of half stage h: weights (int4 codes still packed), digits
    auto frag_a = [&](const L &s, int h, int t) {
        const int c = 4 * h + q, row = (wo * TO + t) * 16 + r;  // c: this lane's 16 columns
        ut_i32x4 x;
        if constexpr (FMT == UT_FMT_INT8) {
            const uint4 v = s.a[row * L::kAC + (c ^ gemm_swz<L::kAC>(row))];
            x = ut_i32x4{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
        } else {
            const uint2 v = ((const uint2 *)&s.a[row * L::kAC + ((c >> 1) ^ gemm_swz<L::kAC>(row))])[c & 1];
            x[0] = (int)v.x;
            x[1] = (int)v.y;
        }
        return x;
    };
    auto frag_b = [&](const L &s, int h, ut_i32x4 (&x)[TM][3]) {
#pragma unroll
        for (int m = 0; m < TM; m++)
#pragma unroll
            for (int p = 0; p < 3; p++) {
                const int row = ((wm * TM + m) * 3 + p) * 16 + r;
                const uint4 v = s.b[row * L::kBC + ((4 * h + q) ^ gemm_swz<L::kBC>(row))];
                x[m][p] = ut_i32x4{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
            }
    };
    auto codes = [](const ut_i32x4 &x) {
        if constexpr (FMT == UT_FMT_INT8) return x;
        else return gemm_i4_codes((uint32_t)x[0], (uint32_t)x[1]);
    };
    auto products = [&](const ut_i32x4 (&f)[TO], const ut_i32x4 (&x)[TM][3]) {
#pragma unroll
        for (int m = 0; m < TM; m++)
#pragma unroll
            for (int p = 0; p < 3; p++)
#pragma unroll
                for (int t = 0; t < TO; t++)
                    acc[t][m][p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f[t], x[m][p], acc[t][m][p], 0, 0, 0);
    };
    struct Frag {
        ut_i32x4 a[TO], b[TM][3];
    };
    auto read = [&](const L &s, int h, Frag &x) {
#pragma unroll
        for (int t = 0; t < TO; t++) x.a[t] = frag_a(s, h, t);
        frag_b(s, h, x.b);
    };
    auto multiply = [&](const Frag &x) {
        ut_i32x4 f[TO];
#pragma unroll
        for (int t = 0; t < TO; t++) f[t] = codes(x.a[t]);
        products(f, x.b);
    };
    Frag f0, f1;
    // step i: its stage has landed, the other buffer is read and gets the next
    auto step = [&](L &s, L &other, int i) {
        gemm_wait_copies();
        copy(other, i + 1);
        if constexpr (PIPE) {
            read(s, 0, f0);
            __builtin_amdgcn_sched_barrier(0);
            if (i) multiply(f1);
            read(s, 1, f1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(f0);
        } else {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                // (unpacked as they are read: after the digits' reads int4
                // 24576 x 1536 at 509 rows took 112 us, 79 so)
                ut_i32x4 f[TO], x[TM][3];
#pragma unroll
                for (int t = 0; t < TO; t++) f[t] = codes(frag_a(s, h, t));
                frag_b(s, h, x);
                products(f, x);
            }
        }
    };
    copy(s0, 0);
    int i = 0;
    for (; i + 2 <= n; i += 2) {
        step(s0, s1, i);
        step(s1, s0, i + 1);
    }
    if (i < n) step(s0, s1, i);
    if constexpr (PIPE) multiply(f1);
    gemm_wait_copies();  // no copy outlives the tile
}

// The exact total of one accumulator element.
__device__ __forceinline__ int64_t gemm_total(const ut_i32x4 (&a)[3], int j) {
    return (int64_t)a[0][j] + ((int64_t)a[1][j] << 8) + ((int64_t)a[2][j] << 16);
}

// A thread's staging chunk: plane row (of 48 TM, tile-major: 16 activation
// rows of one plane after another) and 16-byte chunk within the step.
struct GemmChunk {
    int m, p, off;
};
__device__ __forceinline__ GemmChunk gemm_chunk(int c) {
    const int rr = c >> 3, n = rr / 48, x = rr - 48 * n;
    return {16 * n + (x & 15), x >> 4, ((c & 7) ^ (rr & 7)) * 16};
}

}  // namespace ut
