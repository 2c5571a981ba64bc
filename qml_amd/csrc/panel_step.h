// One 64-wide sub-panel step of a Cholesky block column, shared by the single-matrix factorisation
// (potrf.hip) and the batched one (batched.hip).
#pragma once

#include "chol_panel.h"
#include "linalg.h"
#include "mfma_core.h"

namespace qmlh {

// One 64-wide sub-panel of a block column in one launch: A is its factored w x w diagonal block,
// with m rows below it and ncols more columns of the block column to its right. Every 64 x 64
// block right of the sub-panel before (prev = its width, 0 for the first) still lacks that
// sub-panel's products, but for the diagonal ones, which lack none (of a last one narrower than
// 64 also the rows right below it, up to 64). The workgroups are
//   strip i = 0 .. strips - 1 (64 rows each): its block of this sub-panel minus the products
//     with the previous one, solved against the diagonal block; then, where its rows meet the
//     block column's diagonal, the products of the finished block with itself off the diagonal
//     block there. Strip 0 factors that block: the next sub-panel's.
//   tiles (64 x 64) below the diagonal: the products with the previous sub-panel.
// Every product takes the features in the tile core's order (feature 4 g + q of 16 in lane group
// g), so in FP64 an entry's bits do not depend on which of them a block's products came through.
// No workgroup reads what another one writes, so the chain of a sub-panel is one launch: the
// first strip's, 30 us of latency (loads 3.5, product 2.2, inverses 2.0, solve 2.5, diagonal
// update 3.2, factor 16.3), everything else runs beside it. As two launches, one for the solve
// and one for the update and factor, a sub-panel took 36 us, and each waited for a slot among the
// trailing update's workgroups: factor of order 1000 / 4000 / 8000 / 12,000 / 20,000
// 0.57 / 2.64 / 7.63 / 16.7 / 55.7 ms, now 0.53 / 2.46 / 7.07 / 15.5 / 53.5. (The diagonal block
// of the block column first and then all rows below in one launch: 0.75 / 3.80 / 10.2 / 20.1 /
// 58.7, the rows' own chain of solves comes on top.)
static constexpr int STEP_T = CP_B;
static_assert(STEP_T == WgShape<2>::ROWS, "strips and tiles of one size");
static constexpr int STEP_XS = STEP_T + 4;  // column stride of a strip's solved block in LDS

static constexpr int STEP_PACK = CP_PACK + CP_B / 16 * 16 * 17;  // doubles: packed block, inverses
static_assert(STEP_T * STEP_XS <= WgShape<2>::LDS && STEP_PACK % 2 == 0, "strip and tile LDS");
template <typename T>
static constexpr int STEP_LDS = STEP_PACK + WgShape<2>::LDS * (int)sizeof(T) / (int)sizeof(double);

template <typename T>
struct PanelStep {
    T* A;              // the factored w x w diagonal block
    int64_t lda, m, ncols;
    int64_t col_next;  // column of the matrix that the next diagonal block starts at
    int64_t strips;    // 64-row strips of the m rows
    int32_t* info;
    int32_t w, prev, w_next;
};

// Tiles beside the strips (those on the diagonal and above it return at once).
template <typename T>
static int64_t step_tiles(const PanelStep<T>& st) {
    return st.prev > 0 && st.ncols > 0 ? st.strips * ceil_div(st.ncols, (int64_t)STEP_T) : 0;
}

// A pivot that failed before the next diagonal block (strip 0 may be failing that one now).
template <typename T>
__device__ __forceinline__ bool step_failed(const PanelStep<T>& st) {
    const int32_t failed = *st.info;
    return failed && failed <= st.col_next;
}

template <typename T>
__device__ __forceinline__ void strip_body(const PanelStep<T>& st, PivotRule pr,
                                           double* __restrict__ lds, int64_t strip) {
    constexpr int NB = CP_B / 16;
    T* __restrict__ A = st.A;
    const int64_t lda = st.lda, m = st.m, ncols = st.ncols;
    const int w = st.w, prev = st.prev, w_next = st.w_next;
    double* sp = lds;
    double(*sinv)[16][17] = reinterpret_cast<double(*)[16][17]>(sp + CP_PACK);
    // column-major, STEP_XS apart: the previous sub-panel's block beside the diagonal block, then
    // the strip's solved block
    T* xt = reinterpret_cast<T*>(lds + STEP_PACK);
    __builtin_amdgcn_s_setprio(3);  // on the critical path beside the trailing update's waves
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    T* B = A + w;  // the rows below
    const int lrow = 16 * wave + r;
    const int64_t row = strip * STEP_T + lrow;
    const int64_t rc = row < m ? row : m - 1;
    // The diagonal block in this strip's rows, if the block column has one: wd columns at D.
    const int64_t left = ncols - strip * STEP_T;
    const int wd = left < STEP_T ? (int)left : STEP_T;
    T* D = B + w * lda + strip * STEP_T * (lda + 1);
    const int64_t md = m - strip * STEP_T;  // rows from D on
    // Everything the strip reads, before anything waits: the blocks come from memory (another
    // chiplet wrote them), and one such latency after the other would be a third of the chain.
    Block64<T> diag, beside;
    T mine[NB][4], own[NB][4], dv[NB][4];
    block64_load(diag, A, lda, w, w);
    if (prev > 0) {  // 64 columns
        block64_load(beside, A - (int64_t)prev * lda, lda, w, CP_B);
#pragma unroll
        for (int c = 0; c < NB; ++c)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                // below a narrower diagonal block: rows that had these products with it
                const T v = B[rc + (16 * c + 4 * g + q - (int64_t)prev) * lda];
                own[c][q] = row >= CP_B - w ? v : T(0);
            }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) mine[b][e] = B[rc + cp_clamp(16 * b + g + 4 * e, w) * lda];
    if (left > 0) {
        const int dr = lrow < md ? lrow : (int)(md - 1);
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) dv[b][e] = D[dr + cp_clamp(16 * b + g + 4 * e, wd) * lda];
    }
    block64_pack(sp, diag, w);
    if (prev > 0) {
#pragma unroll
        for (int q = 0; q < CP_B * CP_B / 256; ++q) {
            const int idx = threadIdx.x + 256 * q;
            xt[idx / CP_B * STEP_XS + (idx & (CP_B - 1))] = beside.v[q];
        }
    }
    __syncthreads();
    double4_t acc[NB];  // in the layout of TrsmRows
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[b][e] = (double)mine[b][e];
    if (prev > 0) {
#pragma unroll
        for (int c = 0; c < NB; ++c)
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        -(double)xt[(16 * c + 4 * g + q) * STEP_XS + 16 * b + r],
                        (double)own[c][q], acc[b], 0, 0, 0);
    }
    trsm_inverses(sp, sinv, w);
    __syncthreads();  // the inverses are there, and every wave is done with xt
    TrsmRows X;
    // a block is rounded to the storage type before its solve, as every other update's result is
    trsm_solve16(X, sp, sinv, w, [&](int c, int e) { return (double)(T)acc[c][e]; });
    trsm_store16(X, B, lda, row, m, w);
    if (left <= 0) return;  // the same in every lane
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) xt[(16 * c + g + 4 * e) * STEP_XS + lrow] = (T)X.x[c][e];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[b][e] = (double)dv[b][e];
    __syncthreads();  // the solved block is there, and every wave is done with sp
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            // all four blocks in every wave (those above the diagonal are dropped below): under a
            // condition each LDS read would be waited for by itself, 7.3 us instead of 2.1
            const double x = (double)xt[(16 * c + 4 * g + q) * STEP_XS + lrow];
#pragma unroll
            for (int b = 0; b < NB; ++b)
                acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                    -(double)xt[(16 * c + 4 * g + q) * STEP_XS + 16 * b + r], x, acc[b], 0, 0, 0);
        }
    // the rows of the diagonal block itself are the factor's in strip 0
    const bool factor = strip == 0;
    if (lrow < md && (!factor || lrow >= w_next)) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int col = 16 * b + g + 4 * e;
                if (col <= lrow && col < wd) D[lrow + col * lda] = (T)acc[b][e];
            }
    }
    if (!factor) return;
    potf2_body_sp<T>(
        [&]() {
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int col = 16 * b + g + 4 * e;
                    // as an update stores it: in the storage type
                    if (lrow >= col) sp[pk(lrow, col)] = lrow < w_next ? (double)(T)acc[b][e] : 0.0;
                }
        },
        D, lda, w_next, st.col_next, st.info, sp, pr.floor, pr.bshift, pr.shift_acc, pr.bpivot);
}

template <typename T>
__device__ __forceinline__ void step_tile_body(const PanelStep<T>& st, double* __restrict__ lds,
                                               int64_t tile) {
    const int64_t bi = tile % st.strips, bj = tile / st.strips;
    const int64_t lda = st.lda, m = st.m, ncols = st.ncols;
    if (bi <= bj || bj * STEP_T >= ncols) return;  // on the diagonal or above it, or none of the step's
    const T* P = st.A + st.w - (int64_t)st.prev * lda;
    T* C = st.A + st.w + st.w * lda;
    Operand<T, LAYOUT_COL> rows{P, lda, m, st.prev};
    Operand<T, LAYOUT_COL> cols{P, lda, ncols, st.prev};
    const int wv = threadIdx.x >> 6;
    const int64_t row0 = bi * STEP_T + 32 * (wv >> 1), col0 = bj * STEP_T + 32 * (wv & 1);
    const bool live = row0 < m && col0 < ncols;
    const bool interior = live && row0 + 32 <= m && col0 + 32 <= ncols;
    WaveTile<T, 2> t;
    wave_tile_load_c<T, false>(t, C, lda, row0, col0, m, ncols, live, interior);
    wg_tile_mma_lds<T, LAYOUT_COL, LAYOUT_COL, true>(t, reinterpret_cast<T*>(lds), cols, rows,
                                                     bj * STEP_T, bi * STEP_T, st.prev);
    if (live) wave_tile_store_c<T, false>(t, C, lda, row0, col0, m, ncols, interior);
}

}  // namespace qmlh
