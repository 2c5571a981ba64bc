// Cholesky panel building blocks shared by the single-matrix factorisation (potrf.hip) and the
// batched one (batched.hip): the factor of a <= 64 x 64 diagonal block in LDS, and the
// row-parallel solve of the panel rows below it.
#pragma once

#include "common.h"

namespace qmlh {

static constexpr int CP_B = 64;  // diagonal block / sub-panel width

// Lane `lane`'s value of v in every lane (two scalar reads; lane is a compile-time constant
// where this is used, so no LDS round trip).
__device__ __forceinline__ double readlane_f64(double v, int lane) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, lane);
    const unsigned hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), lane);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Packed lower triangle of a 64 x 64 block in LDS, column-major: element (i, j), i >= j, at
// pk(i, j); column j holds rows j .. 63. 2080 doubles (16.6 KB) instead of a padded square
// (33 KB). Wherever the loops are unrolled the index is a compile-time constant (+ lane).
static constexpr int CP_PACK = CP_B * (CP_B + 1) / 2;
__host__ __device__ constexpr int pk(int i, int j) { return j * CP_B - (j * (j - 1)) / 2 + (i - j); }

// Every lane loads unconditionally from an index clamped into the w x w block and selects
// zero afterwards: a load (and its conversion) under a condition makes the compiler wait for
// it inside the branch, which serialises a run of loads.
__device__ __forceinline__ int cp_clamp(int i, int w) { return i < w ? i : w - 1; }

// A 64 x 64 block spread over 256 lanes: value q of lane t is element (t % 64, t / 64 + 4 q).
template <typename T>
struct Block64 {
    T v[CP_B * CP_B / 256];
};

// The w rows and columns of the block at A (indices clamped), loads issued back to back.
template <typename T>
__device__ __forceinline__ void block64_load(Block64<T>& raw, const T* __restrict__ A, int64_t lda,
                                             int w, int cols) {
    const int t = threadIdx.x;
#pragma unroll
    for (int q = 0; q < CP_B * CP_B / 256; ++q) {
        const int idx = t + 256 * q;
        const int i = idx & (CP_B - 1), j = idx / CP_B;
        raw.v[q] = A[cp_clamp(i, w) + (int64_t)cp_clamp(j, cols) * lda];
    }
}

// Packed LDS <- the lower triangle of a loaded w x w block (zero outside w).
template <typename T>
__device__ __forceinline__ void block64_pack(double* __restrict__ sp, const Block64<T>& raw, int w) {
    const int t = threadIdx.x;
#pragma unroll
    for (int q = 0; q < CP_B * CP_B / 256; ++q) {
        const int idx = t + 256 * q;
        const int i = idx & (CP_B - 1), j = idx / CP_B;
        if (i >= j) sp[pk(i, j)] = (i < w && j < w) ? (double)raw.v[q] : 0.0;
    }
}

// Packed LDS <- the lower triangle of the w x w block at A (zero outside w); 256 lanes.
template <typename T>
__device__ __forceinline__ void stage_packed64(double* __restrict__ sp, const T* __restrict__ A,
                                               int64_t lda, int w) {
    Block64<T> raw;
    block64_load(raw, A, lda, w, w);
    block64_pack(sp, raw, w);
}

// LDS (FP64) <- the lower triangle of the w x w block at A (column-major, lda), zero elsewhere;
// TRANS stores element (i, j) at s[j][i]. All 256 lanes take part; each issues its 16 loads
// back to back before any LDS store.
template <bool TRANS, int LDS_LD, typename T>
__device__ __forceinline__ void stage_lower64(double (*s)[LDS_LD], const T* __restrict__ A,
                                              int64_t lda, int w) {
    const int t = threadIdx.x;
    T raw[CP_B * CP_B / 256];
#pragma unroll
    for (int q = 0; q < CP_B * CP_B / 256; ++q) {
        const int idx = t + 256 * q;
        const int i = idx & (CP_B - 1), j = idx / CP_B;  // consecutive lanes: consecutive rows
        raw[q] = A[cp_clamp(i, w) + (int64_t)cp_clamp(j, w) * lda];
    }
#pragma unroll
    for (int q = 0; q < CP_B * CP_B / 256; ++q) {
        const int idx = t + 256 * q;
        const int i = idx & (CP_B - 1), j = idx / CP_B;
        const double v = (i < w && j < w && i >= j) ? (double)raw[q] : 0.0;
        if (TRANS) s[j][i] = v; else s[i][j] = v;
    }
}

// C(ib, jb) -= L(ib, kb) L(jb, kb)^T on 16 x 16 blocks of the packed block, by one wavefront on
// the FP64 matrix cores (four products deep 4). kb < jb <= ib; on the diagonal only the lower
// part is stored.
__device__ __forceinline__ void potf2_update16(double* __restrict__ sp, int ib, int jb, int kb) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    double4_t acc;
    const int col = 16 * jb + r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int row = 16 * ib + g + 4 * e;
        acc[e] = sp[pk(row > col ? row : col, col)];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int k = 16 * kb + g + 4 * q;
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-sp[pk(16 * ib + r, k)], sp[pk(col, k)], acc, 0,
                                                   0, 0);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int row = 16 * ib + g + 4 * e;
        if (row >= col) sp[pk(row, col)] = acc[e];
    }
}

// Columns c0 .. c0 + 15 of the packed w x w block factored by one wavefront, in registers (lane
// i holds row i; the rows above a column hold scratch). Per column the pivot and the entries of
// the panel's own rows are read from their lanes, so a column is one dependent chain
// (reciprocal square root, scale, update) with no LDS round trip. Returns 0, or c + 1 for the
// first failed pivot c.
static constexpr int CP_PW = 16;  // panel width

// 1/sqrt(piv) from the hardware estimate r (relative error below 2^-20) and one third-order step,
// r + r e (1/2 + 3/8 e) with e = 1 - piv r^2, which leaves less than e^3 beside
// its rounding; sqrt(piv) = piv / sqrt(piv). Four dependent operations on the critical path, two
// fewer than two Newton steps, instead of a correctly rounded square root followed by a division.
__device__ __forceinline__ double potf2_rsqrt(double piv) {
    const double r = __builtin_amdgcn_rsq(piv);
    const double e = fma(-piv * r, r, 1.0);
    return fma(r * e, fma(0.375, e, 0.5), r);
}

__device__ __forceinline__ int potf2_panel16(double* __restrict__ sp, int c0, int w, double floor,
                                             double fail_at) {
    const int lane = threadIdx.x & 63;
    double a[CP_PW];
#pragma unroll
    for (int j = 0; j < CP_PW; ++j) {
        const double v = sp[pk(lane > c0 + j ? lane : c0 + j, c0 + j)];
        a[j] = lane >= c0 + j ? v : 0.0;
    }
    if (!(floor > 0.0)) {
        // No branch between the columns: the pivots are checked on the side and a panel with a
        // failed one (whose later columns are garbage) is done again below from sp. The columns
        // past w are zero and stay out of the check; what they become is never used.
        // Each step starts the next column's chain (its update, pivot and root) and fills that
        // chain's latency with the other columns' updates; the scheduling fence keeps the
        // compiler from collecting updates of many steps, whose lane reads then spill.
        int bad = 0;
        double piv = readlane_f64(a[0], c0);
        double rl = potf2_rsqrt(piv);
#pragma unroll
        for (int c = 0; c < CP_PW; ++c) {
            bad |= (int)!(piv > fail_at) & (int)(c0 + c < w);
            const double x = a[c] * rl;  // the pivot is lane c0 + c's value
            a[c] = x;
            if (c + 1 < CP_PW) {
                a[c + 1] = fma(-x, readlane_f64(x, c0 + c + 1), a[c + 1]);
                piv = readlane_f64(a[c + 1], c0 + c + 1);
                rl = potf2_rsqrt(piv);
            }
#pragma unroll
            for (int j = c + 2; j < CP_PW; ++j) a[j] = fma(-x, readlane_f64(x, c0 + j), a[j]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (!bad) {
#pragma unroll
            for (int j = 0; j < CP_PW; ++j)
                if (lane >= c0 + j) sp[pk(lane, c0 + j)] = a[j];
            return 0;
        }
#pragma unroll
        for (int j = 0; j < CP_PW; ++j) {
            const double v = sp[pk(lane > c0 + j ? lane : c0 + j, c0 + j)];
            a[j] = lane >= c0 + j ? v : 0.0;
        }
    }
    // Column c is always a[0]: the update of the later ones moves them down one register.
    int f = 0;
#pragma unroll 1
    for (int c = c0; c < c0 + CP_PW; ++c) {
        double piv = readlane_f64(a[0], c);
        if (!(piv > floor) && floor > 0.0 && piv == piv) piv = floor;
        if (f == 0 && c < w && !(piv > fail_at)) f = c + 1;
        if (f == 0 && c < w) {
            const double x = (lane == c ? piv : a[0]) * potf2_rsqrt(piv);
            if (lane >= c) sp[pk(lane, c)] = x;
            // entries past the panel (and past lane 63, which wraps) are never stored
#pragma unroll
            for (int j = 1; j < CP_PW; ++j) a[j - 1] = fma(-x, readlane_f64(x, c + j), a[j]);
        } else {
            if (lane >= c) sp[pk(lane, c)] = a[0];
#pragma unroll
            for (int j = 1; j < CP_PW; ++j) a[j - 1] = a[j];
        }
    }
    return f;
}

// Cholesky of the w x w (w <= 64) lower block in packed LDS sp (FP64, zero outside w) by the
// four wavefronts of a workgroup, in four panels of 16 columns: wave 0 factors a panel
// (potf2_panel16) while the other waves apply the previous panel to the blocks right of the
// next one on the matrix cores; the panel's own update of the next 16 columns (at most three
// 16 x 16 blocks, one per wave) is all that lies between two panels. Bound by the latency of
// the 64 column steps, a wavefront's issue of about 60 instructions each: 16.3 us (20 as a launch of
// its own; 17.1 with two Newton steps per root), against 34 us a launch for one wavefront that held
// all 64 columns and sent each through LDS. (Panel columns as a rolled loop, the later ones
// moved down a register each step: 42 us, its lane reads each waited for; unrolled with a
// branch on every pivot: 25 us.)
// Called by all 256 threads (barriers). On exit sp holds L in its lower triangle. Returns 0, or
// c + 1 for the first non-positive (or NaN) pivot c, with the Schur value left on that diagonal
// entry (as LAPACK leaves it) and the columns of later panels not updated by this one; the
// value is the same in every lane. floor > 0 (static pivoting, for factors that only
// precondition): a finite pivot at or below floor is replaced by floor instead of failing; NaN
// still fails. fail_at >= 0: a pivot at or below it fails (0: LAPACK's rule).
__device__ __forceinline__ int potf2_block64(double* __restrict__ sp, int w, double floor = 0.0,
                                             double fail_at = 0.0) {
    __shared__ int s_fail;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (threadIdx.x == 0) s_fail = 0;
#pragma unroll 1
    for (int kb = 0; kb < CP_B / CP_PW && kb * CP_PW < w; ++kb) {
        if (wave == 0) {
            const int f = potf2_panel16(sp, kb * CP_PW, w, floor, fail_at);
            if (f && threadIdx.x == 0) s_fail = f;
        } else if (kb > 0) {
            // blocks right of panel kb by panel kb - 1: at most three, one per wave
            int q = 0;
            for (int jb = kb + 1; jb < 4; ++jb)
                for (int ib = jb; ib < 4; ++ib, ++q)
                    if (q % 3 == wave - 1) potf2_update16(sp, ib, jb, kb - 1);
        }
        __syncthreads();
        if (s_fail) break;
        if (kb + 1 + wave < 4) potf2_update16(sp, kb + 1 + wave, kb + 1, kb);
        __syncthreads();
    }
    return s_fail;
}

// x^T of 16 rows: element e of block c is column 16 c + (lane >> 4) + 4 e of row lane & 15, the
// output layout of the FP64 matrix instruction and, element by element, its second operand for
// the products of later blocks, so the solve never leaves the registers.
struct TrsmRows {
    double4_t x[4];
};

// Diagonal block of a sub-panel, one workgroup: factor the w x w block at A (potf2_block64), write
// L back, set info = col_base + c + 1 on a failed pivot. `info` already set: nothing is done.
// sp: CP_PACK doubles of LDS (potf2_body brings its own; a kernel that has LDS to spare at
// that point passes it).
// Shift on breakdown (shift_acc non-null, bshift > 0; for factors that only precondition): a
// pivot at or below bpivot counts as failed, the block's diagonal first gets *shift_acc (the
// shift earlier blocks settled on), a failed pivot re-factors the block from A with its whole
// diagonal raised by bshift, then 10 bshift (no further: a larger shift would precondition a
// different matrix), and the shift that succeeds is left in *shift_acc for the later blocks. The factor is then the exact Cholesky factor of A + diag(0, .., 0, s1, .., s2, ..):
// zero before the first failing block, nondecreasing after. A block that fails at 10 bshift
// sets info. Diagonal blocks are factored one at a time in column order, each after the
// one before it, so *shift_acc needs no atomics.
// stage(): writes the w x w block to sp (zero outside w), the same values on every call; no
// barriers needed in it.
template <typename T, typename Stage>
__device__ __forceinline__ void potf2_body_sp(Stage stage, T* __restrict__ A, int64_t lda, int w,
                                              int64_t col_base, int32_t* __restrict__ info,
                                              double* __restrict__ sp, double floor = 0.0,
                                              double bshift = 0.0,
                                              double* __restrict__ shift_acc = nullptr,
                                              double bpivot = 0.0) {
    const int t = threadIdx.x;
    const bool shifting = shift_acc != nullptr && bshift > 0.0;
    double shift = shifting ? *shift_acc : 0.0;
    int fail = 0;
    for (int attempt = 0;; ++attempt) {
        stage();
        __syncthreads();
        if (shift > 0.0) {
            if (t < w) sp[pk(t, t)] += shift;
            __syncthreads();
        }
        fail = potf2_block64(sp, w, floor, shifting ? bpivot : 0.0);
        if (!fail || !shifting || shift >= 10.0 * bshift) break;
        shift = shift > 0.0 ? 10.0 * shift : bshift;  // uniform: every lane sees the same fail
        __syncthreads();  // every lane is done with sp and the fail word before both are reset
    }
#pragma unroll
    for (int q = 0; q < CP_B * CP_B / 256; ++q) {
        const int idx = t + 256 * q;
        const int i = idx & (CP_B - 1), j = idx / CP_B;
        if (i < w && j < w && i >= j) A[i + (int64_t)j * lda] = (T)sp[pk(i, j)];
    }
    if (t == 0 && fail) *info = (int32_t)(col_base + fail);
    if (t == 0 && shifting && !fail) *shift_acc = shift;
}

template <typename T>
__device__ __forceinline__ void potf2_body(T* __restrict__ A, int64_t lda, int w,
                                           int64_t col_base, int32_t* __restrict__ info,
                                           double floor = 0.0, double bshift = 0.0,
                                           double* __restrict__ shift_acc = nullptr,
                                           double bpivot = 0.0) {
    __shared__ double sp[CP_PACK];
    if (*info) return;
    __builtin_amdgcn_s_setprio(3);  // one dependent chain beside the trailing update's waves
    potf2_body_sp<T>([&]() { stage_packed64(sp, A, lda, w); }, A, lda, w, col_base, info, sp,
                     floor, bshift, shift_acc, bpivot);
}

// FP64 inverses of the 16 x 16 diagonal blocks of the packed w x w factor sp: each wave inverts
// one, a lane per column (zero past w). One division per lane; what a reciprocal instead of a
// division costs in the last place is undone by the refinement of the solve.
__device__ __forceinline__ void trsm_inverses(const double* __restrict__ sp, double (*sinv)[16][17],
                                              int w) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // column r of the inverse of diagonal block `wave` (the four lane groups do the same work)
    const int b0 = 16 * wave;
    const double rd = b0 + r < w ? 1.0 / sp[pk(b0 + r, b0 + r)] : 0.0;
    double x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = i == r ? 1.0 : 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        x[i] *= readlane_f64(rd, i);
#pragma unroll
        for (int j = i + 1; j < 16; ++j) x[j] = fma(-sp[pk(b0 + j, b0 + i)], x[i], x[j]);
    }
    if (g == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) sinv[wave][i][r] = x[i];
    }
}

// B L^-T for a wavefront's 16 rows, value(c, e) being B's element in the layout of TrsmRows.
//
// A wavefront solves 16 rows in blocks of 16 columns on the FP64 matrix cores: block c takes the
// products with the finished blocks, is multiplied by the FP64 inverse D of L's 16 x 16
// diagonal block and refined once,
//     X = T D^T;  X += (T - X L_cc^T) D^T,
// which brings the residual of the block back to that of a substitution, whatever L_cc's
// condition. 72 products of 64 cycles, 2.5 us; as a launch of its own with the loads and the
// inverses 10.5 us, where one lane per row and 2016 dependent FMAs with as many LDS reads took 21.
template <typename Value>
__device__ __forceinline__ void trsm_solve16(TrsmRows& X, const double* __restrict__ sp,
                                             const double (*sinv)[16][17], int w, Value value) {
    constexpr int NB = CP_B / 16;
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int c = 0; c < NB; ++c) {
        double4_t t;
#pragma unroll
        for (int e = 0; e < 4; ++e) t[e] = 16 * c + g + 4 * e < w ? value(c, e) : 0.0;
#pragma unroll
        for (int k = 0; k < c; ++k)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                t = __builtin_amdgcn_mfma_f64_16x16x4f64(-sp[pk(16 * c + r, 16 * k + g + 4 * q)],
                                                         X.x[k][q], t, 0, 0, 0);
        double4_t x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 4; ++q)
            x = __builtin_amdgcn_mfma_f64_16x16x4f64(sinv[c][r][g + 4 * q], t[q], x, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = g + 4 * q;
            const double l = sp[pk(16 * c + (r > k ? r : k), 16 * c + k)];
            t = __builtin_amdgcn_mfma_f64_16x16x4f64(r >= k ? -l : 0.0, x[q], t, 0, 0, 0);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            x = __builtin_amdgcn_mfma_f64_16x16x4f64(sinv[c][r][g + 4 * q], t[q], x, 0, 0, 0);
        X.x[c] = x;
    }
}

template <typename T>
__device__ __forceinline__ void trsm_store16(const TrsmRows& X, T* __restrict__ B, int64_t lda,
                                             int64_t row, int64_t m, int w) {
    const int g = (threadIdx.x & 63) >> 4;
    if (row >= m) return;
#pragma unroll
    for (int c = 0; c < CP_B / 16; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int col = 16 * c + g + 4 * e;
            if (col < w) B[row + col * lda] = (T)X.x[c][e];
        }
}

}  // namespace qmlh
