// FP64 VALU pairwise tile shared by the pairwise kernels and the batched sweep.
//
// Tiling: a 256-lane workgroup owns a 128 x 128 output tile; each lane owns an 8 x 8 register
// tile (rows 2*tx + 32*r + {0,1}, columns 2*ty + 32*c + {0,1}, tx = t % 16, ty = t / 16).
// Features stream through LDS in chunks of 16, stored k-major so a lane fetches its two
// adjacent rows (or columns) for one feature with a single 16-byte LDS read; 130 doubles between
// features keep the writes (8 lanes a row, 2 features each) free of bank conflicts too. Each lane keeps
// the feature sum of every entry in feature order k = 0, 1, ..., d-1, so an entry equals a
// serial sum over the features.
#pragma once

#include "common.h"

namespace qmlh {

static constexpr int PT_BM = 128;
static constexpr int PT_BN = 128;
static constexpr int PT_BK = 16;
static constexpr int PT_LDS = PT_BM + 2;  // padded k-major row (doubles), keeps 16 B alignment
static constexpr int PT_THREADS = 256;

// Per-feature terms: |a - b|, (a - b)^2, |a - b|^3 and |a - b|^4 by the products binary
// powering forms (x (x x), (x x)(x x)), |a - b|^p for any other p (pow).
enum { OP_L1 = 0, OP_SQ = 1, OP_POW3 = 2, OP_POW4 = 3, OP_POWR = 4 };
// Epilogues of the feature sum s: s, sqrt(s), exp(s0 s), the Sargan polynomial-times-exp in
// the L1 distance, the Matern forms in the L2 distance, s^s0 (the p-norm root).
enum { EPI_IDENTITY = 0, EPI_SQRT = 1, EPI_EXP = 2, EPI_SARGAN = 3, EPI_MATERN = 4, EPI_ROOT = 5 };

static constexpr int PAIR_MAX_GAMMAS = 16;

struct PairEpi {
    double s0, s1;                 // scales (see the epilogues)
    double g[PAIR_MAX_GAMMAS];     // Sargan coefficients gamma_1 ..
    int ng;                        // their count
    int order;                     // Matern order 0, 1, 2
};

// x^n for n >= 0 by binary powering.
__device__ __forceinline__ double pair_powi(double x, int n) {
    double r = (n & 1) ? x : 1.0;
    while (n >>= 1) {
        x = x * x;
        if (n & 1) r = r * x;
    }
    return r;
}

template <int OP>
__device__ __forceinline__ double pair_term(double acc, double a, double b, double p = 0.0) {
    if (OP == OP_L1) {
        return acc + fabs(a - b);
    } else if (OP == OP_SQ) {
        double t = a - b;
        return fma(t, t, acc);
    } else if (OP == OP_POW3) {
        const double x = fabs(a - b);
        return acc + x * (x * x);
    } else if (OP == OP_POW4) {
        const double x = fabs(a - b);
        const double x2 = x * x;
        return acc + x2 * x2;
    } else {
        // |a - b|^p as exp(p log|a - b|): log and exp instead of pow's extended-precision path
        // (relative error about p |log x| ulp, far inside the 1e-12 the kernel is held to);
        // x = 0 gives exp(-inf) = 0 as pow does for p > 0.
        return acc + exp(p * log(fabs(a - b)));
    }
}

template <int EPI>
__device__ __forceinline__ double pair_epilogue(double acc, const PairEpi& e) {
    if (EPI == EPI_EXP) return exp(e.s0 * acc);
    if (EPI == EPI_SQRT) return sqrt(acc);
    if (EPI == EPI_ROOT) return pow(acc, e.s0);
    if (EPI == EPI_SARGAN) {
        // qml/fkernels.f90:513-518: sum_m gamma_m (-inv d)^m, then exp(inv d) (1 + sum).
        const double x = -e.s0 * acc;
        double sum = 0.0;
        for (int m = 0; m < e.ng; ++m) sum = sum + e.g[m] * pair_powi(x, m + 1);
        return exp(e.s0 * acc) * (1 + sum);
    }
    if (EPI == EPI_MATERN) {
        // qml/fkernels.f90:442-482 with acc the squared distance.
        const double d = sqrt(acc);
        if (e.order == 0) return exp(e.s0 * d);
        if (e.order == 1) return exp(e.s0 * d) * (1.0 - e.s0 * d);
        return exp(e.s0 * d) * (1.0 - e.s0 * d + e.s1 * acc);
    }
    return acc;
}

// Tile rows: with few 128 x 128 tiles a launch lasts as long as one tile, so 64- and 32-row tiles
// spread it over more CUs, at more operand reads per pair. Laplacian kernel, 276 features, 128- /
// 64- / 32-row tiles: 64 tiles (1000 x 1000) 101 / 60 / 42 us, 121 tiles 105 / 64 / 61, 225 tiles
// 110 / 99 / 110, 576 tiles 240 / 211 / 221, 1024 tiles 339 / 350 / 388. Launches of fewer 128 x 128
// tiles than these take 64- and 32-row ones.
static constexpr int64_t PAIR_TILES_64 = 800, PAIR_TILES_32 = 160;

// LDS of a tile: two buffers of a k-major chunk of each operand.
static constexpr int PT_ELEMS = 2 * 2 * PT_BK * PT_LDS;

// Two doubles at any 8-byte address.
typedef double pt_pair_t __attribute__((ext_vector_type(2), aligned(8)));

// The rows of an operand that a lane loads: features 2 (t % 8) + {0, 1} of the panel's rows
// t / 8 + 32 q (8 lanes cover a row's 128 bytes of a chunk). N = 4 for 128 rows.
template <int N = 4>
struct PairRows {
    const double* p[N];
};

// Rows row0 .. row0 + 32 N - 1 of X; rows past the last one repeat it (their sums are not used).
template <int N = 4>
__device__ __forceinline__ PairRows<N> pair_rows(const double* __restrict__ X, int64_t ld,
                                                 int64_t n, int64_t row0) {
    PairRows<N> R;
#pragma unroll
    for (int q = 0; q < N; ++q) {
        const int64_t r = row0 + (threadIdx.x >> 3) + 32 * q;
        R.p[q] = X + (r < n ? r : n - 1) * ld + 2 * (threadIdx.x & 7);
    }
    return R;
}

// The rows of X listed in idx[0 .. 127] (LDS).
__device__ __forceinline__ PairRows<4> pair_rows_at(const double* __restrict__ X, int64_t ld,
                                                    const int* __restrict__ idx) {
    PairRows<4> R;
#pragma unroll
    for (int q = 0; q < 4; ++q)
        R.p[q] = X + (int64_t)idx[(threadIdx.x >> 3) + 32 * q] * ld + 2 * (threadIdx.x & 7);
    return R;
}

// acc[r][c] = sum over the first d features of term(A(ri(r)), B(cj(c))) with
// ri(r) = 2 tx + 32 (r / 2) + r % 2 and cj(c) = 2 ty + 32 (c / 2) + c % 2; the tile is 16 R rows
// (R = 2, 4, 8) by 128 columns. Has barriers; lds (PT_ELEMS) is free for the caller on return.
// Two FP64 VALU operations per pair and feature bound it. Chunks are double buffered in LDS, one
// barrier each, and their global loads (16 bytes a lane, unconditional: past the last whole chunk
// they repeat it) run two chunks ahead.
template <int OP, int R>
__device__ __forceinline__ void pair_tile_accumulate(double (&acc)[R][8], double* __restrict__ lds,
                                                     const PairRows<R / 2>& A, const PairRows<4>& B,
                                                     int d, double p = 0.0) {
    const int t = threadIdx.x;
    const int tx = t % 16;
    const int ty = t / 16;
    constexpr int PANEL = PT_BK * PT_LDS;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[r][c] = 0.0;
    double* cur = lds;
    double* nxt = lds + 2 * PANEL;
    pt_pair_t ra[R / 2], rb[4];
    auto fetch = [&](int c) {
#pragma unroll
        for (int q = 0; q < R / 2; ++q)
            ra[q] = *reinterpret_cast<const pt_pair_t*>(A.p[q] + c * PT_BK);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            rb[q] = *reinterpret_cast<const pt_pair_t*>(B.p[q] + c * PT_BK);
    };
    auto stash = [&](double* buf) {
        double* s = buf + 2 * (t & 7) * PT_LDS + (t >> 3);
#pragma unroll
        for (int q = 0; q < R / 2; ++q) {
            s[32 * q] = ra[q].x;
            s[32 * q + PT_LDS] = ra[q].y;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            s[32 * q + PANEL] = rb[q].x;
            s[32 * q + PANEL + PT_LDS] = rb[q].y;
        }
    };
    auto feature = [&](const double* buf, int k) {
        double a[R], b[8];
        const double* sa = buf + k * PT_LDS + 2 * tx;
        const double* sb = buf + PANEL + k * PT_LDS + 2 * ty;
#pragma unroll
        for (int r = 0; r < R / 2; ++r) {
            const double2 va = *reinterpret_cast<const double2*>(sa + 32 * r);
            a[2 * r] = va.x;
            a[2 * r + 1] = va.y;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const double2 vb = *reinterpret_cast<const double2*>(sb + 32 * r);
            b[2 * r] = vb.x;
            b[2 * r + 1] = vb.y;
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < 8; ++c) acc[r][c] = pair_term<OP>(acc[r][c], a[r], b[c], p);
    };
    const int whole = d / PT_BK;
    if (whole > 0) {
        fetch(0);
        stash(cur);
        fetch(whole > 1 ? 1 : 0);
        __syncthreads();
#pragma unroll 1
        for (int c = 0; c < whole; ++c) {
            stash(nxt);
            fetch(c + 2 < whole ? c + 2 : whole - 1);
#pragma unroll 2
            for (int k = 0; k < PT_BK; ++k) feature(cur, k);
            __syncthreads();  // every lane has read this chunk and written the next one
            double* swap = cur;
            cur = nxt;
            nxt = swap;
        }
    }
    const int rest = d - whole * PT_BK;
    if (rest > 0) {
        const int k = 2 * (t & 7);
#pragma unroll
        for (int q = 0; q < R / 2; ++q) {
            const double* pa = A.p[q] + whole * PT_BK;
            ra[q].x = k < rest ? pa[0] : 0.0;
            ra[q].y = k + 1 < rest ? pa[1] : 0.0;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double* pb = B.p[q] + whole * PT_BK;
            rb[q].x = k < rest ? pb[0] : 0.0;
            rb[q].y = k + 1 < rest ? pb[1] : 0.0;
        }
        stash(cur);
        __syncthreads();
#pragma unroll 1
        for (int kk = 0; kk < rest; ++kk) feature(cur, kk);
        __syncthreads();
    }
}

}  // namespace qmlh
