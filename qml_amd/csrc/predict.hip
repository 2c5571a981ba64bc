// Fused KRR prediction: y_q = sum_j k(q, x_j) alpha_j without materialising the kernel,
// the Ks.T.dot(alpha) step of tests/test_energy_krr_cmat.py:108-109.
//
// Batch invariance: the training set is cut into fixed chunks of 128 rows; a workgroup reduces one
// chunk for a block of queries in an order that depends only on the training index, writes one
// partial per (chunk, query), and a second kernel adds the partials of a query in an order that
// depends only on their number. Nothing in a query's arithmetic depends on the other queries or
// on m, so a query's result is bitwise the same alone or in a batch, also where a batch takes
// other tiles: they differ in which workgroup computes what, not in the order of any sum.
#include <mutex>

#include "mfma_core.h"
#include "pair_tile.h"
#include "timer.h"

namespace qmlh {

static constexpr int P_T = 128;      // training rows per chunk
static constexpr int PG_Q = 64;      // queries per Gaussian workgroup
static constexpr int PG_FEW = 16;    // and where there are no more than these

// The Gaussian's chunk sum: units of 32 training rows (two MFMA blocks), each summed by a lane
// over its 8 accumulator entries in (block, element) order, then over the lanes that share the
// query (l, l ^ 16, l ^ 32); the chunk adds its 4 units in order.
__device__ __forceinline__ double gauss_unit_sum(const double4_t& lo, const double4_t& hi,
                                                 int64_t t0, int64_t n, double nq,
                                                 const double* __restrict__ nT,
                                                 const double* __restrict__ alpha, double scale) {
    const int g = (threadIdx.x & 63) >> 4;
    double s = 0.0;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int64_t j = t0 + 16 * a + g + 4 * e;
            if (j < n) {
                double d2 = nq + nT[j] - 2.0 * (a ? hi[e] : lo[e]);
                d2 = d2 > 0.0 ? d2 : 0.0;
                s = fma(exp(scale * d2), alpha[j], s);
            }
        }
    s = s + __shfl_xor(s, 16, 64);
    return s + __shfl_xor(s, 32, 64);
}

template <int NQ>
__device__ __forceinline__ void gauss_chunk_sums(const double (&unit)[4][NQ], int64_t q0, int64_t m,
                                                 int64_t chunk, double* __restrict__ part) {
    const int qi = threadIdx.x;
    if (qi < NQ && q0 + qi < m)
        part[chunk * m + q0 + qi] = ((unit[0][qi] + unit[1][qi]) + unit[2][qi]) + unit[3][qi];
}

// Gaussian, blocks of 64 queries: the cross term on the FP64 matrix cores (64 x 64 tiles, the
// chunk as two of them), FP64 epilogue, per-chunk partials part[chunk * m + q]. Bound by the FP64
// MFMA rate: 512 queries x 50,000 rows x 435 features 423 us = 52.7
// TFLOP/s (760 with operands straight from memory in 64 x 64 blocks per wave).
__global__ __launch_bounds__(256, 4) void predict_gauss_kernel(
    const double* __restrict__ Q, int64_t ldq, int64_t m, const double* __restrict__ nQ,
    const double* __restrict__ T, int64_t ldt, int64_t n, const double* __restrict__ nT,
    const double* __restrict__ alpha, int64_t d, double scale, double* __restrict__ part) {
    static_assert(WgShape<2>::ROWS == PG_Q && 2 * PG_Q == P_T, "a chunk is two tiles");
    __shared__ __attribute__((aligned(16))) double lds[WgShape<2>::LDS];
    __shared__ double unit[4][PG_Q];
    const int64_t q0 = (int64_t)blockIdx.x * PG_Q;
    const int64_t chunk = blockIdx.y;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    Operand<double, LAYOUT_ROW> opT{T, ldt, n, d};
    Operand<double, LAYOUT_ROW> opQ{Q, ldq, m, d};
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
        const int64_t t0 = chunk * P_T + 64 * half;
        const int u = 2 * half + (w & 1), qb = 32 * (w >> 1);
        WaveTile<double, 2> t;
        wave_tile_zero(t);
        // First operand: training rows (accumulator rows), second: queries (columns).
        if (t0 < n) wg_tile_mma_lds<double, LAYOUT_ROW, LAYOUT_ROW>(t, lds, opT, opQ, t0, q0, d);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int64_t q = q0 + qb + 16 * b + (lane & 15);
            const double s = gauss_unit_sum(t.acc[0][b], t.acc[1][b], t0 + 32 * (w & 1), n,
                                            nQ[q < m ? q : m - 1], nT, alpha, scale);
            if (lane < 16) unit[u][qb + 16 * b + lane] = s;
        }
    }
    __syncthreads();
    gauss_chunk_sums<PG_Q>(unit, q0, m, chunk, part);
}

// Gaussian, at most 16 queries in all: bound by reading the training set, so the operands go
// straight from memory to the matrix cores, a wavefront's 32 rows in groups of 64 features with
// the next group's 24 loads of 16 bytes a lane in flight. One query x 50,000 rows: 43 us = 4.1
// TB/s, against 117 in 64-query tiles.
__global__ __launch_bounds__(256, 2) void predict_gauss_few_kernel(
    const double* __restrict__ Q, int64_t ldq, int64_t m, const double* __restrict__ nQ,
    const double* __restrict__ T, int64_t ldt, int64_t n, const double* __restrict__ nT,
    const double* __restrict__ alpha, int64_t d, double scale, double* __restrict__ part) {
    __shared__ double unit[4][PG_FEW];
    const int64_t chunk = blockIdx.x;
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t t0 = chunk * P_T + 32 * w;
    double sum = 0.0;
    if (t0 < n) {
        // rows: two blocks of training rows, the queries; lane (r, g): features 4 g .. of row r
        const double* p[3];
        p[0] = T + (t0 + r < n ? t0 + r : n - 1) * ldt;
        p[1] = T + (t0 + 16 + r < n ? t0 + 16 + r : n - 1) * ldt;
        p[2] = Q + (r < m ? r : m - 1) * ldq;
        // group i: features 64 i + 16 c + 4 g + {0 .. 3}, zero from d on (rows hold an even
        // number of values, so a pair that starts below d can be read whole)
        pt_pair_t v[2][4][3][2];
        const int ng = (int)((d + 63) / 64);
        const int last = (int)((d - 1) & ~(int64_t)1);
        auto fetch = [&](pt_pair_t (&x)[4][3][2], int i) {
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int k = 64 * i + 16 * c + 4 * g + 2 * h;
                    const int ks = k < last ? k : last;
#pragma unroll
                    for (int o = 0; o < 3; ++o)
                        x[c][o][h] = *reinterpret_cast<const pt_pair_t*>(p[o] + ks);
                }
        };
        double4_t acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = {0.0, 0.0, 0.0, 0.0};
        auto multiply = [&](pt_pair_t (&x)[4][3][2], int i) {
            if (i == ng - 1) {
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int k = 64 * i + 16 * c + 4 * g + 2 * h;
#pragma unroll
                        for (int o = 0; o < 3; ++o) {
                            if (k >= d) x[c][o][h].x = 0.0;
                            if (k + 1 >= d) x[c][o][h].y = 0.0;
                        }
                    }
            }
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const double q = s & 1 ? x[c][2][s >> 1].y : x[c][2][s >> 1].x;
                    const double a0 = s & 1 ? x[c][0][s >> 1].y : x[c][0][s >> 1].x;
                    const double a1 = s & 1 ? x[c][1][s >> 1].y : x[c][1][s >> 1].x;
                    acc0 = MfmaTraits<double>::mma(a0, q, acc0);
                    acc1 = MfmaTraits<double>::mma(a1, q, acc1);
                }
        };
        if (ng > 0) {
            fetch(v[0], 0);
#pragma unroll 1
            for (int i = 0; i < ng; i += 2) {
                fetch(v[1], i + 1 < ng ? i + 1 : ng - 1);
                multiply(v[0], i);
                fetch(v[0], i + 2 < ng ? i + 2 : ng - 1);
                if (i + 1 < ng) multiply(v[1], i + 1);
            }
        }
        sum = gauss_unit_sum(acc0, acc1, t0, n, nQ[r < m ? r : m - 1], nT, alpha, scale);
    }
    if (lane < 16) unit[w][lane] = sum;
    __syncthreads();
    gauss_chunk_sums<PG_FEW>(unit, 0, m, chunk, part);
}

// Laplacian: the pairwise kernel's VALU L1 tile, 16 R queries by a chunk of training rows; exp *
// alpha, per-chunk partials (a lane's 8 training columns in order, then the 16 lanes of a query).
// 2,000 queries x 20,000 rows x 435 features: 1.26 ms = 0.70 of the FP64 VALU.
template <int R>
__global__ __launch_bounds__(256, 2) void predict_laplace_kernel(
    const double* __restrict__ Q, int64_t ldq, int64_t m, const double* __restrict__ T,
    int64_t ldt, int64_t n, const double* __restrict__ alpha, int64_t d, double scale,
    double* __restrict__ part) {
    constexpr int NQ = 16 * R;
    static_assert(P_T == PT_BN, "a chunk is the tile's columns");
    __shared__ __attribute__((aligned(16))) double lds[PT_ELEMS];
    static_assert(PT_ELEMS >= 16 * NQ, "the row sums take the tile's place");
    double (*red)[NQ] = reinterpret_cast<double (*)[NQ]>(lds);
    const int64_t row0 = (int64_t)blockIdx.x * NQ;  // queries
    const int64_t chunk = blockIdx.y;
    const int64_t col0 = chunk * P_T;  // training rows
    const int t = threadIdx.x;
    const int tx = t % 16, ty = t / 16;
    double acc[R][8];
    pair_tile_accumulate<OP_L1, R>(acc, lds, pair_rows<R / 2>(Q, ldq, m, row0),
                                   pair_rows(T, ldt, n, col0), (int)d);
    // Row sums over this lane's 8 training columns, in column order.
#pragma unroll
    for (int r = 0; r < R; ++r) {
        double s = 0.0;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int64_t j = col0 + 2 * ty + 32 * (c / 2) + (c % 2);
            if (j < n) s = fma(exp(scale * acc[r][c]), alpha[j], s);
        }
        red[ty][2 * tx + 32 * (r / 2) + (r % 2)] = s;
    }
    __syncthreads();
    if (t < NQ) {
        const int64_t q = row0 + t;
        if (q < m) {
            double s = 0.0;
            for (int g = 0; g < 16; ++g) s = s + red[g][t];
            part[chunk * m + q] = s;
        }
    }
}

// y[q] = the sum of query q's partials: 16 lanes a query, lane i the chunks i, i + 16, .. in order,
// then the 16 lane sums in order. (One lane a query waited for each of its loads' sums: 17 us for
// one query and 391 chunks, 49 us for 512, against 6 and 6.)
__global__ __launch_bounds__(256) void predict_reduce_kernel(const double* __restrict__ part,
                                                             int64_t m, int64_t nchunks,
                                                             double* __restrict__ y) {
    __shared__ double red[16][17];
    const int qi = threadIdx.x & 15, i = threadIdx.x >> 4;
    for (int64_t q0 = (int64_t)blockIdx.x * 16; q0 < m; q0 += (int64_t)gridDim.x * 16) {
        const int64_t q = q0 + qi;
        const double* p = part + (q < m ? q : m - 1);
        double s = 0.0;
#pragma unroll 8
        for (int64_t c = i; c < nchunks; c += 16) s = s + p[c * m];
        red[i][qi] = s;
        __syncthreads();
        if (i == 0 && q < m) {
            double v = red[0][qi];
            for (int k = 1; k < 16; ++k) v = v + red[k][qi];
            y[q] = v;
        }
        __syncthreads();  // the sums are read before the next queries'
    }
}

__global__ void zero_kernel(double* __restrict__ y, int64_t m) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < m) y[q] = 0.0;
}

// ------------------------------------------------------------------------------------------
// Scratch of qmlh_krr_predict_noalloc: the per-(chunk, query) partials in a file-scope device
// array instead of a caller's workspace. Each GPU holds its own copy for the life of the
// process; host code reaches it only through the address hipGetSymbolAddress returns for the
// current device (the array's name on the host is a stand-in, not a device address).
// ------------------------------------------------------------------------------------------
static constexpr int64_t PREDICT_SCRATCH_DOUBLES = (int64_t)2 << 20;  // 16 MiB
static __device__ __align__(256) double scratch[PREDICT_SCRATCH_DOUBLES];

static constexpr int MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static double* g_scratch_ptr[MAX_DEVICES] = {};

// Resolve (once per device) the current device's copy of the scratch array.
int predict_scratch_setup(double** out) {
    int dev = 0;
    QMLH_TRY(check_hip(hipGetDevice(&dev), "predict scratch: hipGetDevice"));
    if (dev < 0 || dev >= MAX_DEVICES)
        return set_error(QMLH_ERR_ARG, "predict scratch: device %d beyond %d", dev, MAX_DEVICES);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        QMLH_TRY(check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)),
                           "predict scratch: hipGetSymbolAddress"));
        if (!p) return set_error(QMLH_ERR_HIP, "predict scratch: null symbol address");
        g_scratch_ptr[dev] = static_cast<double*>(p);
    }
    if (out) *out = g_scratch_ptr[dev];
    return QMLH_OK;
}

size_t predict_workspace_bytes(int64_t m, int64_t n) {
    if (m <= 0 || n <= 0) return 0;
    return (size_t)(ceil_div(n, P_T) * m) * sizeof(double);
}

// The prediction with its partials in `part` (at least predict_workspace_bytes(m, n)).
static int predict_impl(int32_t kind, const double* Xq, int64_t m, int64_t ldq,
                        const double* normsQ, const double* Xt, int64_t n, int64_t ldt,
                        const double* normsT, const double* alpha, int64_t d, double sigma,
                        double* y, double* part, hipStream_t s) {
    if (n == 0) {  // empty training set: y = 0 (a kernel, not a memset, so capture is safe)
        hipLaunchKernelGGL(zero_kernel, dim3((unsigned)ceil_div(m, 256)), dim3(256), 0, s, y, m);
        QMLH_CHECK_LAUNCH("krr_predict zero launch");
        return QMLH_OK;
    }
    const int64_t nchunks = ceil_div(n, P_T);
    TimerScope ts(QMLH_TIMER_PREDICT, (double)m * (double)n, s);
    if (kind == QMLH_PAIR_GAUSSIAN) {
        const double scale = -0.5 / (sigma * sigma);
        if (m <= PG_FEW)
            hipLaunchKernelGGL(predict_gauss_few_kernel, dim3((unsigned)nchunks), dim3(256), 0, s,
                               Xq, ldq, m, normsQ, Xt, ldt, n, normsT, alpha, d, scale, part);
        else
            hipLaunchKernelGGL(predict_gauss_kernel,
                               dim3((unsigned)ceil_div(m, PG_Q), (unsigned)nchunks), dim3(256), 0,
                               s, Xq, ldq, m, normsQ, Xt, ldt, n, normsT, alpha, d, scale, part);
    } else {
        // Query rows per tile: no more than the queries need, and small tiles where few of the
        // large ones would leave CUs idle (the pairwise kernels' lines; whole call with 4 queries,
        // 2,952 rows: 209 us on 128-row tiles, 132 on 32).
        const int64_t tiles = ceil_div(m, 128) * nchunks;
        const int R = m <= 32 || tiles < PAIR_TILES_32 ? 2 : m <= 64 || tiles < PAIR_TILES_64 ? 4 : 8;
        auto kernel = R == 2 ? predict_laplace_kernel<2>
                             : R == 4 ? predict_laplace_kernel<4> : predict_laplace_kernel<8>;
        hipLaunchKernelGGL(kernel, dim3((unsigned)ceil_div(m, 16 * R), (unsigned)nchunks),
                           dim3(256), 0, s, Xq, ldq, m, Xt, ldt, n, alpha, d, -1.0 / sigma, part);
    }
    QMLH_CHECK_LAUNCH("krr_predict launch");
    const int64_t sums = ceil_div(m, 16) < MAX_GRID ? ceil_div(m, 16) : MAX_GRID;
    hipLaunchKernelGGL(predict_reduce_kernel, dim3((unsigned)sums), dim3(256), 0, s, part, m,
                       nchunks, y);
    QMLH_CHECK_LAUNCH("krr_predict reduce launch");
    return QMLH_OK;
}

// Argument checks shared by both entry points (everything but the workspace).
static int predict_check(int32_t kind, const double* Xq, int64_t m, int64_t ldq,
                         const double* normsQ, const double* Xt, int64_t n, int64_t ldt,
                         const double* normsT, const double* alpha, int64_t d, double* y,
                         const char* who) {
    if (m < 0 || n < 0 || d < 0) return set_error(QMLH_ERR_ARG, "%s: negative size", who);
    if (ldq < d || ldt < d) return set_error(QMLH_ERR_ARG, "%s: ld < d", who);
    if (kind != QMLH_PAIR_GAUSSIAN && kind != QMLH_PAIR_LAPLACIAN)
        return set_error(QMLH_ERR_ARG, "%s: kind must be Gaussian or Laplacian", who);
    if (m == 0) return QMLH_OK;
    if (!y) return set_error(QMLH_ERR_ARG, "%s: null pointer", who);
    if (n == 0) return QMLH_OK;
    if (!Xq || !Xt || !alpha) return set_error(QMLH_ERR_ARG, "%s: null pointer", who);
    if (kind == QMLH_PAIR_GAUSSIAN) {
        if (ldq % 4 || ldt % 4)
            return set_error(QMLH_ERR_ARG, "%s: ldq, ldt must be multiples of 4", who);
        if (!normsQ || !normsT) return set_error(QMLH_ERR_ARG, "%s: norms missing", who);
    }
    return QMLH_OK;
}

}  // namespace qmlh

extern "C" size_t qmlh_predict_workspace(int64_t m, int64_t n) {
    return qmlh::predict_workspace_bytes(m, n);
}

extern "C" int qmlh_krr_predict(int32_t kind, const double* Xq, int64_t m, int64_t ldq,
                                const double* normsQ, const double* Xt, int64_t n, int64_t ldt,
                                const double* normsT, const double* alpha, int64_t d,
                                double sigma, double* y, void* ws, size_t ws_bytes,
                                qmlh_stream_t stream) {
    using namespace qmlh;
    QMLH_TRY(predict_check(kind, Xq, m, ldq, normsQ, Xt, n, ldt, normsT, alpha, d, y,
                           "krr_predict"));
    if (m == 0) return QMLH_OK;
    if (n > 0 && (ws_bytes < predict_workspace_bytes(m, n) || !ws))
        return set_error(QMLH_ERR_WORKSPACE, "krr_predict: workspace too small");
    return predict_impl(kind, Xq, m, ldq, normsQ, Xt, n, ldt, normsT, alpha, d, sigma, y,
                        static_cast<double*>(ws), (hipStream_t)stream);
}

extern "C" size_t qmlh_krr_predict_noalloc_capacity(void) {
    return (size_t)qmlh::PREDICT_SCRATCH_DOUBLES * sizeof(double);
}

extern "C" int qmlh_krr_predict_noalloc(int32_t kind, const double* Xq, int64_t m, int64_t ldq,
                                        const double* normsQ, const double* Xt, int64_t n,
                                        int64_t ldt, const double* normsT, const double* alpha,
                                        int64_t d, double sigma, double* y,
                                        qmlh_stream_t stream) {
    using namespace qmlh;
    QMLH_TRY(predict_check(kind, Xq, m, ldq, normsQ, Xt, n, ldt, normsT, alpha, d, y,
                           "krr_predict_noalloc"));
    if (m == 0) return QMLH_OK;
    const size_t need = predict_workspace_bytes(m, n);
    if (need > qmlh_krr_predict_noalloc_capacity())
        return set_error(QMLH_ERR_ARG,
                         "krr_predict_noalloc: %lld queries x %lld training rows need %zu bytes "
                         "of scratch, above its %zu (ceil(n / 128) * m <= %lld)",
                         (long long)m, (long long)n, need, qmlh_krr_predict_noalloc_capacity(),
                         (long long)PREDICT_SCRATCH_DOUBLES);
    double* part = nullptr;
    QMLH_TRY(predict_scratch_setup(&part));
    return predict_impl(kind, Xq, m, ldq, normsQ, Xt, n, ldt, normsT, alpha, d, sigma, y, part,
                        (hipStream_t)stream);
}
