// MFMA tile cores shared by the kernel-matrix builds, the Cholesky updates and the predict.
//
// Element types: double on v_mfma_f64_16x16x4f64, float on v_mfma_f32_16x16x4f32. Both take
// one A value and one B value per lane per 4-deep k step: lane l supplies A(l % 16, l / 16)
// and B(l / 16, l % 16). The 16 x 16 result block is 4 values per lane:
//   f64: D(i, j) in lane j + 16 * (i % 4), element i / 4 (rows interleave across lane groups)
//   f32: D(i, j) in lane j + 16 * (i / 4), element i % 4
// (both pinned on gfx950 by the parity tests; MfmaTraits<T>::acc_row encodes them).
//
// Feature permutation: in a 16-deep chunk, lane group g = l / 16 holds features 4g .. 4g+3 and
// MFMA number s (0..3) consumes feature 4g + s. The four MFMAs cover all 16 features once,
// with the same permutation on both operands, so the product is unchanged.
#pragma once

#include "common.h"

namespace qmlh {

enum { LAYOUT_ROW = 0, LAYOUT_COL = 1 };

template <typename T>
struct MfmaTraits;

template <>
struct MfmaTraits<double> {
    typedef double4_t acc_t;
    typedef double2 pair_t;
    static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // c - a b: the FP64 instruction's last modifier negates its operands, bit 0 the first
    static __device__ __forceinline__ acc_t mma_sub(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 1);
    }
    static __device__ __forceinline__ int acc_row(int lane, int e) { return (lane >> 4) + 4 * e; }
};

template <>
struct MfmaTraits<float> {
    typedef float4_t acc_t;
    typedef float2 pair_t;
    static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ acc_t mma_sub(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(-a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int acc_row(int lane, int e) { return 4 * (lane >> 4) + e; }
};

// Operand view: element (i, k) at p[i * ld + k] (ROW) or p[i + k * ld] (COL).
template <typename T, int LAYOUT>
struct Operand {
    const T* __restrict__ p;
    int64_t ld;
    int64_t rows;  // valid rows; row indices are clamped to rows - 1 when loading
    int64_t kdim;  // valid features; features >= kdim read as zero
};

// One wavefront's block: Q x Q MFMA blocks (64 x 64 for Q = 4, 32 x 32 for Q = 2).
template <typename T, int Q = 4>
struct WaveTile {
    typename MfmaTraits<T>::acc_t acc[Q][Q];
};

template <typename T, int Q>
__device__ __forceinline__ void wave_tile_zero(WaveTile<T, Q>& t) {
#pragma unroll
    for (int a = 0; a < Q; ++a)
#pragma unroll
        for (int b = 0; b < Q; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) t.acc[a][b][e] = T(0);
}

// Output row (within the wave's rows of the first operand) of accumulator element e of
// first-operand block a for this lane; the second-operand index is 16 b + (lane & 15).
template <typename T>
__device__ __forceinline__ int tile_row(int a, int e) {
    return 16 * a + MfmaTraits<T>::acc_row(threadIdx.x & 63, e);
}

// ------------------------------------------------------------------------------------------
// Workgroup tile: 256 lanes own 128 x 128 (2 x 2 waves of 64 x 64; 64 x 64 and 32 x 32 for Q = 2,
// four times the workgroups for outputs too small to fill the chip). Both operands are staged
// through LDS in 16-feature chunks, double buffered, and the fragments of a wave's 64 MFMAs per
// chunk are read half a chunk ahead, so that the matrix cores always have the products of one
// half to work on while the other half's fragments arrive, the next chunk's registers go to LDS
// and the waves meet at the chunk's one barrier. Global loads run two chunks ahead and carry no
// condition (row and feature indices are clamped; features past kdim are zeroed on the way to
// LDS, in the last chunk only): a condition would make the compiler wait for each load where
// the branches join.
// LDS layouts of a panel, both free of bank conflicts in either direction:
//   COL (global loads run down the rows): feature k of row r at k * (rows + 4) + r; a lane reads
//       one value per MFMA, the four lane groups 4 * (rows + 4) elements apart (128 bytes modulo
//       256);
//   ROW (global loads run along the features, 8 lanes a row): pair k / 2 of row r at
//       (k / 2) * (2 rows + 4) + 2 r; a lane reads the pair of two MFMAs.
// What bounds it: the FP64 MFMA rate, and for short products the accumulators' way in and out.
// 8192 x 8192 products, 4096 and 448 deep: 66.8 and 62.4 TFLOP/s of the instruction's 78.6 at the
// nominal clock (54.4 and 52.5 with loads under conditions, one chunk ahead, and all of a chunk's
// fragments read behind its barrier). Workgroup orders that give each XCD a contiguous run of
// tiles change it by less than 1 %: the panels' second readers are not what it waits for.
// ------------------------------------------------------------------------------------------
static constexpr int WG_KC = 16;
template <int Q>
struct WgShape {
    static constexpr int ROWS = 32 * Q;            // the tile's side
    static constexpr int COL_S = ROWS + 4;         // elements between features (COL)
    static constexpr int ROW_S = 2 * ROWS + 4;     // elements between feature pairs (ROW)
    static constexpr int PANEL = WG_KC * COL_S;    // elements per operand panel
    static constexpr int LDS = 2 * 2 * PANEL;      // two buffers x two operands
    static_assert(WG_KC / 2 * ROW_S <= PANEL, "either layout fits a panel");
};
static constexpr int WG_T = WgShape<4>::ROWS;
static constexpr int WG_LDS_ELEMS = WgShape<4>::LDS;

template <typename T, int Q>
struct PanelRegs {
    T v[Q][2];  // 32 Q x 16 panel / 256 lanes
};

// Raw buffer view of `bytes` of memory from p on: loads take a uniform base, a uniform offset and
// the lane's 32-bit offset, so an address costs no vector registers beyond that offset. A load
// past the view gives zeros.
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

// A value that is the same in every lane, in scalar registers (tile coordinates go through vector
// instructions, and a buffer view of a vector pointer costs a loop per load).
__device__ __forceinline__ int64_t uniform_i64(int64_t v) {
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_view(const T* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(p), 0, (int)bytes, 0x00027000);
}
template <typename T>
__device__ __forceinline__ T buffer_load(__amdgpu_buffer_rsrc_t b, uint32_t lane_off) {
    if constexpr (sizeof(T) == 8)
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(b, lane_off, 0, 0));
    else
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(b, lane_off, 0, 0));
}
__device__ __forceinline__ void buffer_load2(double (&x)[2], __amdgpu_buffer_rsrc_t b,
                                             uint32_t lane_off, uint32_t off) {
    const double2 v = __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(b, lane_off, off, 0));
    x[0] = v.x;
    x[1] = v.y;
}
__device__ __forceinline__ void buffer_load2(float (&x)[2], __amdgpu_buffer_rsrc_t b,
                                             uint32_t lane_off, uint32_t off) {
    const float2 v = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(b, lane_off, off, 0));
    x[0] = v.x;
    x[1] = v.y;
}

// Loads of a panel: a uniform pointer per chunk, and the lane's byte offsets, the same for every
// chunk (rows clamped to the operand). L = 16 Q lanes hold the rows of one feature (COL).
// COL: lane t holds rows 2(t%L)+{0,1} of features t/L + (16/Q) u.
// ROW: lane holds features 2(t%8)+{0,1} of rows 8 Q (t/64) + 8u + (t%64)/8.
// Pairs are loaded whole (16 bytes at any multiple of 8). Where a panel ends, a lane's pair may
// not start past the last but one row (COL): the lane whose first row is the last one takes the
// pair's second value for it (`last_row`), and a panel of a single row starts one row earlier.
// Operands of one row only (COL), and of a leading dimension whose offsets within a panel pass 32
// bits (from 4.2e6 doubles on for 128 rows), are loaded value by value at 64-bit addresses
// (`by_value`), as the last partial chunk is. LISTED: the panel's rows are listed in LDS (ROW).
template <typename T, int LAYOUT, int Q, bool LISTED = false>
struct PanelLoader {
    typedef WgShape<Q> S;
    static constexpr int L = 16 * Q;   // lanes per feature (COL)
    static constexpr int PW = 64 / L;  // features per wave and load (COL)
    static constexpr int US = 16 / Q;  // features per workgroup and load (COL)
    // the largest leading dimension for 32-bit offsets: 16 features (COL) or a panel's rows and 16
    // features (ROW) span less than 4 GiB
    static constexpr int64_t MAX_LD = ((int64_t)0xffffffff / (int64_t)sizeof(T) - WgShape<4>::ROWS) /
                                      (LAYOUT == LAYOUT_COL ? WG_KC : S::ROWS - 1);
    const T* base;    // chunk 0; COL: the wave's first feature, row 0; ROW: its first feature
    int64_t step;     // elements between features (COL)
    uint32_t off[Q];  // COL: [0] the lane's rows; ROW: per u the lane's row and features
    uint32_t bytes;   // from a chunk's base to the end of its last feature of the panel's last row
    bool last_row;    // COL: the pair's second value is the lane's first row
    bool by_value;
    const T* p;       // feature 0 of the panel's first row; LISTED: of row 0
    int64_t ld;
    int last;         // last row of the panel
    const int* idx;   // LISTED: its rows

    __device__ __forceinline__ PanelLoader(const Operand<T, LAYOUT>& op, int64_t row0) {
        static_assert(!LISTED, "an operand's rows follow each other");
        const int lane = threadIdx.x & 63;
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int64_t rest = op.rows - 1 - row0;  // rows of the panel: 0 .. last
        last = rest < S::ROWS - 1 ? (int)rest : S::ROWS - 1;
        ld = op.ld;
        idx = nullptr;
        by_value = ld > MAX_LD || (LAYOUT == LAYOUT_COL && op.rows == 1);
        if (LAYOUT == LAYOUT_COL) {
            const int back = last == 0 && op.rows > 1 ? 1 : 0;
            const int pair = last + back > 0 ? last + back - 1 : 0;  // last possible pair start
            const int r = 2 * (lane % L);
            p = op.p + uniform_i64(row0);
            base = op.p + uniform_i64(wave * PW * op.ld + row0 - back);
            step = op.ld;
            bytes = (uint32_t)(((WG_KC - 1 - wave * PW) * op.ld + last + 1 + back) * sizeof(T));
            off[0] = (uint32_t)(((r < pair ? r : pair) + (lane / L) * op.ld) * sizeof(T));
            last_row = op.rows > 1 && r + back > pair;
        } else {
            p = op.p + uniform_i64(row0 * op.ld);
            base = p;
            step = 1;
            bytes = (uint32_t)((last * op.ld + WG_KC) * sizeof(T));
#pragma unroll
            for (int u = 0; u < Q; ++u) {
                const int row = 8 * Q * wave + 8 * u + (lane >> 3);
                off[u] = (uint32_t)(((row < last ? row : last) * op.ld + 2 * (lane & 7)) * sizeof(T));
            }
            last_row = false;
        }
    }
    // The rows of X listed in rows[0 .. 32 Q - 1] (LDS), none below `first` (the same in every lane).
    // wide: they span 4 GiB or more. The caller holds them to X: the view's length does not (it
    // would be one more scalar register in kernels that spill them).
    __device__ __forceinline__ PanelLoader(const T* X, int64_t ldx, const int* rows, int first,
                                           bool wide) {
        static_assert(LISTED && LAYOUT == LAYOUT_ROW, "rows are listed for row-major operands");
        const int lane = threadIdx.x & 63;
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        p = X;
        ld = ldx;
        last = S::ROWS - 1;
        idx = rows;
        by_value = wide;
        base = X + uniform_i64(first * ldx);
        step = 1;
        bytes = 0xffffffffu;
#pragma unroll
        for (int u = 0; u < Q; ++u) {
            const int row = 8 * Q * wave + 8 * u + (lane >> 3);
            off[u] = (uint32_t)(((rows[row] - first) * ldx + 2 * (lane & 7)) * sizeof(T));
        }
        last_row = false;
    }
    __device__ __forceinline__ uint32_t lane_off(int u) const {
        return off[LAYOUT == LAYOUT_COL ? 0 : u];
    }
    __device__ __forceinline__ uint32_t group_off(int u) const {
        return LAYOUT == LAYOUT_COL ? (uint32_t)(US * u * step * sizeof(T)) : 0u;
    }
    // Registers <- whole chunk c.
    __device__ __forceinline__ void load(PanelRegs<T, Q>& R, int64_t c) const {
        const __amdgpu_buffer_rsrc_t b = buffer_view(base + c * WG_KC * step, bytes);
#pragma unroll
        for (int u = 0; u < Q; ++u) buffer_load2(R.v[u], b, lane_off(u), group_off(u));
    }
    // Registers <- the first k <= 16 features of chunk c, value by value, zeros after.
    __device__ __forceinline__ void load_some(PanelRegs<T, Q>& R, int64_t c, int k) const {
        const int lane = threadIdx.x & 63;
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
        for (int u = 0; u < Q; ++u) {
            R.v[u][0] = T(0);
            R.v[u][1] = T(0);
            if (LAYOUT == LAYOUT_COL) {
                const int f = wave * PW + lane / L + US * u, r = 2 * (lane % L);
                const T* x = p + (c * WG_KC + f) * ld;
                if (f < k) {
                    R.v[u][0] = x[r < last ? r : last];
                    R.v[u][1] = x[r + 1 < last ? r + 1 : last];
                }
            } else {
                const int f = 2 * (lane & 7), row = 8 * Q * wave + 8 * u + (lane >> 3);
                if (LISTED && !by_value) {  // nothing kept for it but the offsets
                    const __amdgpu_buffer_rsrc_t b = buffer_view(base + c * WG_KC, bytes);
                    if (f < k) R.v[u][0] = buffer_load<T>(b, off[u]);
                    if (f + 1 < k) R.v[u][1] = buffer_load<T>(b, off[u] + (uint32_t)sizeof(T));
                    continue;
                }
                const T* x = p + (LISTED ? idx[row] : row < last ? row : last) * ld + c * WG_KC + f;
                if (f < k) R.v[u][0] = x[0];
                if (f + 1 < k) R.v[u][1] = x[1];
            }
        }
    }
    // LDS panel <- registers.
    __device__ __forceinline__ void store(T* __restrict__ panel, const PanelRegs<T, Q>& R) const {
        typedef typename MfmaTraits<T>::pair_t P2;
        const int lane = threadIdx.x & 63;
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
        for (int u = 0; u < Q; ++u) {
            P2 v;
            v.x = LAYOUT == LAYOUT_COL && last_row ? R.v[u][1] : R.v[u][0];
            v.y = R.v[u][1];
            const int at = LAYOUT == LAYOUT_COL
                               ? (wave * PW + lane / L + US * u) * S::COL_S + 2 * (lane % L)
                               : (lane & 7) * S::ROW_S + 2 * (8 * Q * wave + 8 * u + (lane >> 3));
            *reinterpret_cast<P2*>(panel + at) = v;
        }
    }
};

// A wave's operand values of half a chunk: MFMAs s = 2h, 2h + 1 of blocks 0 .. 3.
template <typename T, int Q>
struct HalfFrag {
    T v[Q][2];
};

template <typename T, int LAYOUT, int Q>
__device__ __forceinline__ void half_frag_read(HalfFrag<T, Q>& f, const T* __restrict__ panel,
                                               int row0, int h) {
    typedef typename MfmaTraits<T>::pair_t P2;
    typedef WgShape<Q> S;
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        if (LAYOUT == LAYOUT_COL) {
            const T* p = panel + (4 * g + 2 * h) * S::COL_S + row0 + 16 * q + r;
            f.v[q][0] = p[0];
            f.v[q][1] = p[S::COL_S];
        } else {
            const P2 v = *reinterpret_cast<const P2*>(panel + (2 * g + h) * S::ROW_S +
                                                      2 * (row0 + 16 * q + r));
            f.v[q][0] = v.x;
            f.v[q][1] = v.y;
        }
    }
}

template <bool SUB, typename T, int Q>
__device__ __forceinline__ void half_mma(WaveTile<T, Q>& t, const HalfFrag<T, Q>& fa,
                                         const HalfFrag<T, Q>& fb) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int a = 0; a < Q; ++a)
#pragma unroll
            for (int b = 0; b < Q; ++b)
                t.acc[a][b] = SUB ? MfmaTraits<T>::mma_sub(fa.v[a][e], fb.v[b][e], t.acc[a][b])
                                  : MfmaTraits<T>::mma(fa.v[a][e], fb.v[b][e], t.acc[a][b]);
}

// t += F S^T for the panels of two loaders, 32 Q rows each, restricted to this wave's 16 Q x 16 Q
// block (t -= ... with SUB: the first operand is negated, which is exact): wave w owns rows
// 16 Q (w & 1) of the first and 16 Q (w >> 1) of the second. `lds` holds WgShape<Q>::LDS
// elements. All 256 lanes must call this (it has barriers).
template <bool SUB, typename T, int LF, int LS, int Q, bool GF, bool GS>
__device__ __forceinline__ void wg_tile_mma_panels(WaveTile<T, Q>& t, T* __restrict__ lds,
                                                   const PanelLoader<T, LF, Q, GF>& lf,
                                                   const PanelLoader<T, LS, Q, GS>& ls,
                                                   int64_t kdim) {
    if (kdim <= 0) return;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = 16 * Q * (w & 1);
    const int sr = 16 * Q * (w >> 1);
    constexpr int WG_PANEL = WgShape<Q>::PANEL;
    const int64_t whole = lf.by_value || ls.by_value ? 0 : kdim / WG_KC;
    PanelRegs<T, Q> pf, ps;
    T* cur = lds;
    T* nxt = lds + 2 * WG_PANEL;
    if (whole > 0) {
        // Loads, stores and reads are unconditional (past the last chunk they repeat it): under
        // a condition their results would be copied, and waited for, where the branches join.
        lf.load(pf, 0);
        ls.load(ps, 0);
        lf.store(cur, pf);
        ls.store(cur + WG_PANEL, ps);
        lf.load(pf, whole > 1 ? 1 : 0);
        ls.load(ps, whole > 1 ? 1 : 0);
        __syncthreads();
        HalfFrag<T, Q> fa0, fb0, fa1, fb1;
        half_frag_read<T, LF, Q>(fa0, cur, fr, 0);
        half_frag_read<T, LS, Q>(fb0, cur + WG_PANEL, sr, 0);
#pragma unroll 1
        for (int64_t c = 0; c < whole; ++c) {
            const int64_t c2 = c + 2 < whole ? c + 2 : whole - 1;
            half_frag_read<T, LF, Q>(fa1, cur, fr, 1);
            half_frag_read<T, LS, Q>(fb1, cur + WG_PANEL, sr, 1);
            lf.store(nxt, pf);
            ls.store(nxt + WG_PANEL, ps);
            lf.load(pf, c2);
            ls.load(ps, c2);
            half_mma<SUB>(t, fa0, fb0);
            // the fence keeps the wait and the barrier behind the half's products
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();  // every wave has read this chunk and written the next one
            half_frag_read<T, LF, Q>(fa0, nxt, fr, 0);
            half_frag_read<T, LS, Q>(fb0, nxt + WG_PANEL, sr, 0);
            // ... and these reads ahead of the other half's (not merged with the prologue's into
            // one place at the top of the loop)
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            half_mma<SUB>(t, fa1, fb1);
            T* swap = cur;
            cur = nxt;
            nxt = swap;
        }
        __syncthreads();
    }
    // the rest of the features, chunk by chunk (one partial chunk, or all of them by value)
#pragma unroll 1
    for (int64_t k0 = whole * WG_KC; k0 < kdim; k0 += WG_KC) {
        const int k = kdim - k0 < WG_KC ? (int)(kdim - k0) : WG_KC;
        lf.load_some(pf, k0 / WG_KC, k);
        ls.load_some(ps, k0 / WG_KC, k);
        lf.store(cur, pf);
        ls.store(cur + WG_PANEL, ps);
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            HalfFrag<T, Q> fa, fb;
            half_frag_read<T, LF, Q>(fa, cur, fr, h);
            half_frag_read<T, LS, Q>(fb, cur + WG_PANEL, sr, h);
            half_mma<SUB>(t, fa, fb);
        }
        __syncthreads();  // also: the caller may reuse lds
    }
}

// The same for rows f0 .. and s0 .. of two operands.
template <typename T, int LF, int LS, bool SUB = false, int Q = 4>
__device__ __forceinline__ void wg_tile_mma_lds(WaveTile<T, Q>& t, T* __restrict__ lds,
                                                const Operand<T, LF>& F,
                                                const Operand<T, LS>& S, int64_t f0, int64_t s0,
                                                int64_t kdim) {
    if (kdim <= 0) return;
    wg_tile_mma_panels<SUB>(t, lds, PanelLoader<T, LF, Q>(F, f0), PanelLoader<T, LS, Q>(S, s0),
                            kdim);
}

// ------------------------------------------------------------------------------------------
// Accumulators <-> a column-major C block: element e of block (a, b) of this lane is
// C(row0 + 16 b + (lane & 15), col0 + tile_row(a, e)) (first operand = output columns).
// `live`: the wave's block has entries to update; `interior`: every entry of its block
// is inside the M x N matrix (and on or below the diagonal when LOWER), so no masks are needed
// and all loads are issued back to back. Masked entries load as zero and are not stored.
// ------------------------------------------------------------------------------------------
template <typename T, bool LOWER, int Q>
__device__ __forceinline__ void wave_tile_load_c(WaveTile<T, Q>& t, const T* __restrict__ C,
                                                 int64_t ldc, int64_t row0, int64_t col0,
                                                 int64_t M, int64_t N, bool live, bool interior) {
    const int lane = threadIdx.x & 63;
    if (interior) {
#pragma unroll
        for (int a = 0; a < Q; ++a)
#pragma unroll
            for (int b = 0; b < Q; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    t.acc[a][b][e] = C[(row0 + 16 * b + (lane & 15)) + (col0 + tile_row<T>(a, e)) * ldc];
        return;
    }
#pragma unroll
    for (int a = 0; a < Q; ++a)
#pragma unroll
        for (int b = 0; b < Q; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t i = row0 + 16 * b + (lane & 15);
                const int64_t j = col0 + tile_row<T>(a, e);
                const bool ok = live && i < M && j < N && (!LOWER || j <= i);
                t.acc[a][b][e] = ok ? C[i + j * ldc] : T(0);
            }
}

template <typename T, bool LOWER, int Q>
__device__ __forceinline__ void wave_tile_store_c(const WaveTile<T, Q>& t, T* __restrict__ C,
                                                  int64_t ldc, int64_t row0, int64_t col0,
                                                  int64_t M, int64_t N, bool interior) {
    const int lane = threadIdx.x & 63;
    if (interior) {
#pragma unroll
        for (int a = 0; a < Q; ++a)
#pragma unroll
            for (int b = 0; b < Q; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    C[(row0 + 16 * b + (lane & 15)) + (col0 + tile_row<T>(a, e)) * ldc] = t.acc[a][b][e];
        return;
    }
#pragma unroll
    for (int a = 0; a < Q; ++a)
#pragma unroll
        for (int b = 0; b < Q; ++b) {
            const int64_t i = row0 + 16 * b + (lane & 15);
            if (i >= M) continue;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t j = col0 + tile_row<T>(a, e);
                if (j >= N || (LOWER && j > i)) continue;
                C[i + j * ldc] = t.acc[a][b][e];
            }
        }
}

}  // namespace qmlh
