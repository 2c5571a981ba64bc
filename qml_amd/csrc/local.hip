// Local (atom-summed) kernels between molecules:
//   K_s(a, b) = sum over atoms i of molecule a, j of molecule b of exp(inv_s * D(x_i, y_j))
// the quantity of fget_local_kernels_gaussian / fget_local_kernels_laplacian
// (qml/fkernels.f90:23-196) and of fget_vector_kernels_* (qml/fkernels.f90:198-337) behind the
// atomic-kernel wrappers, for several sigmas from one distance tile.
//
// Molecules are grouped into panels of molecules that follow each other in a given order (the
// caller's, by default their index), holding at most LK_TILE atoms and LK_MOLS molecules (a
// molecule larger than LK_TILE atoms is a panel of its own), so that every molecule pair belongs
// to exactly one panel pair and each output entry is written once, by one workgroup, without
// atomics. Atom representations are padded to the largest molecule with trailing zeros, so a
// panel pair's distances need only the features up to the last nonzero one of either panel
// (local_feature_counts_kernel; products: of both): the skipped terms are zeros, which leave every
// sum as it is. Panels of molecules ordered by size make that worth having -- of 5 to 23 atoms,
// size 23 (276 features), the mean over
// panel pairs is 199 features for differences and 105 for products, against 264 and 230 in random
// order. 4,000 such molecules, Gaussian by differences, three widths: 42.9 -> 33.5 ms; 3,000 x 701,
// Laplacian: 9.98 -> 7.50 ms. (Without padding to skip, an order only makes more panels and scatters
// their rows, 5 to 40 % of a call: the caller weighs that, from qmlh_local_feature_counts.) A workgroup computes the atom-pair distance tile of its panel
// pair (128 x 128 atoms: FP64 MFMA expanded form for the Gaussian, the FP64 VALU direct tile
// for the Laplacian and the direct Gaussian), applies exp for each sigma, and reduces the tile
// to molecule-pair sums with two small MFMA products against 0/1 membership matrices:
//   T = V * Sb^T (atom rows x panel molecules of B),  S = Sa * T (molecules of A x of B),
// where Sa(m, i) = [atom i of the tile belongs to the panel's molecule m]. Padding atoms (past
// the panel's end) have no molecule, so ragged panels need no masks. Products with 0 and 1 are
// exact; the sums run in the matrix cores' fixed order, so results are deterministic.
// The four waves' partial sums meet in LDS in wave order (one barrier per wave), then the
// workgroup writes its molecule pairs. For a symmetric call (the same molecules on both sides)
// only panel pairs P <= Q run and every value is mirrored, so K_s is exactly symmetric.
#include "mfma_core.h"
#include "pair_tile.h"
#include "timer.h"

#include <float.h>

#include <vector>

namespace qmlh {

static constexpr int LK_TILE = 128;
static constexpr int LK_MOLS = QMLH_LOCAL_PANEL_MOLS;  // molecules per panel: one MFMA block
static constexpr int LK_NS = 4;                         // sigmas per launch
static_assert(LK_MOLS == 16, "one 16-wide MFMA block of molecules per panel side");

// Workgroups per launch; larger panel-pair counts are covered by a grid-stride loop.
static constexpr int64_t LK_MAX_GRID = 1 << 20;
static constexpr int LK_COUNT_LANES = 1024;
static constexpr int64_t LK_COUNT_PAIRS = QMLH_LOCAL_COUNT_PAIRS;

// LK_GAUSS_WIDE: the expanded form for rows whose offsets within a tile pass 32 bits.
enum { LK_GAUSS_MFMA = 0, LK_GAUSS_VALU = 1, LK_LAPLACE = 2, LK_GAUSS_WIDE = 3 };

struct LkSide {
    const double* X;
    int64_t ld;
    const double* norms;     // squared row norms (MFMA Gaussian only)
    const int64_t* offsets;  // (nmol + 1) atom offsets
    const int64_t* panels;   // (npanels + 1) first place of each panel in the order
    const int64_t* order;    // (nmol) molecule at each place; null: its index
    const int32_t* count;    // (npanels) leading features that hold every nonzero; null: all
    int64_t atoms;           // total atoms (rows of X): no row beyond them is read
};

// Set in a panel's feature count: some value of the panel is not finite.
static constexpr int32_t LK_NOT_FINITE = 1 << 30;

// Features a panel pair's distances need. Differences (PRODUCT false): those that either panel
// has; products: those that both have (0 times a finite value is 0; not so for infinities and NaN,
// and then all of them are taken).
template <bool PRODUCT>
__device__ __forceinline__ int lk_features(const LkSide& A, const LkSide& B, int bi, int bj,
                                           int64_t d) {
    if (!A.count || !B.count) return (int)d;
    const int ca = A.count[bi], cb = B.count[bj];
    if (PRODUCT && ((ca | cb) & LK_NOT_FINITE)) return (int)d;
    const int a = ca & ~LK_NOT_FINITE, b = cb & ~LK_NOT_FINITE;
    const int f = PRODUCT ? (a < b ? a : b) : (a > b ? a : b);
    return f < d ? f : (int)d;
}

// count[panel] := 1 + the last feature that is not zero in any of the panel's atom rows, for the
// panels of side A and then of side B. With norms (products), LK_NOT_FINITE is set where one of the
// panel's is not finite, as it is when a value is not (and when finite ones overflow it: then all
// features are taken without need). One workgroup per panel, four wavefronts per molecule and four
// molecules at a time: a wavefront's rows are one memory latency after the other. Rows are read from
// the end up to their last nonzero feature; a kernel per side that read all of them to see whether
// they are finite took 20,000 molecules of 276 features from 618 (Laplacian) to 631 ms and from
// 253 (Gaussian) to 255.
__global__ __launch_bounds__(LK_COUNT_LANES) void local_feature_counts_kernel(
    LkSide A, int64_t npA, LkSide B, int64_t npB, int64_t d, int32_t* __restrict__ count) {
    constexpr int WAVES = LK_COUNT_LANES / 64;
    __shared__ int s_last[WAVES], s_bad[WAVES];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int64_t p = blockIdx.x; p < npA + npB; p += gridDim.x) {
        const LkSide& S = p < npA ? A : B;
        const int64_t panel = p < npA ? p : p - npA;
        int last = 0, bad = 0;  // per wave
        for (int64_t m = S.panels[panel] + wave / 4; m < S.panels[panel + 1]; m += WAVES / 4) {
            const int64_t mol = S.order ? S.order[m] : m;
            for (int64_t r = S.offsets[mol] + wave % 4; r < S.offsets[mol + 1]; r += 4) {
                const double* x = S.X + r * S.ld;
                if (S.norms) bad |= !(fabs(S.norms[r]) <= DBL_MAX);
                // from the end, 64 features at a time, no further than `last`
                for (int64_t k0 = (d - 1) / 64 * 64; k0 >= 0 && k0 + 64 > last; k0 -= 64) {
                    const int64_t k = k0 + lane;
                    const double v = k < d ? x[k] : 0.0;
                    const unsigned long long nz = __ballot(v != 0.0);
                    if (nz) {
                        const int top = (int)k0 + 64 - __builtin_clzll(nz);
                        last = top > last ? top : last;
                        break;
                    }
                }
            }
        }
        if (lane == 0) {
            s_last[wave] = last;
            s_bad[wave] = bad;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            int l = s_last[0], b = s_bad[0];
            for (int w = 1; w < WAVES; ++w) {
                l = s_last[w] > l ? s_last[w] : l;
                b |= s_bad[w];
            }
            count[p] = l | (b ? LK_NOT_FINITE : 0);
        }
        __syncthreads();
    }
}

struct LkSigmas {
    double inv[4];  // exp argument scale per sigma of this launch
    int n;          // sigmas in this launch (<= LK_NS)
    int64_t first;  // index of inv[0] in the caller's list
};

__device__ __forceinline__ uint32_t lk_byte(uint32_t p, int i) { return (p >> (8 * i)) & 0xffu; }

// sg.inv[s] without a dynamic index into the by-value argument (which would go to scratch).
__device__ __forceinline__ double lk_inv(const LkSigmas& sg, int s) {
    return s == 0 ? sg.inv[0] : s == 1 ? sg.inv[1] : s == 2 ? sg.inv[2] : sg.inv[3];
}

// One side of a panel pair in LDS.
struct LkPanel {
    int mol[LK_MOLS];        // its molecules
    int first[LK_MOLS];      // their first atom rows
    int soff[LK_MOLS + 1];   // atoms of the panel before each molecule, and in all
    int lowest;              // the lowest of the first atom rows
    int slot[LK_TILE];       // tile: the panel molecule of each atom, -1 past the last one
    int row[LK_TILE];        // tile: its row of X (past the last one: the last one's)
};

// Molecules of panel `p` (nm of them), their atoms held to the rows of X; lanes 0 .. 63 of a wave
// call it, a barrier follows.
__device__ __forceinline__ void lk_panel_mols(LkPanel& P, const LkSide& S, int p, int nm) {
    const int m = threadIdx.x & 63;
    int n = 0, low = 0x7fffffff;
    if (m < nm) {
        const int64_t at = S.panels[p] + m;
        const int64_t mol = S.order ? S.order[at] : at;
        int64_t a0 = S.offsets[mol], a1 = S.offsets[mol + 1];
        a0 = a0 < 0 ? 0 : a0;
        a1 = a1 < S.atoms ? a1 : S.atoms;
        n = a1 > a0 ? (int)(a1 - a0) : 0;
        P.mol[m] = (int)mol;
        P.first[m] = (int)a0;
        low = (int)a0;
    }
#pragma unroll
    for (int s = 1; s < LK_MOLS; s <<= 1) {
        const int v = __shfl_xor(low, s, 64);
        low = v < low ? v : low;
    }
    // inclusive sums over the molecules
#pragma unroll
    for (int s = 1; s < LK_MOLS; s <<= 1) {
        const int v = __shfl_up(n, s, 64);
        if (m >= s) n += v;
    }
    if (m < nm) P.soff[m + 1] = n;
    if (m == 0) {
        P.soff[0] = 0;
        P.lowest = low;
    }
}

// Atoms a0 .. a0 + LK_TILE - 1 of the panel; 128 lanes (t) call it, a barrier follows.
__device__ __forceinline__ void lk_panel_atoms(LkPanel& P, int nm, int a0, int t) {
    const int total = P.soff[nm];
    const int a = a0 + t;
    const int c = a < total ? a : total - 1;
    int lo = 0;
    for (int m = 1; m < nm; ++m)
        if (P.soff[m] <= c) lo = m;
    P.slot[t] = a < total ? lo : -1;
    P.row[t] = P.first[lo] + (c - P.soff[lo]);
}

// Loader of a tile's rows. In the molecules' own order they follow each other from the first one
// on; in another they are less than 4 GiB in all (checked by the host).
typedef PanelLoader<double, LAYOUT_ROW, 4, true> LkRows;
template <bool WIDE>
__device__ __forceinline__ LkRows lk_rows(const LkPanel& P, const LkSide& S) {
    return LkRows(S.X, S.ld, P.row, S.order ? P.lowest : P.row[0], WIDE);
}

// Add this wave's molecule-pair sums of one sigma to S.
// Lane layout shared by both tile kinds: value val(r, c) belongs to tile row rowof(r, lane & 15)
// and tile column colof(c, lane >> 4); byte e of rpack[r] is the panel molecule of tile row
// rowof(r, (lane >> 4) + 4e), byte c % 4 of cpack[c / 4] that of tile column colof(c, lane >> 4)
// (0xff: padding, matching no molecule).
// Stage 1, per row set r: T(m, n) = sum_c val(r, c) [cmol[c] = n] (16 rows x 16 molecules);
// stage 2: S(ma, n) += sum_e [rmol[r][e] = ma] T((lane >> 4) + 4e, n).
template <int NR, int NC, typename Val>
__device__ __forceinline__ void lk_reduce(Val val, const uint32_t (&rpack)[NR],
                                          const uint32_t (&cpack)[NC / 4], double4_t& S) {
    typedef MfmaTraits<double> M;
    const uint32_t me = threadIdx.x & 15;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        double4_t T = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int c = 0; c < NC; ++c)
            T = M::mma(val(r, c), lk_byte(cpack[c / 4], c % 4) == me ? 1.0 : 0.0, T);
#pragma unroll
        for (int e = 0; e < 4; ++e) S = M::mma(lk_byte(rpack[r], e) == me ? 1.0 : 0.0, T[e], S);
    }
}

// acc[ma][n] += S in wave order (one barrier per wave); lane element e holds
// S((lane >> 4) + 4e, lane & 15).
__device__ __forceinline__ void lk_accumulate(double* __restrict__ acc, const double4_t& S) {
    const int lane = threadIdx.x & 63;
    const int w = threadIdx.x >> 6;
    for (int w2 = 0; w2 < 4; ++w2) {
        if (w == w2) {
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[((lane >> 4) + 4 * e) * LK_MOLS + (lane & 15)] += S[e];
        }
        __syncthreads();
    }
}

template <int KIND>
__global__ __launch_bounds__(256, 2) void local_kernels_kernel(LkSide A, LkSide B, int64_t d,
                                                               LkSigmas sg, double* __restrict__ K,
                                                               int64_t ldk, int64_t sstride,
                                                               int symmetric, int tiles_a,
                                                               int ntiles) {
    constexpr bool WIDE = KIND == LK_GAUSS_WIDE, PRODUCT = KIND == LK_GAUSS_MFMA || WIDE;
    __shared__ __attribute__((aligned(16))) double lds[PRODUCT ? WG_LDS_ELEMS : PT_ELEMS];
    __shared__ double acc[LK_NS][LK_MOLS * LK_MOLS];
    __shared__ LkPanel PA, PB;

    const int t = threadIdx.x;
    const int lane = t & 63;
    const int w = t >> 6;

    // Atom, molecule and panel indices fit in 32 bits (checked by the host); fewer 64-bit
    // values keep the scalar registers from spilling.
    for (int bid = blockIdx.x; bid < ntiles; bid += gridDim.x) {
        int bi, bj;
        if (symmetric) {
            int64_t j = (int64_t)((sqrt(8.0 * (double)bid + 1.0) - 1.0) * 0.5);
            while (j * (j + 1) / 2 > bid) --j;
            while ((j + 1) * (j + 2) / 2 <= bid) ++j;
            bj = (int)j;
            bi = (int)(bid - j * (j + 1) / 2);
        } else {
            bi = bid % tiles_a;
            bj = bid / tiles_a;
        }
        const int nma = (int)(A.panels[bi + 1] - A.panels[bi]);
        const int nmb = (int)(B.panels[bj + 1] - B.panels[bj]);
        // Panels come from qmlh_local_panels; one with more molecules than the LDS sums hold
        // is skipped rather than overrunning them.
        if (nma > LK_MOLS || nmb > LK_MOLS || nma < 0 || nmb < 0) continue;

        for (int q = t; q < LK_NS * LK_MOLS * LK_MOLS; q += 256) (&acc[0][0])[q] = 0.0;
        if (w == 0) lk_panel_mols(PA, A, bi, nma);
        else if (w == 1) lk_panel_mols(PB, B, bj, nmb);
        __syncthreads();
        const int atoms_a = PA.soff[nma], atoms_b = PB.soff[nmb];
        const int feats = lk_features<PRODUCT>(A, B, bi, bj, d);

        for (int r0 = 0; r0 < atoms_a; r0 += LK_TILE) {
            for (int c0 = 0; c0 < atoms_b; c0 += LK_TILE) {
                if (t < LK_TILE) lk_panel_atoms(PA, nma, r0, t);
                else lk_panel_atoms(PB, nmb, c0, t - LK_TILE);
                __syncthreads();
                if (PRODUCT) {
                    WaveTile<double> tile;
                    wave_tile_zero(tile);
                    wg_tile_mma_panels<false>(tile, lds, lk_rows<WIDE>(PB, B), lk_rows<WIDE>(PA, A),
                                              feats);
                    // Lane value (a, b, e): tile row 64 (w >> 1) + 16 b + (lane & 15),
                    // column 64 (w & 1) + 16 a + (lane >> 4) + 4 e.
                    const int rbase = 64 * (w >> 1), cbase = 64 * (w & 1);
                    uint32_t rpack[4], cpack[4];
                    double ni[4], nj[16];
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        ni[b] = A.norms[PA.row[rbase + 16 * b + (lane & 15)]];
                        uint32_t p = 0;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            p |= (uint32_t)(PA.slot[rbase + 16 * b + (lane >> 4) + 4 * e] & 0xff) << (8 * e);
                        rpack[b] = p;
                    }
#pragma unroll
                    for (int a = 0; a < 4; ++a) {
                        uint32_t p = 0;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int cl = cbase + 16 * a + (lane >> 4) + 4 * e;
                            nj[4 * a + e] = B.norms[PB.row[cl]];
                            p |= (uint32_t)(PB.slot[cl] & 0xff) << (8 * e);
                        }
                        cpack[a] = p;
                    }
                    double d2[4][16];
#pragma unroll
                    for (int b = 0; b < 4; ++b)
#pragma unroll
                        for (int a = 0; a < 4; ++a)
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const double x = ni[b] + nj[4 * a + e] - 2.0 * tile.acc[a][b][e];
                                d2[b][4 * a + e] = x > 0.0 ? x : 0.0;
                            }
#pragma unroll 1
                    for (int s = 0; s < sg.n; ++s) {
                        const double inv = lk_inv(sg, s);
                        double4_t S = {0.0, 0.0, 0.0, 0.0};
                        lk_reduce<4, 16>([&](int r, int c) { return exp(inv * d2[r][c]); },
                                         rpack, cpack, S);
                        lk_accumulate(acc[s], S);
                    }
                } else {
                    double dist[8][8];
                    // Tile rows 2 tx + 32 (r / 2) + r % 2, columns 2 ty + 32 (c / 2) + c % 2
                    // with tx = lane & 15, ty = 4 w + (lane >> 4).
                    if (KIND == LK_LAPLACE)
                        pair_tile_accumulate<OP_L1, 8>(dist, lds, pair_rows_at(A.X, A.ld, PA.row),
                                                       pair_rows_at(B.X, B.ld, PB.row), feats);
                    else
                        pair_tile_accumulate<OP_SQ, 8>(dist, lds, pair_rows_at(A.X, A.ld, PA.row),
                                                       pair_rows_at(B.X, B.ld, PB.row), feats);
                    uint32_t rpack[8], cpack[2];
#pragma unroll
                    for (int r = 0; r < 8; ++r) {
                        uint32_t p = 0;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            p |= (uint32_t)(PA.slot[2 * ((lane >> 4) + 4 * e) + 32 * (r / 2) + r % 2] & 0xff)
                                 << (8 * e);
                        rpack[r] = p;
                    }
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        uint32_t p = 0;
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const int c = 4 * q + u;
                            p |= (uint32_t)(PB.slot[2 * (4 * w + (lane >> 4)) + 32 * (c / 2) + c % 2] & 0xff)
                                 << (8 * u);
                        }
                        cpack[q] = p;
                    }
#pragma unroll 1
                    for (int s = 0; s < sg.n; ++s) {
                        const double inv = lk_inv(sg, s);
                        double4_t S = {0.0, 0.0, 0.0, 0.0};
                        lk_reduce<8, 8>([&](int r, int c) { return exp(dist[r][c] * inv); },
                                        rpack, cpack, S);
                        lk_accumulate(acc[s], S);
                    }
                }
            }
        }
        __syncthreads();

        // Write the panel pair's molecule sums; mirror for a symmetric call.
        const bool diag = symmetric && bi == bj;
        for (int s = 0; s < sg.n; ++s) {
            double* Ks = K + (sg.first + s) * sstride;
            for (int q = t; q < LK_MOLS * LK_MOLS; q += 256) {
                const int ma = q % LK_MOLS, mb = q / LK_MOLS;
                if (ma >= nma || mb >= nmb) continue;
                if (diag && ma > mb) continue;
                const double val = acc[s][ma * LK_MOLS + mb];
                const int64_t ga = PA.mol[ma], gb = PB.mol[mb];
                Ks[ga + gb * ldk] = val;
                if (symmetric && ga != gb) Ks[gb + ga * ldk] = val;
            }
        }
        __syncthreads();
    }
}

template <int KIND>
static void lk_launch(int64_t ntiles, hipStream_t s, const LkSide& A, const LkSide& B,
                      int64_t d, const LkSigmas& sg, double* K, int64_t ldk, int64_t sstride,
                      int symmetric, int64_t tiles_a) {
    const int64_t grid = ntiles < LK_MAX_GRID ? ntiles : LK_MAX_GRID;
    hipLaunchKernelGGL((local_kernels_kernel<KIND>), dim3((unsigned)grid), dim3(256), 0, s, A,
                       B, d, sg, K, ldk, sstride, symmetric, (int)tiles_a, (int)ntiles);
}

}  // namespace qmlh

extern "C" int64_t qmlh_local_panels(const int64_t* offsets_h, int64_t nmol, int64_t* panels_h) {
    using namespace qmlh;
    if (nmol < 0 || !offsets_h || !panels_h)
        return set_error(QMLH_ERR_ARG, "local_panels: bad arguments");
    int64_t np = 0;
    panels_h[0] = 0;
    int64_t start = 0;
    while (start < nmol) {
        int64_t m = start;
        const int64_t a0 = offsets_h[start];
        if (offsets_h[start + 1] < a0) return set_error(QMLH_ERR_ARG, "local_panels: offsets decrease");
        // Take molecules while the panel stays within LK_TILE atoms and LK_MOLS molecules; a
        // first molecule larger than LK_TILE atoms is a panel alone.
        ++m;
        if (offsets_h[m] - a0 <= LK_TILE) {
            while (m < nmol && m - start < LK_MOLS && offsets_h[m + 1] - a0 <= LK_TILE) {
                if (offsets_h[m + 1] < offsets_h[m])
                    return set_error(QMLH_ERR_ARG, "local_panels: offsets decrease");
                ++m;
            }
        }
        panels_h[++np] = m;
        start = m;
    }
    return np;
}

namespace qmlh {

static void launch_counts(const LkSide& A, int64_t npA, const LkSide& B, int64_t npB, int64_t d,
                          int32_t* counts, hipStream_t s) {
    const int64_t panels = npA + npB, most = 16384;
    hipLaunchKernelGGL(local_feature_counts_kernel, dim3((unsigned)(panels < most ? panels : most)),
                       dim3(LK_COUNT_LANES), 0, s, A, npA, B, npB, d, counts);
}

// counts: (npA + npB) int32 for the panels' feature counts, or null to use all features.
static int local_kernels(int32_t kind, const double* A, int64_t atomsA, int64_t lda,
                         const double* normsA, const int64_t* offsA, const int64_t* panelsA,
                         const int64_t* orderA, int64_t npA, const double* B, int64_t atomsB,
                         int64_t ldb, const double* normsB, const int64_t* offsB,
                         const int64_t* panelsB, const int64_t* orderB, int64_t npB, int64_t d,
                         const double* sigmas_h, int32_t nsig, double* K, int64_t ldk,
                         int64_t sstride, int32_t flags, int32_t* counts, qmlh_stream_t stream) {
    if (kind != QMLH_PAIR_GAUSSIAN && kind != QMLH_PAIR_LAPLACIAN)
        return set_error(QMLH_ERR_ARG, "local_kernels: kind %d", kind);
    if (npA < 0 || npB < 0 || atomsA < 0 || atomsB < 0 || d < 0 || nsig < 0)
        return set_error(QMLH_ERR_ARG, "local_kernels: negative size");
    if (lda < d || ldb < d) return set_error(QMLH_ERR_ARG, "local_kernels: ld < d");
    if (npA == 0 || npB == 0 || nsig == 0) return QMLH_OK;
    if (!offsA || !offsB || !panelsA || !panelsB || !K || !sigmas_h)
        return set_error(QMLH_ERR_ARG, "local_kernels: null pointer");
    if ((atomsA > 0 && !A) || (atomsB > 0 && !B))
        return set_error(QMLH_ERR_ARG, "local_kernels: null representation");
    const bool symmetric = (flags & QMLH_SYMMETRIC) != 0;
    if (symmetric && (A != B || offsA != offsB || panelsA != panelsB || orderA != orderB ||
                      npA != npB))
        return set_error(QMLH_ERR_ARG, "local_kernels: symmetric call needs identical sides");
    const bool mfma = kind == QMLH_PAIR_GAUSSIAN && normsA && normsB;
    if (kind == QMLH_PAIR_GAUSSIAN && (normsA != nullptr) != (normsB != nullptr))
        return set_error(QMLH_ERR_ARG, "local_kernels: give both norms or neither");
    for (int32_t s = 0; s < nsig; ++s)
        if (!(sigmas_h[s] > 0.0)) return set_error(QMLH_ERR_ARG, "local_kernels: sigma <= 0");
    // the matrix-core path addresses a panel's rows by 32-bit byte offsets
    if (mfma && ((orderA && (uint64_t)atomsA * lda >= ((uint64_t)1 << 29)) ||
                 (orderB && (uint64_t)atomsB * ldb >= ((uint64_t)1 << 29))))
        return set_error(QMLH_ERR_ARG, "local_kernels: the expanded form takes ordered "
                                       "molecules of less than 4 GiB");
    LkSide sa{A, lda, normsA, offsA, panelsA, orderA, nullptr, atomsA};
    LkSide sb{B, ldb, normsB, offsB, panelsB, orderB, nullptr, atomsB};
    const int64_t grid = symmetric ? npA * (npA + 1) / 2 : npA * npB;
    if (grid > 0x7fffffffLL || atomsA > 0x7fffffffLL - LK_TILE || atomsB > 0x7fffffffLL - LK_TILE)
        return set_error(QMLH_ERR_ARG, "local_kernels: more than 2^31 atoms or panel pairs");
    hipStream_t s = (hipStream_t)stream;
    // Work: atom pairs x features (the pairs of a symmetric call counted once).
    const double pairs = symmetric ? 0.5 * (double)atomsA * (double)(atomsA + 1)
                                   : (double)atomsA * (double)atomsB;
    TimerScope ts(QMLH_TIMER_LOCAL, pairs * (double)d, s);
    // Up to LK_COUNT_PAIRS panel pairs run as one round of workgroups, which lasts as long as its
    // largest molecules' pair whatever the others skip: 100 x 50 molecules, Laplacian, 144 us with
    // the counts and 119 without; 400 x 20, two widths, 164 and 130. 3,000 x 701: 6.97 ms with
    // counts by 16 wavefronts a panel, 7.11 by four.
    if (counts && (symmetric ? npA * (npA + 1) / 2 : npA * npB) > LK_COUNT_PAIRS) {
        launch_counts(sa, npA, sb, symmetric ? 0 : npB, d, counts, s);
        QMLH_CHECK_LAUNCH("local_kernels feature counts launch");
        sa.count = counts;
        sb.count = symmetric ? counts : counts + npA;
    }
    for (int32_t s0 = 0; s0 < nsig; s0 += LK_NS) {
        LkSigmas sg;
        sg.n = nsig - s0 < LK_NS ? (int)(nsig - s0) : LK_NS;
        sg.first = s0;
        for (int q = 0; q < LK_NS; ++q) {
            const double sig = sigmas_h[s0 + (q < sg.n ? q : 0)];
            sg.inv[q] = kind == QMLH_PAIR_GAUSSIAN ? -0.5 / (sig * sig) : -1.0 / sig;
        }
        const int sym = symmetric ? 1 : 0;
        if (mfma && ((!orderA && lda > LkRows::MAX_LD) || (!orderB && ldb > LkRows::MAX_LD)))
            lk_launch<LK_GAUSS_WIDE>(grid, s, sa, sb, d, sg, K, ldk, sstride, sym, npA);
        else if (mfma) lk_launch<LK_GAUSS_MFMA>(grid, s, sa, sb, d, sg, K, ldk, sstride, sym, npA);
        else if (kind == QMLH_PAIR_GAUSSIAN)
            lk_launch<LK_GAUSS_VALU>(grid, s, sa, sb, d, sg, K, ldk, sstride, sym, npA);
        else lk_launch<LK_LAPLACE>(grid, s, sa, sb, d, sg, K, ldk, sstride, sym, npA);
        QMLH_CHECK_LAUNCH("local_kernels launch");
    }
    return QMLH_OK;
}

}  // namespace qmlh

extern "C" int qmlh_local_kernels(int32_t kind, const double* A, int64_t atomsA, int64_t lda,
                                  const double* normsA, const int64_t* offsA,
                                  const int64_t* panelsA, int64_t npA, const double* B,
                                  int64_t atomsB, int64_t ldb, const double* normsB,
                                  const int64_t* offsB, const int64_t* panelsB, int64_t npB,
                                  int64_t d, const double* sigmas_h, int32_t nsig, double* K,
                                  int64_t ldk, int64_t sstride, int32_t flags,
                                  qmlh_stream_t stream) {
    return qmlh::local_kernels(kind, A, atomsA, lda, normsA, offsA, panelsA, nullptr, npA, B,
                               atomsB, ldb, normsB, offsB, panelsB, nullptr, npB, d, sigmas_h,
                               nsig, K, ldk, sstride, flags, nullptr, stream);
}

extern "C" int qmlh_local_feature_counts(const double* A, int64_t atomsA, int64_t lda,
                                         const int64_t* offsA, const int64_t* panelsA,
                                         const int64_t* orderA, int64_t npA, int64_t d,
                                         int32_t* counts, qmlh_stream_t stream) {
    using namespace qmlh;
    if (npA < 0 || atomsA < 0 || d < 0 || lda < d)
        return set_error(QMLH_ERR_ARG, "local_feature_counts: bad shape");
    if (npA == 0) return QMLH_OK;
    if ((atomsA > 0 && !A) || !offsA || !panelsA || !counts)
        return set_error(QMLH_ERR_ARG, "local_feature_counts: null pointer");
    const LkSide side{A, lda, nullptr, offsA, panelsA, orderA, nullptr, atomsA};
    launch_counts(side, npA, side, 0, d, counts, (hipStream_t)stream);
    QMLH_CHECK_LAUNCH("local_feature_counts launch");
    return QMLH_OK;
}

extern "C" size_t qmlh_local_kernels_workspace(int64_t npA, int64_t npB) {
    return npA > 0 && npB > 0 ? (size_t)(npA + npB) * sizeof(int32_t) : 0;
}

extern "C" int qmlh_local_kernels_ordered(
    int32_t kind, const double* A, int64_t atomsA, int64_t lda, const double* normsA,
    const int64_t* offsA, const int64_t* panelsA, const int64_t* orderA, int64_t npA,
    const double* B, int64_t atomsB, int64_t ldb, const double* normsB, const int64_t* offsB,
    const int64_t* panelsB, const int64_t* orderB, int64_t npB, int64_t d, const double* sigmas_h,
    int32_t nsig, double* K, int64_t ldk, int64_t sstride, int32_t flags, void* ws,
    size_t ws_bytes, qmlh_stream_t stream) {
    using namespace qmlh;
    if (ws_bytes < qmlh_local_kernels_workspace(npA, npB) ||
        (!ws && qmlh_local_kernels_workspace(npA, npB) > 0))
        return set_error(QMLH_ERR_WORKSPACE, "local_kernels_ordered: workspace too small");
    return local_kernels(kind, A, atomsA, lda, normsA, offsA, panelsA, orderA, npA, B, atomsB, ldb,
                         normsB, offsB, panelsB, orderB, npB, d, sigmas_h, nsig, K, ldk, sstride,
                         flags, static_cast<int32_t*>(ws), stream);
}
