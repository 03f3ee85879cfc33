// Kriging sums on gfx950: field and variance term of every target point.
//
//   w_k      = M v_k                      (M = krig_mat (K, K), v_k = column k of krig_vecs (K, P))
//   field_k  = cond . w_k
//   error_k  = v_k . w_k                  (variance form only)
//
// Reference contract: the external calc_field_krige(_and_variance)
// (src/gstools/krige/base.py:42-61, called at :307-317); the caller turns
// error into the kriging variance max(sill - error, 0).
//
// Field (both forms): field = (M^T cond) . v_k: a weight vector a (K), then a sum
// over the rows of V in four classes j mod 4, each in steps of 16 rows from the last step
// down, up within a step, added as (0 + 1) + (2 + 3).  The variance form takes it from the rows of V that the
// GEMM stages anyway (a pass over V saved); k_krige_field adds the same numbers
// in the same order, so the field's bits do not depend on the form or on P.
//
// Variance form: error_k = v_k^T M v_k = v_k^T S v_k with S = (M + M^T) / 2
// (the antisymmetric part of M adds nothing to a quadratic form), and with S
// symmetric only the blocks on and right of the diagonal are needed:
//
//   error_k = sum over row blocks r of  v_r^T (M2 V)_r,
//   M2 = S on the diagonal 32 x 32 blocks, 2 S = M + M^T right of them,
//
// so the GEMM W = M2 V runs, for the 32 rows from 32 r on, over the columns from
// 32 r on: about K^2 P flops instead of 2 K^2 P.  Every block owns a 128-row x
// 128-point tile of W, accumulates it on the matrix cores (v_mfma_f64_16x16x4,
// 4 waves in a 2 x 2 arrangement, each four 16-row fragments, every other one of
// the tile's eight, x 64 points, 16 MFMA tiles at 2 waves per SIMD) and reduces
// V o W over its 128 rows into a per-row-tile partial sum (W is never stored).  A
// second kernel adds the partials of the row tiles in a fixed order (bitwise
// reproducible).  Operand tiles (128 x 16 of M2, 16 x 128 of V) are staged
// through LDS with the next stage prefetched into registers.
//
// Bound by the FP64 matrix cores, and on few points by the last round of blocks.
// Field and variance term of 40000 points, K = 301: 299 us with 128 x 128 diagonal
// blocks, pairs of row tiles per block and the field as a pass of its own, 135 without,
// and 117 with staging reads that check nothing (but in the first stage) and the
// epilogue's reads of V in batches; K = 1001 onto 400000: 9.17 -> 8.00 -> 7.11 ms.  Field alone, K = 301 onto 40000: 97 -> 23 us.
//
// Right-hand sides: k_krige_cov writes the covariance rows of V,
// C(|c_i - x_p|) for conditioning points c_i and targets x_p, for models
// with closed-form correlations (the reference evaluates
// model.cov_nugget / model.covariance on scipy's cdist, krige/base.py:357-388;
// the distance here is rounded the same way: differences, squares and sums
// in dimension order, no fused multiply-add).
//
// MFMA operand layouts (v_mfma_f64_16x16x4, 64 lanes, g = lane / 16):
//   A: lane holds row (lane % 16), K element g
//   B: lane holds column (lane % 16), K element g
//   C: lane holds column (lane % 16), rows g, g+4, g+8, g+12 (register r holds
//      row g + 4r; unlike the 16-bit 16x16 MFMAs, whose lanes hold rows 4g..4g+3)
#include "gsx_internal.h"

namespace gsx {

typedef __attribute__((ext_vector_type(4))) double f64x4;

constexpr int kKrRows = 128;  // W rows per block
constexpr int kKrRF = kKrRows / 32;  // 16-row MFMA tiles per wave (two row waves)
constexpr int kKrPts = 128;   // points per block
constexpr int kKrK = 16;      // reduction depth per LDS stage
constexpr int kKrApad = kKrK + 2;  // 16-byte aligned rows, operand reads over all banks
// B rows padded by 16 doubles: the operand reads of K groups g and g + 1
// (rows 144 doubles apart) fall in disjoint LDS banks
constexpr int kKrBpad = kKrPts + 16;

// M2 of the variance form, padded to Rp = 128 * row tiles rows and Kp (K
// rounded up to a multiple of 16) columns, row stride Kp: row i keeps its
// columns from its diagonal block (32 rows) on, zero beyond K (the GEMM's A loads
// then need no bounds checks); the entries left of it reach no product and are not
// written
constexpr int kKrDiag = 32;  // rows per diagonal block: two 16-row fragments, one per row wave
inline int64_t krige_kp(int64_t K) { return ceil_div(K, (int64_t)kKrK) * kKrK; }

// Blocks [0, ceil(K / 64)): a_j = sum_i cond_i M[i, j] for 64 columns, 16 waves of
// every 16th row, added in order.  The blocks after them (variance form): M2.  Both
// read M once and neither waits for the other, so one launch serves them (three took
// 4.5 us each).  first: the launch's first block.
__global__ __launch_bounds__(1024) void k_krige_prepare(int64_t first, int64_t K, int64_t Rp, int64_t Kp,
                                                        const double* __restrict__ M,
                                                        const double* __restrict__ cond, double* __restrict__ a,
                                                        double* __restrict__ M2) {
    __shared__ double red[16][64];
    const int64_t wblocks = (K + 63) / 64;
    const int64_t block = first + blockIdx.x;
    if (block < wblocks) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const int64_t j = block * 64 + lane;
        double s = 0.0;
        if (j < K) {
#pragma unroll 8
            for (int64_t i = wave; i < K; i += 16) s += cond[i] * M[i * K + j];
        }
        red[wave][lane] = s;
        __syncthreads();
        if (wave == 0 && j < K) {
            double r = 0.0;
#pragma unroll
            for (int w = 0; w < 16; ++w) r += red[w][lane];
            a[j] = r;
        }
        return;
    }
    const int64_t idx = (block - wblocks) * 1024 + threadIdx.x;
    if (idx >= Rp * Kp) return;
    const int64_t i = idx / Kp, l = idx - i * Kp;
    const int64_t b0 = (i / kKrDiag) * kKrDiag;
    if (l < b0) return;
    if (i >= K || l >= K) {
        M2[idx] = 0.0;
        return;
    }
    const double s = M[i * K + l] + M[l * K + i];
    M2[idx] = l < b0 + kKrDiag ? 0.5 * s : s;
}

// W = M2 V over the columns from each diagonal block on (K steps in descending
// order); per-row-tile partial sums of V o W; from row tile 0, which passes over
// every row of V, the field.  The staging loads are 16 bytes wide: A (the padded
// M2, row stride Kp) four per thread with no bounds checks; B as point pairs
// (kPairB: P even and V 16-byte aligned), else one point of eight rows per thread.
//
// Row tile r runs about K - 128 r K steps; the blocks of all column tiles' longest
// row tile come first, so the short ones fill the last round.  (Pairs of row tiles
// (u, R - 1 - u) in one block, equally long and one after the other on an XCD so that
// its L2 keeps the column's V, were slower at every size from 1001 x 400000 (8.15
// against 8.00 ms) down to 301 x 40000 (189 against 135 us).)
template <bool kPairB>
__global__ __launch_bounds__(256, 2) void k_krige_gemm(int64_t K, int64_t Kp, int64_t P, int64_t row_tiles,
                                                    int64_t col_tiles, const double* __restrict__ M,
                                                    const double* __restrict__ V,
                                                    const double* __restrict__ wgt,
                                                    double* __restrict__ part_e, double* __restrict__ field) {
    typedef __attribute__((ext_vector_type(2))) double f64x2;
    __shared__ __align__(16) double As[kKrRows * kKrApad];
    __shared__ __align__(16) double Bs[kKrK * kKrBpad];
    __shared__ double red[4][kKrPts];  // [row wave][point], or [row class][point] of the field

    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int wr = __builtin_amdgcn_readfirstlane(wave >> 1), wc = wave & 1;
    const int g = lane >> 4, l16 = lane & 15;
    // XCD-aware order: dispatch puts block b on XCD b % 8, and the grid has R * C8
    // blocks, C8 = col_tiles rounded up to a multiple of 8, so all row tiles of a column
    // tile run on one XCD; padding blocks leave
    const int64_t c8 = (col_tiles + 7) / 8 * 8;
    const int64_t rt_idx = (int64_t)blockIdx.x / c8, ct_idx = (int64_t)blockIdx.x - rt_idx * c8;
    if (ct_idx >= col_tiles) return;  // whole block: before any barrier
    const int64_t p0 = ct_idx * kKrPts;
    const int64_t i0 = rt_idx * kKrRows;

    // staging assignment: A kKrRows x kKrK, 8 consecutive doubles of one row per
    // thread (four 16-byte loads from the padded M2); B kKrK x 128, either point
    // pair (t % 64) * 2 of rows t / 64 + 4u (16-byte loads and LDS stores) or
    // point t % 128 of rows t / 128 + 2u (unit-stride, conflict-free stores)
    static_assert(kKrRows == 128 && kKrK == 16, "staging assignment");
    const int ar = t >> 1, ac = (t & 1) * 8;
    const f64x2* arow = reinterpret_cast<const f64x2*>(M + (i0 + ar) * Kp + ac);
    const int br = __builtin_amdgcn_readfirstlane(kPairB ? t >> 6 : t >> 7);
    const int bc = kPairB ? (t & 63) * 2 : t & 127;
    // columns past P are read from a clamped address and not stored; rows past K, in the first
    // stage only, are zero
    const double* vcol = V + (p0 + bc < P ? p0 + bc : (kPairB ? P - 2 : P - 1)) + br * P;
    f64x2 pa[4];
    f64x2 pb2[4];   // point pairs (P even: a pair is whole or out of range)
    double pb1[8];  // single points
    auto load = [&](int64_t j0, bool whole) {
#pragma unroll
        for (int v = 0; v < 4; ++v) pa[v] = arow[(j0 >> 1) + v];
#pragma unroll
        for (int u = 0; u < (kPairB ? 4 : 8); ++u) {
            const int64_t j = j0 + (kPairB ? 4 : 2) * u;  // row less br
            const bool in = whole || j + br < K;
            if constexpr (kPairB)
                pb2[u] = in ? *reinterpret_cast<const f64x2*>(vcol + j * P) : f64x2{0.0, 0.0};
            else
                pb1[u] = in ? vcol[j * P] : 0.0;
        }
    };
    // the field's terms of the staged rows: class br (pairs), classes br and br + 2
    double f0 = 0.0, f1 = 0.0;
    auto field_terms = [&](int64_t j0, bool whole) {
#pragma unroll
        for (int u = 0; u < (kPairB ? 4 : 8); ++u) {
            const int64_t j = j0 + br + (kPairB ? 4 : 2) * u;
            if (whole || j < K) {
                const double aj = wgt[j];
                if constexpr (kPairB) {
                    f0 = fma_(aj, pb2[u].x, f0);
                    f1 = fma_(aj, pb2[u].y, f1);
                } else if (u & 1) {
                    f1 = fma_(aj, pb1[u], f1);
                } else {
                    f0 = fma_(aj, pb1[u], f0);
                }
            }
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int v = 0; v < 4; ++v) *reinterpret_cast<f64x2*>(&As[ar * kKrApad + ac + 2 * v]) = pa[v];
#pragma unroll
        for (int u = 0; u < (kPairB ? 4 : 8); ++u) {
            if constexpr (kPairB)
                *reinterpret_cast<f64x2*>(&Bs[(br + 4 * u) * kKrBpad + bc]) = pb2[u];
            else
                Bs[(br + 2 * u) * kKrBpad + bc] = pb1[u];
        }
    };

    f64x4 acc[kKrRF][4];
#pragma unroll
    for (int rt = 0; rt < kKrRF; ++rt)
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) acc[rt][ct] = f64x4{0.0, 0.0, 0.0, 0.0};

    // columns left of the diagonal block carry nothing in M2.  The K steps run
    // from the last one down to the diagonal block: every row tile starts at the
    // same rows of V, so the row tiles of one column tile (resident together on
    // one XCD) read each V row at about the same time and share it through L2.
    const int64_t jlast = ((K - 1) / kKrK) * kKrK;
    auto products = [&](int rt_end) {
#pragma unroll
        for (int kk = 0; kk < kKrK; kk += 4) {
            double a[kKrRF], b[4];
#pragma unroll
            for (int rt = 0; rt < kKrRF; ++rt) a[rt] = As[(rt * 32 + wr * 16 + l16) * kKrApad + kk + g];
#pragma unroll
            for (int ct = 0; ct < 4; ++ct) b[ct] = Bs[(kk + g) * kKrBpad + wc * 64 + ct * 16 + l16];
#pragma unroll
            for (int rt = 0; rt < kKrRF; ++rt)
                if (rt < rt_end)
#pragma unroll
                    for (int ct = 0; ct < 4; ++ct)
                        acc[rt][ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[rt], b[ct], acc[rt][ct], 0, 0, 0);
        }
    };
    // row fragments with rows below K (this wave's: 16 of every 32 rows)
    const int64_t rows_left = K - i0 - wr * 16;
    const int rt_rows = rows_left >= kKrRows ? kKrRF : (rows_left > 0 ? (int)((rows_left + 31) >> 5) : 0);
    auto stage = [&](int64_t j0) {
        __syncthreads();
        store();
        if (rt_idx == 0) field_terms(j0, j0 + kKrK <= K);
        __syncthreads();
        if (j0 - kKrK >= i0) load(j0 - kKrK, true);
    };
    load(jlast, jlast + kKrK <= K);
    int64_t j0 = jlast;
    if (i0 + kKrRows <= K)  // every fragment has rows: a straight line of products down to the diagonal
        for (; j0 >= i0 + kKrRows - 32; j0 -= kKrK) {
            stage(j0);
            products(kKrRF);
        }
    for (; j0 >= i0; j0 -= kKrK) {
        // fragments left of their diagonal block or past row K add nothing
        stage(j0);
        const int rt_diag = (int)((j0 - i0) >> 5) + 1;
        products(rt_diag < rt_rows ? rt_diag : rt_rows);
    }

    // epilogue: per column, sum over this wave's kKrRows / 2 rows of V o W (fragments past row
    // K hold zeros).  V is read in two batches of 32 values per lane from clamped addresses:
    // a checked read at a time left 23 us of latency on a block whose loop takes 65.
    double se[4];
#pragma unroll
    for (int c2 = 0; c2 < 4; c2 += 2) {
        double v[2][kKrRF][4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int64_t p = p0 + wc * 64 + (c2 + h) * 16 + l16;
            const double* vp = V + (p < P ? p : P - 1);
#pragma unroll
            for (int rt = 0; rt < kKrRF; ++rt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t i = i0 + rt * 32 + wr * 16 + g + 4 * r;
                    v[h][rt][r] = vp[(i < K ? i : K - 1) * P];
                }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            double e = 0.0;
#pragma unroll
            for (int rt = 0; rt < kKrRF; ++rt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t i = i0 + rt * 32 + wr * 16 + g + 4 * r;
                    e += (i < K ? v[h][rt][r] : 0.0) * acc[rt][c2 + h][r];
                }
            // the four lane groups holding this column, in a fixed order
            e += __shfl_xor(e, 16);
            e += __shfl_xor(e, 32);
            se[c2 + h] = e;
        }
    }
    if (g == 0) {
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) red[wr][wc * 64 + ct * 16 + l16] = se[ct];
    }
    __syncthreads();
    if (t < kKrPts) {
        const int64_t p = p0 + t;
        if (p < P) part_e[rt_idx * P + p] = red[0][t] + red[1][t];
    }
    __syncthreads();  // red is rewritten below
    if (rt_idx == 0) {
        red[br][bc] = f0;
        red[kPairB ? br : br + 2][kPairB ? bc + 1 : bc] = f1;
        __syncthreads();
        if (t < kKrPts && p0 + t < P)
            field[p0 + t] = (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]);
    }
}

__global__ void k_krige_reduce(int64_t tiles, int64_t P, const double* __restrict__ part_e,
                               double* __restrict__ error) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P) return;
    double e = 0.0;
    for (int64_t it = 0; it < tiles; ++it) e += part_e[it * P + p];
    error[p] = e;
}

// field_p = sum_j a_j V[j, p]: 128 points per block (512 blocks for 65536 points,
// where one thread per four points made 64), wave w the rows j = w mod 4 from the last
// 16-row step down, the four sums added as in k_krige_gemm.  kPair (P even, V 16-byte
// aligned): a point pair per lane, else two points 64 apart.  first: the launch's first block.
template <bool kPair>
__global__ __launch_bounds__(256) void k_krige_field(int64_t first, int64_t K, int64_t P, const double* __restrict__ a,
                                                     const double* __restrict__ V, double* __restrict__ field) {
    typedef __attribute__((ext_vector_type(2))) double f64x2;
    __shared__ double red[4][kKrPts];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t p0 = (first + blockIdx.x) * kKrPts;
    const int c0 = kPair ? 2 * lane : lane, c1 = kPair ? 2 * lane + 1 : lane + 64;
    // clamped (valid) addresses past P
    const int64_t q0 = p0 + c0 < P ? p0 + c0 : (kPair ? P - 2 : P - 1), q1 = p0 + c1 < P ? p0 + c1 : P - 1;
    double f0 = 0.0, f1 = 0.0;
    auto step = [&](int64_t j0, bool whole) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int64_t j = j0 + w + 4 * u;
            if (whole || j < K) {
                f64x2 v;
                if constexpr (kPair)
                    v = *reinterpret_cast<const f64x2*>(V + j * P + q0);
                else
                    v = f64x2{V[j * P + q0], V[j * P + q1]};
                f0 = fma_(a[j], v.x, f0);
                f1 = fma_(a[j], v.y, f1);
            }
        }
    };
    int64_t j0 = ((K - 1) / kKrK) * kKrK;
    step(j0, false);
#pragma unroll 4
    for (j0 -= kKrK; j0 >= 0; j0 -= kKrK) step(j0, true);
    red[w][c0] = f0;
    red[w][c1] = f1;
    __syncthreads();
    const int t = threadIdx.x;
    if (t < kKrPts && p0 + t < P) field[p0 + t] = (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]);
}

struct CovModelArgs {
    int kind;           // 0 Gaussian exp(-h^2), 1 Exponential exp(-h), 2 Stable exp(-h^alpha),
                        // 3 Spherical 1 - 1.5 h + 0.5 h^3 (h <= 1)
    double var;         // variance
    double len;         // rescaled length scale: h = r / len
    double alpha;       // Stable shape
    double sill_at_0;   // >= 0: value where r <= 1e-8 (cov_nugget); < 0: none
};

// C(r).  kDiv: h = r / m.len by division; else by inv = 1 / m.len rounded: the product
// corrected by its remainder, the rounded quotient again (for lengths that krige_cov_launch
// passes; a product out of range stays as it is, infinite or NaN like the quotient).
template <int KIND, bool kDiv>
__device__ __forceinline__ double cov_of(const CovModelArgs& m, double inv, double r) {
    double h;
    if constexpr (kDiv) {
        h = r / m.len;
    } else {
        const double q = r * inv;
        h = q < 0x1p+900 ? fma_(fma_(-q, m.len, r), inv, q) : q;
    }
    double c;
    if constexpr (KIND == 0) {
        c = exp(-(h * h));
    } else if constexpr (KIND == 1) {
        c = exp(-h);
    } else if constexpr (KIND == 2) {
        c = exp(-pow(h, m.alpha));
    } else {
        const double g = fmin(h, 1.0);
        c = 1.0 - 1.5 * g + 0.5 * (g * g * g);
    }
    return (m.sill_at_0 >= 0.0 && r <= 1e-8) ? m.sill_at_0 : m.var * c;
}

// out[i * ld + p] = C(|c_i - x_p|), i < K, p < P.  A thread keeps its target in
// registers and writes kCovRows rows (conditioning points i0 .. i0 + kCovRows - 1,
// read as wave-uniform values), so the targets are read once per kCovRows rows.  Bound by
// the vector unit (square root and exponential) and by stores of 512 bytes per wave: a pair
// of points per thread in large launches where P and ld are even and out is 16-byte aligned, the
// model a template argument, the quotient by a reciprocal.  Exponential, 300 x 40000 in 2D: 39 -> 30 us.
constexpr int kCovRows = 16;

template <int DIM, int KIND, bool kPair, bool kDiv>
__global__ __launch_bounds__(256) void k_krige_cov(CovModelArgs m, int64_t K, int64_t P,
                                                   const double* __restrict__ cpos,
                                                   const double* __restrict__ pos, double* __restrict__ out,
                                                   int64_t ld) {
#pragma clang fp contract(off)
    typedef __attribute__((ext_vector_type(2))) double f64x2;
    constexpr int kPts = kPair ? 2 : 1;
    const int64_t p = ((int64_t)blockIdx.x * 256 + threadIdx.x) * kPts;
    const int64_t i0 = (int64_t)blockIdx.y * kCovRows;
    if (p >= P) return;
    double x[kPts][DIM];
#pragma unroll
    for (int e = 0; e < kPts; ++e)
#pragma unroll
        for (int d = 0; d < DIM; ++d) x[e][d] = pos[d * P + p + e];
    const double inv = 1.0 / m.len;
    const int64_t ie = K - i0 < kCovRows ? K : i0 + kCovRows;
#pragma unroll 2
    for (int64_t i = i0; i < ie; ++i) {
        double c[kPts];
#pragma unroll
        for (int e = 0; e < kPts; ++e) {
            double d2 = 0.0;
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                const double t = cpos[d * K + i] - x[e][d];
                d2 += t * t;
            }
            c[e] = cov_of<KIND, kDiv>(m, inv, sqrt(d2));
        }
        if constexpr (kPair)
            *reinterpret_cast<f64x2*>(out + i * ld + p) = f64x2{c[0], c[1]};
        else
            out[i * ld + p] = c[0];
    }
}

template <int DIM>
void krige_cov_launch(const CovModelArgs& m, int64_t K, int64_t P, const double* cpos, const double* pos,
                      double* out, int64_t ld, hipStream_t s) {
    // lengths whose reciprocal and remainders are exact enough: far from the exponent's limits
    const bool div = !(m.len >= 0x1p-400 && m.len <= 0x1p+400);
    // pairs where they leave four blocks per CU: below that single points, twice the blocks, are
    // faster (Stable, 300 x 10000: 37 us in pairs, 30 singly; 300 x 40000: 96 and 100)
    const bool enough = ceil_div(P, (int64_t)512) * ceil_div(K, (int64_t)kCovRows) >= 1024;
    const bool pair = enough && !div && P % 2 == 0 && ld % 2 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
    const dim3 grid((unsigned)ceil_div(P, (int64_t)(pair ? 512 : 256)), (unsigned)ceil_div(K, (int64_t)kCovRows));
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, m, K, P, cpos, pos, out, ld); };
    auto form = [&](auto pairs, auto singles, auto division) { pair ? go(pairs) : div ? go(division) : go(singles); };
    switch (m.kind) {
        case 0: form(k_krige_cov<DIM, 0, true, false>, k_krige_cov<DIM, 0, false, false>,
                     k_krige_cov<DIM, 0, false, true>); break;
        case 1: form(k_krige_cov<DIM, 1, true, false>, k_krige_cov<DIM, 1, false, false>,
                     k_krige_cov<DIM, 1, false, true>); break;
        case 2: form(k_krige_cov<DIM, 2, true, false>, k_krige_cov<DIM, 2, false, false>,
                     k_krige_cov<DIM, 2, false, true>); break;
        default: form(k_krige_cov<DIM, 3, true, false>, k_krige_cov<DIM, 3, false, false>,
                      k_krige_cov<DIM, 3, false, true>);
    }
}

__global__ void k_fill_zero_f64(double* __restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

inline int64_t krige_row_tiles(int64_t K) { return ceil_div(K, (int64_t)kKrRows); }

// field: the weight vector (K); variance form: also the row-tile partials (tiles x P)
// and the padded M2 (128 tiles x Kp), 16-byte aligned after the others
inline int64_t krige_ws_bytes(int64_t K, int64_t P, bool variance) {
    const int64_t field = K;
    if (variance) {
        const int64_t head = krige_row_tiles(K) * P + field;
        return ((head + 1) / 2 * 2 + krige_row_tiles(K) * kKrRows * krige_kp(K)) * (int64_t)sizeof(double);
    }
    return field * (int64_t)sizeof(double);
}

}  // namespace gsx

extern "C" {

int64_t gsx_krige_workspace(int64_t K, int64_t P, int variance) {
    if (K < 0 || P < 0) return GSX_E_INVALID;
    return gsx::krige_ws_bytes(K, P, variance != 0);
}

int gsx_krige_f64(int64_t K, int64_t P, const double* krig_mat, const double* krig_vecs, const double* cond,
                  double* field, double* error, void* workspace, int64_t workspace_bytes, void* stream) {
    if (K < 0 || P < 0) return GSX_E_INVALID;
    if (P == 0) return GSX_OK;
    if (!field) return GSX_E_INVALID;
    hipStream_t s = gsx::as_stream(stream);
    if (K == 0) {
        const unsigned blocks = (unsigned)gsx::ceil_div(P, (int64_t)256);
        hipLaunchKernelGGL(gsx::k_fill_zero_f64, dim3(blocks), dim3(256), 0, s, field, P);
        if (error) hipLaunchKernelGGL(gsx::k_fill_zero_f64, dim3(blocks), dim3(256), 0, s, error, P);
        return gsx::launch_status();
    }
    if (!krig_mat || !krig_vecs || !cond) return GSX_E_INVALID;
    const bool variance = error != nullptr;
    if (!workspace || workspace_bytes < gsx::krige_ws_bytes(K, P, variance)) return GSX_E_WORKSPACE;
    double* ws = static_cast<double*>(workspace);
    const int64_t tiles = gsx::krige_row_tiles(K);
    const int64_t col_blocks = gsx::ceil_div(P, (int64_t)gsx::kKrPts);
    const int64_t Kp = gsx::krige_kp(K), Rp = tiles * gsx::kKrRows;
    if (variance && (tiles * (col_blocks + 8) > 0x7fffffffLL || gsx::ceil_div(Rp * Kp, (int64_t)256) > 0x7fffffffLL))
        return GSX_E_INVALID;
    double* part_e = ws;
    double* a = variance ? ws + tiles * P : ws;
    // M2 16-byte aligned: the workspace is, and its offset is rounded up to an even
    // number of doubles
    double* m2 = ws + (tiles * P + K + 1) / 2 * 2;
    if (variance && reinterpret_cast<uintptr_t>(m2) % 16 != 0) return GSX_E_INVALID;
    const int64_t prep = gsx::ceil_div(K, (int64_t)64) + (variance ? gsx::ceil_div(Rp * Kp, (int64_t)1024) : 0);
    int st = gsx::launch_parts(prep, 1024, [&](int64_t first, dim3 grid) {
        hipLaunchKernelGGL(gsx::k_krige_prepare, grid, dim3(1024), 0, s, first, K, Rp, Kp, krig_mat, cond, a, m2);
    });
    if (st != GSX_OK) return st;
    const bool pair_b = P % 2 == 0 && reinterpret_cast<uintptr_t>(krig_vecs) % 16 == 0;
    if (!variance)
        return gsx::launch_parts(col_blocks, 256, [&](int64_t first, dim3 grid) {
            if (pair_b)
                hipLaunchKernelGGL(gsx::k_krige_field<true>, grid, dim3(256), 0, s, first, K, P, a, krig_vecs, field);
            else
                hipLaunchKernelGGL(gsx::k_krige_field<false>, grid, dim3(256), 0, s, first, K, P, a, krig_vecs, field);
        });
    // error = v^T M2 v over the block upper triangle
    const int64_t col8 = gsx::ceil_div(col_blocks, (int64_t)8) * 8;
    const dim3 grid((unsigned)(col8 * tiles));
    if (pair_b)
        hipLaunchKernelGGL(gsx::k_krige_gemm<true>, grid, dim3(256), 0, s, K, Kp, P, tiles, col_blocks, m2, krig_vecs,
                           a, part_e, field);
    else
        hipLaunchKernelGGL(gsx::k_krige_gemm<false>, grid, dim3(256), 0, s, K, Kp, P, tiles, col_blocks, m2,
                           krig_vecs, a, part_e, field);
    st = gsx::launch_status();
    if (st != GSX_OK) return st;
    hipLaunchKernelGGL(gsx::k_krige_reduce, dim3((unsigned)gsx::ceil_div(P, (int64_t)256)), dim3(256), 0, s, tiles,
                       P, part_e, error);
    return gsx::launch_status();
}

int gsx_krige_cov_f64(int model_kind, double var, double len_rescaled, double alpha, double sill_at_zero,
                      int64_t dim, int64_t K, int64_t P, const double* cond_pos, const double* pos, double* out,
                      int64_t ld_out, void* stream) {
    if (model_kind < 0 || model_kind > 3 || dim < 1 || dim > 3 || K < 0 || P < 0 || ld_out < P) return GSX_E_INVALID;
    if (!(len_rescaled > 0.0)) return GSX_E_INVALID;
    if (K == 0 || P == 0) return GSX_OK;
    if (K > 65535) return GSX_E_INVALID;
    if (!cond_pos || !pos || !out) return GSX_E_INVALID;
    gsx::CovModelArgs m{model_kind, var, len_rescaled, alpha, sill_at_zero};
    hipStream_t s = gsx::as_stream(stream);
    switch (dim) {
        case 1: gsx::krige_cov_launch<1>(m, K, P, cond_pos, pos, out, ld_out, s); break;
        case 2: gsx::krige_cov_launch<2>(m, K, P, cond_pos, pos, out, ld_out, s); break;
        default: gsx::krige_cov_launch<3>(m, K, P, cond_pos, pos, out, ld_out, s);
    }
    return gsx::launch_status();
}

}  // extern "C"
