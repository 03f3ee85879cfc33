// Point-parallel randomisation-method summation on gfx950.
//
//   u(x_i) = sum_j z1_j cos(k_j.x_i) + z2_j sin(k_j.x_i)        (summate)
//   u_c(x_i) = sum_j p_c(k_j) (z1_j cos + z2_j sin)             (summate_incompr)
//
// Reference contract: src/gstools/field/generator.py:193-199 (scalar) and
// :479-494 (incompressible), called at :266-268 and :554-560.
//
// Layout and schedule:
//  * one thread owns PPT points (coalesced loads of the (d, P) position rows,
//    points interleaved by kThreads so every load/store is unit-stride across
//    a wavefront);
//  * modes are staged through LDS in chunks of kChunk: each block turns its
//    chunk of (cov, z1, z2) into a per-mode table -- wavenumbers, amplitude
//    a_j = |z1_j - i z2_j| and phase phi_j = atan2(z2_j, z1_j), so that
//    z1 cos(t) + z2 sin(t) = a cos(t - phi) needs ONE cosine per term;
//  * every lane reads the same table entry (LDS broadcast, no bank conflict).
//
// The Fourier method (generator.py:659-691) is the same sum with a per-mode
// spectrum factor f_j multiplying each term; it is folded into the amplitude
// when the table is built (fac == nullptr for the randomisation method).
//
// Launches of few points share the modes of a point out over the waves of a
// block instead (k_forward_*_split); both forms add the same partial sums in the
// same order, so a point's value does not depend on the launch it is part of.
//
// FP64 path: the phase is the reference's exact product-then-add sequence;
// cos(t - phi) uses the two-term Cody-Waite reduction of gsx_math.h with phi
// folded into the reduction (no rounding of t - phi at large |t|).  A wave
// whose |x|_inf * max_j |k_j|_1 may exceed 2^45 takes a per-term guarded path
// that falls back to the library sincos for |t| > 2^46.  The mode sum runs over
// groups of 64 modes, each from zero, added in order.
//
// FP32 path (gsx_fp32sum.h): the phase is computed in revolutions in FP64
// (t = k/2pi . x - phi/2pi, three FMAs), reduced by magic addition (the low
// word of the sum is the fraction in fixed point, one v_alignbit_b32 makes it
// a float in [1, 2)) for the modes whose |k/2pi|_1 times the largest |x|_inf
// of the point's 2048-point segment stays within 2^18 revolutions, else
// exactly with v_fract_f64 and a conversion, and fed to the hardware cosine
// (v_cos_f32 takes revolutions).  The mode sum
// runs in FP32 for blocks of kSub modes and is then added into an FP64
// accumulator (blocked compensation: FP32 rounding error grows only over
// kSub terms).
#include "gsx_fp32sum.h"
#include "gsx_internal.h"

namespace gsx {

constexpr int kChunk = 256;  // modes per LDS chunk (== kThreads: one mode per thread to build)
constexpr int kGroupF64 = 64;  // modes per FP64 partial sum
constexpr double kSafeK1X = 0x1.0p+45;  // |k|_1 |x|_inf bound of the FP64 fast path

// cos(theta - phi) at any |theta|: the fast reduction where it is exact, else the
// library sincos.  Kept out of line so the fast loop's register budget does not
// pay for the wide-range code.
__device__ __noinline__ double cos_shifted_any(double th, double phi, double phipi) {
    if (fabs(th) <= kFastPhaseMax) return cos_shifted(th, phi, phipi);
    double st, ct, sp, cp;
    sincos(th, &st, &ct);
    sincos(phi, &sp, &cp);
    return ct * cp + st * sp;
}

__device__ __forceinline__ void lds_max_u64(unsigned long long* p, double v) {
    // non-negative doubles order like their bit patterns
    atomicMax(p, (unsigned long long)__double_as_longlong(v));
}

// -------------------------------------------------------------- FP64 --------
template <int D, bool INCOMPR>
struct TabF64 {
    // scalar:  k[D], a, phi, phi/pi ; incompr: k[D], phi, phi/pi, w[D] = p(k) * a
    static constexpr int kW = INCOMPR ? 2 * D + 2 : D + 3;
    static constexpr int kStride = (kW + 1) & ~1;  // 16-byte aligned rows
};

// Table row of mode j; returns |k_j|_1.
template <int D, bool INCOMPR>
__device__ __forceinline__ double f64_build_row(int64_t N, int64_t j, const double* __restrict__ cov,
                                                const double* __restrict__ z1, const double* __restrict__ z2,
                                                const double* __restrict__ fac, double* t) {
    double k[D];
    double k1 = 0.0, k2 = 0.0;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        k[d] = cov[d * N + j];
        t[d] = k[d];
        k1 += fabs(k[d]);
        k2 += k[d] * k[d];
    }
    const double u1 = z1[j], u2 = z2[j];
    const double phi = atan2(u2, u1);
    const double a = fac ? fac[j] * hypot(u1, u2) : hypot(u1, u2);
    if constexpr (INCOMPR) {
        t[D] = phi;
        t[D + 1] = phi * kInvPi;
#pragma unroll
        for (int c = 0; c < D; ++c) {
            const double proj = (c == 0 ? 1.0 : 0.0) - k[c] * k[0] / k2;
            t[D + 2 + c] = proj * a;
        }
    } else {
        t[D] = a;
        t[D + 1] = phi;
        t[D + 2] = phi * kInvPi;
    }
    return k1;
}

// Table rows [m0, m1) into the partial sums of one mode group.  SAFE: every
// phase lies within the fast reduction; else each term is checked and falls
// back to the library sincos.
template <int D, int PPT, bool INCOMPR, bool SAFE>
__device__ __forceinline__ void f64_group_sum(const double* tab, int m0, int m1, const double (&x)[PPT][D],
                                              double (&part)[PPT][INCOMPR ? D : 1]) {
    using T = TabF64<D, INCOMPR>;
    constexpr int NOUT = INCOMPR ? D : 1;
#pragma unroll
    for (int p = 0; p < PPT; ++p)
#pragma unroll
        for (int c = 0; c < NOUT; ++c) part[p][c] = 0.0;
    auto term = [&](int m) {
        const double* t = tab + m * T::kStride;
        double k[D];
#pragma unroll
        for (int d = 0; d < D; ++d) k[d] = t[d];
        const double phi = INCOMPR ? t[D] : t[D + 1];
        const double phipi = INCOMPR ? t[D + 1] : t[D + 2];
        double w[NOUT];
#pragma unroll
        for (int c = 0; c < NOUT; ++c) w[c] = INCOMPR ? t[D + 2 + c] : t[D];
#pragma unroll
        for (int p = 0; p < PPT; ++p) {
            const double th = phase_exact<D>(k, x[p]);
            const double cs = SAFE ? cos_shifted(th, phi, phipi) : cos_shifted_any(th, phi, phipi);
#pragma unroll
            for (int c = 0; c < NOUT; ++c) part[p][c] = fma_(w[c], cs, part[p][c]);
        }
    };
    int m = m0;
    if constexpr (SAFE) {
        // two modes per iteration (by hand: the compiler does not unroll a loop of
        // unknown length around inline assembly)
        for (; m + 1 < m1; m += 2) {
            term(m);
            term(m + 1);
        }
    }
    for (; m < m1; ++m) term(m);
}

template <int D, int PPT, bool INCOMPR, class Pts>
__global__ __launch_bounds__(kThreads) void k_forward_f64(Pts pts, int64_t N, int64_t P,
                                                          const double* __restrict__ cov,
                                                          const double* __restrict__ z1,
                                                          const double* __restrict__ z2,
                                                          const double* __restrict__ fac,
                                                          double* __restrict__ out) {
    using T = TabF64<D, INCOMPR>;
    constexpr int NOUT = INCOMPR ? D : 1;
    __shared__ __align__(16) double tab[kChunk * T::kStride];
    __shared__ unsigned long long s_kmax;

    double x[PPT][D];
    double acc[PPT][NOUT];
    double xmax[PPT];
    const int64_t base = (int64_t)blockIdx.x * (kThreads * PPT) + threadIdx.x;
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
        const int64_t i = base + (int64_t)p * kThreads;
        if (i < P) {
            pts.get(i, x[p]);
        } else {
#pragma unroll
            for (int d = 0; d < D; ++d) x[p][d] = 0.0;
        }
        xmax[p] = 0.0;
#pragma unroll
        for (int d = 0; d < D; ++d) xmax[p] = fmax(xmax[p], fabs(x[p][d]));
#pragma unroll
        for (int c = 0; c < NOUT; ++c) acc[p][c] = 0.0;
    }

    for (int64_t j0 = 0; j0 < N; j0 += kChunk) {
        const int cnt = (int)(N - j0 < kChunk ? N - j0 : kChunk);
        __syncthreads();
        if (threadIdx.x == 0) s_kmax = 0ull;
        __syncthreads();
        if ((int)threadIdx.x < cnt)
            lds_max_u64(&s_kmax, f64_build_row<D, INCOMPR>(N, j0 + threadIdx.x, cov, z1, z2, fac,
                                                           tab + threadIdx.x * T::kStride));
        __syncthreads();
        const double kmax = __longlong_as_double((long long)s_kmax);
        bool safe = true;
#pragma unroll
        for (int p = 0; p < PPT; ++p) safe = safe && (xmax[p] * kmax <= kSafeK1X);
        const bool all_safe = __all(safe);
        for (int m0 = 0; m0 < cnt; m0 += kGroupF64) {
            const int m1 = m0 + kGroupF64 < cnt ? m0 + kGroupF64 : cnt;
            double part[PPT][NOUT];
            if (all_safe)
                f64_group_sum<D, PPT, INCOMPR, true>(tab, m0, m1, x, part);
            else
                f64_group_sum<D, PPT, INCOMPR, false>(tab, m0, m1, x, part);
#pragma unroll
            for (int p = 0; p < PPT; ++p)
#pragma unroll
                for (int c = 0; c < NOUT; ++c) acc[p][c] += part[p][c];
        }
    }

#pragma unroll
    for (int p = 0; p < PPT; ++p) {
        const int64_t i = base + (int64_t)p * kThreads;
        if (i < P) {
#pragma unroll
            for (int c = 0; c < NOUT; ++c) out[c * P + i] = acc[p][c];
        }
    }
}

// Few points: the mode groups of a point are shared out over the waves of a
// block, 16 groups (1024 modes) at a time, and over L equal parts of each
// wave's lanes: a block of 1024 / L threads holds PB = 64 / L * PPT points.
// Every (group, point) partial sum goes through LDS and the groups are added in
// order, so a point's value is the same bits as in k_forward_f64.
constexpr int kSplitModes = 1024;

template <int D, int PPT, int L, bool INCOMPR, class Pts>
__global__ __launch_bounds__(kSplitModes / L) void k_forward_f64_split(Pts pts, int64_t N, int64_t P,
                                                                       const double* __restrict__ cov,
                                                                       const double* __restrict__ z1,
                                                                       const double* __restrict__ z2,
                                                                       const double* __restrict__ fac,
                                                                       double* __restrict__ out) {
    using T = TabF64<D, INCOMPR>;
    constexpr int NOUT = INCOMPR ? D : 1;
    constexpr int kT = kSplitModes / L;             // threads
    constexpr int kG = kSplitModes / kGroupF64;     // groups at a time
    constexpr int kLP = 64 / L;                     // lanes (and points per PPT) of a part
    constexpr int kPB = kLP * PPT;                  // points of the block
    static_assert(kPB * NOUT <= kT, "one thread adds the groups of one output");
    __shared__ __align__(16) double tab[kSplitModes * T::kStride];
    __shared__ double s_part[kG][kPB * NOUT];
    __shared__ unsigned long long s_kmax;

    const int t = (int)threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int grp = wave * L + lane / kLP;          // this lane's group of the 16
    const int64_t p0 = (int64_t)blockIdx.x * kPB;
    double x[PPT][D];
    double xmax = 0.0;
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
        const int64_t i = p0 + p * kLP + lane % kLP;
        if (i < P) {
            pts.get(i, x[p]);
        } else {
#pragma unroll
            for (int d = 0; d < D; ++d) x[p][d] = 0.0;
        }
    }
    // NaN coordinates are left out of the bound (fmax), as in k_forward_f64
#pragma unroll
    for (int p = 0; p < PPT; ++p)
#pragma unroll
        for (int d = 0; d < D; ++d) xmax = fmax(xmax, fabs(x[p][d]));
    double acc = 0.0;  // output t of the block: component t / kPB of point t % kPB

    for (int64_t j0 = 0; j0 < N; j0 += kSplitModes) {
        const int cnt = (int)(N - j0 < kSplitModes ? N - j0 : kSplitModes);
        if (t == 0) s_kmax = 0ull;
        __syncthreads();  // also: the last chunk's table and partial sums are no longer read
#pragma unroll
        for (int q = 0; q < L; ++q) {
            const int m = t + q * kT;
            if (m < cnt)
                lds_max_u64(&s_kmax,
                            f64_build_row<D, INCOMPR>(N, j0 + m, cov, z1, z2, fac, tab + m * T::kStride));
        }
        __syncthreads();
        const double kmax = __longlong_as_double((long long)s_kmax);
        const int m0 = grp * kGroupF64 < cnt ? grp * kGroupF64 : cnt;
        const int m1 = m0 + kGroupF64 < cnt ? m0 + kGroupF64 : cnt;
        double part[PPT][NOUT];
        if (__all(xmax * kmax <= kSafeK1X))
            f64_group_sum<D, PPT, INCOMPR, true>(tab, m0, m1, x, part);
        else
            f64_group_sum<D, PPT, INCOMPR, false>(tab, m0, m1, x, part);
#pragma unroll
        for (int p = 0; p < PPT; ++p)
#pragma unroll
            for (int c = 0; c < NOUT; ++c) s_part[grp][c * kPB + p * kLP + lane % kLP] = part[p][c];
        __syncthreads();
        if (t < kPB * NOUT) {
            const int groups = (cnt + kGroupF64 - 1) / kGroupF64;
            for (int g = 0; g < groups; ++g) acc += s_part[g][t];
        }
    }
    if (t < kPB * NOUT) {
        const int64_t i = p0 + t % kPB;
        if (i < P) out[(int64_t)(t / kPB) * P + i] = acc;
    }
}

// -------------------------------------------------------------- FP32 --------
// One block: kThreads * PPT points (a divisor of the kSeg-point segment), all
// modes through fp32_item_sum (gsx_fp32sum.h).  At least 3 waves per SIMD: the
// two inlined mode loops would otherwise take the 3D sum to 198 VGPRs (2
// waves); bounded, it fits in 168.
template <int D, int PPT, bool INCOMPR, class Pts>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(3))) void k_forward_f32(
    Pts pts, int64_t N, int64_t P, const double* __restrict__ cov, const double* __restrict__ z1,
    const double* __restrict__ z2, const double* __restrict__ fac, float* __restrict__ out) {
    constexpr int NOUT = INCOMPR ? D : 1;
    __shared__ double tabd[kChunk * (D + 1)];
    __shared__ float tabf[kChunk * NOUT];  // a (scalar) or p(k) * a (incompr)
    __shared__ double s_wmax[kWaves];
    __shared__ int s_nmagic[kWaves];

    double x[PPT][D];
    double acc[PPT][NOUT];
    double own = 0.0;
    const int64_t p0 = (int64_t)blockIdx.x * (kThreads * PPT);
    const int64_t base = p0 + threadIdx.x;
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
        const int64_t i = base + (int64_t)p * kThreads;
        if (i < P) {
            pts.get(i, x[p]);
#pragma unroll
            for (int d = 0; d < D; ++d) own = coord_bound(own, x[p][d]);
        } else {
#pragma unroll
            for (int d = 0; d < D; ++d) x[p][d] = 0.0;
        }
#pragma unroll
        for (int c = 0; c < NOUT; ++c) acc[p][c] = 0.0;
    }
    const double xseg = segment_xmax<D, kThreads, kThreads * PPT>(pts, P, p0, own, s_wmax);
    fp32_item_sum<D, PPT, INCOMPR, kChunk>(N, cov, z1, z2, fac, xseg, x, acc, tabd, tabf, s_nmagic);

#pragma unroll
    for (int p = 0; p < PPT; ++p) {
        const int64_t i = base + (int64_t)p * kThreads;
        if (i < P) {
#pragma unroll
            for (int c = 0; c < NOUT; ++c) out[c * P + i] = (float)acc[p][c];
        }
    }
}

// Few points: the mode groups of a point are shared out over the block's waves,
// 1024 modes (8 groups) at a time, two waves per group (the first takes the
// group's first run of at most kSub modes, the second the others); a block of
// 1024 threads holds PB = 64 PPT points.  The FP32 partial sums of every run (at
// most three per group) go through LDS and are added into the FP64 accumulator
// in order, so a point's value is the same bits as in k_forward_f32.
template <int D, int PPT, bool INCOMPR, class Pts>
__global__ __launch_bounds__(kSplitModes) void k_forward_f32_split(
    Pts pts, int64_t N, int64_t P, const double* __restrict__ cov, const double* __restrict__ z1,
    const double* __restrict__ z2, const double* __restrict__ fac, float* __restrict__ out) {
    constexpr int NOUT = INCOMPR ? D : 1;
    constexpr int kG = kSplitModes / kGroup;
    constexpr int kRuns = 3;          // runs of <= kSub modes in a group of two ordered parts
    constexpr int kPB = 64 * PPT;
    static_assert(kGroup == 2 * kSub, "two parts of a group: at most three runs");
    static_assert(kPB * NOUT <= kSplitModes, "one thread adds the runs of one output");
    __shared__ double tabd[kSplitModes * (D + 1)];
    __shared__ float tabf[kSplitModes * NOUT];
    __shared__ float s_part[kG * kRuns][kPB * NOUT];
    __shared__ double s_wmax[kSplitModes / 64];
    __shared__ int s_nmagic[kSplitModes / 64];

    const int t = (int)threadIdx.x;
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int grp = wave >> 1, half = wave & 1;
    const int64_t p0 = (int64_t)blockIdx.x * kPB;
    double x[PPT][D];
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
        const int64_t i = p0 + p * 64 + lane;
        if (i < P) {
            pts.get(i, x[p]);
        } else {
#pragma unroll
            for (int d = 0; d < D; ++d) x[p][d] = 0.0;
        }
    }
    const double xseg = segment_xmax<D, kSplitModes, kPB>(pts, P, p0, 0.0, s_wmax);
    double acc = 0.0;  // output t of the block: component t / kPB of point t % kPB

    for (int64_t j0 = 0; j0 < N; j0 += kSplitModes) {
        const int cnt = (int)(N - j0 < kSplitModes ? N - j0 : kSplitModes);
        fp32_build_table<D, INCOMPR>(N, j0, cnt, cov, z1, z2, fac, xseg, tabd, tabf, s_nmagic);
        const int g0 = grp * kGroup;
        if (g0 < cnt) {
            const int ge = g0 + kGroup < cnt ? g0 + kGroup : cnt;
            const int gm = g0 + s_nmagic[2 * grp] + s_nmagic[2 * grp + 1];
            // runs in order: magic modes [g0, gm) then the others [gm, ge), kSub at a time
            int m = g0;
#pragma unroll 1
            for (int run = 0; run < kRuns; ++run) {
                const int top = m < gm ? gm : ge;
                const int me = m + kSub < top ? m + kSub : top;
                if ((run == 0) == (half == 0)) {
                    float part[PPT][NOUT];
                    if (m < gm)
                        sub_run_f32<D, PPT, NOUT, true>(tabd, tabf, m, me, x, part);
                    else
                        sub_run_f32<D, PPT, NOUT, false>(tabd, tabf, m, me, x, part);
#pragma unroll
                    for (int p = 0; p < PPT; ++p)
#pragma unroll
                        for (int c = 0; c < NOUT; ++c)
                            s_part[grp * kRuns + run][c * kPB + p * 64 + lane] = part[p][c];
                }
                m = me;
            }
        }
        __syncthreads();
        if (t < kPB * NOUT) {
            // runs past a group's last one hold +0, which changes nothing
            const int runs = (cnt + kGroup - 1) / kGroup * kRuns;
            for (int r = 0; r < runs; ++r) acc += (double)s_part[r][t];
        }
    }
    if (t < kPB * NOUT) {
        const int64_t i = p0 + t % kPB;
        if (i < P) out[(int64_t)(t / kPB) * P + i] = (float)acc;
    }
}

// ------------------------------------------------------------ launchers -----
// Points per thread of a plain launch.  Its blocks (256 threads) spread over the 256 CUs in
// whole rounds, so a launch of 600000 points in blocks of 2048 (293 of them) took as long as
// one of 1e6.  Cycles of a CU per round, measured over 1.4e5 to 2.1e6 points and 150 to 2000
// modes in 2D and 3D (a block's mode table and LDS reads spread over its points; the smaller
// FP32 blocks look through the whole segment's coordinates, too):
//   FP32  PPT 8 244 N + 1600, 4 126 N + 2500, 2 67 N + 3300
//   FP64  PPT 4 405 N + 16000, 2 210 N + 5300, 1 117 N + 4000
// a tenth more (FP64: a twentieth) for the largest in a single round, one wave per SIMD,
// and the choice is the least rounds times cost, of equals the largest.  3D, N = 2000, cycles
// of a SIMD per 64 terms: FP32 600000 points 57 -> 41 (PPT 2), 1.3e6 38 -> 32 (4), 4e6 31 (8);
// FP64 140000 points 223 -> 185 (1), 1.3e6 108 -> 104 (4).
// The incompressible sums, d accumulators to a point, start at 4 and 2 points (8 and 4
// would leave 2 waves per SIMD).
template <bool F64, bool INCOMPR>
inline int plain_ppt(int64_t N, int64_t P) {
    constexpr int kTop = (F64 ? 4 : 8) / (INCOMPR ? 2 : 1);
    const double n = (double)N;
    auto cost = [&](int ppt) {
        const double rounds = (double)ceil_div(ceil_div(P, (int64_t)kThreads * ppt), (int64_t)256);
        const double alone = rounds > 1.0 || ppt < (F64 ? 4 : 8) ? 1.0 : (F64 ? 1.05 : 1.1);
        if (F64)
            return alone * rounds *
                   (ppt == 4 ? 405.0 * n + 16000.0 : ppt == 2 ? 210.0 * n + 5300.0 : 117.0 * n + 4000.0);
        return alone * rounds * (ppt == 8 ? 244.0 * n + 1600.0 : ppt == 4 ? 126.0 * n + 2500.0 : 67.0 * n + 3300.0);
    };
    int best = kTop;
    for (int ppt = kTop / 2; ppt >= (F64 ? 1 : 2); ppt /= 2)
        if (cost(ppt) < cost(best)) best = ppt;
    return best;
}

template <int D, int PPT, int L, bool INCOMPR, class Pts>
int launch_f64_split(Pts pts, int64_t N, int64_t P, const double* cov, const double* z1, const double* z2,
                     const double* fac, double* out, hipStream_t s) {
    const int64_t blocks = ceil_div(P, (int64_t)(64 / L * PPT));
    hipLaunchKernelGGL((k_forward_f64_split<D, PPT, L, INCOMPR, Pts>), dim3((unsigned)blocks), dim3(kSplitModes / L),
                       0, s, pts, N, P, cov, z1, z2, fac, out);
    return launch_status();
}

template <int D, int PPT, bool INCOMPR, class Pts>
int launch_f32_split(Pts pts, int64_t N, int64_t P, const double* cov, const double* z1, const double* z2,
                     const double* fac, float* out, hipStream_t s) {
    const int64_t blocks = ceil_div(P, (int64_t)(64 * PPT));
    hipLaunchKernelGGL((k_forward_f32_split<D, PPT, INCOMPR, Pts>), dim3((unsigned)blocks), dim3(kSplitModes), 0, s,
                       pts, N, P, cov, z1, z2, fac, out);
    return launch_status();
}

// Whether the split kernels serve (N, P).  A plain launch of up to one block per CU takes the
// time of one block walking all N modes, and takes the smallest blocks that keep it to that
// (plain_ppt): one point per thread up to 65536 points in FP64, two up to 131072 in FP32, then
// as many more per multiple of that.  A split launch takes rounds of 256 blocks whose waves
// share the modes.  SplitFit: the times of both forms, in us, as fitted to measurements from
// 8000 to 131072 points in FP64, 500000 in FP32 (incompressible 262144: where four rounds end),
// 100 to 4000 modes; plain base + N / rate[m], m multiples less one, split rounds times (start +
// chunk C + N / modes), C chunks of 1024 modes.  Smaller FP32 blocks (up to 65536 points) are
// faster than the split fit and always serve from 129 modes on.
// 10^4 points, 1000 modes in 2D: FP64 84 us plain, 18 split, FP32 58 and 15.  200 modes, 40000
// points in 3D, incompressible, FP64: 21 plain, 34 split; 400 modes, 190000 points, FP32: 39, 46.
struct SplitFit {
    double base, rate[4], start, chunk, modes;
};

template <bool F64, int D, bool INCOMPR>
constexpr SplitFit split_fit() {
    constexpr SplitFit k64[2][3] = {
        {{6.4, {14.3, 9.8, 9.8, 9.8}, 1.6, 7.5, 56.0}, {6.4, {12.6, 9.4, 9.4, 9.4}, 1.6, 8.1, 52.0},
         {6.4, {12.5, 8.3, 8.3, 8.3}, 1.6, 8.2, 48.0}},
        {{}, {5.0, {13.1, 8.4, 8.4, 8.4}, 2.3, 5.7, 45.0}, {5.0, {11.8, 7.0, 7.0, 7.0}, 3.8, 7.6, 40.0}}};
    constexpr SplitFit k32[2][3] = {
        {{8.0, {22.8, 15.5, 14.3, 10.8}, 3.7, 5.3, 66.0}, {8.0, {19.7, 13.9, 11.9, 8.9}, 5.0, 7.4, 57.0},
         {6.8, {18.7, 12.7, 10.2, 8.4}, 6.7, 7.4, 47.0}},
        {{}, {6.0, {17.4, 11.9, 10.6, 8.2}, 4.2, 3.9, 81.0}, {6.0, {15.4, 10.6, 8.7, 7.0}, 5.3, 6.6, 68.0}}};
    return F64 ? k64[INCOMPR][D - 1] : k32[INCOMPR][D - 1];
}

template <bool F64, int D, bool INCOMPR>
inline bool split_pays(int64_t N, int64_t P, int64_t round_points) {
    constexpr SplitFit f = split_fit<F64, D, INCOMPR>();
    const int64_t R = ceil_div(P, round_points), C = ceil_div(N, (int64_t)kSplitModes);
    if (R > 4) return false;
    if (!F64 && P <= 65536 && N > 128) return true;
    const int64_t m = ceil_div(P, (int64_t)(F64 ? 65536 : 131072));  // 1 to 4: R is at most 4
    return (double)R * (f.start + f.chunk * (double)C + (double)N / f.modes) <= f.base + (double)N / f.rate[m - 1];
}

template <int D, bool INCOMPR, class Pts, class OutT>
int launch_forward(Pts pts, int64_t N, int64_t P, const double* cov, const double* z1,
                   const double* z2, const double* fac, OutT* out, hipStream_t s) {
    if constexpr (sizeof(OutT) == 8) {
        // the smallest blocks that keep the launch within one round of 256
        if (split_pays<true, D, INCOMPR>(N, P, 256 * 128)) {
            if (P <= 256 * 32) return launch_f64_split<D, 1, 2, INCOMPR>(pts, N, P, cov, z1, z2, fac, out, s);
            if (P <= 256 * 64) return launch_f64_split<D, 2, 2, INCOMPR>(pts, N, P, cov, z1, z2, fac, out, s);
            return launch_f64_split<D, 2, 1, INCOMPR>(pts, N, P, cov, z1, z2, fac, out, s);
        }
        const int ppt = plain_ppt<true, INCOMPR>(N, P);
        auto plain = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)ceil_div(P, (int64_t)kThreads * ppt)), dim3(kThreads), 0, s, pts,
                               N, P, cov, z1, z2, fac, out);
        };
        if constexpr (!INCOMPR) {
            if (ppt == 4) {
                plain(k_forward_f64<D, 4, INCOMPR, Pts>);
                return launch_status();
            }
        }
        if (ppt == 2)
            plain(k_forward_f64<D, 2, INCOMPR, Pts>);
        else
            plain(k_forward_f64<D, 1, INCOMPR, Pts>);
    } else {
        constexpr int big = INCOMPR ? 4 : 8;  // points per thread of the largest split block
        if (split_pays<false, D, INCOMPR>(N, P, 256 * 64 * big)) {
            if (P <= 256 * 64) return launch_f32_split<D, 1, INCOMPR>(pts, N, P, cov, z1, z2, fac, out, s);
            if (P <= 256 * 128) return launch_f32_split<D, 2, INCOMPR>(pts, N, P, cov, z1, z2, fac, out, s);
            if (P <= 256 * 256) return launch_f32_split<D, 4, INCOMPR>(pts, N, P, cov, z1, z2, fac, out, s);
            return launch_f32_split<D, big, INCOMPR>(pts, N, P, cov, z1, z2, fac, out, s);
        }
        const int ppt = plain_ppt<false, INCOMPR>(N, P);
        auto plain = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)ceil_div(P, (int64_t)kThreads * ppt)), dim3(kThreads), 0, s, pts,
                               N, P, cov, z1, z2, fac, out);
        };
        if constexpr (!INCOMPR) {
            if (ppt == 8) {
                plain(k_forward_f32<D, 8, INCOMPR, Pts>);
                return launch_status();
            }
        }
        if (ppt == 4)
            plain(k_forward_f32<D, 4, INCOMPR, Pts>);
        else
            plain(k_forward_f32<D, 2, INCOMPR, Pts>);
    }
    return launch_status();
}

template <bool INCOMPR, class OutT>
int forward_unstructured(int64_t d, int64_t N, int64_t P, const double* cov, const double* z1,
                         const double* z2, const double* fac, const double* pos, OutT* out,
                         void* stream) {
    if (d < (INCOMPR ? 2 : 1) || d > 3 || N < 0 || P < 0) return GSX_E_INVALID;
    if (P == 0) return GSX_OK;
    if (!pos || !out || (N > 0 && (!cov || !z1 || !z2))) return GSX_E_INVALID;
    if (P > (int64_t)0x7fffffff * kThreads) return GSX_E_INVALID;
    hipStream_t s = as_stream(stream);
    switch (d) {
        case 1: return launch_forward<1, INCOMPR>(UnstructuredPoints<1>{pos, P}, N, P, cov, z1, z2, fac, out, s);
        case 2: return launch_forward<2, INCOMPR>(UnstructuredPoints<2>{pos, P}, N, P, cov, z1, z2, fac, out, s);
        default: return launch_forward<3, INCOMPR>(UnstructuredPoints<3>{pos, P}, N, P, cov, z1, z2, fac, out, s);
    }
}

template <class OutT, bool INCOMPR = false>
int forward_grid(int64_t d, int64_t N, const int64_t* shape, const double* axes, const double* cov,
                 const double* z1, const double* z2, const double* fac, OutT* out, void* stream) {
    if (d < (INCOMPR ? 2 : 1) || d > 3 || N < 0 || !shape) return GSX_E_INVALID;
    int64_t P = 1;
    for (int i = 0; i < d; ++i) {
        if (shape[i] < 0) return GSX_E_INVALID;
        P *= shape[i];
    }
    if (P == 0) return GSX_OK;
    if (P >= ((int64_t)1 << 32)) return GSX_E_INVALID;
    if (!axes || !out || (N > 0 && (!cov || !z1 || !z2))) return GSX_E_INVALID;
    hipStream_t s = as_stream(stream);
    const double* a0 = axes;
    const double* a1 = d > 1 ? a0 + shape[0] : nullptr;
    const double* a2 = d > 2 ? a1 + shape[1] : nullptr;
    const uint32_t n1 = d > 1 ? (uint32_t)shape[1] : 1u;
    const uint32_t n2 = d > 2 ? (uint32_t)shape[2] : 1u;
    if constexpr (INCOMPR) {
        if (d == 2) return launch_forward<2, true>(GridPoints<2>{a0, a1, a2, n1, n2}, N, P, cov, z1, z2, fac, out, s);
        return launch_forward<3, true>(GridPoints<3>{a0, a1, a2, n1, n2}, N, P, cov, z1, z2, fac, out, s);
    } else {
        switch (d) {
            case 1:
                return launch_forward<1, false>(GridPoints<1>{a0, a1, a2, n1, n2}, N, P, cov, z1, z2, fac, out, s);
            case 2:
                return launch_forward<2, false>(GridPoints<2>{a0, a1, a2, n1, n2}, N, P, cov, z1, z2, fac, out, s);
            default:
                return launch_forward<3, false>(GridPoints<3>{a0, a1, a2, n1, n2}, N, P, cov, z1, z2, fac, out, s);
        }
    }
}

}  // namespace gsx

extern "C" {

int gsx_summate_f64(int64_t d, int64_t N, int64_t P, const double* cov, const double* z1,
                    const double* z2, const double* pos, double* out, void* stream) {
    return gsx::forward_unstructured<false>(d, N, P, cov, z1, z2, nullptr, pos, out, stream);
}

int gsx_summate_f32(int64_t d, int64_t N, int64_t P, const double* cov, const double* z1,
                    const double* z2, const double* pos, float* out, void* stream) {
    return gsx::forward_unstructured<false>(d, N, P, cov, z1, z2, nullptr, pos, out, stream);
}

int gsx_summate_incompr_f64(int64_t d, int64_t N, int64_t P, const double* cov, const double* z1,
                            const double* z2, const double* pos, double* out, void* stream) {
    return gsx::forward_unstructured<true>(d, N, P, cov, z1, z2, nullptr, pos, out, stream);
}

int gsx_summate_incompr_f32(int64_t d, int64_t N, int64_t P, const double* cov, const double* z1,
                            const double* z2, const double* pos, float* out, void* stream) {
    return gsx::forward_unstructured<true>(d, N, P, cov, z1, z2, nullptr, pos, out, stream);
}

int gsx_summate_grid_f64(int64_t d, int64_t N, const int64_t* shape, const double* axes,
                         const double* cov, const double* z1, const double* z2, double* out,
                         void* stream) {
    return gsx::forward_grid(d, N, shape, axes, cov, z1, z2, nullptr, out, stream);
}

int gsx_summate_grid_f32(int64_t d, int64_t N, const int64_t* shape, const double* axes,
                         const double* cov, const double* z1, const double* z2, float* out,
                         void* stream) {
    return gsx::forward_grid(d, N, shape, axes, cov, z1, z2, nullptr, out, stream);
}

int gsx_summate_incompr_grid_f64(int64_t d, int64_t N, const int64_t* shape, const double* axes,
                                 const double* cov, const double* z1, const double* z2, double* out,
                                 void* stream) {
    return gsx::forward_grid<double, true>(d, N, shape, axes, cov, z1, z2, nullptr, out, stream);
}

int gsx_summate_incompr_grid_f32(int64_t d, int64_t N, const int64_t* shape, const double* axes,
                                 const double* cov, const double* z1, const double* z2, float* out,
                                 void* stream) {
    return gsx::forward_grid<float, true>(d, N, shape, axes, cov, z1, z2, nullptr, out, stream);
}

// Fourier method: the randomisation sum with per-mode spectrum factors.
int gsx_summate_fourier_f64(int64_t d, int64_t N, int64_t P, const double* spectrum_factor,
                            const double* modes, const double* z1, const double* z2, const double* pos,
                            double* out, void* stream) {
    if (N > 0 && !spectrum_factor) return GSX_E_INVALID;
    return gsx::forward_unstructured<false>(d, N, P, modes, z1, z2, spectrum_factor, pos, out, stream);
}

int gsx_summate_fourier_f32(int64_t d, int64_t N, int64_t P, const double* spectrum_factor,
                            const double* modes, const double* z1, const double* z2, const double* pos,
                            float* out, void* stream) {
    if (N > 0 && !spectrum_factor) return GSX_E_INVALID;
    return gsx::forward_unstructured<false>(d, N, P, modes, z1, z2, spectrum_factor, pos, out, stream);
}

int gsx_summate_fourier_grid_f64(int64_t d, int64_t N, const int64_t* shape, const double* axes,
                                 const double* spectrum_factor, const double* modes, const double* z1,
                                 const double* z2, double* out, void* stream) {
    if (N > 0 && !spectrum_factor) return GSX_E_INVALID;
    return gsx::forward_grid(d, N, shape, axes, modes, z1, z2, spectrum_factor, out, stream);
}

int gsx_summate_fourier_grid_f32(int64_t d, int64_t N, const int64_t* shape, const double* axes,
                                 const double* spectrum_factor, const double* modes, const double* z1,
                                 const double* z2, float* out, void* stream) {
    if (N > 0 && !spectrum_factor) return GSX_E_INVALID;
    return gsx::forward_grid(d, N, shape, axes, modes, z1, z2, spectrum_factor, out, stream);
}

}  // extern "C"
