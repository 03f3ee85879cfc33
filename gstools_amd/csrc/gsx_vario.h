// Device helpers and launch plumbing shared by the variogram kernels.
#pragma once
#include "gsx_internal.h"

namespace gsx {

// Largest b with e[b] <= x for non-decreasing e[0..B]; -1 if x < e[0].
__device__ __forceinline__ int64_t upper_edge(const double* e, int64_t B, double x) {
    int64_t lo = 0, hi = B + 1;  // answer in [lo - 1, hi - 1]
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (e[mid] <= x)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo - 1;
}

// T(e) = the smallest double x >= 0 with sqrt(x) >= e (sqrt correctly rounded,
// hence monotone): sqrt(d2) >= e exactly when d2 >= T(e), so bins can be found on
// squared distances with the reference's sqrt-then-compare decisions.  e <= 0
// gives -1 (every d2 >= 0 passes), e = +inf gives +inf, NaN stays NaN.
static __device__ double sq_threshold(double e) {
    if (e != e) return e;
    if (e <= 0.0) return -1.0;
    double x = e * e;
    while (sqrt(x) < e) x = nextafter(x, __builtin_inf());
    for (;;) {
        const double y = nextafter(x, 0.0);
        if (y >= 0.0 && sqrt(y) >= e && y < x)
            x = y;
        else
            break;
    }
    return x;
}

// Bytes of LDS one block may use on the current device.
int vario_lds_limit(size_t* out);

// gamma / counts of slots [h0, h0 + NH) from per-block partials ([slot][block]):
// sums in a fixed order; accumulate adds to what is there, finish turns the sums
// into estimates (Matheron or Cressie).
int vario_collect(int64_t blocks, int64_t NH, int64_t h0, const double* part_sum, const unsigned long long* part_cnt,
                  double* gamma, int64_t* counts, bool accumulate, bool finish, int cressie, hipStream_t s);

// Omnidirectional estimate of one field (F = 1) on Euclidean distances
// (gsx_vario_iso.hip).  vario_iso_ws: its workspace bytes.
int64_t vario_iso_ws(int64_t P, int64_t dim, int64_t B);
int vario_iso(int64_t P, int64_t dim, int64_t B, const double* f, const double* edges, const double* pos,
              int estimator, double* gamma, int64_t* counts, void* ws, hipStream_t s);

}  // namespace gsx
