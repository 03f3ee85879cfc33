// Omnidirectional empirical variogram of one field: the pair kernel of the
// unstructured estimator on Euclidean distances (reference contract in
// gsx_variogram.hip).
//
// Work unit: 64 points j (one per lane) x 64 points k.  A block is one
// wavefront with one histogram column per lane in LDS (12 bytes per bin and
// lane), so the number of wavefronts in flight is set by the bins alone and not
// rounded down to whole 256-thread blocks (26 bins: 7 per CU instead of 4).  The
// k points are wave-uniform and come through scalar loads: staged in LDS and
// read as broadcasts they took about half of the LDS cycles of a pair, and LDS,
// not the vector unit, set the pace.
//
// Bins.  A pair belongs to the bin of its FP64 distance, rounded as the
// reference rounds it.  For uniformly spaced edges an FP32 distance between
// FP32 coordinates (relative to the centre of the bounding box) gives the
// position q = (d - e0) / w in the bins with an error below eps (derived at
// `eps` below); unless q lies within eps of an edge that decides the bin.
// Otherwise, about once in 10^4 pairs, the whole batch of 4 k points is done
// again in FP64: squared distance with the reference's roundings, compared with
// the thresholds T(edge) (sq_threshold).  Batches that the FP32 form does not
// cover (non-finite coordinates, NaN values, edges that are not uniform or too
// close for FP32) take the FP64 form only.
//
// Order of the points.  Beyond kSortMin points they are sorted by cell along a
// Hilbert curve (counting sort; ties by index, so the order, and with it every
// sum, is reproducible), points with a NaN value are dropped and those with a
// non-finite coordinate go last.  Every 64-point tile has a bounding box; a tile
// pair whose boxes are at least the last edge apart is skipped.  The box
// distance is computed with the operations and roundings of a pair's squared
// distance from per-axis gaps that bound the pair's differences, and rounding is
// monotone, so no pair of a skipped tile lies in a bin.
#include <type_traits>

#include "gsx_vario.h"

namespace gsx {

namespace {

constexpr int64_t kSortMin = 12288;   // points from which sorting pays (prepared in one launch below)
constexpr int kBoxBlocks = 64;        // blocks of the bounding-box pass
constexpr int kCellBits = 15;         // cells 2^15: 15, 7 or 5 bits per axis
constexpr int kCells = 1 << kCellBits;
constexpr unsigned kCellMax = 4096;
constexpr int kBatch = 4;             // k points per step
constexpr int kSlotsMax = 48;         // histogram slots per launch (4 wavefronts per CU)
constexpr int kRowBytes = 64 * 12;    // one histogram row: 64 sums, then 64 counts
constexpr int kTilePad = 64;
constexpr int64_t kLds = 163840;      // LDS of a CU

struct IsoMeta {
    double lo[3];        // of the finite coordinates
    double centre[3];
    double diag;         // of the bounding box
    double cell_scale;   // cells per unit length
    int64_t nv;          // points kept
    int sorted;          // the points are in cell order (else in the given one, all kept)
};

// The edges, looked at once: thp holds -inf, T(e_0) .. T(e_B), +inf.
struct IsoEdges {
    double e0, emax, inv_w;
    double dev;          // largest distance of an edge from uniform spacing, in bins
    int mono, uniform;
};

struct IsoArgs {
    int64_t B;
    int64_t h0, h1;      // slots (bins) of this launch
    int gl2;             // log2 of the k tiles per work item (<= 6)
};

// Workspace layout (bytes, every part 256-byte aligned).
struct IsoLayout {
    int64_t Pp, nt;                                     // padded points, tiles
    int64_t meta, flagged, edges, thp;                  // flagged (int): some tile may have a flag (tile_box)
    int64_t bounds, rec, drec, box, flags;              // prepared points
    int64_t cell, arrival, list, count, start;          // sort
    int64_t part_sum, part_cnt, blocks, slots, total;   // partials
    bool sorted;
};

// Work items: groups of 2^gl2 k tiles for every j tile (half of them left of the
// diagonal); single tile pairs of the upper triangle for gl2 = 0.
__host__ __device__ inline int64_t iso_items(int64_t nt, int gl2) {
    return gl2 == 0 ? nt * (nt + 1) / 2 : nt * ((nt + ((int64_t)1 << gl2) - 1) >> gl2);
}

// k tiles per work item: as many as leave 2^18 items, about 100 per wavefront
// (half of them left of the diagonal; with 17 per wavefront the most loaded one
// took twice the mean)
inline int iso_group_log2(int64_t nt) {
    int g = 6;
    while (g > 0 && iso_items(nt, g) < ((int64_t)1 << 18)) --g;
    return g;
}

inline size_t iso_lds_bytes(int64_t B, int64_t NH) {
    return sizeof(double) * (size_t)(B + 3) + (size_t)(NH + 2) * kRowBytes;
}

// A k point as the pair loop reads it: FP32 coordinates relative to the centre, the
// value as FP64 in the last two words; for the FP64 form the coordinates and value as
// dim + 1 doubles.
constexpr int iso_rec_words(int64_t dim) { return dim == 3 ? 6 : 4; }

inline IsoLayout iso_layout(int64_t P, int64_t dim, int64_t B) {
    IsoLayout l;
    l.nt = ceil_div(P, (int64_t)64);
    l.Pp = l.nt * 64 + kTilePad;
    l.sorted = P >= kSortMin;
    // very many bins: the edges and thresholds take LDS from the histogram
    l.slots = (kLds - (int64_t)iso_lds_bytes(B, 0) - 64 * 4 * 8) / kRowBytes;
    if (l.slots > kSlotsMax) l.slots = kSlotsMax;
    if (l.slots > B) l.slots = B;
    if (l.slots < 1) l.slots = 1;
    // wavefronts that fit the LDS of 256 CUs (at most 16 per CU), four times over: the
    // work of a block is fixed (its sums have a fixed order), so the blocks that start
    // when others end even out what 9 wavefronts on 4 SIMDs do not (1e5 points, 20 bins:
    // 3.15 ms with one round of blocks); enough that no lane sees 2^32 pairs
    int64_t per_cu = kLds / (int64_t)iso_lds_bytes(B, l.slots);
    per_cu = per_cu < 1 ? 1 : (per_cu > 16 ? 16 : per_cu);
    int64_t blocks = 256 * per_cu * 4;
    const double lane_pairs = 64.0 * (double)l.nt * (double)(l.nt + 1);
    if (lane_pairs / 4.0e9 > (double)blocks) blocks = (int64_t)(lane_pairs / 4.0e9) + 1;
    const int64_t items = iso_items(l.nt, iso_group_log2(l.nt));
    if (items < 64 * blocks / 4) {
        // few items per block: one round of blocks with equal numbers of items
        const int64_t each = ceil_div(items, 256 * per_cu);
        blocks = each > 0 ? ceil_div(items, each) : 1;
    }
    l.blocks = blocks;
    int64_t o = 0;
    auto take = [&](int64_t bytes) {
        const int64_t at = o;
        o += ceil_div(bytes, (int64_t)256) * 256;
        return at;
    };
    l.meta = take(sizeof(IsoMeta));
    l.flagged = take(4);
    l.edges = take(sizeof(IsoEdges));
    l.thp = take((B + 3) * 8);
    l.bounds = take((int64_t)kBoxBlocks * 6 * 8);
    l.rec = take(l.Pp * iso_rec_words(dim) * 4);
    l.drec = take(l.Pp * (dim + 1) * 8);
    l.box = take(2 * dim * l.nt * 8);
    l.flags = take(l.nt * 4);
    const int64_t n = l.sorted ? P : 0;
    l.cell = take(n * 4);
    l.arrival = take(n * 4);
    l.list = take(n * 4);
    l.count = take(l.sorted ? (kCells + 2) * 4 : 0);
    l.start = take(l.sorted ? (kCells + 3) * 4 : 0);
    l.part_sum = take(2 * l.blocks * l.slots * 8);
    l.part_cnt = take(2 * l.blocks * l.slots * 8);
    l.total = o;
    return l;
}

// One wavefront: thresholds, order and spacing of the edges.
__device__ void edge_setup(int B, const double* __restrict__ edges, double* __restrict__ thp,
                           IsoEdges* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const double e0 = edges[0], eB = edges[B];
    const double emax = fmax(fabs(e0), fabs(eB));
    const double w = (eB - e0) / B;
    bool mono_l = true;
    double dev = 0.0;
    for (int i = lane; i <= B; i += 64) {
        const double e = edges[i];
        thp[i + 1] = sq_threshold(e);
        if (i < B) mono_l = mono_l && (e <= edges[i + 1]);
        const double x = fabs(e - (e0 + i * w)) / w;
        dev = x <= dev || dev != dev ? dev : x;  // NaN is kept
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double x = __shfl_xor(dev, o);
        dev = x <= dev || dev != dev ? dev : x;
    }
    const bool mono = __all(mono_l);
    // uniform: the FP32 guess of the FP64 form is exact after one threshold step
    // (every edge within w / 4 of uniform, w not below 4e-6 of the edges nor of the
    // distances whose squares underflow FP32)
    const bool uniform = mono && w >= 1.0e-15 && emax < 1.0e18 && w >= 4.0e-6 * emax && dev <= 0.25;
    if (lane == 0) {
        thp[0] = -__builtin_inf();
        thp[B + 2] = __builtin_inf();
        IsoEdges e;
        e.e0 = e0;
        e.emax = emax;
        e.inv_w = uniform ? 1.0 / w : 0.0;
        e.dev = dev;
        e.mono = mono;
        e.uniform = uniform;
        *out = e;
    }
}

// Running bounds over finite coordinates, reduced over the block: bb[0..2] the
// minima, bb[3..5] the maxima (+inf / -inf where there is none).
template <int DIM>
__device__ void block_bounds(int64_t i0, int64_t step, int64_t P, const double* __restrict__ pos, double* bb,
                             double (*red)[6]) {
    double lo[DIM], hi[DIM];
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
        lo[c] = __builtin_inf();
        hi[c] = -__builtin_inf();
    }
#pragma unroll 4
    for (int64_t i = i0; i < P; i += step) {
#pragma unroll
        for (int c = 0; c < DIM; ++c) {
            const double v = pos[c * P + i];
            if (__builtin_isfinite(v)) {
                lo[c] = fmin(lo[c], v);
                hi[c] = fmax(hi[c], v);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < DIM; ++c)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            lo[c] = fmin(lo[c], __shfl_xor(lo[c], o));
            hi[c] = fmax(hi[c], __shfl_xor(hi[c], o));
        }
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int c = 0; c < DIM; ++c) {
            red[threadIdx.x >> 6][c] = lo[c];
            red[threadIdx.x >> 6][3 + c] = hi[c];
        }
    __syncthreads();
    if (threadIdx.x < DIM) {
        double l = red[0][threadIdx.x], h = red[0][3 + threadIdx.x];
        for (int w = 1; w < (int)blockDim.x / 64; ++w) {
            l = fmin(l, red[w][threadIdx.x]);
            h = fmax(h, red[w][3 + threadIdx.x]);
        }
        bb[threadIdx.x] = l;
        bb[3 + threadIdx.x] = h;
    }
    __syncthreads();
}

// Centre, diagonal and cell size from the bounds.
template <int DIM>
__device__ IsoMeta meta_of(const double* bb) {
    IsoMeta m;
    double d2 = 0.0, ext = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        m.lo[c] = 0.0;
        m.centre[c] = 0.0;
    }
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
        double l = bb[c], h = bb[3 + c];
        if (!(l <= h)) l = h = 0.0;
        const double e = h - l;
        m.lo[c] = l;
        m.centre[c] = l + 0.5 * e;
        d2 += e * e;
        ext = fmax(ext, e);
    }
    m.diag = sqrt(d2);
    m.cell_scale = ext > 0.0 ? (double)(1 << (kCellBits / DIM)) / ext : 0.0;
    m.nv = 0;
    m.sorted = 0;
    return m;
}

// Bounds of the points over kBoxBlocks blocks; clears the cell counts.  One more
// block looks at the edges.
template <int DIM>
__global__ __launch_bounds__(256) void k_iso_bounds(int64_t P, const double* __restrict__ pos,
                                                    double* __restrict__ bounds, unsigned* __restrict__ count, int B,
                                                    const double* __restrict__ edges, double* __restrict__ thp,
                                                    IsoEdges* __restrict__ ed) {
    __shared__ double red[4][6], bb[6];
    if (blockIdx.x == kBoxBlocks) {
        if (threadIdx.x < 64) edge_setup(B, edges, thp, ed);
        return;
    }
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    for (int64_t q = i; q < kCells + 2; q += (int64_t)kBoxBlocks * 256) count[q] = 0u;
    block_bounds<DIM>(i, (int64_t)kBoxBlocks * 256, P, pos, bb, red);
    if (threadIdx.x < 6) bounds[blockIdx.x * 6 + threadIdx.x] = (threadIdx.x % 3) < DIM ? bb[threadIdx.x] : 0.0;
}

// Every block reduces the bounds again (64 entries) and sorts its points into
// cells: Hilbert index of the cell, kCells for a non-finite coordinate, kCells + 1
// for a NaN value.  Block 0 writes the metadata.
template <int DIM>
__global__ __launch_bounds__(256) void k_iso_cells(int64_t P, const double* __restrict__ pos,
                                                   const double* __restrict__ f, const double* __restrict__ bounds,
                                                   IsoMeta* __restrict__ meta, unsigned* __restrict__ cell,
                                                   unsigned* __restrict__ arrival, unsigned* __restrict__ count) {
    __shared__ double bb[6];
    if (threadIdx.x < 64) {
        double v[2 * DIM];
#pragma unroll
        for (int c = 0; c < DIM; ++c) {
            v[c] = bounds[threadIdx.x * 6 + c];
            v[DIM + c] = bounds[threadIdx.x * 6 + 3 + c];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                v[c] = fmin(v[c], __shfl_xor(v[c], o));
                v[DIM + c] = fmax(v[DIM + c], __shfl_xor(v[DIM + c], o));
            }
        }
        if (threadIdx.x == 0)
#pragma unroll
            for (int c = 0; c < DIM; ++c) {
                bb[c] = v[c];
                bb[3 + c] = v[DIM + c];
            }
    }
    __syncthreads();
    const IsoMeta m = meta_of<DIM>(bb);
    if (blockIdx.x == 0 && threadIdx.x == 0) *meta = m;  // nv, sorted: k_iso_scan
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= P) return;
    constexpr int bits = kCellBits / DIM;
    unsigned key = 0;
    bool fin = true;
    unsigned q[DIM];
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
        const double v = pos[c * P + i];
        fin = fin && __builtin_isfinite(v);
        q[c] = (unsigned)fmin(fmax((v - m.lo[c]) * m.cell_scale, 0.0), (double)((1 << bits) - 1));
    }
    if constexpr (DIM > 1) {
        // Hilbert index of the cell (J. Skilling, "Programming the Hilbert curve", 2004:
        // undo the excess work bit by bit, then Gray-encode)
        for (unsigned top = 1u << (bits - 1); top > 1u; top >>= 1) {
            const unsigned low = top - 1u;
#pragma unroll
            for (int c = 0; c < DIM; ++c) {
                const unsigned swap = (q[c] & top) ? low : (q[0] ^ q[c]) & low;
                if (!(q[c] & top)) q[c] ^= swap;
                q[0] ^= swap;
            }
        }
#pragma unroll
        for (int c = 1; c < DIM; ++c) q[c] ^= q[c - 1];
        unsigned gray = 0;
        for (unsigned top = 1u << (bits - 1); top > 1u; top >>= 1)
            if (q[DIM - 1] & top) gray ^= top - 1u;
#pragma unroll
        for (int c = 0; c < DIM; ++c) q[c] ^= gray;
    }
#pragma unroll
    for (int b = 0; b < bits; ++b)
#pragma unroll
        for (int c = 0; c < DIM; ++c) key |= ((q[c] >> b) & 1u) << (b * DIM + DIM - 1 - c);
    const double fv = f[i];
    if (!fin) key = kCells;
    if (fv != fv) key = kCells + 1;
    cell[i] = key;
    arrival[i] = atomicAdd(&count[key], 1u);
}

// Exclusive scan of the cell counts (one block); kept points: those before cell
// kCells + 1.  A cell of more than kCellMax points (clustered data, a far outlier) leaves
// the points in the given order: the rank within a cell takes its square.
__global__ __launch_bounds__(1024) void k_iso_scan(int64_t P, const unsigned* __restrict__ count,
                                                   unsigned* __restrict__ start, IsoMeta* __restrict__ meta,
                                                   int* __restrict__ flagged) {
    __shared__ unsigned wsum[16];
    bool crowded = false;
    constexpr int per = kCells / 1024;
    const int t = threadIdx.x, lane = t & 63;
    unsigned v[per], s = 0;
#pragma unroll
    for (int q = 0; q < per; ++q) {
        v[q] = count[t * per + q];
        s += v[q];
        crowded = crowded || v[q] > kCellMax;
    }
    if (t == 0) crowded = crowded || count[kCells] > kCellMax;
    const bool sorted = __syncthreads_or(crowded ? 1 : 0) == 0;
    unsigned inc = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned u = __shfl_up(inc, o);
        if (lane >= o) inc += u;
    }
    if (lane == 63) wsum[t >> 6] = inc;
    __syncthreads();
    unsigned base = 0, total = 0;
    for (int w = 0; w < 16; ++w) {
        if (w < (t >> 6)) base += wsum[w];
        total += wsum[w];
    }
    unsigned at = base + inc - s;
#pragma unroll
    for (int q = 0; q < per; ++q) {
        start[t * per + q] = at;
        at += v[q];
    }
    if (t == 0) {
        const unsigned bad = count[kCells];
        start[kCells] = total;
        start[kCells + 1] = total + bad;
        start[kCells + 2] = total + bad + count[kCells + 1];
        meta->sorted = sorted ? 1 : 0;
        *flagged = bad != 0u || (!sorted && count[kCells + 1] != 0u) ? 1 : 0;
        meta->nv = sorted ? (int64_t)total + bad : P;
    }
}

__global__ __launch_bounds__(256) void k_iso_list(int64_t P, const unsigned* __restrict__ cell,
                                                  const unsigned* __restrict__ arrival,
                                                  const unsigned* __restrict__ start, unsigned* __restrict__ list) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < P) list[start[cell[i]] + arrival[i]] = (unsigned)i;
}

template <int DIM>
__device__ __forceinline__ void put_point(int64_t i, int64_t at, int64_t P, const IsoMeta& m,
                                          const double* __restrict__ pos, const double* __restrict__ f,
                                          uint32_t* __restrict__ rec, double* __restrict__ drec) {
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
        const double v = pos[c * P + i];
        drec[at * (DIM + 1) + c] = v;
        rec[at * iso_rec_words(DIM) + c] = __float_as_uint((float)(v - m.centre[c]));
    }
    const double fv = f[i];
    drec[at * (DIM + 1) + DIM] = fv;
    *reinterpret_cast<double*>(rec + (at + 1) * iso_rec_words(DIM) - 2) = fv;
}

// Points into their sorted places: cell start + rank of the index within the
// cell (the arrival order of the atomics does not matter).
template <int DIM>
__global__ __launch_bounds__(256) void k_iso_place(int64_t P, const IsoMeta* __restrict__ meta,
                                                   const double* __restrict__ pos, const double* __restrict__ f,
                                                   const unsigned* __restrict__ cell,
                                                   const unsigned* __restrict__ start,
                                                   const unsigned* __restrict__ list, uint32_t* __restrict__ rec,
                                                   double* __restrict__ drec) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= P) return;
    int64_t at = i;
    if (meta->sorted) {
        const unsigned key = cell[i];
        if (key == kCells + 1) return;  // dropped
        const unsigned s = start[key], e = start[key + 1];
        unsigned rank = 0;
        for (unsigned q = s; q < e; ++q) rank += list[q] < (unsigned)i ? 1u : 0u;
        at = (int64_t)s + rank;
    }
    put_point<DIM>(i, at, P, *meta, pos, f, rec, drec);
}

// Bounding box and flag of one tile by one wavefront: flag 1 if a point has a
// non-finite coordinate (no box then), 2 if one has a NaN value.
template <int DIM>
__device__ void tile_box(int64_t tile, int64_t nt, int64_t nv, const double* __restrict__ drec,
                         double* __restrict__ box, unsigned* __restrict__ flags) {
    const int lane = threadIdx.x & 63;
    const int64_t i = tile * 64 + lane;
    const bool live = i < nv;
    unsigned flag = 0;
    double v[DIM];
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
        v[c] = live ? drec[i * (DIM + 1) + c] : 0.0;
        if (!__builtin_isfinite(v[c])) flag |= 1u;
    }
    if (live) {
        const double fv = drec[i * (DIM + 1) + DIM];
        if (fv != fv) flag |= 2u;
    }
    flag = (__any(flag & 1u) ? 1u : 0u) | (__any(flag & 2u) ? 2u : 0u);
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
        double lo = live ? v[c] : __builtin_inf(), hi = live ? v[c] : -__builtin_inf();
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            lo = fmin(lo, __shfl_xor(lo, o));
            hi = fmax(hi, __shfl_xor(hi, o));
        }
        if (lane == 0) {
            box[(2 * c) * nt + tile] = lo;
            box[(2 * c + 1) * nt + tile] = hi;
        }
    }
    if (lane == 0) flags[tile] = flag;
}

template <int DIM>
__global__ __launch_bounds__(256) void k_iso_boxes(int64_t nt, const IsoMeta* __restrict__ meta,
                                                   const double* __restrict__ drec, double* __restrict__ box,
                                                   unsigned* __restrict__ flags) {
    const int64_t tile = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tile >= nt) return;  // whole wavefront
    tile_box<DIM>(tile, nt, meta->nv, drec, box, flags);
}

// Few points: bounds (every block over all points), places in the given order
// and boxes in one launch.
template <int DIM>
__global__ __launch_bounds__(1024) void k_iso_prepare(int64_t P, int64_t nt,
                                                      const double* __restrict__ pos, const double* __restrict__ f,
                                                      IsoMeta* __restrict__ meta, uint32_t* __restrict__ rec,
                                                      double* __restrict__ drec, double* __restrict__ box,
                                                      unsigned* __restrict__ flags, int B,
                                                      const double* __restrict__ edges, double* __restrict__ thp,
                                                      IsoEdges* __restrict__ ed, int* __restrict__ flagged) {
    __shared__ double red[16][6], bb[6];
    if (blockIdx.x == gridDim.x - 1) {  // one more block looks at the edges and for odd points
        if (threadIdx.x < 64) edge_setup(B, edges, thp, ed);
        bool odd = false;
#pragma unroll 4
        for (int64_t q = threadIdx.x; q < P; q += 1024) {
            const double fv = f[q];
            odd = odd || fv != fv;
#pragma unroll
            for (int c = 0; c < DIM; ++c) odd = odd || !__builtin_isfinite(pos[c * P + q]);
        }
        const int any = __syncthreads_or(odd ? 1 : 0);
        if (threadIdx.x == 0) *flagged = any;
        return;
    }
    block_bounds<DIM>(threadIdx.x, 1024, P, pos, bb, red);
    IsoMeta m = meta_of<DIM>(bb);
    m.nv = P;
    if (blockIdx.x == 0 && threadIdx.x == 0) *meta = m;
    const int64_t i = (int64_t)blockIdx.x * 1024 + threadIdx.x;
    if (i < P) put_point<DIM>(i, i, P, m, pos, f, rec, drec);
    __syncthreads();  // a tile's points were written by its own wavefront
    const int64_t tile = i >> 6;
    if (tile < nt) tile_box<DIM>(tile, nt, P, drec, box, flags);
}

// One pair into a histogram row; col: LDS offset of this lane's column (8 * lane from the first row).
__device__ __forceinline__ void iso_add(unsigned char* lds, unsigned col, unsigned lane4, int row, double v) {
    const unsigned at = __umul24((unsigned)row, (unsigned)kRowBytes) + col;
    // the column is the lane's own and adds to one location take effect in issue
    // order: every slot adds its pairs in pair order
    __hip_atomic_fetch_add(reinterpret_cast<double*>(lds + at), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(reinterpret_cast<unsigned*>(lds + (at - lane4) + 512u), 1u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Position errors of the FP32 form and whether it serves these edges and points.
struct IsoFast {
    bool on;
    double eps;
};

__device__ __forceinline__ IsoFast iso_fast(const IsoEdges& e, double diag, int B) {
    // Coordinates relative to the centre are rounded to 2^-25 of the extent and
    // differences to 2^-24, so |d32 - d| <= 2^-24 (diag + d) plus 3.5 roundings of the
    // squares, sums and root (v_sqrt_f32: one ulp); scaling and offset add
    // 2^-24 (d / w + |e0| / w + B + 2).  Up to the last edge d <= emax; doubled, and the
    // edges' own deviation from uniform on top.  Squares below 2^-126 count as 0 (v_sqrt_f32
    // takes no denormal numbers): up to sqrt(3) 2^-63 of a distance, below 2^-62.
    IsoFast r;
    r.eps = 0x1p-23 * ((diag + 6.5 * e.emax) * e.inv_w + fabs(e.e0) * e.inv_w + B + 4.0) + e.dev + 0x1p-62 * e.inv_w;
    // (a batch of 256 pairs is done again with a chance of up to 512 eps)
    r.on = e.uniform != 0 && diag < 1.0e18 && r.eps <= 0x1p-11;
    return r;
}

// kBatch k points in scalar registers.
typedef __attribute__((ext_vector_type(8))) uint32_t u32x8;

template <int DIM>
struct KPoints {
    static constexpr int kRec = iso_rec_words(DIM), kVec = kRec * kBatch / 8;
    u32x8 v[kVec];
    __device__ __forceinline__ float x(int u, int c) const {
        return __uint_as_float(v[(u * kRec + c) / 8][(u * kRec + c) % 8]);
    }
    __device__ __forceinline__ double f(int u) const {
        const int w = (u + 1) * kRec - 2;
        return __builtin_bit_cast(double, (uint64_t)v[(w + 1) / 8][(w + 1) % 8] << 32 | v[w / 8][w % 8]);
    }
    __device__ __forceinline__ void load(const uint32_t* __restrict__ rec, int k) {
        const u32x8* r = reinterpret_cast<const u32x8*>(rec + (int64_t)k * kRec);
#pragma unroll
        for (int q = 0; q < kVec; ++q) v[q] = r[q];
    }
    // Waits for the loads before anything that depends on the returned index: scalar
    // loads return out of order, so a later load would be waited for too.
    __device__ __forceinline__ int ready(int k) const {
        if constexpr (kVec == 3)
            asm volatile("" : "+s"(k) : "s"(v[0]), "s"(v[1]), "s"(v[2]));
        else
            asm volatile("" : "+s"(k) : "s"(v[0]), "s"(v[1]));
        return k;
    }
};

// Pairs of all work items into the histograms.  EXACT = false: the FP32 form (with
// single batches again in FP64) for tiles without a flag, where it serves the edges
// (else the launch does nothing); EXACT = true: everything else, in the FP64 form,
// with the k tile staged in LDS (its threshold reads wait for LDS only; behind scalar
// loads they ran at half the rate).  part: 2 x gridDim.x columns of partials, this
// launch's from EXACT * gridDim.x on.
template <int DIM, bool CRESSIE, bool EXACT>
__global__ __launch_bounds__(64, 4) void k_iso_pairs(IsoArgs a, const IsoMeta* __restrict__ meta,
                                                     const int* __restrict__ flagged,
                                                     const IsoEdges* __restrict__ ed, const double* __restrict__ thp,
                                                     const double* __restrict__ edges,
                                                     const uint32_t* __restrict__ rec,
                                                     const double* __restrict__ drec, const double* __restrict__ box,
                                                     const unsigned* __restrict__ flags, int64_t nt_stride,
                                                     double* __restrict__ part_sum,
                                                     unsigned long long* __restrict__ part_cnt) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) unsigned char vlds[];
    const int B = (int)a.B, NH = (int)(a.h1 - a.h0), h0 = (int)a.h0;
    const int lane = (int)threadIdx.x;
    const IsoFast ff = iso_fast(*ed, meta->diag, B);
    const int64_t pcol = (int64_t)blockIdx.x + (EXACT ? gridDim.x : 0), pcols = 2 * (int64_t)gridDim.x;
    if (EXACT ? (ff.on && !*flagged) : !ff.on) {
        for (int h = lane; h < NH; h += 64) {
            part_sum[h * pcols + pcol] = 0.0;
            part_cnt[h * pcols + pcol] = 0ull;
        }
        return;
    }
    double* s_thp = reinterpret_cast<double*>(vlds);  // -inf, T(e_0) .. T(e_B), +inf
    double* s_thr = s_thp + 1;
    double* s_k = s_thp + (B + 3);                    // EXACT: the k tile
    unsigned char* hist =                             // rows 0 and NH + 1: scratch
        reinterpret_cast<unsigned char*>(s_k + (EXACT ? 64 * (DIM + 1) : 0));
    const unsigned col = (unsigned)(hist - vlds) + 8u * lane, lane4 = 4u * lane;

    for (int i = lane; i < B + 3; i += 64) s_thp[i] = thp[i];
    for (int r = 0; r < NH + 2; ++r) {
        reinterpret_cast<double*>(hist + r * kRowBytes)[lane] = 0.0;
        reinterpret_cast<unsigned*>(hist + r * kRowBytes + 512)[lane] = 0u;
    }
    __syncthreads();
    const bool mono = !EXACT || ed->mono != 0, uniform = !EXACT || ed->uniform != 0;
    const float inv_wf = (float)ed->inv_w, qoff = (float)(-ed->e0 * ed->inv_w);
    const float near_f = (float)(0.5 - ff.eps);  // |q - (floor(q) + 1/2)| below this: decided
    const float q1off = qoff + (float)(1 - h0), qtop = (float)NH + 1.5f;
    const double thr_last = s_thr[B];

    const int nv = (int)meta->nv;  // < 2^26 (the launch refuses more)
    const int nt = (nv + 63) >> 6;
    const int ng = (nt + (1 << a.gl2) - 1) >> a.gl2;
    const int64_t items = iso_items(nt, a.gl2);
    double nan_sum = 0.0;  // NaN-distance pairs of this lane (every bin takes them)
    unsigned nan_cnt = 0u;

    for (int64_t it = blockIdx.x; it < items; it += gridDim.x) {
        // skewed, so that a stride that is a multiple of ng still walks all groups
        int tj, gk;
        if (a.gl2 == 0) {
            // it = gk (gk + 1) / 2 + tj, tj <= gk
            gk = (int)((sqrt(8.0 * (double)it + 1.0) - 1.0) * 0.5);
            while ((int64_t)gk * (gk + 1) / 2 > it) --gk;
            while ((int64_t)(gk + 1) * (gk + 2) / 2 <= it) ++gk;
            tj = (int)(it - (int64_t)gk * (gk + 1) / 2);
        } else {
            tj = (int)(it / ng);
            gk = (int)((it + tj) % ng);
        }
        tj = __builtin_amdgcn_readfirstlane(tj);
        gk = __builtin_amdgcn_readfirstlane(gk);
        const int t0 = gk << a.gl2;
        const int t1 = t0 + (1 << a.gl2) < nt ? t0 + (1 << a.gl2) : nt;
        if (t1 <= tj) continue;
        // tiles of this item that may hold a pair within the last edge, of this launch's kind
        unsigned long long todo;
        {
            const int tk = t0 + lane;
            bool in = tk < t1 && tk >= tj;
            if (in) {
                const unsigned flag = flags[tj] | flags[tk];
                if (EXACT ? (ff.on && flag == 0u) : flag != 0u) in = false;
                if (in && mono && (flag & 1u) == 0u) {
                    double d2 = 0.0;
#pragma unroll
                    for (int c = 0; c < DIM; ++c) {
                        const double lo_j = box[(2 * c) * nt_stride + tj], hi_j = box[(2 * c + 1) * nt_stride + tj];
                        const double lo_k = box[(2 * c) * nt_stride + tk], hi_k = box[(2 * c + 1) * nt_stride + tk];
                        const double gap = fmax(fmax(lo_k - hi_j, lo_j - hi_k), 0.0);
                        d2 += gap * gap;
                    }
                    in = !(d2 >= thr_last);
                }
            }
            todo = __ballot(in);
        }
        if (todo == 0ull) continue;
        const int j = tj * 64 + lane;
        const bool live_j = j < nv;
        const int jc = live_j ? j : nv - 1;
        float xj[DIM];
        double pj[DIM];
#pragma unroll
        for (int c = 0; c < DIM; ++c) {
            if (!EXACT) xj[c] = __uint_as_float(rec[(int64_t)jc * iso_rec_words(DIM) + c]);
            pj[c] = drec[(int64_t)jc * (DIM + 1) + c];
        }
        const double fj = drec[(int64_t)jc * (DIM + 1) + DIM];
        auto value = [&](double fk) {
            const double x = fk - fj;
            return CRESSIE ? sqrt(fabs(x)) : x * x;
        };
        // bin of a squared distance for uniform edges: an FP32 guess within one bin of the
        // true one, then one threshold step each way
        auto uniform_bin = [&](double d2) {
            float q = __builtin_fmaf(__builtin_amdgcn_sqrtf((float)d2), inv_wf, qoff);
            if (EXACT) q = (d2 == d2) ? q : -1.0f;
            q = __builtin_amdgcn_fmed3f(q, -1.0f, (float)B);
            const int g0 = (int)q;  // -1 .. B
            return g0 - (s_thp[g0 + 1] > d2 ? 1 : 0) + (s_thp[g0 + 2] <= d2 ? 1 : 0);
        };
        if constexpr (EXACT) {
            double kreg[DIM + 1];  // the next k tile, one point per lane
            auto fetch = [&](int tk) {
                const int k = tk * 64 + lane < nv ? tk * 64 + lane : nv - 1;
#pragma unroll
                for (int c = 0; c <= DIM; ++c) kreg[c] = drec[(int64_t)k * (DIM + 1) + c];
            };
            fetch(t0 + __builtin_ctzll(todo));
            while (todo) {
                const int tk = t0 + __builtin_ctzll(todo);
                todo &= todo - 1ull;
                __syncthreads();  // the last tile is no longer read
#pragma unroll
                for (int c = 0; c <= DIM; ++c) s_k[lane * (DIM + 1) + c] = kreg[c];
                __syncthreads();
                if (todo) fetch(t0 + __builtin_ctzll(todo));
                const int kn = nv - tk * 64 < 64 ? nv - tk * 64 : 64;
                // point kk of the tile is paired with this lane's
                auto counts = [&](int kk, double fk) {
                    return kk < kn && live_j && (tk != tj || kk > lane) && fk == fk && fj == fj;
                };
                if (!mono) {
                    // the reference's comparisons, bin by bin
                    for (int kk = 0; kk < kn; ++kk) {
                        const double* p = s_k + kk * (DIM + 1);
                        double d2 = 0.0;
#pragma unroll
                        for (int c = 0; c < DIM; ++c) {
                            const double dd = p[c] - pj[c];
                            d2 += dd * dd;
                        }
                        const double dist = sqrt(d2), v = value(p[DIM]);
                        const bool ok = counts(kk, p[DIM]);
                        for (int b = 0; ok && b < NH; ++b)
                            if (!(dist < edges[h0 + b] || dist >= edges[h0 + b + 1]))
                                iso_add(vlds, col, lane4, b + 1, v);
                    }
                    continue;
                }
                // eight pairs per step, their threshold reads overlapping.  CLEAN: a whole tile
                // right of the diagonal with finite coordinates and no NaN value
                auto run = [&](auto uni, auto clean) {
                    constexpr bool UNI = decltype(uni)::value, CLEAN = decltype(clean)::value;
                    for (int k8 = 0; k8 < kn; k8 += 8) {
                        int row[8];
                        double val[8];
#pragma unroll
                        for (int u = 0; u < 8; ++u) {
                            const double* p = s_k + (k8 + u) * (DIM + 1);
                            double d2 = 0.0;
#pragma unroll
                            for (int c = 0; c < DIM; ++c) {
                                const double dd = p[c] - pj[c];
                                d2 += dd * dd;
                            }
                            val[u] = value(p[DIM]);
                            bool ok = true;
                            if constexpr (!CLEAN) {
                                ok = counts(k8 + u, p[DIM]);
                                const bool dnan = d2 != d2;  // in every bin by the reference's comparisons
                                nan_sum += (dnan && ok) ? val[u] : 0.0;
                                nan_cnt += (dnan && ok) ? 1u : 0u;
                                ok = ok && !dnan;
                            }
                            int g = UNI ? uniform_bin(d2) : (int)upper_edge(s_thr, B, d2);
                            // opaque, so that the search stays unconditional and its reads overlap
                            asm volatile("" : "+v"(g));
                            const unsigned sl = (unsigned)(g - h0);
                            row[u] = (ok && sl < (unsigned)NH) ? (int)sl + 1 : 0;
                        }
#pragma unroll
                        for (int u = 0; u < 8; ++u) iso_add(vlds, col, lane4, row[u], val[u]);
                    }
                };
                const bool clean = kn == 64 && tk != tj && (flags[tj] | flags[tk]) == 0u;
                if (uniform) {
                    if (clean)
                        run(std::true_type{}, std::true_type{});
                    else
                        run(std::true_type{}, std::false_type{});
                } else {
                    if (clean)
                        run(std::false_type{}, std::true_type{});
                    else
                        run(std::false_type{}, std::false_type{});
                }
            }
        } else {
            // FP32 positions in the bins (plus one, in q1) and values of a batch; returns 1
            // if one lies too close to an edge.  MASK: k points from kk on; those at or past
            // kn, and on the diagonal those not past the lane, go to the scratch row
            auto fast_batch = [&](auto mask, const KPoints<DIM>& p, float (&q1)[kBatch], double (&val)[kBatch],
                                  int kk = 0, int kn = 0, bool diagonal = false) {
                constexpr bool MASK = decltype(mask)::value;
                float far = 0.0f;
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    float d2 = 0.0f;
#pragma unroll
                    for (int c = 0; c < DIM; ++c) {
                        const float dd = p.x(u, c) - xj[c];
                        d2 = c == 0 ? dd * dd : __builtin_fmaf(dd, dd, d2);
                    }
                    float q = __builtin_fmaf(__builtin_amdgcn_sqrtf(d2), inv_wf, q1off);
                    q = __builtin_amdgcn_fmed3f(q, 0.5f, qtop);
                    if constexpr (MASK) q = (kk + u < kn && (!diagonal || lane < kk + u)) ? q : 0.5f;
                    q1[u] = q;
                    far = fmaxf(far, fabsf(__builtin_amdgcn_fractf(q) - 0.5f));
                    val[u] = value(p.f(u));
                }
                return __ballot(far > near_f) != 0ull ? 1u : 0u;
            };
            auto add_batch = [&](const float (&q1)[kBatch], const double (&val)[kBatch]) {
#pragma unroll
                for (int u = 0; u < kBatch; ++u) iso_add(vlds, col, lane4, (int)q1[u], val[u]);
            };
            while (todo) {
                const int tk = t0 + __builtin_ctzll(todo);
                todo &= todo - 1ull;
                const int k0 = tk * 64;
                const int kn = nv - k0 < 64 ? nv - k0 : 64;
                unsigned redo = 0u;  // batches for the FP64 form
                if (tk == tj || kn < 64) {
                    for (int s = 0; s * kBatch < kn; ++s) {
                        KPoints<DIM> k;
                        float q[kBatch];
                        double v[kBatch];
                        k.load(rec, k0 + s * kBatch);
                        const unsigned close = fast_batch(std::true_type{}, k, q, v, s * kBatch, kn, tk == tj);
                        redo |= close << s;
                        if (!close) add_batch(q, v);
                    }
                } else {
                    // Two batches per step; the scalar loads of the next are in flight while
                    // one is worked on, and a batch is added before the next is worked out (the
                    // wait for scalar loads also waits for the LDS adds before it).
                    KPoints<DIM> ka, kb;
                    float qa[kBatch], qb[kBatch];
                    double va[kBatch], vb[kBatch];
                    ka.load(rec, k0);
#pragma unroll 1
                    for (int s = 0; s < 16; s += 2) {
                        kb.load(rec, ka.ready(k0 + (s + 1) * kBatch));
                        if (s > 0 && !(redo >> (s - 1) & 1u)) add_batch(qb, vb);
                        redo |= fast_batch(std::false_type{}, ka, qa, va) << s;
                        ka.load(rec, kb.ready(k0 + (s + 2) * kBatch));  // past the tile: padding or the next
                        if (!(redo >> s & 1u)) add_batch(qa, va);
                        redo |= fast_batch(std::false_type{}, kb, qb, vb) << (s + 1);
                    }
                    if (!(redo >> 15 & 1u)) add_batch(qb, vb);
                }
                while (redo) {
                    const int s = __builtin_ctz(redo) * kBatch;
                    redo &= redo - 1u;
                    int row[kBatch];
                    double val[kBatch];
#pragma unroll
                    for (int u = 0; u < kBatch; ++u) {
                        const double* p = drec + (int64_t)(k0 + s + u) * (DIM + 1);
                        double d2 = 0.0;
#pragma unroll
                        for (int c = 0; c < DIM; ++c) {
                            const double dd = p[c] - pj[c];
                            d2 += dd * dd;
                        }
                        val[u] = value(p[DIM]);
                        const bool ok = s + u < kn && (tk != tj || s + u > lane);
                        const unsigned sl = (unsigned)(uniform_bin(ok ? d2 : 0.0) - h0);
                        row[u] = (ok && sl < (unsigned)NH) ? (int)sl + 1 : 0;
                    }
#pragma unroll
                    for (int u = 0; u < kBatch; ++u) iso_add(vlds, col, lane4, row[u], val[u]);
                }
            }
        }
    }
    if (EXACT && nan_cnt)
        for (int r = 1; r <= NH; ++r) {
            reinterpret_cast<double*>(hist + r * kRowBytes)[lane] += nan_sum;
            reinterpret_cast<unsigned*>(hist + r * kRowBytes + 512)[lane] += nan_cnt;
        }
    __syncthreads();
    // block partials: lane h adds the 64 columns of slot h, starting at its own
    // column (no bank conflicts)
    for (int h = lane; h < NH; h += 64) {
        const double* rs = reinterpret_cast<const double*>(hist + (h + 1) * kRowBytes);
        const unsigned* rc = reinterpret_cast<const unsigned*>(hist + (h + 1) * kRowBytes + 512);
        double s = 0.0;
        unsigned long long c = 0;
#pragma unroll 16
        for (int i = 0; i < 64; ++i) {
            s += rs[(i + h) & 63];
            c += rc[(i + h) & 63];
        }
        part_sum[h * pcols + pcol] = s;
        part_cnt[h * pcols + pcol] = c;
    }
}

template <int DIM, bool CRESSIE, bool EXACT>
int launch_iso_pairs(const IsoArgs& a, const IsoLayout& l, char* ws, const double* edges, hipStream_t s) {
    const size_t lds = iso_lds_bytes(a.B, a.h1 - a.h0) + (EXACT ? 64 * (DIM + 1) * sizeof(double) : 0);
    if (lds > 65536 &&
        hipFuncSetAttribute(reinterpret_cast<const void*>(&k_iso_pairs<DIM, CRESSIE, EXACT>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return GSX_E_LAUNCH;
    hipLaunchKernelGGL((k_iso_pairs<DIM, CRESSIE, EXACT>), dim3((unsigned)l.blocks), dim3(64), lds, s, a,
                       reinterpret_cast<const IsoMeta*>(ws + l.meta), reinterpret_cast<const int*>(ws + l.flagged),
                       reinterpret_cast<const IsoEdges*>(ws + l.edges),
                       reinterpret_cast<const double*>(ws + l.thp), edges, reinterpret_cast<const uint32_t*>(ws + l.rec),
                       reinterpret_cast<const double*>(ws + l.drec), reinterpret_cast<const double*>(ws + l.box),
                       reinterpret_cast<const unsigned*>(ws + l.flags), l.nt,
                       reinterpret_cast<double*>(ws + l.part_sum),
                       reinterpret_cast<unsigned long long*>(ws + l.part_cnt));
    return launch_status();
}

template <int DIM, bool CRESSIE>
int launch_iso(const IsoArgs& a, const IsoLayout& l, char* ws, const double* edges, hipStream_t s) {
    const int st = launch_iso_pairs<DIM, CRESSIE, false>(a, l, ws, edges, s);
    return st != GSX_OK ? st : launch_iso_pairs<DIM, CRESSIE, true>(a, l, ws, edges, s);
}

template <int DIM>
int iso_run(const IsoLayout& l, int64_t P, int64_t B, const double* f, const double* edges, const double* pos,
            int estimator, double* gamma, int64_t* counts, char* ws, hipStream_t s) {
    IsoMeta* meta = reinterpret_cast<IsoMeta*>(ws + l.meta);
    uint32_t* rec = reinterpret_cast<uint32_t*>(ws + l.rec);
    double* drec = reinterpret_cast<double*>(ws + l.drec);
    double* box = reinterpret_cast<double*>(ws + l.box);
    unsigned* flags = reinterpret_cast<unsigned*>(ws + l.flags);
    double* thp = reinterpret_cast<double*>(ws + l.thp);
    IsoEdges* ed = reinterpret_cast<IsoEdges*>(ws + l.edges);
    int* flagged = reinterpret_cast<int*>(ws + l.flagged);
    int st;
    if (l.sorted) {
        double* bounds = reinterpret_cast<double*>(ws + l.bounds);
        unsigned* cell = reinterpret_cast<unsigned*>(ws + l.cell);
        unsigned* arrival = reinterpret_cast<unsigned*>(ws + l.arrival);
        unsigned* list = reinterpret_cast<unsigned*>(ws + l.list);
        unsigned* count = reinterpret_cast<unsigned*>(ws + l.count);
        unsigned* start = reinterpret_cast<unsigned*>(ws + l.start);
        const dim3 grid((unsigned)ceil_div(P, (int64_t)256)), block(256);
        hipLaunchKernelGGL(k_iso_bounds<DIM>, dim3(kBoxBlocks + 1), block, 0, s, P, pos, bounds, count,
                           (int)B, edges, thp, ed);
        if ((st = launch_status()) != GSX_OK) return st;
        hipLaunchKernelGGL(k_iso_cells<DIM>, grid, block, 0, s, P, pos, f, bounds, meta, cell, arrival, count);
        if ((st = launch_status()) != GSX_OK) return st;
        hipLaunchKernelGGL(k_iso_scan, dim3(1), dim3(1024), 0, s, P, count, start, meta, flagged);
        if ((st = launch_status()) != GSX_OK) return st;
        hipLaunchKernelGGL(k_iso_list, grid, block, 0, s, P, cell, arrival, start, list);
        if ((st = launch_status()) != GSX_OK) return st;
        hipLaunchKernelGGL(k_iso_place<DIM>, grid, block, 0, s, P, meta, pos, f, cell, start, list, rec, drec);
        if ((st = launch_status()) != GSX_OK) return st;
        hipLaunchKernelGGL(k_iso_boxes<DIM>, dim3((unsigned)ceil_div(l.nt, (int64_t)4)), block, 0, s, l.nt, meta,
                           drec, box, flags);
    } else {
        hipLaunchKernelGGL(k_iso_prepare<DIM>, dim3((unsigned)ceil_div(l.nt * 64, (int64_t)1024) + 1), dim3(1024), 0,
                           s, P, l.nt, pos, f, meta, rec, drec, box, flags, (int)B, edges, thp, ed,
                           flagged);
    }
    if ((st = launch_status()) != GSX_OK) return st;
    for (int64_t h0 = 0; h0 < B; h0 += l.slots) {
        IsoArgs a;
        a.B = B;
        a.h0 = h0;
        a.h1 = h0 + l.slots < B ? h0 + l.slots : B;
        a.gl2 = iso_group_log2(l.nt);
        st = estimator ? launch_iso<DIM, true>(a, l, ws, edges, s) : launch_iso<DIM, false>(a, l, ws, edges, s);
        if (st != GSX_OK) return st;
        st = vario_collect(2 * l.blocks, a.h1 - h0, h0, reinterpret_cast<double*>(ws + l.part_sum),
                           reinterpret_cast<unsigned long long*>(ws + l.part_cnt), gamma, counts, false, true,
                           estimator, s);
        if (st != GSX_OK) return st;
    }
    return GSX_OK;
}

}  // namespace

int64_t vario_iso_ws(int64_t P, int64_t dim, int64_t B) { return iso_layout(P, dim, B).total; }

int vario_iso(int64_t P, int64_t dim, int64_t B, const double* f, const double* edges, const double* pos,
              int estimator, double* gamma, int64_t* counts, void* ws, hipStream_t s) {
    const IsoLayout l = iso_layout(P, dim, B);
    size_t limit = 0;
    const int st = vario_lds_limit(&limit);
    if (st != GSX_OK) return st;
    if (iso_lds_bytes(B, l.slots) + 64 * 4 * 8 > limit) return GSX_E_UNSUPPORTED;
    char* w = static_cast<char*>(ws);
    switch (dim) {
        case 1: return iso_run<1>(l, P, B, f, edges, pos, estimator, gamma, counts, w, s);
        case 2: return iso_run<2>(l, P, B, f, edges, pos, estimator, gamma, counts, w, s);
        default: return iso_run<3>(l, P, B, f, edges, pos, estimator, gamma, counts, w, s);
    }
}

}  // namespace gsx
