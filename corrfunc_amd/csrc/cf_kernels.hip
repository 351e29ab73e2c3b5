// cf_kernels.hip -- HIP kernels of the MI355X theory pair-counting engine (gfx950).
//
// Device pipeline of one countpairs* call:
//   k_minmax / k_minmax_final     data extent              (reference gridlink_utils.c.src:52-70)
//   k_bucket_count (_few)         cell index per particle, cell histogram
//                                                          (gridlink_impl.c.src:162-201)
//   k_scan_*                      exclusive prefix sum of the cell histogram
//   k_index_scatter               particle indices in cell order
//   k_build_small / _big          per cell: Hilbert order, records in HBM (FP64 + quantized
//                                 cell-local positions for the integer pair filter), the
//                                 bounding boxes of the cell (gridlink_impl.c.src:292-316)
//                                 and of its groups
//   k_cellpair_flag / _emit       neighbour-cell work list with periodic wraps and
//                                 min-separation culling   (gridlink_impl.c.src:439-625)
//   k_pairs_plain                 FP64 pair kernel, one workgroup per cell pair
//   k_pairs_tuned                 integer filter + FP64 replay, persistent waves, LDS histograms
//
// All FP64 arithmetic that decides a pair's bin is written in the reference's
// operation order; this file is compiled with -ffp-contract=off so the compiler
// never fuses it, and fma() appears only where the reference's AVX512F kernels
// use an FMA.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <float.h>
#include "cf_device.h"

namespace cfamd {

// ---------------------------------------------------------------- helpers
__device__ __forceinline__ int lane_id() { return __lane_id(); }

__device__ __forceinline__ double wave_min_d(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ double wave_max_d(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

// ------------------------------------------------------------ extent (a2)
// Extent of the points i, i + step, ... below end, reduced over a workgroup of
// 256 into out[0..5].
template <typename T>
__device__ __forceinline__ void minmax_block(int64_t i, int64_t end, int64_t step, const T* __restrict__ X,
                                             const T* __restrict__ Y, const T* __restrict__ Z,
                                             double* __restrict__ out)
{
    double mn[3] = {DBL_MAX, DBL_MAX, DBL_MAX}, mx[3] = {-DBL_MAX, -DBL_MAX, -DBL_MAX};
    for (; i < end; i += step) {
        const double v[3] = {(double)X[i], (double)Y[i], (double)Z[i]};
        for (int d = 0; d < 3; d++) { mn[d] = fmin(mn[d], v[d]); mx[d] = fmax(mx[d], v[d]); }
    }
    __shared__ double s[6][256];
    for (int d = 0; d < 3; d++) { s[d][threadIdx.x] = mn[d]; s[3 + d][threadIdx.x] = mx[d]; }
    __syncthreads();
    for (int st = blockDim.x / 2; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st)
            for (int d = 0; d < 3; d++) {
                s[d][threadIdx.x] = fmin(s[d][threadIdx.x], s[d][threadIdx.x + st]);
                s[3 + d][threadIdx.x] = fmax(s[3 + d][threadIdx.x], s[3 + d][threadIdx.x + st]);
            }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int d = 0; d < 6; d++) out[d] = s[d][0];
}
template <typename T>
__global__ void k_minmax(int64_t n, const T* __restrict__ X, const T* __restrict__ Y, const T* __restrict__ Z,
                         double* __restrict__ partial)
{
    minmax_block(blockIdx.x * (int64_t)blockDim.x + threadIdx.x, n, (int64_t)gridDim.x * blockDim.x, X, Y, Z,
                 partial + blockIdx.x * 6);
}

// One wave: the lanes reduce strided subsets of the block partials, then the
// wave (min/max are exact, so the order does not matter).
__device__ __forceinline__ void minmax_reduce(int nblocks, const double* __restrict__ partial,
                                              double* __restrict__ out)
{
    const int lane = (int)threadIdx.x;
    double r[6] = {DBL_MAX, DBL_MAX, DBL_MAX, -DBL_MAX, -DBL_MAX, -DBL_MAX};
    for (int b = lane; b < nblocks; b += 64)
        for (int d = 0; d < 3; d++) {
            r[d] = fmin(r[d], partial[b * 6 + d]);
            r[3 + d] = fmax(r[3 + d], partial[b * 6 + 3 + d]);
        }
    for (int d = 0; d < 3; d++) {
        r[d] = wave_min_d(r[d]);
        r[3 + d] = wave_max_d(r[3 + d]);
    }
    if (lane == 0)
        for (int d = 0; d < 6; d++) out[d] = r[d];
}
__global__ void k_minmax_final(int nblocks, const double* __restrict__ partial, double* __restrict__ out)
{
    minmax_reduce(nblocks, partial, out);
}

// --------------------------------------------------------- gridding (a5)
struct GridArgs {
    double xmin, ymin, zmin;
    double xinv, yinv, zinv;
    double xbs, ybs, zbs;
    int nx, ny, nz;
    double qinv;  // quanta per unit length of the quantized positions
};

// Quantized cell-local coordinate: rint(v * qinv) clamped to [-kQMax, kQMax].
__device__ __forceinline__ int quantize(double v, double qinv)
{
    const double t = fmin(fmax(v * qinv, -(double)kQMax), (double)kQMax);
    return (int)rint(t);
}
__device__ __forceinline__ uint2 quantize_pos(double dx, double dy, double dz, double qinv)
{
    const int qx = quantize(dx, qinv), qy = quantize(dy, qinv), qz = quantize(dz, qinv);
    return make_uint2(((unsigned)qx & 0xffffu) | ((unsigned)qy << 16), (unsigned)qz);
}

// Cell index exactly as the reference computes it (gridlink_impl.c.src:167-178).
__device__ __forceinline__ int cell_of(const GridArgs& g, double X, double Y, double Z, int* oob)
{
    int ix = (int)((X - g.xmin) * g.xinv);
    int iy = (int)((Y - g.ymin) * g.yinv);
    int iz = (int)((Z - g.zmin) * g.zinv);
    if (ix > g.nx - 1) ix--;
    if (iy > g.ny - 1) iy--;
    if (iz > g.nz - 1) iz--;
    *oob = ix < 0 || ix >= g.nx || iy < 0 || iy >= g.ny || iz < 0 || iz >= g.nz;
    return (ix * g.ny + iy) * g.nz + iz;
}

// Adds the active lanes to counts[c] of their cells and returns each one's rank in
// its cell. Lanes that share a cell are added by one of them: an atomic per particle
// is serialized on its cell (~30 ns each; 1M points in four clumps, to the end of
// gridding: 6.1 ms, 3.1 with the sharing). The search for shared cells ends with the
// second lane that has its cell to itself, so particles in random order on a fine
// grid pay two rounds of it.
__device__ __forceinline__ int claim_ranks(int* __restrict__ counts, int c)
{
    const int lane = lane_id();
    int leader = lane, before = 0, n = 1, alone = 0;
    unsigned long long todo = __builtin_amdgcn_ballot_w64(true);
    while (todo && alone < 2) {
        const int f = __builtin_ctzll(todo);
        const unsigned long long m = todo & __builtin_amdgcn_ballot_w64(c == __builtin_amdgcn_readlane(c, f));
        if ((m >> lane) & 1ull) {
            leader = f;
            before = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
            n = __popcll(m);
        }
        alone += __popcll(m) == 1;
        todo &= ~m;
    }
    int base = 0;
    if (lane == leader) base = atomicAdd(&counts[c], n);
    return __shfl(base, leader, 64) + before;
}

// The particle's cell and its rank among the cell's particles (the order of
// the atomics, so any order), which the index scatter needs no second atomic for.
template <typename T>
__device__ __forceinline__ void bucket_count_one(int64_t i, const T* __restrict__ X, const T* __restrict__ Y,
                                                 const T* __restrict__ Z, const GridArgs& g, int* __restrict__ bucket,
                                                 int* __restrict__ rank, int* __restrict__ counts,
                                                 unsigned long long* __restrict__ oob_count)
{
    int oob;
    const int c = cell_of(g, (double)X[i], (double)Y[i], (double)Z[i], &oob);
    if (oob) {
        atomicAdd(oob_count, 1ull);
        bucket[i] = -1;
        return;
    }
    bucket[i] = c;
    rank[i] = claim_ranks(counts, c);
}

template <typename T>
__global__ void k_bucket_count(int64_t n, const T* __restrict__ X, const T* __restrict__ Y, const T* __restrict__ Z,
                               GridArgs g, int* __restrict__ bucket, int* __restrict__ rank,
                               int* __restrict__ counts, unsigned long long* __restrict__ oob_count)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < n) bucket_count_one(i, X, Y, Z, g, bucket, rank, counts, oob_count);
}

// The same for few, crowded cells (ncells <= kFewCells): a workgroup counts its
// kFewItems particles in LDS and adds each cell's number once, so a cell's atomics
// are n / kFewItems instead of one per wave that meets it.
constexpr int kFewCells = 2048;
constexpr int kFewItems = 2048;
template <typename T>
__global__ __launch_bounds__(256) void k_bucket_count_few(int64_t n, const T* __restrict__ X,
                                                          const T* __restrict__ Y, const T* __restrict__ Z,
                                                          GridArgs g, int ncells, int* __restrict__ bucket,
                                                          int* __restrict__ rank, int* __restrict__ counts,
                                                          unsigned long long* __restrict__ oob_count)
{
    __shared__ int local[kFewCells];
    for (int c = threadIdx.x; c < ncells; c += 256) local[c] = 0;
    __syncthreads();
    const int64_t i0 = blockIdx.x * (int64_t)kFewItems + threadIdx.x;
    int cell[kFewItems / 256], r[kFewItems / 256];
#pragma unroll
    for (int k = 0; k < kFewItems / 256; k++) {
        const int64_t i = i0 + 256 * k;
        cell[k] = -1;
        if (i >= n) continue;
        int oob;
        const int c = cell_of(g, (double)X[i], (double)Y[i], (double)Z[i], &oob);
        if (oob)
            atomicAdd(oob_count, 1ull);
        else
            cell[k] = c;
        bucket[i] = cell[k];
        if (!oob) r[k] = atomicAdd(&local[c], 1);
    }
    __syncthreads();
    for (int c = threadIdx.x; c < ncells; c += 256)
        if (local[c]) local[c] = atomicAdd(&counts[c], local[c]);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kFewItems / 256; k++)
        if (cell[k] >= 0) rank[i0 + 256 * k] = local[cell[k]] + r[k];
}

// Particle indices in cell order.
__global__ void k_index_scatter(int64_t n, const int* __restrict__ bucket, const int* __restrict__ rank,
                                const int* __restrict__ bstart, int* __restrict__ idx)
{
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int b = bucket[i];
    if (b >= 0) idx[bstart[b] + rank[i]] = (int)i;  // b < 0: outside the grid, reported by the host
}

// Exclusive scan over int32 counts, three phases, 1024 items per block; the
// total goes to out[n] (written by the kernels: a copy of 4 bytes costs a launch).
constexpr int kScanBlock = 256;
constexpr int kScanItems = 4;

__device__ int block_exclusive_scan(int v, int* total)
{
    __shared__ int ws[kScanBlock / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int incl = v;
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(incl, o, 64);
        if (lane >= o) incl += t;
    }
    if (lane == 63) ws[w] = incl;
    __syncthreads();
    int off = 0, tot = 0;
    for (int k = 0; k < kScanBlock / 64; k++) {
        if (k < w) off += ws[k];
        tot += ws[k];
    }
    __syncthreads();
    *total = tot;
    return off + incl - v;
}

__global__ void k_scan_blocks(int64_t n, const int* __restrict__ in, int* __restrict__ out, int* __restrict__ block_sums)
{
    const int64_t base = (int64_t)blockIdx.x * kScanBlock * kScanItems + (int64_t)threadIdx.x * kScanItems;
    int v[kScanItems], s = 0;
    for (int k = 0; k < kScanItems; k++) {
        v[k] = base + k < n ? in[base + k] : 0;
        s += v[k];
    }
    int tot;
    int ex = block_exclusive_scan(s, &tot);
    for (int k = 0; k < kScanItems; k++) {
        if (base + k < n) out[base + k] = ex;
        ex += v[k];
    }
    if (threadIdx.x == 0) {
        block_sums[blockIdx.x] = tot;
        if (gridDim.x == 1) out[n] = tot;
    }
}

__global__ void k_scan_add(int64_t n, int* __restrict__ out, const int* __restrict__ block_offsets)
{
    const int64_t base = (int64_t)blockIdx.x * kScanBlock * kScanItems + (int64_t)threadIdx.x * kScanItems;
    const int add = block_offsets[blockIdx.x];
    for (int k = 0; k < kScanItems; k++)
        if (base + k < n) out[base + k] += add;
    if (threadIdx.x == 0 && blockIdx.x == gridDim.x - 1) out[n] = block_offsets[gridDim.x];
}

// Position of (x, y, z), b bits each, on the 3-D Hilbert curve (J. Skilling,
// "Programming the Hilbert curve", 2004: inverse undo of the excess work, then
// Gray encoding).
__device__ __forceinline__ unsigned hilbert3(unsigned x, unsigned y, unsigned z, int b)
{
    unsigned v[3] = {x, y, z};
    for (int k = b - 1; k > 0; k--) {
        const unsigned q = 1u << k, m = q - 1u;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const unsigned t = (v[0] ^ v[d]) & m;
            const bool up = (v[d] & q) != 0;
            v[0] ^= up ? m : t;
            if (d > 0) v[d] ^= up ? 0u : t;
        }
    }
    v[1] ^= v[0];
    v[2] ^= v[1];
    unsigned t = 0;
    for (int k = b - 1; k > 0; k--)
        if (v[2] & (1u << k)) t ^= (1u << k) - 1u;
    unsigned h = 0;
    for (int k = b - 1; k >= 0; k--)
        h = (h << 3) | ((((v[0] ^ t) >> k) & 1u) << 2) | ((((v[1] ^ t) >> k) & 1u) << 1) | (((v[2] ^ t) >> k) & 1u);
    return h;
}

// Cells up to kSmallCell particles are sorted by one wave each, larger ones by
// a workgroup of kBigThreads.
constexpr int kSmallCell = 512;
constexpr int kSmallBins = 512;
constexpr int kBigBins = 4096;
constexpr int kBigThreads = 1024;
constexpr int kMaxSegments = 8;

template <int NT>
__device__ __forceinline__ void build_sync()
{
    __threadfence_block();
    if (NT == 64)
        __builtin_amdgcn_wave_barrier();
    else
        __syncthreads();
}

// Orders the particles of cell c along a Hilbert curve through the cell (a
// counting sort over up to MAXBINS sub-cells in LDS, `hist`), so that runs of
// consecutive particles are compact, and writes their FP64 records, quantized
// cell-local positions, the cell's bounding box and the bounding boxes of its
// groups of kGroup. A cell longer in z than in x and y is cut into cubic
// segments along z, one curve each. Two gathers of the particles' coordinates
// (key, placement) instead of one pass that keeps them in registers: the
// second hits L2, and any cell size takes the same code. The whole of NT
// threads (`tid` in it) works on one cell; `red` holds 6 NT / 64 doubles (NT > 64).
template <typename T, int NT, int MAXBINS>
__device__ __forceinline__ void build_cell(int64_t c, int tid, const T* __restrict__ X, const T* __restrict__ Y,
                                           const T* __restrict__ Z, const T* __restrict__ W, const GridArgs& g,
                                           const int* __restrict__ bstart, const int* __restrict__ idx,
                                           int* __restrict__ keys, double4* d4, uint2* __restrict__ q,
                                           double* __restrict__ bounds, double* __restrict__ gbox,
                                           float* __restrict__ rr, int* hist, double* red)
{
    const int s = bstart[c], n = bstart[c + 1] - s;
    const int lane = tid & 63;
    double b[6] = {DBL_MAX, -DBL_MAX, DBL_MAX, -DBL_MAX, DBL_MAX, -DBL_MAX};
    const int ic = (int)c, iz = ic % g.nz, ixy = ic / g.nz, iy = ixy % g.ny, ix = ixy / g.ny;
    const double ox = g.xmin + ix * g.xbs, oy = g.ymin + iy * g.ybs, oz = g.zmin + iz * g.zbs;
    if (n > 0) {
        const double side = fmax(g.xbs, g.ybs);
        int nseg = side > 0 ? (int)fmin((double)kMaxSegments, g.zbs / side + 0.5) : 1;
        nseg = nseg < 1 ? 1 : nseg;
        int nb = 0;
        while (nb < 5 && (nseg << (3 * (nb + 1))) <= min(MAXBINS, 2 * n)) nb++;
        const int bins = nseg << (3 * nb), top = (1 << nb) - 1;
        const double scale = (double)(1 << nb);
        for (int k = tid; k < bins; k += NT) hist[k] = 0;
        build_sync<NT>();
        for (int k = tid; k < n; k += NT) {
            const int i = idx[s + k];
            const double xv = (double)X[i], yv = (double)Y[i], zv = (double)Z[i];
            b[0] = xv < b[0] ? xv : b[0];
            b[1] = xv > b[1] ? xv : b[1];
            b[2] = yv < b[2] ? yv : b[2];
            b[3] = yv > b[3] ? yv : b[3];
            b[4] = zv < b[4] ? zv : b[4];
            b[5] = zv > b[5] ? zv : b[5];
            const int hx = (int)fmin(fmax((xv - ox) * g.xinv * scale, 0.0), (double)top);
            const int hy = (int)fmin(fmax((yv - oy) * g.yinv * scale, 0.0), (double)top);
            const int zt = (nseg << nb) - 1;
            const int hz = (int)fmin(fmax((zv - oz) * g.zinv * scale * nseg, 0.0), (double)zt);
            const int key = ((hz >> nb) << (3 * nb)) + (int)hilbert3(hx, hy, hz & top, nb);
            keys[s + k] = key;
            atomicAdd(&hist[key], 1);
        }
        build_sync<NT>();
        // exclusive scan of the bins by the first wave
        if (tid < 64) {
            int carry = 0;
            for (int k0 = 0; k0 < bins; k0 += 64) {
                const int k = k0 + lane;
                const int v = k < bins ? hist[k] : 0;
                int incl = v;
                for (int o = 1; o < 64; o <<= 1) {
                    const int t = __shfl_up(incl, o, 64);
                    if (lane >= o) incl += t;
                }
                if (k < bins) hist[k] = carry + incl - v;
                carry += __shfl(incl, 63, 64);
            }
        }
        build_sync<NT>();
        for (int k = tid; k < n; k += NT) {
            const int i = idx[s + k];
            const double xv = (double)X[i], yv = (double)Y[i], zv = (double)Z[i];
            const int pos = s + atomicAdd(&hist[keys[s + k]], 1);
            d4[pos] = make_double4(xv, yv, zv, W ? (double)W[i] : 0.0);
            q[pos] = quantize_pos(xv - ox, yv - oy, zv - oz, g.qinv);
            if (rr) rr[pos] = (float)(2.0 * (xv * xv + yv * yv + zv * zv));
        }
    }
    // cell bounds (min / max are exact, so the order of the reduction does not
    // matter); empty cells get (+DBL_MAX, -DBL_MAX)
    for (int o = 32; o > 0; o >>= 1) {
#pragma unroll
        for (int d = 0; d < 6; d += 2) {
            const double lo = __shfl_xor(b[d], o, 64), hi = __shfl_xor(b[d + 1], o, 64);
            b[d] = lo < b[d] ? lo : b[d];
            b[d + 1] = hi > b[d + 1] ? hi : b[d + 1];
        }
    }
    if (NT > 64) {
        if (lane == 0)
            for (int d = 0; d < 6; d++) red[(tid >> 6) * 6 + d] = b[d];
        __syncthreads();
        if (tid < 6) {
            double v = red[tid];
            for (int w = 1; w < NT / 64; w++) {
                const double t = red[w * 6 + tid];
                v = (tid & 1) ? (t > v ? t : v) : (t < v ? t : v);
            }
            bounds[c * 6 + tid] = v;
        }
    } else if (lane == 0) {
        for (int d = 0; d < 6; d++) bounds[c * 6 + d] = b[d];
    }
    // group boxes, kGroup lanes per group, from the records just written
    build_sync<NT>();
    const int64_t g0 = group_index(s, c);
    for (int gk = tid / kGroup; gk * kGroup < n; gk += NT / kGroup) {
        const int k = gk * kGroup + (tid & (kGroup - 1));
        double e[6] = {DBL_MAX, -DBL_MAX, DBL_MAX, -DBL_MAX, DBL_MAX, -DBL_MAX};
        if (k < n) {
            const double4 r = d4[s + k];
            // a particle with a NaN coordinate is in no pair; the unbounded box keeps
            // its group off the paths that rely on finite separations
            const bool nan = r.x != r.x || r.y != r.y || r.z != r.z;
            e[0] = nan ? -DBL_MAX : r.x; e[1] = nan ? DBL_MAX : r.x;
            e[2] = nan ? -DBL_MAX : r.y; e[3] = nan ? DBL_MAX : r.y;
            e[4] = nan ? -DBL_MAX : r.z; e[5] = nan ? DBL_MAX : r.z;
        }
        for (int o = kGroup / 2; o > 0; o >>= 1) {
#pragma unroll
            for (int d = 0; d < 6; d += 2) {
                e[d] = fmin(e[d], __shfl_xor(e[d], o, 64));
                e[d + 1] = fmax(e[d + 1], __shfl_xor(e[d + 1], o, 64));
            }
        }
        const int d = tid & (kGroup - 1);
        const double v = d == 0 ? e[0] : d == 1 ? e[1] : d == 2 ? e[2] : d == 3 ? e[3] : d == 4 ? e[4] : e[5];
        if (d < 6) gbox[(g0 + gk) * 6 + d] = v;
    }
}

// One wave per cell; cells above kSmallCell particles are left to
// k_build_big, listed at big[1 ...] with their number at big[0].
template <typename T>
__device__ __forceinline__ void build_small(int64_t ncells, const T* X, const T* Y, const T* Z, const T* W,
                                            const GridArgs& g, const int* bstart, const int* idx, int* keys,
                                            double4* d4, uint2* q, double* bounds, double* gbox, float* rr, int* big)
{
    __shared__ int hist[4][kSmallBins];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t c = blockIdx.x * (int64_t)(blockDim.x >> 6) + wave;
    if (c >= ncells) return;  // uniform per wave
    if (bstart[c + 1] - bstart[c] > kSmallCell) {
        if (lane == 0) big[1 + atomicAdd(big, 1)] = (int)c;
        return;
    }
    build_cell<T, 64, kSmallBins>(c, lane, X, Y, Z, W, g, bstart, idx, keys, d4, q, bounds, gbox, rr,
                                      hist[wave], nullptr);
}
template <typename T>
__device__ __forceinline__ void build_big(const T* X, const T* Y, const T* Z, const T* W, const GridArgs& g,
                                          const int* bstart, const int* idx, int* keys, double4* d4, uint2* q,
                                          double* bounds, double* gbox, float* rr, const int* big)
{
    __shared__ int hist[kBigBins];
    __shared__ double red[6 * kBigThreads / 64];
    const int nbig = big[0];
    for (int t = blockIdx.x; t < nbig; t += gridDim.x) {
        build_cell<T, kBigThreads, kBigBins>(big[1 + t], threadIdx.x, X, Y, Z, W, g, bstart, idx, keys, d4, q, bounds,
                                             gbox, rr, hist, red);
        __syncthreads();
    }
}
template <typename T>
__global__ __launch_bounds__(256) void k_build_small(int64_t ncells, const T* X, const T* Y, const T* Z, const T* W,
                                                     GridArgs g, const int* bstart, const int* idx, int* keys,
                                                     double4* d4, uint2* q, double* bounds, double* gbox, float* rr,
                                                     int* big)
{
    build_small(ncells, X, Y, Z, W, g, bstart, idx, keys, d4, q, bounds, gbox, rr, big);
}
template <typename T>
__global__ __launch_bounds__(kBigThreads) void k_build_big(const T* X, const T* Y, const T* Z, const T* W, GridArgs g,
                                                           const int* bstart, const int* idx, int* keys, double4* d4,
                                                           uint2* q, double* bounds, double* gbox, float* rr,
                                                           const int* big)
{
    build_big(X, Y, Z, W, g, bstart, idx, keys, d4, q, bounds, gbox, rr, big);
}

// Sums of the weights and of their squares over the grid-ordered records
// (workgroups of 256).
__device__ __forceinline__ void weight_sums_block(int64_t i, int64_t end, int64_t step,
                                                  const double4* __restrict__ d4, double* __restrict__ out)
{
    double s = 0, s2 = 0;
    for (; i < end; i += step) {
        const double w = d4[i].w;
        s += w;
        s2 += w * w;
    }
    for (int o = 32; o > 0; o >>= 1) {
        s += __shfl_xor(s, o, 64);
        s2 += __shfl_xor(s2, o, 64);
    }
    // one atomic per workgroup and sum (they are serialized, ~14 ns each)
    __shared__ double part[2][4];
    if ((threadIdx.x & 63) == 0) {
        part[0][threadIdx.x >> 6] = s;
        part[1][threadIdx.x >> 6] = s2;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const double* p = part[threadIdx.x];
        atomicAdd(&out[threadIdx.x], (p[0] + p[1]) + (p[2] + p[3]));
    }
}
__global__ void k_weight_sums(int64_t n, const double4* __restrict__ d4, double* __restrict__ out)
{
    weight_sums_block(blockIdx.x * (int64_t)blockDim.x + threadIdx.x, n, (int64_t)gridDim.x * blockDim.x, d4, out);
}

// Device-to-device copy: n16 16-byte words through the vector path (grid-stride),
// then the byte tail. Reads and writes exactly the bytes asked for, which also
// makes it the reference kernel for scaling the HBM byte counters.
__global__ void k_copy16(int64_t n16, const uint4* __restrict__ src, uint4* __restrict__ dst, int tail,
                         const unsigned char* __restrict__ src_tail, unsigned char* __restrict__ dst_tail)
{
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n16; i += stride) dst[i] = src[i];
    if (blockIdx.x == 0 && (int)threadIdx.x < tail) dst_tail[threadIdx.x] = src_tail[threadIdx.x];
}

// ------------------------------------------------------- cell pairs (a6)
struct NgbArgs {
    int nx, ny, nz;
    int rx, ry, rz;
    int px, py, pz;
    int autocorr, min_sep_opt, dupcheck;
    double xwrap, ywrap, zwrap;
    double max3, max2, max1;
};

__device__ __forceinline__ int64_t cell_count(const int* bstart, int64_t c)
{
    return (int64_t)bstart[c + 1] - bstart[c];
}

// Evaluates neighbour k of primary cell icell in the reference's loop order
// (iix outer, iiy, iiz inner). Returns 1 and fills rec when the reference would
// append this cell pair (before its duplicate check).
__device__ int eval_neighbour(const NgbArgs& a, int64_t icell, int k, const int* __restrict__ bs1,
                              const int* __restrict__ bs2, const double* __restrict__ bd1,
                              const double* __restrict__ bd2, CellPairRec* rec)
{
    const int ny_n = 2 * a.ry + 1, nz_n = 2 * a.rz + 1;
    const int iix = k / (ny_n * nz_n) - a.rx;
    const int iiy = (k / nz_n) % ny_n - a.ry;
    const int iiz = k % nz_n - a.rz;
    const int iz = (int)(icell % a.nz);
    const int ix = (int)(icell / ((int64_t)a.ny * a.nz));
    const int iy = (int)((icell - iz - (int64_t)ix * a.nz * a.ny) / a.nz);
    const int iiix = a.px ? (ix + iix + a.nx) % a.nx : ix + iix;
    if (iiix < 0 || iiix >= a.nx) return 0;
    const int iiiy = a.py ? (iy + iiy + a.ny) % a.ny : iy + iiy;
    if (iiiy < 0 || iiiy >= a.ny) return 0;
    const int iiiz = a.pz ? (iz + iiz + a.nz) % a.nz : iz + iiz;
    if (iiiz < 0 || iiiz >= a.nz) return 0;
    const int wx = (ix + iix >= 0 && ix + iix < a.nx) ? 0 : (ix + iix < 0 ? 1 : -1);
    const int wy = (iy + iiy >= 0 && iy + iiy < a.ny) ? 0 : (iy + iiy < 0 ? 1 : -1);
    const int wz = (iz + iiz >= 0 && iz + iiz < a.nz) ? 0 : (iz + iiz < 0 ? 1 : -1);
    const int64_t icell2 = iiiz + (int64_t)a.nz * iiiy + (int64_t)a.nz * a.ny * iiix;
    if ((a.autocorr == 1 && icell2 > icell) || cell_count(bs2, icell2) == 0) return 0;
    const double offx = wx * a.xwrap, offy = wy * a.ywrap, offz = wz * a.zwrap;
    double cx = 0, cy = 0, cz = 0, mdx = 0, mdy = 0, mdz = 0;
    if (a.min_sep_opt) {
        const double* f = bd1 + icell * 6;
        const double* s = bd2 + icell2 * 6;
        const double xl = f[0] + offx, xh = f[1] + offx;
        const double yl = f[2] + offy, yh = f[3] + offy;
        const double zl = f[4] + offz, zh = f[5] + offz;
        cx = iix < 0 ? xl : (iix > 0 ? xh : 0.0);
        cy = iiy < 0 ? yl : (iiy > 0 ? yh : 0.0);
        cz = iiz < 0 ? zl : (iiz > 0 ? zh : 0.0);
        mdx = iix != 0 ? ((iix < 0 ? xl : xh) - (iix < 0 ? s[1] : s[0])) : 0.0;
        mdy = iiy != 0 ? ((iiy < 0 ? yl : yh) - (iiy < 0 ? s[3] : s[2])) : 0.0;
        mdz = iiz != 0 ? ((iiz < 0 ? zl : zh) - (iiz < 0 ? s[5] : s[4])) : 0.0;
        if (a.max3 > 0) {
            const double t = mdx * mdx + mdy * mdy + mdz * mdz;
            if (t >= a.max3 * a.max3) return 0;
        }
        if (a.max2 > 0) {
            const double t = mdx * mdx + mdy * mdy;
            if (t >= a.max2 * a.max2) return 0;
        }
        if (a.max1 > 0 && iiz != 0) {
            if (mdz * mdz >= a.max1 * a.max1) return 0;
        }
    }
    rec->c1 = (int)icell;
    rec->c2 = (int)icell2;
    rec->wx = (signed char)wx;
    rec->wy = (signed char)wy;
    rec->wz = (signed char)wz;
    rec->same = (a.autocorr == 1 && icell2 == icell) ? 1 : 0;
    rec->pad = 0;
    rec->mdx = mdx; rec->mdy = mdy; rec->mdz = mdz;
    rec->cx = cx; rec->cy = cy; rec->cz = cz;
    return 1;
}

__device__ int neighbour_added(const NgbArgs& a, int64_t icell, int k, const int* bs1, const int* bs2,
                               const double* bd1, const double* bd2, CellPairRec* rec)
{
    if (cell_count(bs1, icell) == 0) return 0;
    if (!eval_neighbour(a, icell, k, bs1, bs2, bd1, bd2, rec)) return 0;
    if (a.dupcheck) {
        // the reference skips a neighbour already appended for this primary cell with
        // the same secondary cell and the same wrap (gridlink_utils.h.src:46-72).
        // prev is initialized: eval_neighbour writes it only when it returns 1, and a
        // compiler may evaluate the comparisons below on an unwritten record and
        // combine them with the result (observed: neighbours dropped depending on
        // leftover register contents)
        CellPairRec prev = {};
        for (int kk = 0; kk < k; kk++) {
            const int added = eval_neighbour(a, icell, kk, bs1, bs2, bd1, bd2, &prev);
            if (added && prev.c2 == rec->c2 && prev.wx == rec->wx && prev.wy == rec->wy && prev.wz == rec->wz)
                return 0;
        }
    }
    return 1;
}

// The tests of a kept cell pair.
__device__ __forceinline__ double pair_tests(const CellPairRec& r, const int* __restrict__ bs1,
                                             const int* __restrict__ bs2)
{
    const double n1 = (double)cell_count(bs1, r.c1), n2 = (double)cell_count(bs2, r.c2);
    return r.same ? n1 * (n1 - 1) * 0.5 : n1 * n2;
}

// Adds a workgroup's (256 threads) sum of `my` to *out, one atomic per workgroup
// (integers below 2^53: exact in any order).
__device__ __forceinline__ void add_tests(double my, double* __restrict__ out)
{
    __shared__ double part[4];
    for (int o = 32; o > 0; o >>= 1) my += __shfl_xor(my, o, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = my;
    __syncthreads();
    if (threadIdx.x == 0) {
        const double s = part[0] + part[1] + part[2] + part[3];
        if (s != 0) atomicAdd(out, s);
    }
}

// Flags the candidates that are kept; the pairs tested are added to
// tested[0 .. kTestedSlots - 1], spread because atomics on one address are
// serialized (~14 ns each).
constexpr int kTestedSlots = 64;
__global__ __launch_bounds__(256) void k_cellpair_flag(NgbArgs a, int64_t ncells, int nngb,
                                                       const int* __restrict__ bs1, const int* __restrict__ bs2,
                                                       const double* __restrict__ bd1,
                                                       const double* __restrict__ bd2, int* __restrict__ flags,
                                                       double* __restrict__ tested)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    double my = 0;
    if (t < ncells * nngb) {
        CellPairRec r = {};
        const int f = neighbour_added(a, t / nngb, (int)(t % nngb), bs1, bs2, bd1, bd2, &r);
        flags[t] = f;
        if (f) my = pair_tests(r, bs1, bs2);
    }
    add_tests(my, &tested[blockIdx.x % kTestedSlots]);
}

// The records of the flagged candidates at their scan positions (a kept candidate
// only needs its record again, not the duplicate check).
__global__ __launch_bounds__(256) void k_cellpair_emit(NgbArgs a, int64_t ncells, int nngb,
                                                       const int* __restrict__ bs1, const int* __restrict__ bs2,
                                                       const double* __restrict__ bd1,
                                                       const double* __restrict__ bd2, const int* __restrict__ flags,
                                                       const int* __restrict__ pos, CellPairRec* __restrict__ out,
                                                       int cat)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (t >= ncells * nngb || !flags[t]) return;
    CellPairRec r = {};
    if (eval_neighbour(a, t / nngb, (int)(t % nngb), bs1, bs2, bd1, bd2, &r)) {
        r.pad = cat;
        out[pos[t]] = r;
    }
}

// ------------------------------------------------- exact pair replay (a8-a12)
__device__ __forceinline__ double r2_3d(int f, double dx, double dy, double dz)
{
    switch (f) {
    case R2_FMA_DZ_DY_DX: return fma(dz, dz, fma(dy, dy, dx * dx));
    case R2_X_SUM_YZ: return dx * dx + (dy * dy + dz * dz);
    case R2_FMA_DX_DY_DZ: return fma(dx, dx, fma(dy, dy, dz * dz));
    default: return (dx * dx + dy * dy) + dz * dz;
    }
}

__device__ __forceinline__ double rp2_f(int f, double dx, double dy)
{
    return f == RP_FMA ? fma(dy, dy, dx * dx) : dx * dx + dy * dy;
}

// first k from the top with r2 >= rupp_sqr[k-1] (countpairs_kernels.c.src:982-993)
__device__ __forceinline__ int find_kbin(const double* __restrict__ e, int nbin, int sorted, double r2)
{
    if (sorted) {
        int lo = 0, hi = nbin - 1;  // count of e[0..nbin-2] <= r2
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (e[mid] <= r2) lo = mid + 1; else hi = mid;
        }
        return lo;
    }
    for (int k = nbin - 1; k >= 1; k--)
        if (r2 >= e[k - 1]) return k;
    return 0;
}

// On-sky pair (mocks/DDrppi_mocks/countpairs_rp_pi_mocks_kernels.c.src:1240-1290,
// mocks/DDsmu_mocks/countpairs_s_mu_mocks_kernels.c.src fallback): s = x_j - x_i,
// l = x_i + x_j; rp-pi: pi^2 = (s.l)^2 / |l|^2, rp^2 = s^2 - pi^2; s-mu:
// mu^2 = (s.l)^2 / (|l|^2 s^2). Returns 0 for a rejected pair, else the squared
// separation that selects the bin (*key: rp^2 or s^2) and the pi / mu column
// (*j2; n2 where pi^2 >= pimax^2 or mu^2 >= mu_max^2, as the reference).
__device__ __forceinline__ int los_split(const PairParams& P, int mode, double xi, double yi, double zi, double xj,
                                         double yj, double zj, double* key, int* j2)
{
    const double parx = xi + xj, pary = yi + yj, parz = zi + zj;
    const double perpx = xj - xi, perpy = yj - yi, perpz = zj - zi;
    const double sqr_s = perpx * perpx + perpy * perpy + perpz * perpz;
    const double s_dot_l = parx * perpx + pary * perpy + parz * perpz;
    const double sqr_l = parx * parx + pary * pary + parz * parz;
    const double sqr_s_dot_l = s_dot_l * s_dot_l;
    const double sqr_lim = P.sqr_mu_max;
    if (mode == MODE_RPPI_MOCKS) {
        if (sqr_s >= P.sqr_rmax) return 0;
        if (sqr_s_dot_l >= sqr_l * sqr_lim) return 0;
        const double sqr_par = sqr_s_dot_l / sqr_l;
        *j2 = sqr_par >= sqr_lim ? P.n2 : (int)(sqrt(sqr_par) * P.inv_d2);
        const double sqr_perp = sqr_s - sqr_par;
        if (sqr_perp >= P.sqr_rpmax || sqr_perp < P.sqr_rmin) return 0;
        *key = sqr_perp;
        return 1;
    }
    if (sqr_s >= P.sqr_rmax || sqr_s < P.sqr_rmin) return 0;
    const double sqr_mu = sqr_s_dot_l / (sqr_l * sqr_s);
    *j2 = sqr_mu >= sqr_lim ? P.n2 : (int)(sqrt(sqr_mu) * P.inv_d2);
    *key = sqr_s;
    return 1;
}

struct ITerms {
    double xpos, ypos, zpos;
    double max_dz, target;
    int skip;
};

// The reference kernels' per-particle prologue (countpairs_kernels.c.src:900-950 and
// the rp_pi / s_mu / wp / xi counterparts): position + wrap, minimum separation of
// this particle to the secondary cell, z window.
__device__ __forceinline__ void i_terms(const PairParams& P, int mode, const CellPairRec& cp, double xi, double yi,
                                        double zi, ITerms* t)
{
    t->xpos = xi + cp.wx * P.xwrap;
    t->ypos = yi + cp.wy * P.ywrap;
    t->zpos = zi + cp.wz * P.zwrap;
    if (cp.same) {
        t->skip = 0;
        t->max_dz = (mode == MODE_RPPI || mode == MODE_WP) ? P.pimax : P.max_all_dz_same;
        t->target = t->zpos - t->max_dz;
        return;
    }
    const double mdx = cp.mdx > 0 ? cp.mdx + fabs(t->xpos - cp.cx) : cp.mdx;
    const double mdy = cp.mdy > 0 ? cp.mdy + fabs(t->ypos - cp.cy) : cp.mdy;
    const double mdz = cp.mdz > 0 ? cp.mdz + fabs(t->zpos - cp.cz) : cp.mdz;
    if (mode == MODE_RPPI || mode == MODE_WP) {
        t->skip = (mdx * mdx + mdy * mdy) >= P.sqr_rmax || mdz >= P.pimax;
        t->max_dz = P.pimax;
        t->target = t->zpos - P.pimax;
    } else if (mode == MODE_SMU) {
        t->skip = ((mdx * mdx + mdy * mdy) + mdz * mdz) >= P.sqr_rmax || mdz >= P.pimax;
        const double sq = (P.sqr_rmax - mdx * mdx) - mdy * mdy;
        t->max_dz = sq < P.pimax * P.pimax ? sqrt(sq) : P.pimax;
        t->target = t->zpos - t->max_dz;
    } else {
        t->skip = ((mdx * mdx + mdy * mdy) + mdz * mdz) >= P.sqr_rmax;
        t->max_dz = sqrt((P.sqr_rmax - mdx * mdx) - mdy * mdy);
        t->target = t->zpos - t->max_dz;
    }
}

// Decides one (i, j) pair exactly as the reference does. Returns the histogram
// slot or -1; *sep receives sqrt(r^2) (or sqrt(s^2)).
// `window` = 0 skips the z-window / per-particle tests, which the caller may do
// only when it has shown the pair lies outside the edge windows (see k_pairs_tuned).
__device__ __forceinline__ int replay_pair(const PairParams& P, int mode, const ITerms& t, int same, int window,
                                           double xj, double yj, double zj, const double* __restrict__ e,
                                           double* sep)
{
    const double dx = xj - t.xpos, dy = yj - t.ypos, dz = zj - t.zpos;
    if (mode == MODE_RPPI || mode == MODE_WP) {
        if (window && ((!same && (t.skip || zj <= t.target)))) return -1;
        if (dz <= -P.pimax || dz >= P.pimax) return -1;
        const double adz = fabs(dz);
        const double r2 = rp2_f(P.r2form, dx, dy);
        if (r2 >= P.sqr_rmax || r2 < P.sqr_rmin) return -1;
        const int k = find_kbin(e, P.nbin, P.sorted_edges, r2);
        if (k == 0) return -1;
        *sep = sqrt(r2);
        if (mode == MODE_WP) return k;
        if (P.float_index) return (int)((double)k * (double)(P.n2 + 1) + adz * P.inv_d2);
        int pb = (int)(adz * P.inv_d2);
        pb = pb > P.n2 ? P.n2 : pb;
        return k * (P.n2 + 1) + pb;
    }
    if (window) {
        if (t.skip) return -1;
        if (zj <= t.target) return -1;
        if (dz >= t.max_dz) return -1;
    }
    if (mode == MODE_RPPI_MOCKS || mode == MODE_SMU_MOCKS) {
        double key;
        int j2;
        if (!los_split(P, mode, t.xpos, t.ypos, t.zpos, xj, yj, zj, &key, &j2)) return -1;
        const int k = find_kbin(e, P.nbin, P.sorted_edges, key);
        if (k == 0) return -1;
        *sep = sqrt(key);
        return k * (P.n2 + 1) + j2;
    }
    if (mode == MODE_SMU) {
        const double sqr_dz = dz * dz;
        const double s2 = P.r2form == R2_FMA_DX_DY_DZ ? fma(dx, dx, fma(dy, dy, sqr_dz)) : (dx * dx + dy * dy) + sqr_dz;
        if (s2 >= P.sqr_rmax || s2 < P.sqr_rmin) return -1;
        if (sqr_dz >= s2 * P.sqr_mu_max) return -1;
        const double mu = sqrt(sqr_dz / s2);
        const int k = find_kbin(e, P.nbin, P.sorted_edges, s2);
        if (k == 0) return -1;
        *sep = sqrt(s2);
        if (P.float_index) return (int)((double)k * (double)(P.n2 + 1) + mu * P.inv_d2);
        int mb = (int)(mu * P.inv_d2);
        mb = mb > P.n2 ? P.n2 : mb;
        return k * (P.n2 + 1) + mb;
    }
    const double r2 = r2_3d(P.r2form, dx, dy, dz);
    if (r2 >= P.sqr_rmax || r2 < P.sqr_rmin) return -1;
    const int k = find_kbin(e, P.nbin, P.sorted_edges, r2);
    if (k == 0) return -1;
    *sep = sqrt(r2);
    return k;
}

// Histogram of one workgroup in LDS: counts (u64), sum of separations, sum of weights.
struct LdsHist {
    unsigned long long* np;
    double* avg;
    double* w;
};

__device__ __forceinline__ void hist_add(const PairParams& P, LdsHist& h, int slot, double sep, double wprod)
{
    atomicAdd(&h.np[slot], 1ull);
    if (P.need_avg) atomicAdd(&h.avg[slot], sep);
    if (P.need_w) atomicAdd(&h.w[slot], wprod);
}

__device__ void hist_flush(const PairParams& P, LdsHist& h, unsigned long long* g_np, double* g_avg, double* g_w)
{
    for (int s = threadIdx.x; s < P.nslots; s += blockDim.x) {
        const unsigned long long c = h.np[s];
        if (c) {
            atomicAdd(&g_np[s], c);
            if (P.need_avg) atomicAdd(&g_avg[s], h.avg[s]);
            if (P.need_w) atomicAdd(&g_w[s], h.w[s]);
        }
    }
}

__device__ void hist_init(const PairParams& P, LdsHist& h)
{
    for (int s = threadIdx.x; s < P.nslots; s += blockDim.x) {
        h.np[s] = 0;
        h.avg[s] = 0;
        h.w[s] = 0;
    }
}

// -------------------------------------------------- plain FP64 pair kernel
// One workgroup per cell pair; every (i, j) of the pair is decided in FP64 with
// the full reference predicate. This is the "plain GPU form". Its histogram is
// FP64 in LDS (GH = false), or the global histogram itself (GH = true) when
// the slots do not fit the workgroup's LDS.
template <bool GH>
__global__ __launch_bounds__(128) void k_pairs_plain(PairParams P, DevLattice L1, DevLattice L2,
                                                     const CellPairRec* __restrict__ cps,
                                                     const double* __restrict__ rupp_sqr,
                                                     unsigned long long* __restrict__ g_np,
                                                     double* __restrict__ g_avg, double* __restrict__ g_w)
{
    extern __shared__ unsigned long long smem_u64[];
    LdsHist h;
    const double* e;
    if (GH) {
        // no LDS: histogram and edges in global memory
        h.np = g_np;
        h.avg = g_avg;
        h.w = g_w;
        e = rupp_sqr;
    } else {
        h.np = smem_u64;
        h.avg = reinterpret_cast<double*>(smem_u64 + P.nslots);
        h.w = h.avg + P.nslots;
        double* el = h.w + P.nslots;
        hist_init(P, h);
        for (int s = threadIdx.x; s < P.nbin; s += blockDim.x) el[s] = rupp_sqr[s];
        e = el;
        __syncthreads();
    }
    const CellPairRec cp = cps[blockIdx.x];
    const int mode = P.mode;
    const int i0 = L1.bstart[cp.c1], i1 = L1.bstart[cp.c1 + 1];
    const int j0 = L2.bstart[cp.c2], j1 = L2.bstart[cp.c2 + 1];
    for (int i = i0 + threadIdx.x; i < i1; i += blockDim.x) {
        ITerms t = {};
        const double4 pi = L1.d4[i];
        i_terms(P, mode, cp, pi.x, pi.y, pi.z, &t);
        if (t.skip) continue;
        const int jstart = cp.same ? i + 1 : j0;
        for (int j = jstart; j < j1; j++) {
            double sep = 0;
            const double4 pj = L2.d4[j];
            const int slot = replay_pair(P, mode, t, cp.same, 1, pj.x, pj.y, pj.z, e, &sep);
            if (slot >= 0) hist_add(P, h, slot, sep, P.need_w ? pi.w * pj.w : 0.0);
        }
    }
    if (GH) return;
    __syncthreads();
    hist_flush(P, h, g_np, g_avg, g_w);
}
template __global__ void k_pairs_plain<false>(PairParams, DevLattice, DevLattice, const CellPairRec*, const double*,
                                              unsigned long long*, double*, double*);
template __global__ void k_pairs_plain<true>(PairParams, DevLattice, DevLattice, const CellPairRec*, const double*,
                                             unsigned long long*, double*, double*);

// ------------------------------------------------- tuned pair kernel
// Work item: (cell pair, chunk of <= 64 consecutive primary particles).
// Each wave pulls work items from a device counter until the list is exhausted.
// Lane l holds primary particle i0+l. The secondary particles of the cell pair
// come in groups of kGroup with a bounding box each; the lanes test 64 groups at
// a time against the chunk's box, and runs of groups within reach are read with
// scalar loads: the index is wave-uniform, so a secondary lands in scalar
// registers that every lane's vector instructions read directly (no per-lane
// load, no broadcast instruction). Two paths per group:
//  * dense (enough of its pairs are in range): each (i, j) is decided in FP64 in
//    lockstep from a 32-byte (x, y, z, w) record;
//  * sparse: an integer test on quantized cell-local positions (packed 16-bit
//    differences, one dot-product instruction per pair), with thresholds that
//    provably pass every pair the FP64 test can accept, rejects the pairs that
//    cannot be in range; the survivors are compacted into a per-wave LDS queue
//    and decided 64 at a time in FP64.
// Either way every counted pair is decided by the reference's FP64 arithmetic.
constexpr int kQueues = 8;          // work sub-queues (one counter each)
constexpr int kCounterStride = 32;  // ints between sub-queue counters (128 B)
// Secondary windows up to this many groups are not box-tested: the test's chain of
// loads costs what the skipped groups save (uniform DD, kernel, with 2 / 4 / 8: 43
// particles per cell 1.50 / 1.38 / 1.38 ms, 57 2.00 / 1.93 / 1.91, 115 5.32 / 5.32 / 5.49).
constexpr int kFewGroups = 4;
constexpr int kBlockJ = 4;          // secondaries per scalar load of the sparse path
// Survivor buffer per wave: entries (j << 6) | lane at [head, tail). Drains take
// 64 * DP entries from the head (DP survivors per lane: 1, or 2 with both pairs'
// records loaded before either is decided); a scan runs while fewer than that
// wait, a block adds <= 64 kBlockJ, and lanes without a survivor write up to 127
// slots past the tail (see enqueue); once head >= kCompactAt the remaining
// entries move to the front. At a block's start head <= 64 (DP = 1; head
// advances by 64 and is reset at 128) or head = 0 (DP = 2: every drain round
// ends with the move) and tail - head < 64 DP, so tail <= 127 and the
// furthest write is 127 + 64 (kBlockJ - 1) + 127 < kQueueAlloc.
constexpr int kCompactAt = 128;
constexpr int kQueueAlloc = kCompactAt + 64 + 64 * (kBlockJ - 1) + 127;
// Queue entries hold secondary indices relative to the first one of the 64
// groups being scanned, ((j - jbase) << 6) | lane.

// Read-only particle data seen through the constant address space: loads with a
// wave-uniform index become scalar loads.
typedef const __attribute__((address_space(4))) double KDouble;
typedef const __attribute__((address_space(4))) unsigned KUint;
__device__ __forceinline__ double4 kload_d4(KDouble* p, int j)
{
    return make_double4(p[4 * (int64_t)j], p[4 * (int64_t)j + 1], p[4 * (int64_t)j + 2], p[4 * (int64_t)j + 3]);
}
__device__ __forceinline__ uint2 kload_u2(KUint* p, int j)
{
    return make_uint2(p[2 * (int64_t)j], p[2 * (int64_t)j + 1]);
}
typedef short short2v __attribute__((ext_vector_type(2)));

// sqrt(r2) to ~1e-14 relative from y = the hardware FP32 reciprocal square root
// of f = (float)r2: s = f y, one FP32 Newton step (to about half an ulp of FP32),
// one in FP64. One transcendental (a quarter of the FMA rate), shared with the mu
// bin, instead of a square root and a reciprocal. Lanes below 1e-30 take sqrt; the
// test is one branch of the whole wave.
__device__ __forceinline__ double fast_sqrt(double r2, float f, float y)
{
    const float h = 0.5f * y, s0 = f * y;
    const float s = fmaf(fmaf(-s0, s0, f), h, s0);
    const double sd = (double)s;
    double r = fma(fma(-sd, sd, r2), (double)h, sd);
    if (__builtin_amdgcn_ballot_w64(!(f > 1e-30f))) {
        double q = sqrt(r2);
        asm volatile("" : "+v"(q));  // keeps the branch: the compiler would compute q always and select
        r = f > 1e-30f ? r : q;
    }
    return r;
}

// Histogram of one workgroup of the tuned kernel, replicated R ways with layout
// [slot][R]: lanes of one wave that land in the same slot add to different
// copies, which sit in different banks. Counts u64, sums FP64 (native
// ds_add_u64 / ds_add_f64: the LDS atomics issue on the LDS pipe, not on the
// VALU, which bounds this kernel). GH kernels (histograms larger than the
// workgroup's LDS) add to the global histogram instead.
struct KernelLds {
    unsigned long long* np;
    double* avg;
    double* w;
    int rshift;                // log2 R
    int lane_copy;             // lane & (R - 1)
    const double* e;           // rupp_sqr[0..nbin-1]
    const unsigned short* lut; // bin lookup
    unsigned long long* gnp;   // the global histogram (GH)
    double* gavg;
    double* gw;
};

// Per-launch flags of the tuned kernel as compile-time constants: FL >= 0 is the
// mask of the launch's separation sums (kFlAvg), weight sums (kFlW) and
// single-step bin lookup (kFlLut1: sorted edges, at most one edge per lookup
// bucket); FL = kFlRuntime reads them from P (the global-histogram kernels).
// Read from P, every such test in the per-pair code is a uniform branch on a
// scalar lane mask held across the persistent loop, and the masks crowd the
// scalar registers into spills.
constexpr int kFlAvg = 1, kFlW = 2, kFlLut1 = 4, kFlRuntime = -1;
template <int FL>
__device__ __forceinline__ bool fl_avg(const PairParams& P)
{
    return FL < 0 ? P.need_avg != 0 : (FL & kFlAvg) != 0;
}
template <int FL>
__device__ __forceinline__ bool fl_w(const PairParams& P)
{
    return FL < 0 ? P.need_w != 0 : (FL & kFlW) != 0;
}
template <int FL>
__device__ __forceinline__ bool fl_lut1(const PairParams& P)
{
    return FL < 0 ? (P.sorted_edges != 0 && P.lut_single != 0) : (FL & kFlLut1) != 0;
}
// The reference's AVX512F flattened (rp, pi) / (s, mu) index rule: used exactly
// when the rounding order replayed is the AVX512F kernel's (the host sets
// P.float_index by the same rule).
template <int MODE, int R2F>
__device__ __forceinline__ constexpr bool float_index_of()
{
    return (MODE == MODE_RPPI && R2F == RP_FMA) || (MODE == MODE_SMU && R2F == R2_FMA_DX_DY_DZ);
}

// Adds a counted pair (slot, squared separation r2, weight product) to the
// histogram; f = (float)r2, y its reciprocal square root.
template <bool GH, int FL>
__device__ __forceinline__ void hist_pair(const PairParams& P, KernelLds& S, int slot, double r2, float f, float y,
                                          double wprod)
{
    if (GH) {
        atomicAdd(&S.gnp[slot], 1ull);
        if (fl_avg<FL>(P)) atomicAdd(&S.gavg[slot], fast_sqrt(r2, f, y));
        if (fl_w<FL>(P)) atomicAdd(&S.gw[slot], wprod);
        return;
    }
    const int a = (slot << S.rshift) + S.lane_copy;
    atomicAdd(&S.np[a], 1ull);
    if (fl_avg<FL>(P)) atomicAdd(&S.avg[a], fast_sqrt(r2, f, y));
    if (fl_w<FL>(P)) atomicAdd(&S.w[a], wprod);
}

// Number of edges e[0..nbin-2] <= r2 (the reference's top-down bin search,
// countpairs_kernels.c.src:982-993, for non-decreasing edges), for e[0] <= r2 <
// e[nbin-1]: start from the lookup table's lower bound for the 1/16-octave bucket
// of f = (float)r2 and step up. (The table ends above the bucket of e[nbin-1], so
// only its start needs a clamp: e[0] may be 0.) 0 only for unsorted edges.
template <int FL>
__device__ __forceinline__ int lut_kbin(const PairParams& P, const KernelLds& S, double r2, float f)
{
    if (!fl_lut1<FL>(P) && !P.sorted_edges) return find_kbin(S.e, P.nbin, 0, r2);
    const unsigned idx = __builtin_elementwise_sub_sat(__float_as_uint(f) >> 19, (unsigned)P.lut_base);
    int k = S.lut[idx];
    if (fl_lut1<FL>(P)) return k + (S.e[k] <= r2 ? 1 : 0);  // e[nbin-1] = rmax^2 > r2
    while (k < P.nbin - 1 && S.e[k] <= r2) k++;
    return k;
}

// slot of bin k, column m (24-bit multiply: an LDS histogram has fewer slots).
template <bool GH>
__device__ __forceinline__ int slot_of(const PairParams& P, int k, int m)
{
    return GH ? k * (P.n2 + 1) + m : (int)__umul24((unsigned)k, (unsigned)(P.n2 + 1)) + m;
}

// Whether the integer part of an FP32 estimate t with error below 1e-6 (t + 1) is
// certain (false for NaN and infinities).
__device__ __forceinline__ bool column_sure(float t)
{
    return fabsf(__builtin_amdgcn_fractf(t) - 0.5f) <= fmaf(-1e-6f, t, 0.499999f);
}

// a / b, correctly rounded for operands whose quotient and reciprocal are normal
// (Markstein: two Newton steps on the hardware reciprocal, then one on the
// quotient with its exact remainder); the general division also scales and fixes
// up the ranges that squared comoving distances do not reach.
__device__ __forceinline__ double quotient(double a, double b)
{
    double r = __builtin_amdgcn_rcp(b);
    r = fma(fma(-b, r, 1.0), r, r);
    r = fma(fma(-b, r, 1.0), r, r);
    const double q = a * r;
    return fma(fma(-b, q, a), r, q);
}

// FP64 separation in the rounding order R2F of the reference kernel being replayed.
template <int R2F>
__device__ __forceinline__ double sep2(double dx, double dy, double dz)
{
    if (R2F == R2_FMA_DZ_DY_DX) return fma(dz, dz, fma(dy, dy, dx * dx));
    if (R2F == R2_X_SUM_YZ) return dx * dx + (dy * dy + dz * dz);
    if (R2F == R2_FMA_DX_DY_DZ) return fma(dx, dx, fma(dy, dy, dz * dz));
    if (R2F == RP_FMA) return fma(dy, dy, dx * dx);
    if (R2F == RP_SUM) return dx * dx + dy * dy;
    return (dx * dx + dy * dy) + dz * dz;
}

// The same pointer, opaque to the compiler: loads through it are issued where
// they are written (not hoisted, not merged with earlier ones), which keeps
// values that only rare paths need out of the registers of the hot loops.
template <typename T>
__device__ __forceinline__ const T* fresh(const T* p)
{
    asm volatile("" : "+s"(p));
    return p;
}
// The same for read-only data seen through the constant address space, so the
// loads are scalar.
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T* fresh_k(const T* p)
{
    asm volatile("" : "+s"(p));
    return (const __attribute__((address_space(4))) T*)(const void*)p;
}

// Decides one (i, j) pair in FP64 exactly as the reference does and adds it to
// the LDS histogram. (xpos, ypos, zpos) = primary position plus the cell pair's
// wrap; (xj, yj, zj) = secondary position. `ok` masks lanes without a pair. UNI:
// cpp and l1p are the same in all lanes.
template <int MODE, int R2F, bool GH, int FL, bool UNI = true>
__device__ __forceinline__ void exact_pair(const PairParams& P, const CellPairRec* cpp, const DevLattice* l1p, int i,
                                           int ok, double xpos, double ypos, double zpos, double wi, double xj,
                                           double yj, double zj, double wj, KernelLds& S)
{
    constexpr bool is2d = MODE == MODE_RPPI || MODE == MODE_WP;
    constexpr bool onsky = MODE == MODE_RPPI_MOCKS || MODE == MODE_SMU_MOCKS;
    const double dx = xj - xpos, dy = yj - ypos, dz = zj - zpos;
    if (onsky) {
        // as los_split, with the pi / mu column from an FP32 estimate: each factor
        // rounded once and the hardware roots (1 ulp) put t within 7e-7 of its value,
        // so its integer part is the reference's unless t is within 1e-6 (t + 1) of an
        // integer; only those pairs take the FP64 root (and, for mu, the quotient)
        const double parx = xpos + xj, pary = ypos + yj, parz = zpos + zj;
        const double sqr_s = dx * dx + dy * dy + dz * dz;
        const double s_dot_l = parx * dx + pary * dy + parz * dz;
        const double sqr_l = parx * parx + pary * pary + parz * parz;
        const double sqr_s_dot_l = s_dot_l * s_dot_l;
        const double sqr_lim = P.sqr_mu_max;
        bool in = ok && sqr_s < P.sqr_rmax;
        double key;
        int j2;
        if (MODE == MODE_RPPI_MOCKS) {
            if (!(in && sqr_s_dot_l < sqr_l * sqr_lim)) return;
            const double sqr_par = quotient(sqr_s_dot_l, sqr_l);
            key = sqr_s - sqr_par;
            if (!(key < P.sqr_rpmax && key >= P.sqr_rmin)) return;
            const float t = __builtin_amdgcn_sqrtf((float)sqr_par) * (float)P.inv_d2;
            j2 = (int)t;
            if (!column_sure(t)) j2 = sqr_par >= sqr_lim ? P.n2 : (int)(sqrt(sqr_par) * P.inv_d2);
        } else {
            if (!(in && sqr_s >= P.sqr_rmin)) return;
            key = sqr_s;
            const float t = fabsf((float)s_dot_l) * __builtin_amdgcn_rsqf((float)sqr_l) *
                            __builtin_amdgcn_rsqf((float)sqr_s) * (float)P.inv_d2;
            j2 = (int)fminf(t, (float)P.n2);
            if (!column_sure(t)) {
                const double sqr_mu = sqr_s_dot_l / (sqr_l * sqr_s);
                j2 = sqr_mu >= sqr_lim ? P.n2 : (int)(sqrt(sqr_mu) * P.inv_d2);
            }
        }
        // pruning replay for pairs near the 3-D limit (the 3-D kernels' rules)
        if (sep2<R2F>(dx, dy, dz) >= P.near_lo2) {
            const CellPairRec* c = UNI ? fresh(cpp) : cpp;
            const DevLattice* l1 = UNI ? fresh(l1p) : l1p;
            ITerms t = {};
            const double4 p = l1->d4[i];
            i_terms(P, MODE, *c, p.x, p.y, p.z, &t);
            if (t.skip || zj <= t.target || dz >= t.max_dz) return;
        }
        const float f = (float)key;
        const int k = lut_kbin<FL>(P, S, key, f);
        if (!fl_lut1<FL>(P) && k == 0) return;
        hist_pair<GH, FL>(P, S, slot_of<GH>(P, k, j2), key, f, __builtin_amdgcn_rsqf(f), wi * wj);
        return;
    }
    const double sqr_dz = dz * dz;
    const double r2 = sep2<R2F>(dx, dy, dz);
    const double adz = fabs(dz);
    bool in = ok && r2 < P.sqr_rmax && r2 >= P.sqr_rmin;
    if (is2d) in = in && adz < P.pimax;
    if (MODE == MODE_SMU) in = in && sqr_dz < r2 * P.sqr_mu_max;
    if (!in) return;
    // The reference's pruning tests (per-particle minimum separation, z window)
    // can only reject pairs within a few ulps of the coordinate scale of rmax or
    // pimax; only such pairs replay them.
    const bool near = r2 >= P.near_lo2 || (MODE != MODE_DD && MODE != MODE_XI && adz >= P.near_lodz);
    if (near) {
        // the cell pair record and the primary set, loaded here
        const CellPairRec* c = UNI ? fresh(cpp) : cpp;
        const DevLattice* l1 = UNI ? fresh(l1p) : l1p;
        ITerms t = {};
        const double4 p = l1->d4[i];
        i_terms(P, MODE, *c, p.x, p.y, p.z, &t);
        if (is2d) {
            if (!c->same && (t.skip || zj <= t.target)) return;
        } else {
            if (t.skip || zj <= t.target || dz >= t.max_dz) return;
        }
    }
    const bool findex = FL < 0 ? P.float_index != 0 : float_index_of<MODE, R2F>();
    const float f = (float)r2;
    const int k = lut_kbin<FL>(P, S, r2, f);
    if (!fl_lut1<FL>(P) && k == 0) return;
    const float y = MODE == MODE_SMU || fl_avg<FL>(P) ? __builtin_amdgcn_rsqf(f) : 0.0f;
    int slot = k;
    if (MODE == MODE_RPPI) {
        if (findex) {
            slot = (int)((double)k * (double)(P.n2 + 1) + adz * P.inv_d2);
        } else {
            int pb = (int)(adz * P.inv_d2);
            slot = slot_of<GH>(P, k, pb > P.n2 ? P.n2 : pb);
        }
    } else if (MODE == MODE_SMU) {
        // mu bin from an FP32 estimate t ~ mu * inv_dmu: |dz|, s^2 and inv_dmu
        // rounded to FP32 (2^-24 each), the hardware reciprocal square root (1
        // ulp) and two products put t within 4e-7 * t of the reference's FP64
        // value, so its integer part is the reference's unless t lies within
        // 1e-6 * (t + 1) of an integer; only those pairs (and non-finite
        // estimates) compute mu = sqrt(dz^2 / s^2) in FP64 as the reference does
        // (countpairs_s_mu_kernels.c.src:1154-1171).
        const float t = (float)adz * y * (float)P.inv_d2;
        if (column_sure(t)) {
            slot = slot_of<GH>(P, k, min((int)t, P.n2));
        } else {
            const double mu = sqrt(sqr_dz / r2);
            if (findex) {
                slot = (int)((double)k * (double)(P.n2 + 1) + mu * P.inv_d2);
            } else {
                const int mb = (int)(mu * P.inv_d2);
                slot = slot_of<GH>(P, k, mb > P.n2 ? P.n2 : mb);
            }
        }
    }
    hist_pair<GH, FL>(P, S, slot, r2, f, y, wi * wj);
}

// Decides up to 64 queued survivors (entries ((j - jbase) << 6) | lane) in FP64.
template <int MODE, int R2F, bool GH, int FL>
__device__ __forceinline__ void drain_queue(const PairParams& P, const CellPairRec& cp, const CellPairRec* cpp,
                                            const DevLattice* l1p, const double4* d4_1, const double4* d4_2,
                                            const double3& wrap, int i0, int istride, const unsigned* qe,
                                            const double4* prim, unsigned head, int ndrain, int jbase,
                                            KernelLds& S)
{
    const int lane = lane_id();
    if (lane < ndrain) {
        const unsigned e = qe[head + lane];
        const int j = jbase + (int)(e >> 6), l = (int)(e & 63);
        const int i = i0 + l * istride;
        double4 pi;
        if (P.prim_cache) {
            pi = prim[l];  // the primary's wrapped position and weight
        } else {
            pi = d4_1[i];
            pi.x += wrap.x;
            pi.y += wrap.y;
            pi.z += wrap.z;
        }
        const double4 pj = d4_2[j];
        exact_pair<MODE, R2F, GH, FL>(P, cpp, l1p, i, 1, pi.x, pi.y, pi.z, pi.w, pj.x, pj.y, pj.z, pj.w, S);
    }
}

// Decides up to 128 queued survivors, two per lane: both pairs' records are
// loaded before either is decided, so two gathers are in flight per lane (the
// DP = 2 kernels, for launches whose LDS already limits the waves per SIMD to
// five or fewer: the extra registers then cost no residency).
template <int MODE, int R2F, bool GH, int FL>
__device__ __forceinline__ void drain_queue2(const PairParams& P, const CellPairRec& cp, const CellPairRec* cpp,
                                             const DevLattice* l1p, const double4* d4_1, const double4* d4_2,
                                             const double3& wrap, int i0, int istride, const unsigned* qe,
                                             const double4* prim, unsigned head, int ndrain, int jbase,
                                             KernelLds& S)
{
    const int lane = lane_id();
    const int oka = lane < ndrain, okb = lane + 64 < ndrain;
    // entries past the tail read as 0: j = jbase, primary i0 (valid indices)
    const unsigned ea0 = qe[head + lane], eb0 = qe[head + 64 + lane];
    const unsigned ea = oka ? ea0 : 0u, eb = okb ? eb0 : 0u;
    const int ja = jbase + (int)(ea >> 6), la = (int)(ea & 63);
    const int jb = jbase + (int)(eb >> 6), lb = (int)(eb & 63);
    const int ia = i0 + la * istride, ib = i0 + lb * istride;
    double4 pia, pib;
    if (P.prim_cache) {
        pia = prim[la];
        pib = prim[lb];
    } else {
        pia = d4_1[ia];
        pib = d4_1[ib];
        pia.x += wrap.x;
        pia.y += wrap.y;
        pia.z += wrap.z;
        pib.x += wrap.x;
        pib.y += wrap.y;
        pib.z += wrap.z;
    }
    const double4 pja = d4_2[ja], pjb = d4_2[jb];
    exact_pair<MODE, R2F, GH, FL>(P, cpp, l1p, ia, oka, pia.x, pia.y, pia.z, pia.w, pja.x, pja.y, pja.z, pja.w, S);
    exact_pair<MODE, R2F, GH, FL>(P, cpp, l1p, ib, okb, pib.x, pib.y, pib.z, pib.w, pjb.x, pjb.y, pjb.z, pjb.w, S);
}

// Integer pair filter on quantized cell-local positions (secondary s, primary
// qxy / qz). 3-D: (dqx^2 + dqy^2 + dqz^2 + qlo) mod 2^32 < qrange; projected:
// the same on (dqx, dqy) and |dqz| < zq, as (dqz + zq - 1) unsigned < 2 zq - 1
// with zoff = zq - 1 - qz. Differences fit 16 bits and sums of squares 32 bits
// (|q| <= kQMax), so the only rounding is that of the positions themselves.
//
// On-sky (rp, pi) adds a test of rp: with l = x_i + x_j, s.l = |x_j|^2 - |x_i|^2 and
// |l|^2 = 2 |x_i|^2 + 2 |x_j|^2 - s^2, so rp^2 < rpmax^2 means (s^2 - rpmax^2) |l|^2 <
// (s.l)^2. In FP32 from the quantized s^2 and the stored 2 |x|^2: the left side is
// taken too small (s^2 less the quantization's 4 h smax, |l|^2 with smax^2 for s^2 and
// less 2^-20 of the largest |x|^2, at least 0) and |s.l| too large (by 2^-20 of it),
// which covers the rounding, so every pair the FP64 test can accept passes (NaN passes). Of the
// pairs within the 3-D limit 64 % are out of rp range (rpmax 25, pimax 40), and
// eight instructions here replace their share of a decision of about 85.
struct QFilter {
    float los_r, los_a, los_c1, los_c0, los_t0;  // 2 |x_i|^2 and the test's terms
    unsigned qxy;
    int qz, qlo, zoff;
    unsigned qrange, zspan;
    int ilim;                  // same cell: the lane takes j > ilim
};
// The wave's mask of lanes whose pair with secondary s (index j) survives.
template <int MODE, bool SAME>
__device__ __forceinline__ unsigned long long qpass(const QFilter& f, uint2 s, float rj, int j)
{
    const short2v d = __builtin_bit_cast(short2v, s.x) - __builtin_bit_cast(short2v, f.qxy);
    unsigned long long m;
    if (MODE == MODE_RPPI || MODE == MODE_WP) {
        const int r = __builtin_amdgcn_sdot2(d, d, f.qlo, false);
        m = __builtin_amdgcn_ballot_w64((unsigned)r < f.qrange) &
            __builtin_amdgcn_ballot_w64((unsigned)((int)s.y + f.zoff) < f.zspan);
    } else {
        const int dz = (int)s.y - f.qz;
        const int r = __builtin_amdgcn_sdot2(d, d, __mul24(dz, dz) + f.qlo, false);
        m = __builtin_amdgcn_ballot_w64((unsigned)r < f.qrange);
        if (MODE == MODE_RPPI_MOCKS) {
            const float u = fmaf((float)(unsigned)r, f.los_c1, f.los_c0);
            const float t = fabsf(rj - f.los_r) + f.los_t0;
            m &= __builtin_amdgcn_ballot_w64(!(u * fmaxf(rj + f.los_a, 0.0f) > t * t));
        }
    }
    // same cell: the lane's own j > i (lanes without a primary have quantized
    // positions no secondary passes)
    return SAME ? m & __builtin_amdgcn_ballot_w64(j > f.ilim) : m;
}

// Per-lane select by a lane mask: the lane's bit of m set ? a : b (one
// v_cndmask; a C select here tends to become a branch around the computation of a).
__device__ __forceinline__ unsigned lane_select(unsigned long long m, unsigned a, unsigned b)
{
    unsigned r;
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(r) : "v"(b), "v"(a), "s"(m));
    return r;
}

// Appends the lanes of m (nonzero) to the survivor buffer at tail with entry
// (j << 6) | lane. Branch-free: the other lanes write slot tail + 64 + lane, past
// this secondary's survivors, where a later survivor overwrites it or it stays
// beyond the tail.
__device__ __forceinline__ void enqueue(unsigned* qe, unsigned long long m, unsigned& tail, unsigned entry)
{
    const unsigned lane = (unsigned)lane_id();
    const unsigned b =
        (unsigned)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
    unsigned* qt = qe + __builtin_amdgcn_readfirstlane(tail);
    qt[lane_select(m, b, 64u + lane)] = entry;
    tail += (unsigned)__popcll(m);
}

// A block of kBlockJ quantized secondaries in scalar registers.
struct QBlock {
    uint2 s[kBlockJ];
    float r[kBlockJ];  // on-sky (rp, pi)
};
typedef const __attribute__((address_space(4))) float KFloat;
template <int MODE>
__device__ __forceinline__ QBlock qload(KUint* qs, KFloat* rs, int jb)
{
    KUint* p = qs + 2 * (int64_t)jb;
    QBlock b;
#pragma unroll
    for (int t = 0; t < kBlockJ; t++) {
        b.s[t] = make_uint2(p[2 * t], p[2 * t + 1]);
        b.r[t] = MODE == MODE_RPPI_MOCKS ? rs[(int64_t)jb + t] : 0.0f;
    }
    return b;
}

// Filters block b (secondaries jb .. jb + kBlockJ - 1, of which the first
// `nlive` exist) and enqueues the survivors relative to jbase.
template <int MODE, bool SAME, bool PARTIAL>
__device__ __forceinline__ void qblock(const QFilter& f, const QBlock& b, int jb, int nlive, unsigned* qe,
                                       unsigned& tail, int jbase)
{
    unsigned long long m[kBlockJ];
#pragma unroll
    for (int t = 0; t < kBlockJ; t++) {
        m[t] = qpass<MODE, SAME>(f, b.s[t], b.r[t], jb + t);
        if (PARTIAL) m[t] = t < nlive ? m[t] : 0ull;
    }
    const unsigned e0 = ((unsigned)(jb - jbase) << 6) | (unsigned)lane_id();
#pragma unroll
    for (int t = 0; t < kBlockJ; t++)
        if (m[t]) enqueue(qe, m[t], tail, e0 + 64u * t);
}

// Filters the full blocks from jb on and enqueues their survivors, until fewer
// than kBlockJ secondaries are left or 64 survivors are waiting; returns the next
// jb. On entry and exit `a` holds the block at jb: the loop alternates between
// two register blocks so that each block is loaded one block ahead (q is padded
// by kQPad entries, so the look-ahead stays inside the array).
template <int MODE, bool SAME, int DRAIN>
__device__ __forceinline__ int qscan(const QFilter& f, KUint* qs, KFloat* rs, int jb, int jhi, QBlock& a, unsigned* qe,
                                     unsigned head, unsigned& tail, int jbase)
{
    int nfull = (jhi - jb) / kBlockJ;
    for (;;) {
        if (nfull <= 0 || tail - head >= DRAIN) return jb;
        const QBlock b = qload<MODE>(qs, rs, jb + kBlockJ);
        qblock<MODE, SAME, false>(f, a, jb, kBlockJ, qe, tail, jbase);
        jb += kBlockJ;
        if (--nfull <= 0 || tail - head >= DRAIN) {
            a = b;
            return jb;
        }
        a = qload<MODE>(qs, rs, jb + kBlockJ);
        qblock<MODE, SAME, false>(f, b, jb, kBlockJ, qe, tail, jbase);
        jb += kBlockJ;
        --nfull;
    }
}

// Next run of consecutive groups of the mask m (nonzero; cleared from it): the
// secondaries [j, je) of a cell whose group 0 of the mask starts at jbase.
__device__ __forceinline__ void next_run(unsigned long long& m, int jbase, int jend, int& j, int& je)
{
    const int g = __builtin_ctzll(m);
    const unsigned long long rest = ~(m >> g);
    const int run = rest ? __builtin_ctzll(rest) : 64;
    m = g + run < 64 ? m & (~0ull << (g + run)) : 0ull;
    j = jbase + g * kGroup;
    je = min(j + run * kGroup, jend);
}

// The path of 1-D counts (no sums) for groups whose separations from the chunk
// fall into at most kMaxRegBins bins: bins k0 .. k0 + NB - 1, the last without an
// upper edge unless `touch`, which says that its upper edge is rmax. Every (i, j)
// is decided in FP64 in lockstep as on the dense path, but the bin comes from NB
// compares that count in registers until the groups of this bin range are done: no
// lookup (two dependent LDS reads) and no LDS atomic per pair. (With sums it loses:
// the accumulators spill the rest of the kernel's registers, and a root, a masked
// add per bin and sum cost what the lookup and the atomics do.)
constexpr int kMaxRegBins = 4;
template <int MODE, int R2F, int NB>
__device__ __forceinline__ void reg_groups(const PairParams& P, const CellPairRec* cpp, const DevLattice* l1p, int i,
                                           bool ivalid, double xpos, double ypos, double zpos, KDouble* ds,
                                           unsigned long long m, int jbase, int jend, int k0, bool touch,
                                           KernelLds& S)
{
    double e[NB];
    unsigned cnt[NB];  // cumulative: pairs below e[b]
#pragma unroll
    for (int b = 0; b < NB; b++) {
        // (no edge above rmax: the last line of a bin file may end below an earlier one,
        // and the differences of the cumulative counts need edges in order)
        e[b] = b < NB - 1 || touch ? fmin(S.e[min(k0 + b, P.nbin - 1)], P.sqr_rmax) : DBL_MAX;
        if (!ivalid) e[b] = -1.0;  // no pair of a lane without a primary
        cnt[b] = 0;
    }
    auto decide = [&](double xj, double yj, double zj) {
        const double dx = xj - xpos, dy = yj - ypos, dz = zj - zpos;
        double r2 = sep2<R2F>(dx, dy, dz);
        if (touch) {
            // (a lane without a primary has a position, but no record i to replay)
            const bool near = ivalid && r2 >= P.near_lo2 && r2 < P.sqr_rmax;
            if (__builtin_amdgcn_ballot_w64(near)) {
                if (near) {
                    // the reference's pruning tests (see exact_pair)
                    const CellPairRec* c = fresh(cpp);
                    const DevLattice* l1 = fresh(l1p);
                    ITerms t = {};
                    const double4 p = l1->d4[i];
                    i_terms(P, MODE, *c, p.x, p.y, p.z, &t);
                    const bool out = MODE == MODE_WP ? !c->same && (t.skip || zj <= t.target)
                                                     : t.skip || zj <= t.target || dz >= t.max_dz;
                    if (out) r2 = P.sqr_rmax;  // in no bin
                }
            }
        }
#pragma unroll
        for (int b = 0; b < NB; b++) cnt[b] += r2 < e[b] ? 1u : 0u;
    };
    // two records per step, loaded one step ahead (the next run's first two after
    // a run's last), at 32-bit offsets from the batch's first record: the scalar
    // unit, which issues the loads and the loop, would bound a simpler loop
    // (2M points, counts, 14 % per launch; d4 is padded)
    typedef const __attribute__((address_space(4))) char KChar;
    KChar* base = (KChar*)(ds + 4 * (int64_t)jbase);
    auto rec = [&](unsigned o) { return kload_d4((KDouble*)(base + o), 0); };
    int j, je;
    next_run(m, 0, jend - jbase, j, je);
    unsigned o = (unsigned)j * 32u;
    double4 a0 = rec(o), a1 = rec(o + 32u);
    for (;;) {
        const unsigned oe = (unsigned)je * 32u;
        const bool more = m != 0;
        unsigned no = o;
        if (more) {
            next_run(m, 0, jend - jbase, j, je);
            no = (unsigned)j * 32u;
        }
        for (;;) {
            const unsigned on = o + 64u < oe ? o + 64u : no;
            const double4 b0 = rec(on), b1 = rec(on + 32u);
            decide(a0.x, a0.y, a0.z);
            o += 32u;
            if (o < oe) {
                decide(a1.x, a1.y, a1.z);
                o += 32u;
            }
            a0 = b0;
            a1 = b1;
            if (o >= oe) break;
        }
        if (!more) break;
        o = no;
    }
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const unsigned n = cnt[b] - (b > 0 ? cnt[b > 0 ? b - 1 : 0] : 0u);
        if (k0 + b > 0 && n) atomicAdd(&S.np[((k0 + b) << S.rshift) + S.lane_copy], (unsigned long long)n);
    }
}

// One lane's value from its neighbour in the row of 16 lanes (a DPP row rotation).
static_assert(kGroup == 16, "a group of secondaries is held by a row of 16 lanes");
__device__ __forceinline__ double row_next(double v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x121, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x121, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// One work item of the tuned kernel (see the comment above kQueues).
template <int MODE, int R2F, bool GH, int DP, int FL>
__device__ __forceinline__ void process_item(const PairParams& P, const DevLattice* l1p, const DevLattice* l2p,
                                             const CellPairRec& cp, const CellPairRec* cpp, const WorkItem& it,
                                             KernelLds& S, unsigned* qe, double4* prim)
{
    // the lattices and the set-up parameters are loaded per item (fresh), so
    // that they do not occupy registers across the persistent loop
    const __attribute__((address_space(4))) DevLattice& L1 = *fresh_k(l1p);
    const __attribute__((address_space(4))) DevLattice& L2 = *fresh_k(l2p);
    const PairParams& Pi = P;
    const int lane = lane_id();
    const int i0 = __builtin_amdgcn_readfirstlane(it.i0), i1 = __builtin_amdgcn_readfirstlane(it.i1);
    const int flags = __builtin_amdgcn_readfirstlane(it.flags);
    // with P.dense_stride, dense cross-cell items take strided primaries (a
    // whole-cell sample per wave, spreading the lanes' pairs over more
    // histogram slots); else 64 consecutive ones
    const int stride = flags >> kStrideShift;
    const int i = i0 + lane * (stride > 0 ? stride : 1);
    const int ivalid = i < i1;
    const int c2 = cp.c2;
    const int same = cp.same;
    // a lane takes secondary j iff j > ilim (its primary exists; same cell: j > i)
    const int ilim = !ivalid ? INT_MAX : (same ? i : INT_MIN);
    const double3 wrap = make_double3(cp.wx * Pi.xwrap, cp.wy * Pi.ywrap, cp.wz * Pi.zwrap);
    const double4* d4_1 = L1.d4;
    const double4* d4_2 = L2.d4;
    double xpos, ypos, zpos, wi;
    {
        // (a lane without a primary holds the chunk's last one)
        const double4 pi = d4_1[ivalid ? i : i1 - 1];
        xpos = pi.x + wrap.x;
        ypos = pi.y + wrap.y;
        zpos = pi.z + wrap.z;
        wi = pi.w;
    }
    // groups of kGroup secondaries of the cell; same cell: from the chunk's own on
    const int s2 = __builtin_amdgcn_readfirstlane(L2.bstart[c2]), e2 = __builtin_amdgcn_readfirstlane(L2.bstart[c2 + 1]);
    int glo = same ? (i0 - s2) / kGroup : 0, ghi = (e2 - s2 + kGroup - 1) / kGroup;
    {
        const int nparts = __builtin_amdgcn_readfirstlane(it.nparts);
        if (nparts > 1) {
            const int part = __builtin_amdgcn_readfirstlane(it.part);
            const int64_t len = ghi - glo;
            const int a = glo + (int)(len * part / nparts), b = glo + (int)(len * (part + 1) / nparts);
            glo = a;
            ghi = b;
        }
    }
    if (ghi <= glo) return;
    // with at most kFewGroups groups the cell pair's own dense estimate decides
    // (the cell pair list has culled by the cells' boxes)
    const bool few = ghi - glo <= kFewGroups;
    const double* gb2 = L2.gbox + group_index(s2, c2) * 6;
    // sparse path: quantize the wave's primaries relative to the secondary cell
    const int iz2 = c2 % L2.nz, ixy2 = c2 / L2.nz, iy2 = ixy2 % L2.ny, ix2 = ixy2 / L2.ny;
    const double ox = L2.xmin + ix2 * L2.xbs, oy = L2.ymin + iy2 * L2.ybs, oz = L2.zmin + iz2 * L2.zbs;
    // a lane without a primary gets (qx, qy) = (-32768, -32768): every difference
    // to a secondary (0 <= q <= kQMax) wraps to |dq| >= 32768 - kQMax per axis, so
    // its squared distance exceeds any threshold (which is < (kQMax + 2)^2 + 1)
    // without overflowing 32 bits
    uint2 qi = quantize_pos(xpos - ox, ypos - oy, zpos - oz, L2.qinv);
    if (!ivalid) qi = make_uint2(0x80008000u, 0u);
    QFilter f;
    f.qxy = qi.x;
    f.qz = (int)qi.y;
    f.qlo = L2.qlo_neg;
    f.qrange = L2.qrange;
    f.zoff = L2.qz - 1 - f.qz;
    f.zspan = 2u * (unsigned)L2.qz - 1u;
    f.ilim = ilim;
    const int istride = stride > 0 ? stride : 1;
    unsigned head = 0, tail = 0;
    // the wave's primaries (wrapped, FP64) for the drains
    if (P.prim_cache) {
        prim[lane] = make_double4(xpos, ypos, zpos, wi);
        __builtin_amdgcn_wave_barrier();
    }
    KDouble* ds = (KDouble*)(const void*)d4_2;
    KUint* qs = (KUint*)(const void*)L2.q;
    KFloat* rs = nullptr;
    if (MODE == MODE_RPPI_MOCKS) {
        rs = (KFloat*)(const void*)L2.rr;
        f.los_r = (float)(2.0 * (xpos * xpos + ypos * ypos + zpos * zpos));
        f.los_a = f.los_r - L2.los_a0;
        f.los_c1 = L2.los_c1;
        f.los_c0 = L2.los_c0;
        f.los_t0 = L2.los_t0;
    }
    constexpr int kDrain = 64 * DP;
    for (int g0 = glo; g0 < ghi; g0 += 64) {
        // lane l tests group g0 + l against the chunk's box: out of reach,
        // dense (enough of its pairs in range), or sparse
        unsigned long long mdense, msparse, mreg = 0;
        int keyv = 0;  // bin range of the lane's group: k0 | NB << 16 | touch << 20
        constexpr bool regs = (MODE == MODE_DD || MODE == MODE_XI || MODE == MODE_WP) && !GH && FL == kFlLut1;
        if (few) {
            const unsigned long long ml = ~0ull >> (64 - (ghi - glo));
            const bool dns = Pi.dense_mode == 0 ? (flags & kItemDense) != 0 : Pi.dense_mode == 1;
            mdense = dns ? ml : 0ull;
            msparse = dns ? 0ull : ml;
        } else {
            // the chunk's bounding box (wrapped): the union of its groups' boxes, or
            // the cell's for strided primaries (recomputed per 64 groups: kept
            // across the scans it costs 12 registers there)
            double A[6];
            {
                const int c1 = cp.c1;
                const int s1 = __builtin_amdgcn_readfirstlane(L1.bstart[c1]);
                KDouble* ub = (KDouble*)(const void*)(stride > 0 ? L1.bounds + (int64_t)c1 * 6
                                                                 : L1.gbox + (group_index(s1, c1) + (i0 - s1) / kGroup) * 6);
                const int ng = stride > 0 ? 1 : (i1 - i0 + kGroup - 1) / kGroup;
#pragma unroll
                for (int d = 0; d < 6; d++) A[d] = ub[d];
                for (int k = 1; k < ng; k++)
#pragma unroll
                    for (int d = 0; d < 6; d += 2) {
                        A[d] = fmin(A[d], ub[6 * k + d]);
                        A[d + 1] = fmax(A[d + 1], ub[6 * k + d + 1]);
                    }
                A[0] += wrap.x; A[1] += wrap.x;
                A[2] += wrap.y; A[3] += wrap.y;
                A[4] += wrap.z; A[5] += wrap.z;
            }
            const bool have = g0 + lane < ghi;
            const double* bx = gb2 + (int64_t)(have ? g0 + lane : glo) * 6;
            const double x0 = bx[0], x1 = bx[1], y0 = bx[2], y1 = bx[3], z0 = bx[4], z1 = bx[5];
            const double nx = fmax(fmax(x0 - A[1], A[0] - x1), 0.0), ny = fmax(fmax(y0 - A[3], A[2] - y1), 0.0),
                         nz = fmax(fmax(z0 - A[5], A[4] - z1), 0.0);
            const double fx = fmax(x1 - A[0], A[1] - x0), fy = fmax(y1 - A[2], A[3] - y0),
                         fz = fmax(z1 - A[4], A[5] - z0);
            constexpr bool is2d = MODE == MODE_RPPI || MODE == MODE_WP;
            const double near2 = is2d ? nx * nx + ny * ny : nx * nx + ny * ny + nz * nz;
            const double far2 = is2d ? fx * fx + fy * fy : fx * fx + fy * fy + fz * fz;
            // the margins cover the rounding of the pairs' own separations
            bool live = have && near2 <= P.sqr_rmax * (1.0 + 1e-9) && nz <= P.zreach * (1.0 + 1e-9) + P.box_margin;
            if (MODE == MODE_RPPI_MOCKS) {
                // the filter's line-of-sight test (QFilter) on the boxes' ranges of |x|^2, and
                // pi < pimax by (s.l)^2 < pimax^2 |l|^2
                const double x0s = x0 * x0, x1s = x1 * x1, y0s = y0 * y0, y1s = y1 * y1, z0s = z0 * z0, z1s = z1 * z1;
                const double hi2 = fmax(x0s, x1s) + fmax(y0s, y1s) + fmax(z0s, z1s);
                const double lo2 = (x0 * x1 > 0 ? fmin(x0s, x1s) : 0.0) + (y0 * y1 > 0 ? fmin(y0s, y1s) : 0.0) +
                                   (z0 * z1 > 0 ? fmin(z0s, z1s) : 0.0);
                double hi1 = 0, lo1 = 0;
#pragma unroll
                for (int d = 0; d < 6; d += 2) {
                    const double u = A[d] * A[d], v = A[d + 1] * A[d + 1];
                    hi1 += fmax(u, v);
                    lo1 += A[d] * A[d + 1] > 0 ? fmin(u, v) : 0.0;
                }
                const double slack = 1e-9 * (hi1 + hi2);
                const double tmax = fmax(hi2 - lo1, hi1 - lo2) + slack, tmin = fmax(fmax(lo2 - hi1, lo1 - hi2) - slack, 0.0);
                const double lmin = fmax(2.0 * (lo1 + lo2) - P.sqr_rmax - slack, 0.0), lmax = 2.0 * (hi1 + hi2) + slack;
                live = live && !((near2 * (1.0 - 1e-9) - P.sqr_rpmax) * lmin > tmax * tmax) &&
                       !(tmin * tmin > P.sqr_mu_max * lmax);
            }
            double num = P.sqr_rmax - near2, den = far2 - near2;
            bool dns = num >= (double)P.dense_frac * den;
            if (is2d) {
                // times the share of |dz| below pimax
                const double zn = fmax(P.pimax - nz, 0.0), zd = fz - nz;
                dns = fmin(num, den) * fmin(zn, zd) >= (double)P.dense_frac * (den * zd);
            }
            if (Pi.dense_mode != 0) dns = Pi.dense_mode == 1;
            if (stride > 0) dns = true;
            unsigned long long ml = __builtin_amdgcn_ballot_w64(live);
            if constexpr (regs) {
                // the group's bin range, from its nearest and farthest separation with
                // the same margins; not for separations FP32 cannot hold (nor NaN)
                const double lo = near2 * (1.0 - 1e-9), hi = far2 * (1.0 + 1e-9);
                const bool touch = !(hi < P.near_lo2);
                bool ok = live && dns && lo < P.sqr_rmax && far2 < 1e30;
                if (MODE == MODE_WP) ok = ok && fz * (1.0 + 1e-9) < P.near_lodz;
                if (same) ok = ok && s2 + (g0 + lane) * kGroup >= i1;  // every j > every i
                ok = ok && stride == 0 && Pi.dense_mode == 0;
                if (ok) {
                    const int k0 = lo < P.sqr_rmin ? 0 : lut_kbin<FL>(P, S, lo, (float)lo);
                    const int k1 = touch ? P.nbin : (hi < P.sqr_rmin ? 0 : lut_kbin<FL>(P, S, hi, (float)hi));
                    const int nb = k1 - k0 + (touch ? 0 : 1);
                    ok = nb <= kMaxRegBins;
                    keyv = k0 | nb << 16 | (touch ? 1 << 20 : 0);
                }
                mreg = __builtin_amdgcn_ballot_w64(ok);
                ml &= ~mreg;
            }
            mdense = ml & __builtin_amdgcn_ballot_w64(dns);
            msparse = ml & ~mdense;
        }
        if constexpr (regs) {
            while (mreg) {
                const int key = __builtin_amdgcn_readlane(keyv, __builtin_ctzll(mreg));
                const unsigned long long m = mreg & __builtin_amdgcn_ballot_w64(keyv == key);
                mreg &= ~m;
                const int k0 = key & 0xffff, nb = (key >> 16) & 15;
                const bool touch = key >> 20;
                const int jb0 = s2 + g0 * kGroup;
                if (nb == 1)
                    reg_groups<MODE, R2F, 1>(P, cpp, l1p, i, ivalid, xpos, ypos, zpos, ds, m, jb0, e2, k0, touch, S);
                else if (nb == 2)
                    reg_groups<MODE, R2F, 2>(P, cpp, l1p, i, ivalid, xpos, ypos, zpos, ds, m, jb0, e2, k0, touch, S);
                else if (nb == 3)
                    reg_groups<MODE, R2F, 3>(P, cpp, l1p, i, ivalid, xpos, ypos, zpos, ds, m, jb0, e2, k0, touch, S);
                else if (nb == 4)
                    reg_groups<MODE, R2F, 4>(P, cpp, l1p, i, ivalid, xpos, ypos, zpos, ds, m, jb0, e2, k0, touch, S);
            }
        }
        // DDsmu's dense path: every row of 16 lanes holds a group's secondaries and
        // rotates them, so the lanes of a histogram update have 16 different
        // secondaries. With one secondary for all lanes, compact chunks put many lanes
        // into one (s, mu) slot, and the same-address atomics serialize: 31 % of the
        // cycles on clustered data x randoms, 389 -> 314 ms; the rotation's 8 moves
        // cost 4 % where the points are uniform. (DDrppi, whose pi columns already
        // spread a compact chunk: 3 % slower; on-sky modes are bound by the decision's
        // arithmetic.)
        constexpr bool rotate = MODE == MODE_SMU;
        if constexpr (rotate) {
            const int r = lane & (kGroup - 1);
            while (mdense) {
                const int g = __builtin_ctzll(mdense);
                mdense &= mdense - 1;
                const int j0 = s2 + (g0 + g) * kGroup;
                int j = j0 + r;
                double4 cur = d4_2[min(j, e2 - 1)];
                int left = kGroup;
                for (;;) {
                    exact_pair<MODE, R2F, GH, FL>(P, cpp, l1p, i, j > ilim && j < e2, xpos, ypos, zpos, wi, cur.x,
                                                  cur.y, cur.z, fl_w<FL>(P) ? cur.w : 0.0, S);
                    if (--left == 0) break;
                    cur.x = row_next(cur.x);
                    cur.y = row_next(cur.y);
                    cur.z = row_next(cur.z);
                    if (fl_w<FL>(P)) cur.w = row_next(cur.w);
                    // (row_ror 1: lane l takes lane l - 1's)
                    j = j0 + ((j - j0 + kGroup - 1) & (kGroup - 1));
                }
            }
        }
        while (mdense) {
            // a run of consecutive dense groups: FP64 lockstep; the secondary
            // record is a scalar load (d4 is padded, so the look-ahead load of
            // j + 1 stays inside the array)
            int j, je;
            next_run(mdense, s2 + g0 * kGroup, e2, j, je);
            double4 cur = kload_d4(ds, j);
            for (; j < je; j++) {
                const double4 nxt = kload_d4(ds, j + 1);
                exact_pair<MODE, R2F, GH, FL>(P, cpp, l1p, i, j > ilim, xpos, ypos, zpos, wi, cur.x, cur.y, cur.z,
                                              fl_w<FL>(P) ? cur.w : 0.0, S);
                cur = nxt;
            }
        }
        // sparse runs: filter into the queue and drain full rounds; what is left
        // is drained after the batch's last run, so that queue entries can hold
        // j relative to the batch's first secondary
        const int jbase = s2 + g0 * kGroup;
        int jb = 0, jhi = 0;  // the run being scanned
        QBlock a = {};        // its block at jb
        bool last = msparse == 0;
        while (!last) {
            if (jb >= jhi) {
                if (msparse) {
                    next_run(msparse, jbase, e2, jb, jhi);
                    a = qload<MODE>(qs, rs, jb);
                } else {
                    last = true;
                }
            }
            if (!last) {
                if (same)
                    jb = qscan<MODE, true, kDrain>(f, qs, rs, jb, jhi, a, qe, head, tail, jbase);
                else
                    jb = qscan<MODE, false, kDrain>(f, qs, rs, jb, jhi, a, qe, head, tail, jbase);
                if (jb < jhi && jb + kBlockJ > jhi && tail - head < kDrain) {
                    // the last, partial block
                    if (same)
                        qblock<MODE, true, true>(f, a, jb, jhi - jb, qe, tail, jbase);
                    else
                        qblock<MODE, false, true>(f, a, jb, jhi - jb, qe, tail, jbase);
                    jb = jhi;
                }
            }
            while (tail - head >= (last ? 1u : (unsigned)kDrain)) {
                const unsigned nd = min(tail - head, (unsigned)kDrain);
                __builtin_amdgcn_wave_barrier();
                if (DP == 2)
                    drain_queue2<MODE, R2F, GH, FL>(P, cp, cpp, l1p, d4_1, d4_2, wrap, i0, istride, qe, prim, head,
                                                    (int)nd, jbase, S);
                else
                    drain_queue<MODE, R2F, GH, FL>(P, cp, cpp, l1p, d4_1, d4_2, wrap, i0, istride, qe, prim, head,
                                                   (int)nd, jbase, S);
                __builtin_amdgcn_wave_barrier();
                head += nd;
            }
            if (last) head = tail = 0;
            if (head >= kCompactAt) {
                // move the < kDrain waiting entries to the front
                const unsigned n = tail - head;
                unsigned v[DP];
#pragma unroll
                for (int p = 0; p < DP; p++) {
                    v[p] = 0;
                    if ((unsigned)(lane + 64 * p) < n) v[p] = qe[head + lane + 64 * p];
                }
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int p = 0; p < DP; p++)
                    if ((unsigned)(lane + 64 * p) < n) qe[lane + 64 * p] = v[p];
                __builtin_amdgcn_wave_barrier();
                head = 0;
                tail = n;
            }
        }
    }
}

// Adds a (replicated) LDS histogram region to the global histogram at `base`
// and clears it; `t0`/`tstep` split the slots among the calling threads.
__device__ __forceinline__ void flush_region(const PairParams& P, KernelLds& S, int R, int64_t base, int t0,
                                             int tstep, unsigned long long* g_np, double* g_avg, double* g_w)
{
    for (int sl = t0; sl < P.nslots; sl += tstep) {
        unsigned long long c = 0;
        double sa = 0, sw = 0;
        for (int r = 0; r < R; r++) {
            c += S.np[sl * R + r];
            S.np[sl * R + r] = 0;
            if (P.need_avg) { sa += S.avg[sl * R + r]; S.avg[sl * R + r] = 0; }
            if (P.need_w) { sw += S.w[sl * R + r]; S.w[sl * R + r] = 0; }
        }
        if (c) {
            atomicAdd(&g_np[base + sl], c);
            if (P.need_avg) atomicAdd(&g_avg[base + sl], sa);
            if (P.need_w) atomicAdd(&g_w[base + sl], sw);
        }
    }
}

// The tuned pair kernel. lats[0], lats[1]: primary / secondary particle sets;
// in a batch (BATCH = true) every cell pair carries its catalog index k in
// `pad`, both sets are lats[k], each wave keeps its own LDS histogram for the
// catalog it is working on, and the histogram of catalog k lives at
// g_*[k*nslots ...]. GH = true: no LDS histogram; every counted pair is added
// to the global histogram (histograms too large for the workgroup's LDS).
// DP = survivors per lane per drain (1: compiled for six waves per SIMD, <= 80
// VGPRs; 2: for five, <= 96 VGPRs). FL = the launch's flags (fl_avg etc.):
// a mask for the LDS-histogram kernels, kFlRuntime for the GH ones.
template <int MODE, int R2F, bool BATCH, bool GH, int DP, int FL>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(DP == 2 ? 5 : 6))) void k_pairs_tuned(PairParams P, const DevLattice* __restrict__ lats,
                                                     const CellPairRec* __restrict__ cps,
                                                     const WorkItem* __restrict__ items,
                                                     const int* __restrict__ nitems_p, int* __restrict__ counter,
                                                     const double* __restrict__ rupp_sqr,
                                                     const unsigned short* __restrict__ lut_g,
                                                     unsigned long long* __restrict__ g_np,
                                                     double* __restrict__ g_avg, double* __restrict__ g_w,
                                                     unsigned long long* __restrict__ cp_ticks,
                                                     int* __restrict__ cp_cu, const int* __restrict__ single_p)
{
    extern __shared__ unsigned long long smem_u64[];
    KernelLds S;
    const int R = GH ? 1 : P.hist_copies;
    const int nwaves = blockDim.x >> 6;
    const int nrep = GH ? 0 : P.nslots * R;         // one histogram region
    const int nreg = BATCH ? nrep * nwaves : nrep;  // all regions of the workgroup
    const int wave = threadIdx.x >> 6, lane = lane_id();
    unsigned long long* np0 = smem_u64;
    double* avg0 = reinterpret_cast<double*>(smem_u64 + nreg);
    double* w0 = avg0 + (P.need_avg ? nreg : 0);
    double* e = w0 + (P.need_w ? nreg : 0);
    const int roff = BATCH ? wave * nrep : 0;
    S.np = np0 + roff;
    S.avg = avg0 + roff;
    S.w = w0 + roff;
    S.rshift = __builtin_ctz(R);
    S.lane_copy = lane & (R - 1);
    S.gnp = g_np;
    S.gavg = g_avg;
    S.gw = g_w;
    unsigned short* lut = reinterpret_cast<unsigned short*>(e + P.nbin);
    int* qbase = reinterpret_cast<int*>(lut + ((P.lut_n + 1) & ~1));
    S.e = e;
    S.lut = lut;
    unsigned* qe = reinterpret_cast<unsigned*>(qbase) + __builtin_amdgcn_readfirstlane(wave) * kQueueAlloc;
    // primaries cache: 16-byte aligned after the queues
    // (offsets from the LDS base, so the pointer stays an LDS pointer)
    const size_t poff = ((size_t)(reinterpret_cast<char*>(qbase + nwaves * kQueueAlloc) -
                                  reinterpret_cast<char*>(smem_u64)) + 15) & ~(size_t)15;
    double4* prim = reinterpret_cast<double4*>(reinterpret_cast<char*>(smem_u64) + poff) + wave * 64;
    for (int s = threadIdx.x; s < P.nbin; s += blockDim.x) e[s] = rupp_sqr[s];
    for (int s = threadIdx.x; s < P.lut_n; s += blockDim.x) lut[s] = lut_g[s];
    for (int s = threadIdx.x; s < nreg; s += blockDim.x) {
        np0[s] = 0;
        if (P.need_avg) avg0[s] = 0;
        if (P.need_w) w0[s] = 0;
    }
    __syncthreads();
    const int nitems = *nitems_p;
    const DevLattice* l1p = lats;
    const DevLattice* l2p = lats + (BATCH ? 0 : 1);
    int cur = -1;  // catalog whose histogram the wave's LDS region holds (BATCH)
    // Work queue: the list is cut into blocks of B = 2^qblock_log2 consecutive
    // items, and block b belongs to sub-queue b % kQueues (the cost order is kept
    // inside every sub-queue): the k-th item of sub-queue q is
    // g = ((k / B) * kQueues + q) * B + k % B. Sub-queue q has its own counter at
    // counter[q * kCounterStride], so the device-wide atomics spread over kQueues
    // addresses. A wave starts at sub-queue blockIdx.x % kQueues -- workgroups are
    // dispatched to the XCDs round-robin, so that is mostly the wave's own XCD --
    // and moves on to the next when that one is exhausted, until all are. Blocks
    // keep the items of a cell pair, which scan the same secondary window, on one
    // XCD and its L2. Items below *single_p (the heavy cell pairs the scheduler
    // puts first) are taken one at a time; the others P.fetch per atomic while
    // more than 2 P.fetch items per wave of the grid remain (as last seen), then
    // one at a time.
    // The loop has no lane-divergent branch around its wave-wide steps: every
    // lane executes the queue atomic (lane 0 adds the batch, the others 0) and
    // the broadcast reads lane 0's result. A divergent `if (lane == 0)` here lets
    // the compiler start the next iteration's broadcast without lane 0
    // (observed in the generated code).
    const int tail_zone = (int)min((long)nitems, (long)gridDim.x * nwaves * P.fetch * 2);
    const int n_single = *single_p;
    const int home = blockIdx.x & (kQueues - 1);
    const int lb = P.qblock_log2, bmask = (1 << lb) - 1;
    const long round = (long)kQueues << lb;  // items of one block per sub-queue
    int qi = 0, q = 0, next = 0, end = 0, last = 0;
    for (;;) {
        if (next >= end) {
            bool got = false;
            while (qi < kQueues) {
                q = (home + qi) & (kQueues - 1);
                const long full = (long)nitems / round;
                const long rem = (long)nitems - full * round - ((long)q << lb);
                const int cnt = (int)((full << lb) + (rem < 0 ? 0 : (rem > bmask ? bmask + 1 : rem)));
                const int want = (last >= n_single && last < nitems - tail_zone) ? P.fetch : 1;
                const int fetched = atomicAdd(&counter[q * kCounterStride], lane == 0 ? want : 0);
                const int k = __builtin_amdgcn_readlane(fetched, 0);
                if (k < cnt) {
                    next = k;
                    end = min(k + want, cnt);
                    got = true;
                    break;
                }
                qi++;
            }
            if (!got) break;
        }
        const int item = (((next >> lb) * kQueues + q) << lb) + (next & bmask);
        next++;
        last = item;
        const WorkItem it = items[item];
        const CellPairRec* cpp = cps + __builtin_amdgcn_readfirstlane(it.cp);
        const CellPairRec cp = *cpp;
        if (BATCH) {
            const int k = __builtin_amdgcn_readfirstlane(cp.pad);
            if (k != cur) {
                if (cur >= 0) {
                    __builtin_amdgcn_wave_barrier();
                    flush_region(P, S, R, (int64_t)cur * P.nslots, lane, 64, g_np, g_avg, g_w);
                    __builtin_amdgcn_wave_barrier();
                }
                cur = k;
                l1p = lats + k;
                l2p = l1p;
            }
        }
        // per-cell-pair cost record: wall-clock ticks of the wave on this item
        // (branch-free in the lanes: lane 0 adds dt, the others 0; every lane
        // stores the same compute-unit id)
        const unsigned long long t0 = cp_ticks ? wall_clock64() : 0ull;
        process_item<MODE, R2F, GH, DP, FL>(P, l1p, l2p, cp, cpp, it, S, qe, prim);
        if (cp_ticks) {
            const unsigned long long dt = wall_clock64() - t0;
            atomicAdd(&cp_ticks[it.cp], lane == 0 ? dt : 0ull);
            cp_cu[it.cp] = (int)__smid();
        }
    }
    if (GH) return;
    if (BATCH) {
        if (cur >= 0) {
            __builtin_amdgcn_wave_barrier();
            flush_region(P, S, R, (int64_t)cur * P.nslots, lane, 64, g_np, g_avg, g_w);
        }
        return;
    }
    __syncthreads();
    flush_region(P, S, R, 0, threadIdx.x, blockDim.x, g_np, g_avg, g_w);
}

#define CF_TUNED_INST0(M, F, B, G, D, FL)                                                                      \
    template __global__ void k_pairs_tuned<M, F, B, G, D, FL>(PairParams, const DevLattice*, const CellPairRec*, \
                                                              const WorkItem*, const int*, int*, const double*,  \
                                                              const unsigned short*, unsigned long long*,         \
                                                              double*, double*, unsigned long long*, int*,        \
                                                              const int*);
// LDS-histogram kernels: one per flag mask; global-histogram kernels: runtime flags
#define CF_TUNED_INST_FL(M, F, B, D)                                                                           \
    CF_TUNED_INST0(M, F, B, false, D, 0) CF_TUNED_INST0(M, F, B, false, D, 1)                                   \
    CF_TUNED_INST0(M, F, B, false, D, 2) CF_TUNED_INST0(M, F, B, false, D, 3)                                   \
    CF_TUNED_INST0(M, F, B, false, D, 4) CF_TUNED_INST0(M, F, B, false, D, 5)                                   \
    CF_TUNED_INST0(M, F, B, false, D, 6) CF_TUNED_INST0(M, F, B, false, D, 7)
#define CF_TUNED_INST(M, F, B) CF_TUNED_INST_FL(M, F, B, 1) CF_TUNED_INST_FL(M, F, B, 2)
#define CF_TUNED_INST2(M, F)                                                                                   \
    CF_TUNED_INST(M, F, false) CF_TUNED_INST0(M, F, false, true, 1, kFlRuntime)                                 \
    CF_TUNED_INST0(M, F, false, true, 2, kFlRuntime)
CF_TUNED_INST2(MODE_DD, R2_SUM_XY_Z)
CF_TUNED_INST2(MODE_DD, R2_FMA_DZ_DY_DX)
CF_TUNED_INST2(MODE_XI, R2_SUM_XY_Z)
CF_TUNED_INST2(MODE_XI, R2_X_SUM_YZ)
CF_TUNED_INST2(MODE_XI, R2_FMA_DZ_DY_DX)
CF_TUNED_INST2(MODE_RPPI, RP_SUM)
CF_TUNED_INST2(MODE_RPPI, RP_FMA)
CF_TUNED_INST2(MODE_WP, RP_SUM)
CF_TUNED_INST2(MODE_WP, RP_FMA)
CF_TUNED_INST2(MODE_SMU, R2_SUM_XY_Z)
CF_TUNED_INST2(MODE_SMU, R2_FMA_DX_DY_DZ)
CF_TUNED_INST2(MODE_RPPI_MOCKS, R2_SUM_XY_Z)
CF_TUNED_INST2(MODE_SMU_MOCKS, R2_SUM_XY_Z)
CF_TUNED_INST(MODE_DD, R2_SUM_XY_Z, true)
CF_TUNED_INST(MODE_DD, R2_FMA_DZ_DY_DX, true)
#undef CF_TUNED_INST2
#undef CF_TUNED_INST
#undef CF_TUNED_INST_FL
#undef CF_TUNED_INST0

// Light cell pairs (at most `light` tests each): one lane per cell pair, which
// tests its few pairs in FP64 one after the other; the work list of the persistent
// kernel leaves them out. On sparse grids (a few particles per cell) an item of that
// kernel is one cell pair: a queue atomic and a chain of dependent loads, some
// microseconds a wave, for a handful of tests. Wave w takes the chunks w, w + W, ...
// of `chunk` consecutive cell pairs (a multiple of 64); batched, each wave keeps the
// histogram of the catalog it is working on.
template <int MODE, int R2F, bool BATCH>
__global__ __launch_bounds__(256) void k_pairs_light(PairParams P, const DevLattice* __restrict__ lats,
                                                     const CellPairRec* __restrict__ cps, int ncp, int light,
                                                     int chunk, const double* __restrict__ rupp_sqr,
                                                     const unsigned short* __restrict__ lut_g,
                                                     unsigned long long* __restrict__ g_np,
                                                     double* __restrict__ g_avg, double* __restrict__ g_w)
{
    extern __shared__ unsigned long long smem_u64[];
    KernelLds S;
    const int R = P.hist_copies, nwaves = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = lane_id();
    const int nrep = P.nslots * R, nreg = BATCH ? nrep * nwaves : nrep;
    double* avg0 = reinterpret_cast<double*>(smem_u64 + nreg);
    double* w0 = avg0 + (P.need_avg ? nreg : 0);
    double* e = w0 + (P.need_w ? nreg : 0);
    unsigned short* lut = reinterpret_cast<unsigned short*>(e + P.nbin);
    const int roff = BATCH ? wave * nrep : 0;
    S.np = smem_u64 + roff;
    S.avg = avg0 + roff;
    S.w = w0 + roff;
    S.rshift = __builtin_ctz(R);
    S.lane_copy = lane & (R - 1);
    S.e = e;
    S.lut = lut;
    for (int s = threadIdx.x; s < P.nbin; s += blockDim.x) e[s] = rupp_sqr[s];
    for (int s = threadIdx.x; s < P.lut_n; s += blockDim.x) lut[s] = lut_g[s];
    for (int s = threadIdx.x; s < nreg; s += blockDim.x) {
        smem_u64[s] = 0;
        if (P.need_avg) avg0[s] = 0;
        if (P.need_w) w0[s] = 0;
    }
    __syncthreads();
    int cur = -1;
    const int64_t step = (int64_t)gridDim.x * nwaves * chunk;
    for (int64_t c0 = ((int64_t)blockIdx.x * nwaves + wave) * chunk; c0 < ncp; c0 += step) {
        const int64_t c1 = min(c0 + chunk, (int64_t)ncp);
        for (int64_t t0 = c0; t0 < c1; t0 += 64) {
            const int64_t t = t0 + lane;
            const CellPairRec* cpp = cps + (t < c1 ? t : c0);
            const CellPairRec cp = *cpp;
            const int cat = BATCH ? cp.pad : 0;
            const DevLattice* l1p = lats + cat;
            const DevLattice* l2p = lats + (BATCH ? cat : 1);
            int s1 = 0, e1 = 0, s2 = 0, e2 = 0;
            if (t < c1) {
                s1 = l1p->bstart[cp.c1];
                e1 = l1p->bstart[cp.c1 + 1];
                s2 = l2p->bstart[cp.c2];
                e2 = l2p->bstart[cp.c2 + 1];
            }
            if ((int64_t)(e1 - s1) * (e2 - s2) > light) e1 = s1;
            const double wx = cp.wx * P.xwrap, wy = cp.wy * P.ywrap, wz = cp.wz * P.zwrap;
            const double4 *d1 = l1p->d4, *d2 = l2p->d4;
            unsigned long long todo = __ballot(e1 > s1);
            while (todo) {
                // the lanes of one catalog at a time
                int k = 0;
                unsigned long long mine = todo;
                if (BATCH) {
                    k = __builtin_amdgcn_readlane(cat, __builtin_ctzll(todo));
                    mine = todo & __ballot(cat == k);
                    if (k != cur) {
                        if (cur >= 0) {
                            __builtin_amdgcn_wave_barrier();
                            flush_region(P, S, R, (int64_t)cur * P.nslots, lane, 64, g_np, g_avg, g_w);
                            __builtin_amdgcn_wave_barrier();
                        }
                        cur = k;
                    }
                }
                todo &= ~mine;
                if ((mine >> lane) & 1ull) {
                    int i = s1, j = cp.same ? s1 + 1 : s2;
                    double4 pi = d1[i];
                    pi.x += wx;
                    pi.y += wy;
                    pi.z += wz;
                    while (i < e1) {
                        if (j < e2) {
                            const double4 pj = d2[j];
                            exact_pair<MODE, R2F, false, kFlRuntime, false>(P, cpp, l1p, i, 1, pi.x, pi.y, pi.z, pi.w,
                                                                            pj.x, pj.y, pj.z, pj.w, S);
                            j++;
                        }
                        if (j >= e2) {
                            i++;
                            j = cp.same ? i + 1 : s2;
                            if (i < e1) {
                                pi = d1[i];
                                pi.x += wx;
                                pi.y += wy;
                                pi.z += wz;
                            }
                        }
                    }
                }
            }
        }
    }
    if (BATCH) {
        if (cur >= 0) {
            __builtin_amdgcn_wave_barrier();
            flush_region(P, S, R, (int64_t)cur * P.nslots, lane, 64, g_np, g_avg, g_w);
        }
        return;
    }
    __syncthreads();
    flush_region(P, S, R, 0, threadIdx.x, blockDim.x, g_np, g_avg, g_w);
}

// Largest squared separation between the bounding boxes of a cell pair
// (primary box shifted by the wrap), per the geometry of the mode, and whether
// the pair takes the dense path: every pair of its particles is inside the range,
// or the estimated in-range fraction -- the share of the squared-separation span
// [min_sep^2, max_sep^2] below rmax^2 (times the |dz| share below pimax in the
// projected modes) -- reaches P.dense_frac.
__device__ __forceinline__ int cp_dense(const PairParams& P, const CellPairRec& cp, const double* b1,
                                        const double* b2, double* maxsep2)
{
    const double ox = cp.wx * P.xwrap, oy = cp.wy * P.ywrap, oz = cp.wz * P.zwrap;
    const double mx = fmax(fabs(b2[1] - (b1[0] + ox)), fabs((b1[1] + ox) - b2[0]));
    const double my = fmax(fabs(b2[3] - (b1[2] + oy)), fabs((b1[3] + oy) - b2[2]));
    const double mz = fmax(fabs(b2[5] - (b1[4] + oz)), fabs((b1[5] + oz) - b2[4]));
    const bool is2d = P.mode == MODE_RPPI || P.mode == MODE_WP;
    const double hi = is2d ? mx * mx + my * my : mx * mx + my * my + mz * mz;
    *maxsep2 = hi;
    if (is2d ? (hi < 0.98 * P.sqr_rmax && mz < 0.98 * P.pimax) : hi < 0.98 * P.sqr_rmax) return 1;
    const double lo = cp.mdx * cp.mdx + cp.mdy * cp.mdy + (is2d ? 0.0 : cp.mdz * cp.mdz);
    double f = hi > lo ? (P.sqr_rmax - lo) / (hi - lo) : 0.0;
    f = fmin(1.0, fmax(0.0, f));
    if (is2d) f *= mz > cp.mdz ? fmin(1.0, fmax(0.0, (P.pimax - cp.mdz) / (mz - cp.mdz))) : 1.0;
    return f >= (double)P.dense_frac;
}

// A predicted log2 cost clamped to [0, kCostTop] (NaN -> 0), so that any model
// output gives a valid bucket and a finite total.
__device__ __forceinline__ float sane_cost(float c)
{
    return c >= 0.f ? (c <= kCostTop ? c : kCostTop) : 0.f;
}

// Work-item construction: chunks of 64 primary particles per cell pair, each
// split into `parts` slices of its secondary window. Position t of the list
// holds cell pair order[t] (order == nullptr: t). With a cost array (log2
// units), a chunk whose predicted cost exceeds total / cap_div is split into
// ceil(cost / cap) parts (at most kMaxParts).
// ncp_dev (optional): a device count that bounds ncp; entries of the count
// array past it are 0 (a graph-captured batch scans its whole capacity).
__global__ void k_count_chunks(int ncp, const int* __restrict__ order, const CellPairRec* __restrict__ cps,
                               const DevLattice* __restrict__ lats, int batch, const float* __restrict__ cost,
                               const double* __restrict__ total, double cap_div, int* __restrict__ nparts,
                               int* __restrict__ nitems, const int* __restrict__ ncp_dev = nullptr, int light = 0)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ncp) return;
    if (ncp_dev && t >= *ncp_dev) {
        nitems[t] = 0;
        return;
    }
    const int c = order ? order[t] : t;
    const int* bs1 = lats[batch ? cps[c].pad : 0].bstart;
    const int n = (int)cell_count(bs1, cps[c].c1);
    const int nch = (n + 63) / 64;
    if (light > 0) {
        // k_pairs_light's share
        const int n2 = (int)cell_count(lats[batch ? cps[c].pad : 1].bstart, cps[c].c2);
        if ((int64_t)n * n2 <= light) {
            nitems[t] = 0;
            return;
        }
    }
    int parts = 1;
    if (cost && nch > 0) {
        const double cap = *total / cap_div;
        const double per_chunk = exp2((double)sane_cost(cost[c])) / nch;
        if (cap > 0 && per_chunk > cap) parts = (int)fmin((double)kMaxParts, ceil(per_chunk / cap));
    }
    if (nparts) nparts[t] = parts;
    nitems[t] = nch * parts;
}

// Items are written only below items_cap (a graph-captured batch's capacity).
__global__ void k_emit_chunks(int ncp, const int* __restrict__ order, const CellPairRec* __restrict__ cps,
                              const DevLattice* __restrict__ lats, int batch, PairParams P,
                              const int* __restrict__ off, const int* __restrict__ nparts,
                              WorkItem* __restrict__ items, const int* __restrict__ ncp_dev = nullptr,
                              int items_cap = INT_MAX, int light = 0)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ncp || (ncp_dev && t >= *ncp_dev)) return;
    if (light > 0 && off[t + 1] == off[t]) return;
    const int c = order ? order[t] : t;
    const CellPairRec cp = cps[c];
    const int* bs1 = lats[batch ? cp.pad : 0].bstart;
    const double* bd1 = lats[batch ? cp.pad : 0].bounds;
    const double* bd2 = lats[batch ? cp.pad : 1].bounds;
    double maxsep2;
    const int dense = cp_dense(P, cp, bd1 + (int64_t)cp.c1 * 6, bd2 + (int64_t)cp.c2 * 6, &maxsep2);
    const int s = bs1[cp.c1], e = bs1[cp.c1 + 1];
    const int parts = nparts ? nparts[t] : 1;
    int o = off[t];
    const int nch = (e - s + 63) / 64;
    for (int ch = 0; ch < nch; ch++) {
        WorkItem w;
        w.cp = c;
        if (dense && P.dense_stride && !cp.same) {
            w.i0 = s + ch;
            w.i1 = e;
            w.flags = kItemDense | (nch << kStrideShift);
        } else {
            w.i0 = s + 64 * ch;
            w.i1 = w.i0 + 64 < e ? w.i0 + 64 : e;
            w.flags = dense ? kItemDense : 0;
        }
        w.nparts = parts;
        for (int p = 0; p < parts; p++) {
            w.part = p;
            if (o < items_cap) items[o] = w;
            o++;
        }
    }
}

// dst[0] = src[0] (a device-side gather of a count computed by a scan).
__global__ void k_copy_int(const int* __restrict__ src, int* __restrict__ dst)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *dst = *src;
}

// *single = item index where the light cell pairs start: the work-list offset
// of ordered position *nheavy.
__global__ void k_single_boundary(const int* __restrict__ nheavy, const int* __restrict__ off,
                                  int* __restrict__ single)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *single = off[*nheavy];
}

}  // namespace cfamd
