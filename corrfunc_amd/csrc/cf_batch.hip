// cf_batch.hip -- gridding and cell pairs of all catalogs of a batch at once.
//
// A batch of many small catalogs is bound by kernel launches when every catalog
// takes its own (96 catalogs of 2,000-20,000 points: 2,757 launches, 11.6 ms a
// call with 1 ms of pair counting). Here the catalogs' particles, cells and
// candidate cell pairs lie in concatenated arrays, and every step is one launch
// over all of them: a block belongs to one catalog, which it finds by bisection
// in a table (BatchSet, first block of each catalog); the scans run over the
// concatenations, so that cell starts and cell-pair positions come out global.
#include "cf_device.h"

namespace cfamd {

// One catalog: its input, grid, and first element in the concatenations.
struct BatchSet {
    const void *X, *Y, *Z, *W;
    int64_t n;
    int64_t p0, c0, t0;      // first particle, cell, candidate cell pair
    int64_t ncells, ncand;   // cells, candidates (ncells * nngb)
    int mb0, pb0, cb0, tb0;  // first block of the extent, particle, cell and candidate kernels
    int nngb;
    GridArgs g;
    NgbArgs a;
};
constexpr int kExtentItems = 4096;  // particles per block of the extent and weight kernels
constexpr int kEmitItems = 4096;    // candidates per block of the cell-pair kernels

// The catalog whose blocks (first one: member F) contain block b; s[ncat].*F is
// the number of blocks, and a catalog may have none.
template <int BatchSet::*F>
__device__ __forceinline__ int batch_find(const BatchSet* __restrict__ s, int ncat, int b)
{
    int lo = 0, hi = ncat - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (s[mid].*F <= b) lo = mid; else hi = mid - 1;
    }
    return lo;
}

template <typename T>
__global__ __launch_bounds__(256) void kb_minmax(const BatchSet* __restrict__ sets, int ncat,
                                                 double* __restrict__ partial)
{
    const int k = batch_find<&BatchSet::mb0>(sets, ncat, blockIdx.x);
    const BatchSet& s = sets[k];
    const int64_t i0 = (int64_t)(blockIdx.x - s.mb0) * kExtentItems;
    minmax_block(i0 + threadIdx.x, min(i0 + kExtentItems, s.n), (int64_t)blockDim.x, (const T*)s.X, (const T*)s.Y,
                 (const T*)s.Z, partial + (int64_t)blockIdx.x * 6);
}

// One wave per catalog.
__global__ void kb_minmax_final(const BatchSet* __restrict__ sets, const double* __restrict__ partial,
                                double* __restrict__ out)
{
    const int k = blockIdx.x;
    const int b0 = sets[k].mb0, b1 = sets[k + 1].mb0;
    minmax_reduce(b1 - b0, partial + (int64_t)b0 * 6, out + 6 * (int64_t)k);
}

template <typename T>
__global__ void kb_bucket_count(const BatchSet* __restrict__ sets, int ncat, int* __restrict__ bucket,
                                int* __restrict__ rank, int* __restrict__ counts,
                                unsigned long long* __restrict__ oob)
{
    const BatchSet& s = sets[batch_find<&BatchSet::pb0>(sets, ncat, blockIdx.x)];
    const int64_t i = (int64_t)(blockIdx.x - s.pb0) * blockDim.x + threadIdx.x;
    if (i < s.n)
        bucket_count_one(i, (const T*)s.X, (const T*)s.Y, (const T*)s.Z, s.g, bucket + s.p0, rank + s.p0,
                         counts + s.c0, oob);
}

__global__ void kb_index_scatter(const BatchSet* __restrict__ sets, int ncat, const int* __restrict__ bucket,
                                 const int* __restrict__ rank, const int* __restrict__ bstart, int* __restrict__ idx)
{
    const BatchSet& s = sets[batch_find<&BatchSet::pb0>(sets, ncat, blockIdx.x)];
    const int64_t i = (int64_t)(blockIdx.x - s.pb0) * blockDim.x + threadIdx.x;
    if (i >= s.n) return;
    const int b = bucket[s.p0 + i];
    if (b >= 0) idx[bstart[s.c0 + b] + rank[s.p0 + i]] = (int)i;
}

// As k_build_small / k_build_big; bstart, d4, ... are the concatenations, and
// the list of big cells holds global cell numbers.
template <typename T>
__global__ __launch_bounds__(256) void kb_build_small(const BatchSet* __restrict__ sets, int ncat, const int* bstart,
                                                      const int* idx, int* keys, double4* d4, uint2* q,
                                                      double* bounds, double* gbox, int* big)
{
    __shared__ int hist[4][kSmallBins];
    const BatchSet& s = sets[batch_find<&BatchSet::cb0>(sets, ncat, blockIdx.x)];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t c = (int64_t)(blockIdx.x - s.cb0) * 4 + wave;
    if (c >= s.ncells) return;  // uniform per wave
    const int* bs = bstart + s.c0;
    if (bs[c + 1] - bs[c] > kSmallCell) {
        if (lane == 0) big[1 + atomicAdd(big, 1)] = (int)(s.c0 + c);
        return;
    }
    build_cell<T, 64, kSmallBins>(c, lane, (const T*)s.X, (const T*)s.Y, (const T*)s.Z, (const T*)s.W, s.g, bs, idx,
                                  keys, d4, q, bounds + 6 * s.c0, gbox + 6 * s.c0, nullptr,
                                  hist[wave], nullptr);
}
template <typename T>
__global__ __launch_bounds__(kBigThreads) void kb_build_big(const BatchSet* __restrict__ sets, int ncat,
                                                            const int* bstart, const int* idx, int* keys, double4* d4,
                                                            uint2* q, double* bounds, double* gbox, const int* big)
{
    __shared__ int hist[kBigBins];
    __shared__ double red[6 * kBigThreads / 64];
    const int nbig = big[0];
    for (int t = blockIdx.x; t < nbig; t += gridDim.x) {
        const int gc = big[1 + t];
        int lo = 0, hi = ncat - 1;  // the last catalog with c0 <= gc (catalogs have cells)
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (sets[mid].c0 <= gc) lo = mid; else hi = mid - 1;
        }
        const BatchSet& s = sets[lo];
        build_cell<T, kBigThreads, kBigBins>(gc - s.c0, threadIdx.x, (const T*)s.X, (const T*)s.Y, (const T*)s.Z,
                                             (const T*)s.W, s.g, bstart + s.c0, idx, keys, d4, q, bounds + 6 * s.c0,
                                             gbox + 6 * s.c0, nullptr, hist, red);
        __syncthreads();
    }
}

// The pairs tested of a catalog are added to tested[catalog].
__global__ __launch_bounds__(256) void kb_cellpair_flag(const BatchSet* __restrict__ sets, int ncat,
                                                        const int* __restrict__ bstart,
                                                        const double* __restrict__ bounds, int* __restrict__ flags,
                                                        double* __restrict__ tested)
{
    const int k = batch_find<&BatchSet::tb0>(sets, ncat, blockIdx.x);
    const BatchSet& s = sets[k];
    const int* bs = bstart + s.c0;
    const double* bd = bounds + 6 * s.c0;
    const int64_t t0 = (int64_t)(blockIdx.x - s.tb0) * kEmitItems, t1 = min(t0 + kEmitItems, s.ncand);
    double my = 0;
    for (int64_t t = t0 + threadIdx.x; t < t1; t += blockDim.x) {
        CellPairRec r = {};
        const int f = neighbour_added(s.a, t / s.nngb, (int)(t % s.nngb), bs, bs, bd, bd, &r);
        flags[s.t0 + t] = f;
        if (f) my += pair_tests(r, bs, bs);
    }
    add_tests(my, &tested[k]);
}

// The flagged candidates' records at their scan positions.
__global__ __launch_bounds__(256) void kb_cellpair_emit(const BatchSet* __restrict__ sets, int ncat,
                                                        const int* __restrict__ bstart,
                                                        const double* __restrict__ bounds,
                                                        const int* __restrict__ flags, const int* __restrict__ pos,
                                                        CellPairRec* __restrict__ out)
{
    const int k = batch_find<&BatchSet::tb0>(sets, ncat, blockIdx.x);
    const BatchSet& s = sets[k];
    const int* bs = bstart + s.c0;
    const double* bd = bounds + 6 * s.c0;
    const int64_t t0 = (int64_t)(blockIdx.x - s.tb0) * kEmitItems, t1 = min(t0 + kEmitItems, s.ncand);
    for (int64_t t = t0 + threadIdx.x; t < t1; t += blockDim.x) {
        CellPairRec r = {};
        if (flags[s.t0 + t] && eval_neighbour(s.a, t / s.nngb, (int)(t % s.nngb), bs, bs, bd, bd, &r)) {
            r.pad = k;
            out[pos[s.t0 + t]] = r;
        }
    }
}

// Sums of weights and squared weights of catalog k at out[2 k] (blocks as kb_minmax).
__global__ __launch_bounds__(256) void kb_weight_sums(const BatchSet* __restrict__ sets, int ncat,
                                                      const double4* __restrict__ d4, double* __restrict__ out)
{
    const int k = batch_find<&BatchSet::mb0>(sets, ncat, blockIdx.x);
    const BatchSet& s = sets[k];
    const int64_t i0 = (int64_t)(blockIdx.x - s.mb0) * kExtentItems;
    weight_sums_block(i0 + threadIdx.x, min(i0 + kExtentItems, s.n), (int64_t)blockDim.x, d4 + s.p0, out + 2 * k);
}

}  // namespace cfamd
