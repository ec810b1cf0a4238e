// Counting and distribution as a two-pass Morton bucket sort of the cloud.
//
// The cloud arrives in arbitrary spatial order, so counting it straight into the level-0 grid and
// scattering every point to its leaf costs one random global atomic and a handful of random
// partial-line stores per point. Here the points are sorted by the Morton code of their level-0
// cell instead (child slot order: x bit 4, y bit 2, z bit 1, as point_count_propagation.cuh:62-70),
// in two passes that only use LDS atomics per point:
//   kBucketHist     per-workgroup LDS histogram of coarse buckets (level-lc cells) -> bucket sizes
//   kBucketScatter  each workgroup ranks its chunk of points per bucket in LDS, reserves one
//                   range per bucket with a single global atomic, stages the chunk in bucket order
//                   in LDS and writes sorted-point records (coordinates, point index, colour) plus
//                   the 3*lc-bit fine code as contiguous runs
//   kFineSort       one workgroup per bucket: LDS histogram over the bucket's (2^lc)^3 level-0
//                   cells, exclusive scan, dense counts of levels 0..lc of the count pyramid,
//                   then the permutation into full Morton order (4-byte indices)
// In Morton order every octree node is one contiguous range, so after the merge a leaf's points
// are the range [sortedStart, sortedStart + count). The records move once more, then: gathered
// through the permutation and ordered within every leaf by its parent's subsampling cells
// (kLeafCellOrder, with the subsampling kernels), or in plain Morton order (kGatherSorted) when
// the root is the only leaf. The distribution is a coalesced copy of the leaf ranges of that
// sorted cloud into the leaf data blocks (kDistributeSorted).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "device_common.h"
#include "kernels_chunking.h"
#include "scan.h"
#include "types.h"

namespace oc {

constexpr uint32_t MAX_COARSE_LEVEL = 5;                               // (2^5)^3 level-0 cells per bucket
constexpr uint32_t MAX_FINE_CELLS   = 1u << (3 * MAX_COARSE_LEVEL);    // 32768
constexpr uint32_t SMALL_FINE_CELLS = 1u << (3 * (MAX_COARSE_LEVEL - 1));

// Bucket level of a single cloud's sort. A 256^3 grid has 16^3 buckets, as a 512^3 one: with 8^3 it had
// fewer occupied ones than compute units, each with a histogram eight times as large (1.5M points:
// kFineSort 73 -> 46 us, kLeafCellOrder 41 -> 36, kBucketScatter 41 -> 47). Smaller grids keep 8^3, whose
// cells are few (64^3 grid, 50K points: kFineSort 9.2 us, 12.3 with 16^3).
constexpr uint32_t coarseLevel(uint32_t depth)
{
    const uint32_t above = depth >= 8 ? 4 : 3;
    const uint32_t level = depth > above ? depth - above : 0;
    return level < MAX_COARSE_LEVEL ? level : MAX_COARSE_LEVEL;
}
constexpr uint32_t MAX_BUCKETS      = 4096;                            // (512 >> 5)^3
constexpr int SORT_THREADS          = 1024;
constexpr int SORT_WAVES            = SORT_THREADS / 64;
constexpr int SCATTER_THREADS       = 1024;
constexpr int STAGE_ITEMS           = 4;
constexpr uint32_t STAGE_CHUNK      = SCATTER_THREADS * STAGE_ITEMS;   // points per scatter workgroup
constexpr int HIST_THREADS          = 512;
constexpr uint32_t COMPUTE_UNITS    = 256;
constexpr uint32_t XCD_COUNT        = 8;  // workgroup b runs on XCD b mod 8, each XCD with its own L2

// The item of a work list of `count` entries that this workgroup takes when XCD x is to take the
// x-th eighth of the list, front to back (~0u: none). Neighbouring items then share one L2 instead
// of being spread over eight. The grid must hold at least count rounded up to a multiple of 8.
__device__ __forceinline__ uint32_t xcdItem(uint32_t count)
{
    const uint32_t per = (count + XCD_COUNT - 1) / XCD_COUNT;
    const uint32_t at  = blockIdx.x / XCD_COUNT;
    if (at >= per)
        return ~0u;
    const uint32_t item = (blockIdx.x % XCD_COUNT) * per + at;
    return item < count ? item : ~0u;
}

// A point of the sorted cloud: the original coordinates, its index in the input cloud and its
// colour (r | g << 8 | b << 16).
template <typename T>
struct alignas(sizeof(T) == 8 ? 16 : 4) SortedPoint
{
    T x, y, z;
    uint32_t idx;
    uint32_t rgb;
};
static_assert(sizeof(SortedPoint<double>) == 32, "double sorted point is 32 bytes");
static_assert(sizeof(SortedPoint<float>) == 20, "float sorted point is 20 bytes");
static_assert(STAGE_CHUNK <= 65535, "staged slots are 16-bit");

// Exclusive scan over a 1024-thread workgroup; `total` receives the sum. Contains barriers.
__device__ __forceinline__ uint32_t sortBlockExclusiveScan(uint32_t v, uint32_t& total, uint32_t* lds)
{
    const uint32_t inc = waveInclusiveScan(v);
    const int w        = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 63)
        lds[w] = inc;
    __syncthreads();
    uint32_t off = 0, sum = 0;
#pragma unroll
    for (int i = 0; i < SORT_WAVES; ++i)
    {
        const uint32_t s = lds[i];
        off += (i < w) ? s : 0u;
        sum += s;
    }
    __syncthreads();
    total = sum;
    return inc - v + off;
}

// Exclusive scan over a workgroup of THREADS threads (a multiple of 64); `total` receives the sum.
// Contains barriers.
template <int THREADS>
__device__ __forceinline__ uint32_t sortBlockExclusiveScanN(uint32_t v, uint32_t& total, uint32_t* lds)
{
    const uint32_t inc = waveInclusiveScan(v);
    const int w        = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 63)
        lds[w] = inc;
    __syncthreads();
    uint32_t off = 0, sum = 0;
#pragma unroll
    for (int i = 0; i < THREADS / 64; ++i)
    {
        const uint32_t s = lds[i];
        off += (i < w) ? s : 0u;
        sum += s;
    }
    __syncthreads();
    total = sum;
    return inc - v + off;
}

// Level-0 Morton code of a point, or ~0u when it lies outside the grid.
__device__ __forceinline__ uint32_t pointMorton(double x, double y, double z, const Gridding& g)
{
    uint32_t ix, iy, iz;
    gridCoords(x, y, z, g, ix, iy, iz);
    if (ix >= g.gridSize || iy >= g.gridSize || iz >= g.gridSize)
        return ~0u;
    return morton3(ix, iy, iz);
}

template <typename T>
static __global__ __launch_bounds__(HIST_THREADS) void kBucketHist(const uint8_t* __restrict__ cloud, uint32_t n,
                                                             uint32_t stride, Gridding g, uint32_t fineBits,
                                                             uint32_t buckets, uint32_t* __restrict__ bucketCount,
                                                             uint32_t* __restrict__ err)
{
    __shared__ uint32_t h[MAX_BUCKETS];
    for (uint32_t b = threadIdx.x; b < buckets; b += HIST_THREADS)
        h[b] = 0;
    __syncthreads();
    bool outside = false;
    auto take    = [&](double x, double y, double z) {
        const uint32_t m = pointMorton(x, y, z, g);
        if (m == ~0u)
            outside = true;
        else
            atomicAdd(h + (m >> fineBits), 1u);
    };
    __shared__ RecordStage stages[HIST_THREADS / 64];
    forRecords<T, HIST_THREADS>(cloud, n, stride, stages, take);
    if (outside)
        atomicOr(err, ERR_OUTSIDE);
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < buckets; b += HIST_THREADS)
        if (h[b])
            atomicAdd(bucketCount + b, h[b]);
}

// bucket sizes -> bucket starts (exclusive) and the scatter cursors
struct BucketStartOut
{
    uint32_t* start;
    uint32_t* cursor;
    __device__ void operator()(uint64_t i, uint32_t prefix, uint32_t) const
    {
        start[i]  = prefix;
        cursor[i] = prefix;
    }
};

// Buckets above FINE_SPLIT points are sorted by several workgroups (kFineChunkHist,
// kFineSplitScan, kFineChunkPerm): one workgroup's time grows with its bucket, and a dense
// cluster puts more than a million points in one bucket while the median holds a quarter of that.
constexpr uint32_t FINE_SPLIT = 196608;

__device__ __forceinline__ uint32_t splitChunksOf(uint32_t points)
{
    return points > FINE_SPLIT ? (points + FINE_SPLIT - 1) / FINE_SPLIT : 0u;
}

// The bucket tables in one scan: per bucket its points (low 32 bits), whether it holds any (bits
// 32-47) and its chunks in the split path (bits 48-63; at most 2 n / FINE_SPLIT + 1 in all).
struct BucketIn
{
    const uint32_t* count;
    __device__ uint64_t operator()(uint64_t b) const
    {
        const uint32_t c = count[b];
        return (static_cast<uint64_t>(splitChunksOf(c)) << 48) | (c ? 1ull << 32 : 0ull) | c;
    }
};

// starts, scatter cursors, the list of the buckets that hold points, and the split chunks (entry:
// bucket << 32 | part)
struct BucketTablesOut
{
    uint32_t* start;  // buckets + 1
    uint32_t* cursor;
    uint32_t* occupied;
    uint64_t* chunks;
    uint32_t buckets;
    __device__ void operator()(uint64_t b, uint64_t prefix, uint64_t v) const
    {
        const uint32_t first = static_cast<uint32_t>(prefix), points = static_cast<uint32_t>(v);
        start[b]  = first;
        cursor[b] = first;
        if (b + 1 == buckets)
            start[buckets] = first + points;
        if (points)
            occupied[(prefix >> 32) & 0xFFFF] = static_cast<uint32_t>(b);
        for (uint32_t k = 0; k < (v >> 48); ++k)
            chunks[(prefix >> 48) + k] = (b << 32) | k;
    }
};

// Each workgroup takes a chunk of ITEMS consecutive points per thread, ranks them per bucket in LDS,
// reserves one range per occupied bucket with a single global atomic, stages the records in LDS
// in bucket order and writes them out so that consecutive lanes write consecutive records of one
// bucket.
// LDS of one bucket-scatter workgroup
template <typename T, int ITEMS = STAGE_ITEMS>
struct ScatterLds
{
    SortedPoint<T> stage[SCATTER_THREADS * ITEMS];
    uint32_t delta[MAX_BUCKETS];           // counts, then global start - local start
    uint16_t localStart[MAX_BUCKETS];      // first staged slot of every bucket
    uint32_t scratch[SCATTER_THREADS / 64];
};

// One chunk (all threads of the workgroup; ends with the LDS free again).
template <typename T, int ITEMS = STAGE_ITEMS>
__device__ __forceinline__ void bucketScatterChunk(uint32_t chunk, const uint8_t* __restrict__ cloud, uint32_t n,
                                                   uint32_t stride, const Gridding& g, uint32_t fineBits,
                                                   uint32_t* __restrict__ cursor, SortedPoint<T>* __restrict__ dst,
                                                   uint16_t* __restrict__ fineCode, ScatterLds<T, ITEMS>& lds)
{
    SortedPoint<T>* stage = lds.stage;
    uint32_t* delta       = lds.delta;
    uint16_t* localStart  = lds.localStart;
    uint32_t* scratch     = lds.scratch;
    for (uint32_t b = threadIdx.x; b < MAX_BUCKETS; b += SCATTER_THREADS)
        delta[b] = 0;
    __syncthreads();

    const uint64_t base = static_cast<uint64_t>(chunk) * (SCATTER_THREADS * ITEMS);
    uint32_t code[ITEMS], rank[ITEMS];
    SortedPoint<T> p[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
    {
        const uint64_t i = base + static_cast<uint64_t>(j) * SCATTER_THREADS + threadIdx.x;
        code[j]          = ~0u;
        rank[j]          = 0;
        if (i < n)
        {
            const uint8_t* rec = cloud + i * stride;
            __builtin_memcpy(&p[j].x, rec, 3 * sizeof(T));
            const uint8_t* col = rec + 3 * sizeof(T);
            p[j].idx           = static_cast<uint32_t>(i);
            p[j].rgb = static_cast<uint32_t>(col[0]) | (static_cast<uint32_t>(col[1]) << 8) |
                       (static_cast<uint32_t>(col[2]) << 16);
            code[j] = pointMorton(static_cast<double>(p[j].x), static_cast<double>(p[j].y),
                                  static_cast<double>(p[j].z), g);
            if (code[j] != ~0u)
                rank[j] = atomicAdd(delta + (code[j] >> fineBits), 1u);
        }
    }
    __syncthreads();

    // exclusive scan of the bucket counts (MAX_BUCKETS / SCATTER_THREADS consecutive per thread),
    // one global reservation per occupied bucket
    constexpr int PER = MAX_BUCKETS / SCATTER_THREADS;
    uint32_t cnt[PER], sum = 0;
#pragma unroll
    for (int k = 0; k < PER; ++k)
    {
        cnt[k] = delta[PER * threadIdx.x + k];
        sum += cnt[k];
    }
    uint32_t total;
    uint32_t off = sortBlockExclusiveScanN<SCATTER_THREADS>(sum, total, scratch);
#pragma unroll
    for (int k = 0; k < PER; ++k)
    {
        const uint32_t b = PER * threadIdx.x + k;
        localStart[b]    = static_cast<uint16_t>(off);
        if (cnt[k])
            delta[b] = atomicAdd(cursor + b, cnt[k]) - off;
        off += cnt[k];
    }
    __syncthreads();
    // records into LDS in bucket order
    const uint32_t fineMask = (1u << fineBits) - 1u;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
        if (code[j] != ~0u)
            stage[localStart[code[j] >> fineBits] + rank[j]] = p[j];
    __syncthreads();

    // a staged record's bucket is recomputed from its coordinates (a few FP64 operations) rather
    // than searched for among the buckets' first slots (a dozen dependent LDS reads). The records of a
    // wave go out word by word, consecutive lanes storing consecutive words: a record stored by its own
    // lane, and a fine code from the unsorted points, were a request of the L2 each (chunks of 4 float points
    // per thread, 25.8M / 5.1M: 660 -> 608 / 134 -> 118 us; 119.7M double points 2.5 ms either way).
    using Word              = std::conditional_t<sizeof(T) == 8, uint4, uint32_t>;
    constexpr uint32_t W    = sizeof(SortedPoint<T>) / sizeof(Word);
    const uint32_t lane     = threadIdx.x & 63;
    for (uint32_t j0 = threadIdx.x - lane; j0 < total; j0 += SCATTER_THREADS)
    {
        const uint32_t j = j0 + lane;
        uint32_t d       = ~0u;
        if (j < total)
        {
            const uint32_t m  = pointMorton(static_cast<double>(stage[j].x), static_cast<double>(stage[j].y),
                                            static_cast<double>(stage[j].z), g);  // in the grid: it was staged
            const uint32_t at = j + delta[m >> fineBits];
            if (at < n)  // always: the histogram and this pass compute the same codes
            {
                d           = at;
                fineCode[d] = static_cast<uint16_t>(m & fineMask);
            }
        }
        const Word* src = reinterpret_cast<const Word*>(stage + j0);
#pragma unroll
        for (uint32_t r = 0; r < W; ++r)
        {
            const uint32_t w  = 64 * r + lane, rec = w / W;
            const uint32_t at = __shfl(d, static_cast<int>(rec), 64);
            if (at != ~0u)
                reinterpret_cast<Word*>(dst)[static_cast<uint64_t>(at) * W + (w - rec * W)] = src[w];
        }
    }
    __syncthreads();
}

// Points per thread of a single cloud's scatter. A workgroup's runs in the buckets are the longer the more
// points it stages, and it takes a global atomic for each: as many as a CU's LDS holds (25.8M float points
// with 2 / 4 / 6 per thread: 965 / 608 / 495 us). Clouds that would leave most CUs without a chunk take
// smaller ones (50K points with 1 / 2 / 4: 8.3 / 9.9 / 13.6 us; 200K with 1 / 2: 17.3 / 15.2 us).
template <typename T>
constexpr int LARGE_STAGE_ITEMS = sizeof(T) == 4 ? 6 : STAGE_ITEMS;
constexpr uint32_t SCATTER_ONE_POINTS = 1u << 17, SCATTER_TWO_POINTS = 1u << 19;

template <typename T, int ITEMS>
static __global__ __launch_bounds__(SCATTER_THREADS) void kBucketScatter(const uint8_t* __restrict__ cloud, uint32_t n,
                                                                uint32_t stride, Gridding g, uint32_t fineBits,
                                                                uint32_t buckets, uint32_t* __restrict__ cursor,
                                                                SortedPoint<T>* __restrict__ dst,
                                                                uint16_t* __restrict__ fineCode)
{
    __shared__ ScatterLds<T, ITEMS> lds;
    bucketScatterChunk<T, ITEMS>(blockIdx.x, cloud, n, stride, g, fineBits, cursor, dst, fineCode, lds);
}

struct FineSortParams
{
    uint32_t lc;                   // coarse level: a bucket is one level-lc cell
    uint32_t bucketGrid;           // buckets per axis (chunking grid >> lc)
    uint32_t levelOffset[MAX_LEVELS];
    uint32_t levelGrid[MAX_LEVELS];
};

// Place of fine cell c in the LDS histogram: the five bits that choose the bank take in the ten above
// them. The counts are read along x, whose bits lie three apart in a Morton code, so unswizzled a
// wave's 64 reads fell in 4 banks on level 0 and in one on the levels above.
__device__ __forceinline__ uint32_t fineSlot(uint32_t c)
{
    return c ^ (((c >> 5) ^ (c >> 10)) & 31u);
}

// Dense counts of bucket b's cells on levels 0..lc (kernelPropagatePointCounts,
// point_count_propagation.cuh:34-86, as differences of the Morton prefix h over the bucket's
// fine cells) and their occupancy bits. Only what is not zero is written: the bitmap is clear, and the
// counts below level lc are read for occupied cells only (storing those levels' zero counts was 77 MB
// per 512^3 build whatever the cloud's size: with a pass for the bits it took 147 + 35 us of a
// 200K-point build). A row of a bucket's level is `side` cells from a multiple of `side`: a word, a
// half-word or a byte of the bitmap is stored whole by one lane, shorter rows (20 a bucket) are ored.
__device__ __forceinline__ void bucketCounts(uint32_t b, const FineSortParams& fp, const uint32_t* h,
                                             uint32_t* __restrict__ count, uint32_t* __restrict__ occ)
{
    const uint32_t bx = compact3(b >> 2), by = compact3(b >> 1), bz = compact3(b);
    for (uint32_t k = 0; k <= fp.lc; ++k)
    {
        const uint32_t side   = 1u << (fp.lc - k);
        const uint32_t n3     = side * side * side;
        const uint64_t gk     = fp.levelGrid[k];
        const uint64_t offset = fp.levelOffset[k];
        for (uint32_t j = threadIdx.x; j < n3; j += SORT_THREADS)
        {
            const uint32_t lx = j & (side - 1), ly = (j >> (fp.lc - k)) & (side - 1), lz = j >> (2 * (fp.lc - k));
            const uint32_t m  = morton3(lx, ly, lz);
            const uint32_t v  = h[fineSlot((m + 1) << (3 * k))] - h[fineSlot(m << (3 * k))];
            const uint64_t gx = static_cast<uint64_t>(bx) * side + lx, gy = static_cast<uint64_t>(by) * side + ly,
                           gz = static_cast<uint64_t>(bz) * side + lz;
            const uint64_t d = offset + gx + gy * gk + gz * gk * gk;
            if (v)
                count[d] = v;
            // the lanes of a row are together here or none of them is (n3 is a multiple of side)
            const uint64_t set = (__ballot(v != 0) >> (threadIdx.x & (64 - side) & 63)) & ((1ull << side) - 1);
            if (lx == 0 && set)
            {
                if (side == 32)
                    occ[d >> 5] = static_cast<uint32_t>(set);
                else if (side == 16)
                    reinterpret_cast<uint16_t*>(occ)[d >> 4] = static_cast<uint16_t>(set);
                else if (side == 8)
                    reinterpret_cast<uint8_t*>(occ)[d >> 3] = static_cast<uint8_t>(set);
                else
                    atomicOr(occ + (d >> 5), static_cast<uint32_t>(set) << (d & 31));
            }
        }
    }
}

// In place: the exclusive prefix of the histogram h of `cells` cells (entries at fineSlot), the total
// in entry `cells`. All threads; cells is a power of two (8^lc). Each thread scans a run of
// R = cells / SORT_THREADS consecutive entries around one workgroup scan of the runs' sums (a
// workgroup scan per SORT_THREADS entries would take 32 of them, 64 barriers, per 32^3-cell
// bucket); fineSlot puts the lanes' k-th entries in different banks.
__device__ __forceinline__ void bucketScan(uint32_t* h, uint32_t cells, uint32_t* scratch)
{
    if (cells <= SORT_THREADS)
    {
        const uint32_t c = threadIdx.x;
        const uint32_t v = c < cells ? h[fineSlot(c)] : 0u;
        uint32_t total;
        const uint32_t ex = sortBlockExclusiveScan(v, total, scratch);
        if (c < cells)
            h[fineSlot(c)] = ex;
        if (threadIdx.x == 0)
            h[fineSlot(cells)] = total;
        __syncthreads();
        return;
    }
    const uint32_t R     = cells / SORT_THREADS;
    const uint32_t first = threadIdx.x * R;
    uint32_t sum         = 0;
    for (uint32_t k = 0; k < R; ++k)
        sum += h[fineSlot(first + k)];
    uint32_t total;
    uint32_t acc = sortBlockExclusiveScan(sum, total, scratch);
    for (uint32_t k = 0; k < R; ++k)
    {
        const uint32_t i = fineSlot(first + k);
        const uint32_t v = h[i];
        h[i]             = acc;
        acc += v;
    }
    if (threadIdx.x == 0)
        h[fineSlot(cells)] = total;
    __syncthreads();
}

// Fine codes per thread and step of the fine-sort loops: all of a step's loads are in flight
// before its LDS atomics (a load -> atomic -> load chain waits out the memory latency per code).
constexpr uint32_t FINE_ITEMS = 8;

// LDS histogram of fineCode[lo, hi) into h (at fineSlot).
__device__ __forceinline__ void fineHistogram(const uint16_t* __restrict__ fineCode, uint32_t lo, uint32_t hi,
                                              uint32_t* h)
{
    uint32_t i = lo + threadIdx.x;
    for (; i + (FINE_ITEMS - 1) * SORT_THREADS < hi; i += FINE_ITEMS * SORT_THREADS)
    {
        uint32_t c[FINE_ITEMS];
#pragma unroll
        for (uint32_t k = 0; k < FINE_ITEMS; ++k)
            c[k] = fineCode[i + k * SORT_THREADS];
#pragma unroll
        for (uint32_t k = 0; k < FINE_ITEMS; ++k)
            atomicAdd(h + fineSlot(c[k]), 1u);
    }
    for (; i < hi; i += SORT_THREADS)
        atomicAdd(h + fineSlot(fineCode[i]), 1u);
}

// perm[base + slot] = i for every i in [lo, hi), slot taken from the running starts at h[fineSlot(code)].
__device__ __forceinline__ void finePermute(const uint16_t* __restrict__ fineCode, uint32_t lo, uint32_t hi,
                                            uint32_t* h, uint32_t base, uint32_t* __restrict__ perm)
{
    uint32_t i = lo + threadIdx.x;
    for (; i + (FINE_ITEMS - 1) * SORT_THREADS < hi; i += FINE_ITEMS * SORT_THREADS)
    {
        uint32_t c[FINE_ITEMS];
#pragma unroll
        for (uint32_t k = 0; k < FINE_ITEMS; ++k)
            c[k] = fineCode[i + k * SORT_THREADS];
        uint32_t slot[FINE_ITEMS];
#pragma unroll
        for (uint32_t k = 0; k < FINE_ITEMS; ++k)
            slot[k] = atomicAdd(h + fineSlot(c[k]), 1u);
#pragma unroll
        for (uint32_t k = 0; k < FINE_ITEMS; ++k)
            perm[base + slot[k]] = i + k * SORT_THREADS;
    }
    for (; i < hi; i += SORT_THREADS)
    {
        const uint32_t slot = atomicAdd(h + fineSlot(fineCode[i]), 1u);
        perm[base + slot]   = i;
    }
}

// One bucket (all threads of the workgroup; h holds MAX_FINE_CELLS + 1 values). Ends with a barrier.
__device__ __forceinline__ void fineSortBucket(uint32_t b, const uint16_t* __restrict__ fineCode,
                                               const uint32_t* __restrict__ bucketStart, const FineSortParams& fp,
                                               uint32_t* __restrict__ count, uint32_t* __restrict__ perm, uint32_t* h,
                                               uint32_t* scratch, uint32_t* __restrict__ occ)
{
    const uint32_t cells = 1u << (3 * fp.lc);
    const uint32_t lo = bucketStart[b], hi = bucketStart[b + 1];
    if (hi - lo > FINE_SPLIT)
        return;  // sorted by the split path
    if (lo == hi)
        return;  // an empty bucket (most of them in a sparse cloud)

    for (uint32_t c = threadIdx.x; c <= cells; c += SORT_THREADS)
        h[c] = 0;
    __syncthreads();
    fineHistogram(fineCode, lo, hi, h);
    __syncthreads();
    bucketScan(h, cells, scratch);
    bucketCounts(b, fp, h, count, occ);
    __syncthreads();

    // the permutation into Morton order: 4-byte scattered stores instead of 32-byte records
    finePermute(fineCode, lo, hi, h, lo, perm);
}

// The occupied buckets (list of `totals` bits 32-47), one or two workgroups per compute unit taking the
// next one from a counter: with the 132 KB of LDS of 32^3 cells one fits, and a grid over all
// buckets spent 16 rounds of launches on the empty ones (512^3 grid: 4096, a few hundred occupied).
template <uint32_t CELLS>
static __global__ __launch_bounds__(SORT_THREADS) void kFineSort(const uint16_t* __restrict__ fineCode,
                                                           const uint32_t* __restrict__ bucketStart,
                                                           const uint32_t* __restrict__ occupied,
                                                           const uint64_t* __restrict__ totals,
                                                           uint32_t* __restrict__ next, FineSortParams fp,
                                                           uint32_t* __restrict__ count, uint32_t* __restrict__ perm,
                                                           uint32_t* __restrict__ occ)
{
    __shared__ uint32_t h[CELLS + 32];  // fineSlot moves an entry by up to 31, the total's too
    __shared__ uint32_t scratch[SORT_WAVES];
    __shared__ uint32_t mine;
    const uint32_t buckets = static_cast<uint32_t>(*totals >> 32) & 0xFFFF;
    for (;;)
    {
        if (threadIdx.x == 0)
            mine = atomicAdd(next, 1u);
        __syncthreads();
        const uint32_t i = mine;
        if (i >= buckets)
            return;
        fineSortBucket(occupied[i], fineCode, bucketStart, fp, count, perm, h, scratch, occ);
        __syncthreads();
    }
}

// chunks of the buckets above FINE_SPLIT points: entry = bucket << 32 | part
struct SplitChunksIn
{
    const uint32_t* bucketStart;
    __device__ uint32_t operator()(uint64_t b) const { return splitChunksOf(bucketStart[b + 1] - bucketStart[b]); }
};

struct SplitChunksOut
{
    uint64_t* list;
    __device__ void operator()(uint64_t b, uint32_t prefix, uint32_t v) const
    {
        for (uint32_t k = 0; k < v; ++k)
            list[prefix + k] = (b << 32) | k;
    }
};

// Split path, 1: the histogram of one chunk over the bucket's fine cells, to chunkHist[chunk].
__device__ __forceinline__ void fineChunkHist(uint32_t chunk, const uint16_t* __restrict__ fineCode,
                                              const uint32_t* __restrict__ bucketStart,
                                              const uint64_t* __restrict__ chunks, uint32_t lc,
                                              uint32_t* __restrict__ chunkHist, uint32_t* h)
{
    const uint32_t cells = 1u << (3 * lc);
    const uint64_t e     = chunks[chunk];
    const uint32_t b = static_cast<uint32_t>(e >> 32), part = static_cast<uint32_t>(e);
    const uint32_t lo = bucketStart[b] + part * FINE_SPLIT;
    const uint32_t hi = min(bucketStart[b + 1], lo + FINE_SPLIT);
    for (uint32_t c = threadIdx.x; c < cells; c += SORT_THREADS)
        h[c] = 0;
    __syncthreads();
    fineHistogram(fineCode, lo, hi, h);
    __syncthreads();
    uint32_t* dst = chunkHist + static_cast<uint64_t>(chunk) * MAX_FINE_CELLS;
    for (uint32_t c = threadIdx.x; c < cells; c += SORT_THREADS)
        dst[c] = h[fineSlot(c)];
}

static __global__ __launch_bounds__(SORT_THREADS) void kFineChunkHist(const uint16_t* __restrict__ fineCode,
                                                                const uint32_t* __restrict__ bucketStart,
                                                                const uint64_t* __restrict__ chunks,
                                                                const uint64_t* __restrict__ totals, uint32_t lc,
                                                                uint32_t* __restrict__ chunkHist)
{
    __shared__ uint32_t h[MAX_FINE_CELLS];
    if (blockIdx.x >= *totals >> 48)
        return;  // the whole workgroup
    fineChunkHist(blockIdx.x, fineCode, bucketStart, chunks, lc, chunkHist, h);
}

// Split path, 2: per split bucket (the workgroup of its part-0 chunk), the bucket's histogram as
// the sum of its chunks', its scan and dense counts. The permutation is then written by
// partitions of the bucket's fine cells, one per chunk: partition k starts at the first cell
// whose points start at or after k * FINE_SPLIT in the bucket, so each writes one contiguous
// range of the permutation (chunks of points would interleave their runs in every cell). The
// first chunk's slot receives the cells' starts; word 0 of chunk k's slot (k >= 1) the first cell
// of partition k.
// (all threads; chunk is the first chunk of its bucket)
__device__ __forceinline__ void fineSplitScan(uint32_t chunk, const uint32_t* __restrict__ bucketStart,
                                              const uint64_t* __restrict__ chunks, const FineSortParams& fp,
                                              uint32_t* __restrict__ count, uint32_t* __restrict__ chunkHist,
                                              uint32_t* h, uint32_t* scratch, uint32_t* __restrict__ occ)
{
    const uint32_t b     = static_cast<uint32_t>(chunks[chunk] >> 32);
    const uint32_t parts = (bucketStart[b + 1] - bucketStart[b] + FINE_SPLIT - 1) / FINE_SPLIT;
    const uint32_t cells = 1u << (3 * fp.lc);
    uint32_t* first      = chunkHist + static_cast<uint64_t>(chunk) * MAX_FINE_CELLS;
    for (uint32_t c = threadIdx.x; c < cells; c += SORT_THREADS)
    {
        uint32_t v = 0;
        for (uint32_t k = 0; k < parts; ++k)
            v += first[static_cast<uint64_t>(k) * MAX_FINE_CELLS + c];
        h[fineSlot(c)] = v;
    }
    __syncthreads();
    bucketScan(h, cells, scratch);  // every chunk histogram has been read
    bucketCounts(b, fp, h, count, occ);
    for (uint32_t c = threadIdx.x; c < cells; c += SORT_THREADS)
        first[c] = h[fineSlot(c)];
    for (uint32_t k = 1 + threadIdx.x; k < parts; k += SORT_THREADS)
    {
        // the first cell c with h[c] >= k * FINE_SPLIT (k * FINE_SPLIT < the total, so c <= cells)
        const uint32_t target = k * FINE_SPLIT;
        uint32_t lo = 0, hi = cells;
        while (lo < hi)
        {
            const uint32_t mid = (lo + hi) >> 1;
            if (h[fineSlot(mid)] < target)
                lo = mid + 1;
            else
                hi = mid;
        }
        first[static_cast<uint64_t>(k) * MAX_FINE_CELLS] = lo;
    }
}

static __global__ __launch_bounds__(SORT_THREADS) void kFineSplitScan(const uint32_t* __restrict__ bucketStart,
                                                                const uint64_t* __restrict__ chunks,
                                                                const uint64_t* __restrict__ totals,
                                                                FineSortParams fp, uint32_t* __restrict__ count,
                                                                uint32_t* __restrict__ chunkHist,
                                                                uint32_t* __restrict__ occ)
{
    __shared__ uint32_t h[MAX_FINE_CELLS + 1];
    __shared__ uint32_t scratch[SORT_WAVES];
    if (blockIdx.x >= *totals >> 48 || static_cast<uint32_t>(chunks[blockIdx.x]) != 0)
        return;  // the whole workgroup: not the first chunk of a bucket
    fineSplitScan(blockIdx.x, bucketStart, chunks, fp, count, chunkHist, h, scratch, occ);
}

// Split path, 3: partition `part` of the bucket's fine cells: every point of the bucket is read,
// those in the partition's cells [cLo, cHi) take their slots from the cells' running starts.
__device__ __forceinline__ void fineChunkPerm(uint32_t chunk, const uint16_t* __restrict__ fineCode,
                                              const uint32_t* __restrict__ bucketStart,
                                              const uint64_t* __restrict__ chunks, uint32_t lc,
                                              const uint32_t* __restrict__ chunkHist, uint32_t* __restrict__ perm,
                                              uint32_t* h)
{
    const uint32_t cells = 1u << (3 * lc);
    const uint64_t e     = chunks[chunk];
    const uint32_t b = static_cast<uint32_t>(e >> 32), part = static_cast<uint32_t>(e);
    const uint32_t base  = bucketStart[b];
    const uint32_t end   = bucketStart[b + 1];
    const uint32_t parts = (end - base + FINE_SPLIT - 1) / FINE_SPLIT;
    const uint32_t* start = chunkHist + static_cast<uint64_t>(chunk - part) * MAX_FINE_CELLS;
    const uint32_t cLo    = part ? chunkHist[static_cast<uint64_t>(chunk) * MAX_FINE_CELLS] : 0u;
    const uint32_t cHi    = part + 1 < parts ? chunkHist[static_cast<uint64_t>(chunk + 1) * MAX_FINE_CELLS] : cells;
    const uint32_t span   = cHi - cLo;
    for (uint32_t c = threadIdx.x; c < span; c += SORT_THREADS)
        h[c] = start[cLo + c];
    __syncthreads();
    uint32_t i = base + threadIdx.x;
    for (; i + (FINE_ITEMS - 1) * SORT_THREADS < end; i += FINE_ITEMS * SORT_THREADS)
    {
        uint32_t c[FINE_ITEMS];
#pragma unroll
        for (uint32_t k = 0; k < FINE_ITEMS; ++k)
            c[k] = static_cast<uint32_t>(fineCode[i + k * SORT_THREADS]) - cLo;  // wraps below the partition
#pragma unroll
        for (uint32_t k = 0; k < FINE_ITEMS; ++k)
            if (c[k] < span)
                perm[base + atomicAdd(h + c[k], 1u)] = i + k * SORT_THREADS;
    }
    for (; i < end; i += SORT_THREADS)
    {
        const uint32_t c = static_cast<uint32_t>(fineCode[i]) - cLo;
        if (c < span)
            perm[base + atomicAdd(h + c, 1u)] = i;
    }
}

static __global__ __launch_bounds__(SORT_THREADS) void kFineChunkPerm(const uint16_t* __restrict__ fineCode,
                                                                const uint32_t* __restrict__ bucketStart,
                                                                const uint64_t* __restrict__ chunks,
                                                                const uint64_t* __restrict__ totals, uint32_t lc,
                                                                const uint32_t* __restrict__ chunkHist,
                                                                uint32_t* __restrict__ perm)
{
    __shared__ uint32_t h[MAX_FINE_CELLS];
    // the partitions of one bucket read the same fine codes: on one XCD, from one L2
    const uint32_t chunk = xcdItem(static_cast<uint32_t>(*totals >> 48));
    if (chunk == ~0u)
        return;  // the whole workgroup
    fineChunkPerm(chunk, fineCode, bucketStart, chunks, lc, chunkHist, perm, h);
}

// The sorted cloud: gathered records, written in order. The permutation only moves a record
// inside its bucket, so the reads of one output range hit one bucket's lines. Workgroup b runs on
// XCD b mod 8, and XCD x gathers the x-th eighth of the output front to back: each bucket's lines
// are fetched into a single L2 and reused by all of its points instead of by up to eight L2s.
constexpr int GATHER_ITEMS      = 4;
constexpr uint32_t GATHER_TILE  = BLOCK * GATHER_ITEMS;

// Workgroups of kGatherSorted for n points (a multiple of XCD_COUNT).
inline unsigned gatherGrid(uint32_t n)
{
    const uint64_t tiles = (static_cast<uint64_t>(n) + GATHER_TILE - 1) / GATHER_TILE;
    const uint64_t perXcd = (tiles + XCD_COUNT - 1) / XCD_COUNT;
    return static_cast<unsigned>((perXcd ? perXcd : 1) * XCD_COUNT);
}

template <typename T>
static __global__ __launch_bounds__(BLOCK) void kGatherSorted(const SortedPoint<T>* __restrict__ bucketed,
                                                        const uint32_t* __restrict__ perm, uint32_t n,
                                                        SortedPoint<T>* __restrict__ sorted, uint64_t* stamp)
{
    stampStart(stamp);
    const uint32_t perXcd = gridDim.x / XCD_COUNT;
    const uint64_t tile   = static_cast<uint64_t>(blockIdx.x % XCD_COUNT) * perXcd + blockIdx.x / XCD_COUNT;
    const uint64_t base   = tile * GATHER_TILE + threadIdx.x;
#pragma unroll
    for (int k = 0; k < GATHER_ITEMS; ++k)
    {
        const uint64_t j = base + static_cast<uint64_t>(k) * BLOCK;
        if (j < n)
            sorted[j] = bucketed[perm[j]];
    }
}

// K5: kernelDistributePoints (point_distributing.cuh:31-76) over the sorted cloud. The leaf of a
// point is the one of its level-0 cell (cellLeaf); its slot is its offset in the leaf's sorted
// range, so consecutive threads write consecutive records of one leaf block.
constexpr int DIST_ITEMS = 4;

template <typename T>
static __global__ __launch_bounds__(BLOCK) void kDistributeSorted(const SortedPoint<T>* __restrict__ sorted, uint32_t n,
                                                            Gridding g, const uint32_t* __restrict__ cellLeaf,
                                                            const uint32_t* __restrict__ sortedStart,
                                                            const uint64_t* __restrict__ dataIdx,
                                                            uint32_t* __restrict__ lut, OutRecord* __restrict__ out,
                                                            double sx, double sy, double sz)
{
    // DIST_ITEMS records per thread and step, each level of the load chain (record, its leaf,
    // the leaf's placement) issued for all of them before the next
    const uint64_t stride = globalStride();
    auto cellOf = [&](const SortedPoint<T>& p, uint32_t& cell) {
        uint32_t ix, iy, iz;
        gridCoords(static_cast<double>(p.x), static_cast<double>(p.y), static_cast<double>(p.z), g, ix, iy, iz);
        cell = ix + iy * g.gridSize + iz * g.gridSize * g.gridSize;
        return ix < g.gridSize && iy < g.gridSize && iz < g.gridSize;  // only in-grid points are sorted
    };
    for (uint64_t s0 = globalThread(); s0 < n; s0 += stride * DIST_ITEMS)
    {
        if (s0 + (DIST_ITEMS - 1) * stride < n)
        {
            SortedPoint<T> p[DIST_ITEMS];
            uint32_t leaf[DIST_ITEMS];
            bool in[DIST_ITEMS];
#pragma unroll
            for (int k = 0; k < DIST_ITEMS; ++k)
                p[k] = sorted[s0 + k * stride];
            // the lookups go to cell 0 for a point outside the grid (none is sorted), so every
            // load is unconditional and only the stores are predicated
#pragma unroll
            for (int k = 0; k < DIST_ITEMS; ++k)
            {
                uint32_t cell;
                in[k]   = cellOf(p[k], cell);
                leaf[k] = cellLeaf[in[k] ? cell : 0u];
            }
            uint64_t pos[DIST_ITEMS];
#pragma unroll
            for (int k = 0; k < DIST_ITEMS; ++k)
                pos[k] = dataIdx[leaf[k]] + (s0 + k * stride - sortedStart[leaf[k]]);
#pragma unroll
            for (int k = 0; k < DIST_ITEMS; ++k)
                if (in[k])
                {
                    lut[pos[k]] = p[k].idx;
                    storeRecord(out + pos[k], quantizePoint(p[k].x, p[k].y, p[k].z, p[k].rgb, g, sx, sy, sz));
                }
            continue;
        }
        for (uint64_t s = s0; s < n; s += stride)
        {
            const SortedPoint<T> p = sorted[s];
            uint32_t cell;
            if (!cellOf(p, cell))
                continue;
            const uint32_t leaf = cellLeaf[cell];
            const uint64_t pos  = dataIdx[leaf] + (s - sortedStart[leaf]);
            lut[pos]            = p.idx;
            storeRecord(out + pos, quantizePoint(p.x, p.y, p.z, p.rgb, g, sx, sy, sz));
        }
    }
}

}  // namespace oc
