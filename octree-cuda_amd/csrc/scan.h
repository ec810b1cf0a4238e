// Device-wide exclusive prefix sum for the builder (sparse ids, leaf blocks, table slices, slots).
//
// Reduce-then-scan in two launches with no inter-workgroup waiting: (1) each workgroup reduces its
// contiguous range of tiles of SCAN_TILE items, (2) each workgroup adds up the sums of the ranges
// before its own (at most SCAN_GRID values, one or a few per thread, from L2), rescans its tiles in
// order from there and hands (index, exclusive prefix, value) to an output functor. A launch in
// between that scans the sums took 4-10 us per scan, 28 to 116 us per build.
// A tile is held striped: thread t holds items k * SCAN_THREADS + t (k < SCAN_ITEMS), so each load
// and store instruction of a wave covers 64 consecutive items, and a full tile is read with no
// bounds test, all SCAN_ITEMS loads in flight at once. Its scan is SCAN_ITEMS row scans (row k =
// the SCAN_THREADS items k * SCAN_THREADS ..): a wave64 shuffle scan per row, the wave totals of
// all rows through LDS, one barrier. Inputs and outputs are functors so the flags / values are
// generated and consumed in the same pass as the scan (e.g. occupancy flags straight from the
// counting grid); an output functor is called once per item, in no particular order. Scans of at
// most SCAN_DIRECT_TILES tiles take one launch (small builds make many small scans): one workgroup
// per tile, which reduces the tiles before its own by itself.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace oc {

constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS   = 8;
constexpr int SCAN_TILE    = SCAN_THREADS * SCAN_ITEMS;
constexpr int SCAN_WAVES   = SCAN_THREADS / 64;

template <typename T>
__device__ __forceinline__ T waveInclusiveScan(T v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
    {
        T n = __shfl_up(v, o, 64);
        if (lane >= o)
            v += n;
    }
    return v;
}

// Exclusive scan of one value per thread over the workgroup; *total gets the workgroup sum.
template <typename T>
__device__ __forceinline__ T blockExclusiveScan(T v, T& total, T* lds)
{
    T inc        = waveInclusiveScan(v);
    const int w  = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 63)
        lds[w] = inc;
    __syncthreads();
    T off = 0, sum = 0;
#pragma unroll
    for (int i = 0; i < SCAN_WAVES; ++i)
    {
        T s = lds[i];
        off += (i < w) ? s : T(0);
        sum += s;
    }
    __syncthreads();
    total = sum;
    return inc - v + off;
}

// The SCAN_ITEMS items of this thread in the tile starting at tileBase (zero past n).
template <typename T, typename In>
__device__ __forceinline__ void loadTile(In in, uint64_t tileBase, uint64_t n, T (&v)[SCAN_ITEMS])
{
    const uint64_t first = tileBase + threadIdx.x;
    if (tileBase + SCAN_TILE <= n)
    {
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k)
            v[k] = in(first + static_cast<uint64_t>(k) * SCAN_THREADS);
    }
    else
    {
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k)
        {
            const uint64_t i = first + static_cast<uint64_t>(k) * SCAN_THREADS;
            v[k]             = i < n ? in(i) : T(0);
        }
    }
}

// Exclusive prefix within the tile of each item of this thread; returns the tile total.
// lds holds SCAN_ITEMS * SCAN_WAVES values.
template <typename T>
__device__ __forceinline__ T tileExclusiveScan(const T (&v)[SCAN_ITEMS], T (&pre)[SCAN_ITEMS], T* lds)
{
    const int w = threadIdx.x >> 6;
    T inc[SCAN_ITEMS];
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k)
        inc[k] = waveInclusiveScan(v[k]);
    if ((threadIdx.x & 63) == 63)
    {
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k)
            lds[k * SCAN_WAVES + w] = inc[k];
    }
    __syncthreads();
    T carry = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k)
    {
        T row = 0, before = 0;
#pragma unroll
        for (int i = 0; i < SCAN_WAVES; ++i)
        {
            const T s = lds[k * SCAN_WAVES + i];
            before += (i < w) ? s : T(0);
            row += s;
        }
        pre[k] = carry + before + (inc[k] - v[k]);
        carry += row;
    }
    __syncthreads();
    return carry;
}

// The same where tiles of zeros are common (bitmaps): they need no scan.
template <typename T>
__device__ __forceinline__ T sparseTileScan(const T (&v)[SCAN_ITEMS], T (&pre)[SCAN_ITEMS], T* lds)
{
    bool any = false;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k)
    {
        any |= v[k] != 0;
        pre[k] = 0;
    }
    return __syncthreads_or(any) ? tileExclusiveScan(v, pre, lds) : T(0);
}

// out(i, offset + exclusive prefix, value) for each item i of this thread in the tile (items past n
// skipped).
template <typename T, typename Out>
__device__ __forceinline__ void storeTile(Out out, uint64_t tileBase, uint64_t n, const T (&v)[SCAN_ITEMS],
                                          const T (&pre)[SCAN_ITEMS], T offset)
{
    const uint64_t first = tileBase + threadIdx.x;
    if (tileBase + SCAN_TILE <= n)
    {
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k)
            out(first + static_cast<uint64_t>(k) * SCAN_THREADS, offset + pre[k], v[k]);
        return;
    }
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k)
    {
        const uint64_t i = first + static_cast<uint64_t>(k) * SCAN_THREADS;
        if (i < n)
            out(i, offset + pre[k], v[k]);
    }
}

// Workgroup b of a grid of G takes the contiguous tiles [b * per, (b + 1) * per), per = ceil(tiles / G).
__device__ __forceinline__ void tileRange(uint64_t tiles, uint64_t& first, uint64_t& last)
{
    const uint64_t per = (tiles + gridDim.x - 1) / gridDim.x;
    first              = blockIdx.x * per;
    last               = first + per < tiles ? first + per : tiles;
}

// The number of items: known to the host, or on the device as the difference of two words.
struct HostCount
{
    uint64_t n;
    __device__ uint64_t operator()() const { return n; }
};

struct DeviceCount
{
    const uint32_t* end;
    const uint32_t* begin;
    __device__ uint64_t operator()() const { return *end - *begin; }
};

__host__ __device__ inline uint64_t scanTiles(uint64_t n)
{
    return (n + SCAN_TILE - 1) / SCAN_TILE;
}

template <typename T, typename In, typename Size>
static __global__ __launch_bounds__(SCAN_THREADS) void kScanReduce(In in, Size size, T* blockSums)
{
    __shared__ T lds[SCAN_WAVES];
    const uint64_t n = size();
    uint64_t first, last;
    tileRange(scanTiles(n), first, last);
    T s = 0;
    for (uint64_t tile = first; tile < last; ++tile)
    {
        T v[SCAN_ITEMS];
        loadTile<T>(in, tile * SCAN_TILE, n, v);
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k)
            s += v[k];
    }
    T total;
    (void)blockExclusiveScan(s, total, lds);
    if (threadIdx.x == 0)
        blockSums[blockIdx.x] = total;
}

// Sum of v over the workgroup, in every thread. Contains barriers.
template <typename T>
__device__ __forceinline__ T blockSum(T v, T* lds)
{
    T total;
    (void)blockExclusiveScan(v, total, lds);
    return total;
}

// Sum of the range sums before this workgroup's range.
template <typename T>
__device__ __forceinline__ T sumBefore(const T* blockSums, T* lds)
{
    T before = 0;
    for (uint32_t b = threadIdx.x; b < blockIdx.x; b += SCAN_THREADS)
        before += blockSums[b];
    return blockSum(before, lds);
}

template <typename T, typename In, typename Out, typename Size>
static __global__ __launch_bounds__(SCAN_THREADS) void kScanDown(In in, Out out, Size size, const T* blockSums, T* total)
{
    __shared__ T lds[SCAN_ITEMS * SCAN_WAVES];
    const uint64_t n = size();
    uint64_t first, last;
    tileRange(scanTiles(n), first, last);
    T carry = sumBefore(blockSums, lds);
    for (uint64_t tile = first; tile < last; ++tile)
    {
        T v[SCAN_ITEMS], pre[SCAN_ITEMS];
        loadTile<T>(in, tile * SCAN_TILE, n, v);
        const T chunk = sparseTileScan(v, pre, lds);
        storeTile<T>(out, tile * SCAN_TILE, n, v, pre, carry);
        carry += chunk;
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0 && total)
        *total = carry;
}

// One launch, workgroup b for tile b: the sum of the tiles before it (two tiles' loads in flight),
// then its own tile. The input is read while other workgroups write their outputs, so an output
// must not write what the input reads.
template <typename T, typename In, typename Out>
static __global__ __launch_bounds__(SCAN_THREADS) void kScanDirect(In in, Out out, uint64_t n, T* total)
{
    __shared__ T lds[SCAN_ITEMS * SCAN_WAVES];
    const uint64_t own = static_cast<uint64_t>(blockIdx.x) * SCAN_TILE;
    T v[SCAN_ITEMS], pre[SCAN_ITEMS];
    loadTile<T>(in, own, n, v);
    T before = 0;
    constexpr uint64_t STEP = 2 * SCAN_ITEMS * SCAN_THREADS;
    uint64_t i              = threadIdx.x;
    for (; i - threadIdx.x + STEP <= own; i += STEP)
    {
        T w[2 * SCAN_ITEMS];
#pragma unroll
        for (int k = 0; k < 2 * SCAN_ITEMS; ++k)
            w[k] = in(i + static_cast<uint64_t>(k) * SCAN_THREADS);
#pragma unroll
        for (int k = 0; k < 2 * SCAN_ITEMS; ++k)
            before += w[k];
    }
    if (i < own)  // an odd tile: own is a whole number of tiles
    {
        T w[SCAN_ITEMS];
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k)
            w[k] = in(i + static_cast<uint64_t>(k) * SCAN_THREADS);
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k)
            before += w[k];
    }
    const T carry = blockSum(before, lds);
    const T chunk = tileExclusiveScan(v, pre, lds);
    storeTile<T>(out, own, n, v, pre, carry);
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0 && total)
        *total = carry + chunk;
}

// Small inputs: one workgroup walks the tiles in order with a running carry. All SCAN_THREADS
// threads of the workgroup call it with the same lds (SCAN_ITEMS * SCAN_WAVES values); the outputs
// are visible to the workgroup after a barrier.
template <typename T, typename In, typename Out>
__device__ __forceinline__ void blockScanAll(In in, Out out, uint64_t n, T* total, T* lds)
{
    T carry = 0;
    for (uint64_t tileBase = 0; tileBase < n; tileBase += SCAN_TILE)
    {
        T v[SCAN_ITEMS], pre[SCAN_ITEMS];
        loadTile<T>(in, tileBase, n, v);
        const T chunk = tileExclusiveScan(v, pre, lds);
        storeTile<T>(out, tileBase, n, v, pre, carry);
        carry += chunk;
    }
    if (threadIdx.x == 0 && total)
        *total = carry;
}

// Inputs up to this many tiles are scanned by kScanDirect: its last workgroup reads
// all of them, SCAN_DIRECT_TILES / 2 dependent rounds of loads (16 tiles: ~6 us; one workgroup
// walking them took ~25 us, two launches take ~9 us).
constexpr uint64_t SCAN_DIRECT_TILES = 16;
// Workgroups of a two-launch scan: eight of 256 threads fill each of 256 compute units.
constexpr uint64_t SCAN_GRID = 2048;

// Exclusive scan of in(0..n-1); out(i, prefix, value) for each i; *total (device) = sum. out must not write
// what in reads. tileScratch must hold min(scanTiles(n), SCAN_GRID) values.
template <typename T, typename In, typename Out>
void scanExclusive(uint64_t n, In in, Out out, T* tileScratch, T* total, hipStream_t stream)
{
    const uint64_t tiles = scanTiles(n);
    if (tiles <= SCAN_DIRECT_TILES)
    {
        kScanDirect<T, In, Out><<<static_cast<unsigned>(tiles ? tiles : 1), SCAN_THREADS, 0, stream>>>(in, out, n,
                                                                                                       total);
        return;
    }
    const unsigned grid = static_cast<unsigned>(tiles < SCAN_GRID ? tiles : SCAN_GRID);
    kScanReduce<T><<<grid, SCAN_THREADS, 0, stream>>>(in, HostCount{n}, tileScratch);
    kScanDown<T><<<grid, SCAN_THREADS, 0, stream>>>(in, out, HostCount{n}, tileScratch, total);
}

// The same over a number of items that only the device knows, n(); bound: the most it can be.
// tileScratch must hold min(scanTiles(bound), SCAN_GRID) values.
template <typename T, typename Size, typename In, typename Out>
void scanExclusive(Size n, uint64_t bound, In in, Out out, T* tileScratch, T* total, hipStream_t stream)
{
    const uint64_t tiles = scanTiles(bound);
    const unsigned grid  = static_cast<unsigned>(tiles < SCAN_GRID ? (tiles ? tiles : 1) : SCAN_GRID);
    kScanReduce<T><<<grid, SCAN_THREADS, 0, stream>>>(in, n, tileScratch);
    kScanDown<T><<<grid, SCAN_THREADS, 0, stream>>>(in, out, n, tileScratch, total);
}

}  // namespace oc
