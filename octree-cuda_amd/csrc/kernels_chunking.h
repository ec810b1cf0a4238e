// Kernels of the merging phase: count pyramid, canonical sparse ids, node links and flags, leaf
// data blocks and the level-0 cell -> leaf map.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_common.h"
#include "scan.h"
#include "types.h"

namespace oc {

constexpr int BLOCK    = 256;

// scalar slots (u64) in itsScalars
enum ScalarSlot : int
{
    SC_ERROR       = 0,
    SC_M           = 1,
    SC_LEAF_TOTAL  = 2,  // packed (leaf chunks << 32 | leaf points)
    SC_SEG_TOTAL   = 3,  // packed (tiles << 32 | inputs)
    SC_TABLE_TOTAL = 4,
    SC_BUCKETS     = 5,  // totals of the bucket tables (BucketIn)
    SC_NEXT_BUCKET = 6,  // the fine sort's next occupied bucket
    SC_INTERNAL    = 7,  // internal nodes
    SC_LEVEL_START = 8,  // u32[MAX_LEVELS + 1] packed into the following slots
    SC_STAMP       = 14,  // clock at the start of the build, of the merge and of the distribution
    SC_COUNT       = 17
};

constexpr uint32_t ERR_OUTSIDE  = 1u;
constexpr uint32_t ERR_CAPACITY = 2u;
constexpr uint32_t ERR_OVERFLOW = 4u;  // N + I > E (A14)

inline unsigned gridFor(uint64_t n, uint64_t cap = 65536)
{
    uint64_t b = (n + BLOCK - 1) / BLOCK;
    if (b == 0)
        b = 1;
    return static_cast<unsigned>(b < cap ? b : cap);
}


// What a build starts from, cleared in one launch: the scalars, the bucket counts, the occupancy
// bitmap and the counts [first, last) of the bucket level and the levels above.
static __global__ __launch_bounds__(BLOCK) void kBuildInit(uint64_t* __restrict__ sc, uint32_t* __restrict__ bucketCount,
                                                     uint32_t buckets, uint32_t* __restrict__ occ, uint64_t words,
                                                     uint32_t* __restrict__ count, uint64_t first, uint64_t last)
{
    const uint64_t i = globalThread();
    if (i < SC_COUNT)
        sc[i] = i == SC_STAMP ? wall_clock64() : 0;
    for (uint64_t b = i; b < buckets; b += globalStride())
        bucketCount[b] = 0;
    for (uint64_t w = i; w < words; w += globalStride())
        occ[w] = 0;
    for (uint64_t d = first + i; d < last; d += globalStride())
        count[d] = 0;
}

// K2 (counts only): kernelPropagatePointCounts (point_count_propagation.cuh:34-86). Child slot k
// of parent (x, y, z) is (2x + (k>>2 & 1), 2y + (k>>1 & 1), 2z + (k & 1)).
__device__ __forceinline__ void propagateOne(uint32_t idx, uint32_t* __restrict__ count, uint32_t offset,
                                             uint32_t grid, uint32_t childOffset, uint32_t childGrid)
{
    const uint32_t cxy = childGrid * childGrid;
    uint32_t xy        = grid * grid;
    uint32_t z = idx / xy, y = (idx - z * xy) / grid, x = (idx - z * xy) % grid;
    const uint32_t* c = count + childOffset + 2 * z * cxy + 2 * y * childGrid + 2 * x;
    uint32_t sum      = c[0] + c[1] + c[childGrid] + c[childGrid + 1] + c[cxy] + c[cxy + 1] + c[cxy + childGrid] +
                   c[cxy + childGrid + 1];
    count[offset + idx] = sum;
}

struct LevelOffsets
{
    uint32_t offset[MAX_LEVELS];
    uint32_t levels;
};

// The levels above the bucket level, at most 8^3 + 4^3 + 2^3 + 1 cells: one workgroup.
__device__ __forceinline__ void propagateTop(uint32_t* count, const LevelOffsets& lo, uint32_t lc,
                                             uint32_t chunkingGrid)
{
    for (uint32_t l = lc + 1; l < lo.levels; ++l)
    {
        const uint32_t grid = chunkingGrid >> l;
        for (uint32_t i = threadIdx.x; i < grid * grid * grid; i += blockDim.x)
            propagateOne(i, count, lo.offset[l], grid, lo.offset[l - 1], 2 * grid);
        __syncthreads();
    }
}

// Occupancy bitmap (bit d: dense cell d holds points) of the 32 cells of word w, from their counts.
__device__ __forceinline__ uint32_t occupancyWord(const uint32_t* count, uint64_t w, uint64_t dense)
{
    uint32_t bits    = 0;
    const uint64_t d = 32 * w;
    if (d + 32 <= dense)
    {
        const uint4* c = reinterpret_cast<const uint4*>(count + d);
#pragma unroll
        for (int k = 0; k < 8; ++k)
        {
            const uint4 v = c[k];
            bits |= ((v.x ? 1u : 0u) | (v.y ? 2u : 0u) | (v.z ? 4u : 0u) | (v.w ? 8u : 0u)) << (4 * k);
        }
    }
    else
        for (uint32_t k = 0; d + k < dense; ++k)
            bits |= (count[d + k] ? 1u : 0u) << k;
    return bits;
}

// First pass of the id scan over the tiles [first, last) of the bitmap's words: the number of set bits,
// in thread 0. All threads. The fine sort has marked the levels up to the bucket level; the workgroups
// with words of the levels above, the last few of all, first sum up those levels (twice if two
// workgroups share them: the same values) and make the words from the counts.
__device__ __forceinline__ uint32_t occupancyTiles(uint32_t* occ, uint32_t* count, uint64_t dense,
                                                   const LevelOffsets& lo, uint32_t lc, uint32_t chunkingGrid,
                                                   uint64_t first, uint64_t last, uint32_t* lds)
{
    const uint64_t words  = (dense + 31) / 32;
    const uint64_t marked = lo.offset[lc + 1] / 32;  // the level above the buckets is never past the root
    if (first < last && last * SCAN_TILE > marked)
        propagateTop(count, lo, lc, chunkingGrid);
    uint32_t bits = 0;
    for (uint64_t tile = first; tile < last; ++tile)
    {
        const uint64_t base = tile * SCAN_TILE;
        if (base + SCAN_TILE <= marked)
        {
            uint32_t v[SCAN_ITEMS];
            loadTile<uint32_t>([occ](uint64_t w) { return occ[w]; }, base, words, v);
#pragma unroll
            for (int k = 0; k < SCAN_ITEMS; ++k)
                bits += __popc(v[k]);
        }
        else
            for (uint64_t w = base + threadIdx.x; w < base + SCAN_TILE && w < words; w += SCAN_THREADS)
            {
                uint32_t v;
                if (w < marked)
                    v = occ[w];
                else
                    occ[w] = v = occupancyWord(count, w, dense);
                bits += __popc(v);
            }
    }
    return blockSum(bits, lds);
}

static __global__ __launch_bounds__(SCAN_THREADS) void kOccupancy(uint32_t* occ, uint32_t* count, uint64_t dense,
                                                           LevelOffsets lo, uint32_t lc,
                                                           uint32_t chunkingGrid, uint32_t* __restrict__ sums,
                                                           uint64_t* stamp)
{
    __shared__ uint32_t lds[SCAN_WAVES];
    stampStart(stamp);
    uint64_t first, last;
    tileRange(scanTiles((dense + 31) / 32), first, last);
    const uint32_t bits = occupancyTiles(occ, count, dense, lo, lc, chunkingGrid, first, last, lds);
    if (threadIdx.x == 0)
        sums[blockIdx.x] = bits;
}

// Sparse ids (A2): the exclusive rank of an occupied dense cell; its node key and dense count are
// written in the same pass, and the first id of every level (ids ascend with the dense index and a
// level is one dense range).
struct IdTables
{
    const uint32_t* occ;
    const uint32_t* count;
    uint32_t* idBase;
    uint32_t* nodeKey;
    uint32_t* nodeCount;
    uint32_t* levelStart;
    LevelOffsets levels;
};

// The id of an occupied dense cell: the first id of its bitmap word (there for the words of the tiles
// that hold any occupied cell) and the set bits below it. Bitmap and bases are 38 MB at a 512 grid and
// stay in cache; an array of an id per dense cell was 613 MB.
struct IdMap
{
    const uint32_t* occ;
    const uint32_t* idBase;
    // the cell is occupied
    __device__ __forceinline__ uint32_t at(uint32_t d) const
    {
        return idBase[d >> 5] + __popc(occ[d >> 5] & ((1u << (d & 31)) - 1u));
    }
    // -1: it is not
    __device__ __forceinline__ int32_t find(uint32_t d) const
    {
        const uint32_t w = occ[d >> 5];
        return (w >> (d & 31)) & 1u ? static_cast<int32_t>(idBase[d >> 5] + __popc(w & ((1u << (d & 31)) - 1u))) : -1;
    }
};

// Set bits of a tile that are listed in LDS at a time.
constexpr uint32_t ID_LIST  = 8192;
constexpr uint32_t ID_ITEMS = 8;

struct IdLds
{
    uint32_t scan[SCAN_ITEMS * SCAN_WAVES];
    uint16_t list[ID_LIST];
};

// The tiles [first, last) of the bitmap's words from id `carry` on (all threads); returns the next
// id. A tile's set bits are listed in LDS in order and then written one per thread, coalesced: a
// thread walking the bits of its own words wrote every node from one lane, 40 us of a 200K-point
// build and 284 us of a 7.3M-node one, now 15 and 166.
__device__ __forceinline__ uint32_t occupiedIds(const IdTables& t, uint64_t words, uint64_t first, uint64_t last,
                                                uint32_t carry, IdLds& lds)
{
    for (uint64_t tile = first; tile < last; ++tile)
    {
        uint32_t w[SCAN_ITEMS], v[SCAN_ITEMS], pre[SCAN_ITEMS];
        loadTile<uint32_t>([&t](uint64_t i) { return t.occ[i]; }, tile * SCAN_TILE, words, w);
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k)
            v[k] = __popc(w[k]);
        const uint32_t ids  = sparseTileScan(v, pre, lds.scan);
        const uint64_t cell = 32 * tile * SCAN_TILE;  // of the tile's first bit
        for (uint32_t l = 0; l < t.levels.levels; ++l)
        {
            const uint32_t d = t.levels.offset[l];
            if (d < cell || d - cell >= 32 * SCAN_TILE)
                continue;
            const uint32_t item = static_cast<uint32_t>(d - cell) >> 5;
#pragma unroll
            for (int k = 0; k < SCAN_ITEMS; ++k)
                if (item == k * SCAN_THREADS + threadIdx.x)
                    t.levelStart[l] = carry + pre[k] + __popc(w[k] & ((1u << (d & 31)) - 1u));
        }
        if (ids)
#pragma unroll
            for (int k = 0; k < SCAN_ITEMS; ++k)
                if (const uint64_t i = tile * SCAN_TILE + k * SCAN_THREADS + threadIdx.x; i < words)
                    t.idBase[i] = carry + pre[k];
        for (uint32_t base = 0; base < ids; base += ID_LIST)
        {
#pragma unroll
            for (int k = 0; k < SCAN_ITEMS; ++k)
            {
                uint32_t at = pre[k] - base;  // wraps below the listed range
                if (v[k] == 0 || pre[k] >= base + ID_LIST || pre[k] + v[k] <= base)
                    continue;
                for (uint32_t bits = w[k]; bits; bits &= bits - 1u, ++at)
                    if (at < ID_LIST)
                        lds.list[at] = static_cast<uint16_t>(32 * (k * SCAN_THREADS + threadIdx.x) +
                                                             static_cast<uint32_t>(__builtin_ctz(bits)));
            }
            __syncthreads();
            // a terrain's cells fill a few tiles: several counts in flight per thread
            const uint32_t n = ids - base < ID_LIST ? ids - base : ID_LIST;
            for (uint32_t j0 = threadIdx.x; j0 < n; j0 += ID_ITEMS * SCAN_THREADS)
            {
                uint32_t d[ID_ITEMS], c[ID_ITEMS];
#pragma unroll
                for (uint32_t k = 0; k < ID_ITEMS; ++k)
                {
                    const uint32_t j = j0 + k * SCAN_THREADS;
                    d[k]             = static_cast<uint32_t>(cell) + lds.list[j < n ? j : j0];
                    c[k]             = t.count[d[k]];
                }
#pragma unroll
                for (uint32_t k = 0; k < ID_ITEMS; ++k)
                    if (const uint32_t j = j0 + k * SCAN_THREADS; j < n)
                    {
                        const uint32_t id = carry + base + j;
                        t.nodeKey[id]     = d[k];
                        t.nodeCount[id]   = c[k];
                    }
            }
            __syncthreads();
        }
        carry += ids;
    }
    return carry;
}

// second pass of the id scan; *m: the number of nodes
static __global__ __launch_bounds__(SCAN_THREADS) void kOccupiedIds(IdTables t, uint64_t words, const uint32_t* sums,
                                                             uint32_t* __restrict__ m)
{
    __shared__ IdLds lds;
    uint64_t first, last;
    tileRange(scanTiles(words), first, last);
    const uint32_t next = occupiedIds(t, words, first, last, sumBefore(sums, lds.scan), lds);
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0)
        *m = next;
}

struct LevelParams
{
    uint32_t offset[MAX_LEVELS];
    uint32_t grid[MAX_LEVELS];
    uint32_t depth;
    uint32_t threshold;
};

__device__ __forceinline__ uint32_t levelOfKey(uint32_t key, const LevelParams& lp)
{
    uint32_t l = 0;
    for (uint32_t k = 1; k <= lp.depth; ++k)
        if (key >= lp.offset[k])
            l = k;
    return l;
}

// The leaf of a level-0 cell (the first finished ancestor-or-self, point_distributing.cuh:56-60): the
// first node on the way up whose parent is internal, or the root.
__device__ __forceinline__ uint32_t leafOfCell(uint32_t id, uint32_t x, uint32_t y, uint32_t z, const LevelParams& lp,
                                               const uint32_t* __restrict__ nodeCount, const IdMap& ids)
{
    for (uint32_t l = 1; l <= lp.depth; ++l)
    {
        const uint32_t g = lp.grid[l];
        const uint32_t p = ids.at(lp.offset[l] + (x >> l) + (y >> l) * g + (z >> l) * g * g);
        if (nodeCount[p] >= lp.threshold)
            return id;
        id = p;
    }
    return id;
}

// Start of a node's range in the sorted cloud (full Morton order of the level-0 cells): the points of
// all buckets before its own, which are numbered in Morton order, and below the bucket level lc those
// of the lower-slot siblings of the node and of its ancestors inside the bucket.
__device__ __forceinline__ uint32_t sortedStartOf(uint32_t l, uint32_t x, uint32_t y, uint32_t z, uint32_t lc,
                                                  const LevelParams& lp, const uint32_t* __restrict__ bucketStart,
                                                  const IdMap& ids, const uint32_t* __restrict__ nodeCount)
{
    uint32_t start = 0;
    for (; l < lc; ++l)
    {
        const uint32_t g    = lp.grid[l];
        const uint32_t slot = ((x & 1) << 2) | ((y & 1) << 1) | (z & 1);
        for (uint32_t k = 0; k < slot; ++k)
        {
            const uint32_t sx = (x & ~1u) + (k >> 2), sy = (y & ~1u) + ((k >> 1) & 1), sz = (z & ~1u) + (k & 1);
            const int32_t c = ids.find(lp.offset[l] + sx + sy * g + sz * g * g);
            if (c >= 0)
                start += nodeCount[c];
        }
        x >>= 1;
        y >>= 1;
        z >>= 1;
    }
    return start + bucketStart[morton3(x, y, z) << (3 * (l - lc))];
}

// Node links and flags: kernelInitLeafNodes (octree_initialization.cuh:24-52) and the structural
// part of kernelMergeHierarchical (hierarchical_merging.cuh:35-122):
//   internal  = level >= 1 && count >= threshold
//   finished  = parent is internal (the root is always finished, A13)
//   pointCount = internal ? 0 : count
// For a leaf also its range of the sorted cloud, and for a level-0 node its leaf, over its cell's
// count (nothing reads that again), so the distribution needs one lookup per point.
__device__ __forceinline__ void nodeLinksOf(uint32_t id, const LevelParams& lp, const uint32_t* __restrict__ nodeKey,
                                            const uint32_t* __restrict__ nodeCount, const IdMap& ids,
                                            uint32_t* __restrict__ pointCount,
                                            uint64_t* __restrict__ dataIdx, int32_t* __restrict__ parent,
                                            int32_t* __restrict__ children, uint8_t* __restrict__ flags,
                                            uint32_t* __restrict__ subtree, uint32_t lc,
                                            const uint32_t* __restrict__ bucketStart,
                                            uint32_t* __restrict__ sortedStart, uint32_t* __restrict__ cellLeaf)
{
    const uint32_t key = nodeKey[id];
    const uint32_t l   = levelOfKey(key, lp);
    const uint32_t g   = lp.grid[l];
    const uint32_t lin = key - lp.offset[l];
    const uint32_t x = lin % g, y = (lin / g) % g, z = lin / (g * g);
    const uint32_t cnt  = nodeCount[id];
    const bool internal = l >= 1 && cnt >= lp.threshold;

    int32_t p = -1;
    if (l < lp.depth)
    {
        const uint32_t pg = lp.grid[l + 1];  // the parent of an occupied cell is occupied
        p = static_cast<int32_t>(ids.at(lp.offset[l + 1] + (x >> 1) + (y >> 1) * pg + (z >> 1) * pg * pg));
    }
    const bool finished = (p < 0) ? true : (nodeCount[p] >= lp.threshold);

    for (int k = 0; k < 8; ++k)
    {
        int32_t c = -1;
        if (l >= 1)
        {
            const uint32_t cg = lp.grid[l - 1];
            const uint32_t cx = 2 * x + ((k >> 2) & 1), cy = 2 * y + ((k >> 1) & 1), cz = 2 * z + (k & 1);
            c = ids.find(lp.offset[l - 1] + cx + cy * cg + cz * cg * cg);
        }
        children[8 * static_cast<uint64_t>(id) + k] = c;
    }
    pointCount[id] = internal ? 0u : cnt;
    dataIdx[id]    = 0;
    parent[id]     = p;
    flags[id]      = static_cast<uint8_t>((finished ? NODE_FINISHED : 0) | (internal ? NODE_INTERNAL : 0));
    subtree[id]    = 0;
    if (finished && !internal)
        sortedStart[id] = sortedStartOf(l, x, y, z, lc, lp, bucketStart, ids, nodeCount);
    if (l == 0)
        cellLeaf[key] = leafOfCell(id, x, y, z, lp, nodeCount, ids);
}

static __global__ __launch_bounds__(BLOCK) void kNodeLinks(uint32_t m, LevelParams lp, const uint32_t* __restrict__ nodeKey,
                                                     const uint32_t* __restrict__ nodeCount, IdMap ids,
                                                     uint32_t* __restrict__ pointCount, uint64_t* __restrict__ dataIdx,
                                                     int32_t* __restrict__ parent, int32_t* __restrict__ children,
                                                     uint8_t* __restrict__ flags, uint32_t* __restrict__ subtree,
                                                     uint32_t lc, const uint32_t* __restrict__ bucketStart,
                                                     uint32_t* __restrict__ sortedStart, uint32_t* __restrict__ cellLeaf,
                                                     uint64_t* __restrict__ cursor, uint32_t points)
{
    for (uint64_t i = globalThread(); i < m; i += globalStride())
        nodeLinksOf(static_cast<uint32_t>(i), lp, nodeKey, nodeCount, ids, pointCount, dataIdx, parent,
                    children, flags, subtree, lc, bucketStart, sortedStart, cellLeaf);
    if (globalThread() == 0)
        *cursor = points;  // the output cursor before the first subsampling step
}

// Internal nodes (level >= 1 and at least `threshold` points), in id order.
struct InternalNodeIn
{
    const uint32_t* nodeCount;
    const uint32_t* levelStart;
    uint32_t threshold;
    __device__ uint32_t operator()(uint64_t i) const { return nodeCount[levelStart[1] + i] >= threshold ? 1u : 0u; }
};

struct InternalNodeOut
{
    uint32_t* list;
    const uint32_t* levelStart;
    __device__ void operator()(uint64_t i, uint32_t prefix, uint32_t v) const
    {
        if (v)
            list[prefix] = levelStart[1] + static_cast<uint32_t>(i);
    }
};

struct ArrayIn
{
    const uint32_t* v;
    __device__ uint32_t operator()(uint64_t i) const { return v[i]; }
};

struct ExclusiveToArray
{
    uint32_t* dst;
    __device__ void operator()(uint64_t i, uint32_t prefix, uint32_t) const { dst[i] = prefix; }
};

// Leaf data offsets (A4): an internal node's block of leaf children starts at the exclusive scan of
// the block sizes in sparse-id order (= parent level, parent linear index), one item per node;
// children follow in slot order.
struct LeafBlockIn
{
    const uint8_t* flags;
    const int32_t* children;
    const uint32_t* pointCount;
    __device__ uint32_t operator()(uint64_t id) const
    {
        uint32_t block = 0;
        if (flags[id] & NODE_INTERNAL)
            for (int k = 0; k < 8; ++k)
            {
                const int32_t c = children[8 * id + k];
                if (c >= 0 && !(flags[c] & NODE_INTERNAL))
                    block += pointCount[c];
            }
        return block;
    }
};

struct LeafBlockOut
{
    LeafBlockIn in;
    uint64_t* dataIdx;
    __device__ void operator()(uint64_t id, uint32_t prefix, uint32_t v) const
    {
        if (v == 0)
            return;
        uint64_t r = prefix;
        for (int k = 0; k < 8; ++k)
        {
            const int32_t c = in.children[8 * id + k];
            if (c >= 0 && !(in.flags[c] & NODE_INTERNAL))
            {
                dataIdx[c] = r;
                r += in.pointCount[c];
            }
        }
    }
};

}  // namespace oc
