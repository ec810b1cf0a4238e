// Kernels of the level-batched subsampling and the final DFS post-order placement.
//
// All internal nodes of one octree level are processed together (in memory-bounded batches of
// nodes). Each node of a batch owns an occupancy bitmap over its g^3 subsampling grid and the
// exclusive popcount prefix of that bitmap's words, i.e. a rank dictionary: the occupied cells of
// the batch get dense indices in (node, cell index) order; the cell index groups the grid's x-rows
// into 4 x 4 pencils or is a Morton code (CellOrder). Per batch:
//   kMark        input point -> cell (the reference's mapPointToGrid with the node's gridding),
//                set the cell's bit
//   prefix scan  popcounts of all bitmap words -> dense index of every occupied cell
//   kAccumulate  winner per cell (atomicMin of rank<<32 | input position), packed colour sums,
//                per-cell point counts for the weighted filter
//   (kMarkLarge, kAccumulateLarge and kAccumulateRest on the levels of large builds)
//   kScatterPayload (weighted only) each point's offset from its cell centre + colour, and its
//                winner key, in cell order
//   kEmit        one staged point per occupied cell, in ascending cell order per node
//                (kEmitWeighted for the distance-weighted filter)
// and after the last level kPlaceNodes and kPermute, which write the staged points' records.
// Leaf points come from the sorted cloud, whose leaf ranges kLeafCellOrder has put in the cell
// order of each leaf's parent grid, so a level's first reads of them follow the bitmap.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "cell_order.h"
#include "device_common.h"
#include "kernels_chunking.h"
#include "kernels_sort.h"
#include "types.h"

namespace oc {

constexpr uint32_t TILE = 256;  // inputs per workgroup in the per-input kernels

constexpr uint32_t EMIT_CHUNK = 32;  // consecutive cell blocks of the weighted emit per XCD turn
constexpr uint32_t XCD_TILE_RUN = 32;  // consecutive input tiles of kMark / kScatterPayload per XCD turn

// Workgroup b runs on XCD b mod 8, each XCD with its own L2. The work item of workgroup b when
// every XCD is to take runs of `run` consecutive items: rounds of 8 * run items, XCD x taking
// items x * run .. x * run + run - 1 of each round. Grids are rounded up to whole rounds.
__device__ __forceinline__ uint32_t xcdRunItem(uint32_t b, uint32_t run)
{
    return (b / (XCD_COUNT * run)) * (XCD_COUNT * run) + (b % XCD_COUNT) * run + (b / XCD_COUNT) % run;
}

__host__ __forceinline__ uint32_t xcdRunGrid(uint64_t items, uint32_t run)
{
    const uint64_t round = static_cast<uint64_t>(XCD_COUNT) * run;
    return static_cast<uint32_t>((items + round - 1) / round * round);
}

// Order of a node grid's cells in its bitmap, and so of a node's staged points and of the leaf points
// that the node reads: rows in pencils where the colour filter walks neighbourhoods, Morton order
// (child-slot groups, as the octree's) where it does not. Then the up to eight cells of a child that
// make one cell of its parent are consecutive, as are the parent's cells: a wave's inputs are a few long
// runs of one cell each, and a bitmap word is a 4 x 4 x 2 block instead of a row of 32 that a surface
// meets in a few cells (25.8M points, intra-cell colours: kAccumulate 1447 -> 981 us).
enum CellOrder : uint32_t
{
    CELLS_PENCIL_ROWS,
    CELLS_MORTON
};

__host__ __device__ __forceinline__ CellOrder cellOrderOf(uint32_t colorMode, uint32_t g)
{
    const bool neighbours = colorMode == COLOR_INTER || colorMode == COLOR_INTER_WEIGHTED;
    return neighbours || (g & (g - 1)) != 0 || g < PENCIL ? CELLS_PENCIL_ROWS : CELLS_MORTON;
}

__device__ __forceinline__ uint32_t cellIndex(uint32_t x, uint32_t y, uint32_t z, uint32_t g, CellOrder order)
{
    return order == CELLS_MORTON ? morton3(x, y, z) : rowIndex(y, z, g) * g + x;
}

// Colours of the staged points. An average of packed sums can take 16 bits (their fields wrap), so the
// filters on packed sums keep the packed form; no filter and the distance-weighted one keep 8 bits each.
struct StagedColors
{
    uint32_t* rgb;     // r | g << 8 | b << 16, or null
    uint64_t* packed;  // encodeColors, or null
};

// The points a subsampling level reads: leaf points at positions [0, N) of the sorted cloud (a
// leaf's points are one contiguous range there) and already subsampled points of lower
// levels at positions [N, N + I) (staging, in level order until the final DFS post-order
// placement). A staged point is its index, exact coordinates and colour; its output record is derived
// from them by the placement exactly as a leaf point's is by the distribution (kept as records of 18
// bytes beside the coordinates, a level wrote 34 bytes per float point instead of 20 to 24).
template <typename T>
struct PointStore
{
    const SortedPoint<T>* sorted;
    uint32_t* stLut;
    T* stPts;
    StagedColors staged;
    uint32_t N;
    __device__ __forceinline__ uint32_t index(uint32_t pos) const
    {
        return pos < N ? sorted[pos].idx : stLut[pos - N];
    }
    // r | g << 8 | b << 16 (no filter, distance-weighted filter)
    __device__ __forceinline__ uint32_t rgb(uint32_t pos) const
    {
        return pos < N ? sorted[pos].rgb : staged.rgb[pos - N];
    }
    // encodeColors (filters on packed sums)
    __device__ __forceinline__ uint64_t packed(uint32_t pos) const
    {
        if (pos >= N)
            return staged.packed[pos - N];
        const uint32_t c = sorted[pos].rgb;
        return encodeColors(c & 0xFF, (c >> 8) & 0xFF, (c >> 16) & 0xFF);
    }
    __device__ __forceinline__ void xyz(uint32_t pos, T& x, T& y, T& z) const
    {
        if (pos < N)
        {
            const SortedPoint<T>& p = sorted[pos];
            x                        = p.x;
            y                        = p.y;
            z                        = p.z;
            return;
        }
        const T* q = stPts + 3 * static_cast<uint64_t>(pos - N);
        x          = q[0];
        y          = q[1];
        z          = q[2];
    }
};

struct SubsampleParams
{
    double cubicMin[3];
    double sideHalf[MAX_LEVELS];  // side of level L / 2 (the child offset when descending from L)
    double side;                  // side of the current level
    uint32_t level;
    uint32_t depth;
    uint32_t levelOffset;
    uint32_t levelGrid;
    uint32_t g;  // subsampling grid
    uint64_t seed;
};

// internal nodes of a level (batched builds)
struct InternalIn
{
    const uint8_t* flags;
    uint32_t levelStart;
    __device__ uint32_t operator()(uint64_t i) const { return (flags[levelStart + i] & NODE_INTERNAL) ? 1u : 0u; }
};

// Subsampling grid of the node with linear index lin at level `level` (grid gl per axis): the
// node minimum accumulated top-down exactly like the reference's DFS (calculateChildMinBB,
// tools.cu:29-61; rp_subsampling.cu:16-60): x = min.x; for every step down whose slot has the x
// bit, x = x + side/2 of that step; the extent is bbSize = (min.x + side) - min.x.
__device__ __forceinline__ Gridding nodeGridding(uint32_t lin, uint32_t gl, uint32_t level, uint32_t depth,
                                                 const double* cubicMin, const double* sideHalf, double side,
                                                 uint32_t g)
{
    const uint32_t x = lin % gl, y = (lin / gl) % gl, z = lin / (gl * gl);
    double mx = cubicMin[0], my = cubicMin[1], mz = cubicMin[2];
    for (uint32_t L = depth; L > level; --L)
    {
        const uint32_t b = L - 1 - level;
        if ((x >> b) & 1)
            mx = mx + sideHalf[L];
        if ((y >> b) & 1)
            my = my + sideHalf[L];
        if ((z >> b) & 1)
            mz = mz + sideHalf[L];
    }
    return gridding(mx, my, mz, (mx + side) - mx, g);
}

// What one node's subsampling needs, from its key.
__device__ __forceinline__ NodeGrid nodeGridOf(uint32_t id, uint32_t key, uint32_t levelOffset, uint32_t levelGrid,
                                               uint32_t level, uint32_t depth, const double* cubicMin,
                                               const double* sideHalf, double side, uint32_t g, uint64_t seed)
{
    NodeGrid ng;
    ng.grid        = nodeGridding(key - levelOffset, levelGrid, level, depth, cubicMin, sideHalf, side, g);
    const double t = ng.grid.bbSize / g;
    const double d = sqrt((t * 3) * (t * 3) * 3) / 2.0;
    ng.cell        = static_cast<float>(t);
    ng.weight      = static_cast<float>((-10.0 * 1.4426950408889634) / (d * d));
    ng.salt        = nodeSalt(seed, key);
    ng.id          = id;
    return ng;
}

// Per internal node k of the level: its eight input segments (children in slot order, the leaf's
// range of the sorted cloud or the child's staged subsample) and its gridding (nodeGridding).
struct LevelTables
{
    const uint32_t* nodeKey;
    const uint8_t* flags;
    const int32_t* children;
    const uint32_t* pointCount;
    const uint32_t* sortedStart;
    const uint32_t* stage;
    uint32_t* internalList;
    uint32_t* segCount;
    uint32_t* segSrc;
    uint32_t* segTile;
    uint32_t* segInput;
    uint32_t* tileList;
    NodeGrid* nodeGrid;
};

__device__ __forceinline__ void segmentsOf(uint64_t k, const SubsampleParams& sp, const LevelTables& lt)
{
    const uint32_t id = lt.internalList[k];
    for (int s = 0; s < 8; ++s)
    {
        const int32_t c = lt.children[8 * static_cast<uint64_t>(id) + s];
        uint32_t cnt = 0, src = 0;
        if (c >= 0)
        {
            cnt = lt.pointCount[c];
            src = (lt.flags[c] & NODE_INTERNAL) ? lt.stage[c] : lt.sortedStart[c];
        }
        lt.segCount[8 * k + s] = cnt;
        lt.segSrc[8 * k + s]   = src;
    }
    lt.nodeGrid[k] = nodeGridOf(id, lt.nodeKey[id], sp.levelOffset, sp.levelGrid, sp.level, sp.depth, sp.cubicMin,
                                sp.sideHalf, sp.side, sp.g, sp.seed);
}

// The sorted cloud in leaf and cell order. The fine sort's permutation puts the points in Morton
// order of their finest cells, so every leaf is one range; within a leaf that order says nothing
// about the parent's subsampling grid (a leaf spans 64^3 of the parent's 128^3 cells), and
// subsampling would see consecutive points in unrelated bitmap words and cells, making every
// atomic, rank lookup and payload store of the level random. So the records are gathered through
// the permutation leaf by leaf and reordered by bitmap word in the parent grid (the cell rows of
// the leaf's octant in the bitmap's pencil order, 32 cells per word): every leaf range is cut into
// chunks of at most LEAF_CHUNK points, one workgroup sorts a chunk with a counting sort over an
// LDS histogram and stores every record at its place in the chunk's range. Chunks bound the work
// of one workgroup (a dense cluster puts 10^5 points in one finest cell). Points within a leaf
// are unordered by definition (node point sets are compared), so the order is free to choose;
// the key only orders, so a point the parent grid clamps lands in an edge key.
constexpr int LEAF_THREADS    = 1024;
constexpr int LEAF_ITEMS      = 4;                          // points per thread, held in registers
constexpr uint32_t LEAF_KEYS  = 8192;                       // word keys (histogram entries)
constexpr uint32_t LEAF_CHUNK = LEAF_THREADS * LEAF_ITEMS;  // points per workgroup
constexpr uint32_t LEAF_LAUNCH_CHUNKS = 1u << 21;           // of one launch (fewer than 2^32 work-items)

struct LeafOrderParams
{
    double cubicMin[3];
    double sideHalf[MAX_LEVELS];
    double side[MAX_LEVELS];  // node side per level
    LevelParams lp;
    uint32_t g;         // subsampling grid (>= 2)
    uint32_t keyShift;  // word keys >> keyShift < LEAF_KEYS
    CellOrder order;
};

// What one leaf chunk reads of the level tables and node sides, by pointer: into the kernel
// argument (single cloud) or into the cloud's table in device memory (batches), so that no copy
// of the per-level arrays is made per chunk.
struct LeafOrderView
{
    const double* cubicMin;  // 3
    const double* sideHalf;  // per level
    const double* side;      // per level
    const uint32_t* offset;  // per level
    const uint32_t* grid;    // per level
    uint32_t depth, g, keyShift;
    CellOrder order;
};

__device__ __forceinline__ LeafOrderView leafOrderView(const LeafOrderParams& p)
{
    return LeafOrderView{p.cubicMin, p.sideHalf, p.side, p.lp.offset, p.lp.grid, p.lp.depth, p.g, p.keyShift,
                         p.order};
}

// Keys a leaf chunk can take: the bitmap words of a leaf's octant of the parent grid, shifted.
__host__ __device__ __forceinline__ uint32_t leafKeyCount(uint32_t g, uint32_t keyShift)
{
    const uint32_t h    = g > 1 ? g / 2 : 1;
    const uint64_t keys = rowsPerNode(h) * ((h + 31) / 32);
    return static_cast<uint32_t>(((keys - 1) >> keyShift) + 1);
}

// chunks of a leaf that a subsampling level reads (finished, not internal, with a parent)
struct LeafIn
{
    const uint8_t* flags;
    const int32_t* parent;
    const uint32_t* count;
    __device__ uint32_t operator()(uint64_t i) const
    {
        return ((flags[i] & (NODE_FINISHED | NODE_INTERNAL)) == NODE_FINISHED && parent[i] >= 0)
                       ? (count[i] + LEAF_CHUNK - 1) / LEAF_CHUNK
                       : 0u;
    }
};

// work list entry per chunk: chunk number << 32 | leaf id
struct LeafOut
{
    uint64_t* list;
    __device__ void operator()(uint64_t i, uint32_t prefix, uint32_t v) const
    {
        for (uint32_t c = 0; c < v; ++c)
            list[prefix + c] = (static_cast<uint64_t>(c) << 32) | i;
    }
};

// histogram slot of a key: one pad word per 32 keys, so the per-thread runs of the scan fall in
// distinct banks
__device__ __forceinline__ uint32_t leafSlot(uint32_t key)
{
    return key + (key >> 5);
}

__device__ __forceinline__ uint32_t leafLocal(uint32_t i, uint32_t origin, uint32_t h)
{
    return i < origin ? 0u : i - origin < h ? i - origin : h - 1;
}

// Word key of a point: its cell in the parent grid (multiplied by 1 / t instead of divided by t:
// the key only orders, so a point next to a cell face may take either side) relative to the leaf's
// octant, in the bitmap's order: (pencil row, x / 32), or the Morton code without its lowest bits (the
// octant is a whole run of the parent's code): as many cells to a key as a row has, up to a word's 32. With a
// word's in every grid, the points of the few cells that a small one has came in no order (421K points, g =
// 4: kAccumulate 903 us instead of 45).
struct LeafKeyer
{
    Gridding grid;
    uint32_t ox, oy, oz, h, wordsPerRow, shift, mortonShift;
    CellOrder order;
    __device__ __forceinline__ uint32_t operator()(double x, double y, double z) const
    {
        const double top = grid.gridSize - 1.0;
        const uint32_t ix = static_cast<uint32_t>(static_cast<int32_t>(fmin((x - grid.minX) * grid.inv, top)));
        const uint32_t iy = static_cast<uint32_t>(static_cast<int32_t>(fmin((y - grid.minY) * grid.inv, top)));
        const uint32_t iz = static_cast<uint32_t>(static_cast<int32_t>(fmin((z - grid.minZ) * grid.inv, top)));
        const uint32_t lx = leafLocal(ix, ox, h), ly = leafLocal(iy, oy, h), lz = leafLocal(iz, oz, h);
        const uint32_t word = order == CELLS_MORTON ? morton3(lx, ly, lz) >> mortonShift : rowIndex(ly, lz, h) * wordsPerRow + (lx >> 5);
        return word >> shift;
    }
};

struct LeafOrderLds
{
    uint32_t hist[LEAF_KEYS + LEAF_KEYS / 32];
    uint32_t scanLds[LEAF_THREADS / 64];
};

// One chunk of one leaf (all threads; the LDS is free again on return).
template <typename T>
__device__ __forceinline__ void leafCellOrderChunk(uint64_t entry, const LeafOrderView& p,
                                                   const uint32_t* __restrict__ nodeKey,
                                                   const int32_t* __restrict__ parent,
                                                   const uint32_t* __restrict__ count,
                                                   const uint32_t* __restrict__ sortedStart,
                                                   const SortedPoint<T>* __restrict__ bucketed,
                                                   const uint32_t* __restrict__ perm, SortedPoint<T>* __restrict__ out,
                                                   LeafOrderLds& lds)
{
    uint32_t* hist    = lds.hist;
    uint32_t* scanLds = lds.scanLds;
    const uint32_t leaf  = static_cast<uint32_t>(entry);
    const uint32_t first = static_cast<uint32_t>(entry >> 32) * LEAF_CHUNK;
    const uint32_t total = count[leaf];
    const uint32_t src   = sortedStart[leaf] + first;
    const uint32_t cnt   = total - first < LEAF_CHUNK ? total - first : LEAF_CHUNK;
    const uint32_t pkey  = nodeKey[static_cast<uint32_t>(parent[leaf])];
    uint32_t pl = 0;
    for (uint32_t k = 1; k <= p.depth; ++k)
        if (pkey >= p.offset[k])
            pl = k;
    LeafKeyer keyer;
    keyer.grid = nodeGridding(pkey - p.offset[pl], p.grid[pl], pl, p.depth, p.cubicMin, p.sideHalf, p.side[pl], p.g);
    // the leaf's octant of the parent grid: the low bit of its coordinates one level down
    const uint32_t ll = pl - 1, lgl = p.grid[ll], llin = nodeKey[leaf] - p.offset[ll];
    keyer.h           = p.g > 1 ? p.g / 2 : 1;  // cells per axis of the leaf's octant (1 for a 1-cell grid)
    keyer.ox          = ((llin % lgl) & 1u) * keyer.h;
    keyer.oy          = (((llin / lgl) % lgl) & 1u) * keyer.h;
    keyer.oz          = ((llin / (lgl * lgl)) & 1u) * keyer.h;
    keyer.wordsPerRow = (keyer.h + 31) / 32;
    keyer.shift       = p.keyShift;
    keyer.mortonShift = keyer.h >= 32 ? 5 : static_cast<uint32_t>(__builtin_ctz(keyer.h));
    keyer.order       = p.order;

    // only the keys this grid can produce take part (1024 of the 8192 at g = 64)
    const uint32_t keys = leafKeyCount(p.g, p.keyShift);
    for (uint32_t i = threadIdx.x; i < leafSlot(keys); i += LEAF_THREADS)
        hist[i] = 0;
    __syncthreads();
    // all loads in flight first, then the keys and their ranks within the key
    // every record is gathered once, kept in registers and stored at its place in the chunk's
    // range (a few hundred KB, so the scattered stores merge into whole lines in L2)
    uint32_t key[LEAF_ITEMS], rank[LEAF_ITEMS];
    SortedPoint<T> rec[LEAF_ITEMS];
    {
        uint32_t from[LEAF_ITEMS];
#pragma unroll
        for (int k = 0; k < LEAF_ITEMS; ++k)
        {
            const uint32_t i = threadIdx.x + k * LEAF_THREADS;
            if (i < cnt)
                from[k] = perm[src + i];
        }
#pragma unroll
        for (int k = 0; k < LEAF_ITEMS; ++k)
            if (threadIdx.x + k * LEAF_THREADS < cnt)
                rec[k] = bucketed[from[k]];
#pragma unroll
        for (int k = 0; k < LEAF_ITEMS; ++k)
            if (threadIdx.x + k * LEAF_THREADS < cnt)
            {
                key[k]  = keyer(static_cast<double>(rec[k].x), static_cast<double>(rec[k].y),
                                static_cast<double>(rec[k].z));
                rank[k] = atomicAdd(hist + leafSlot(key[k]), 1u);
            }
    }
    __syncthreads();

    // exclusive scan of the histogram, up to LEAF_KEYS / LEAF_THREADS consecutive keys per thread
    constexpr uint32_t PER = LEAF_KEYS / LEAF_THREADS;
    const uint32_t base    = threadIdx.x * PER;
    uint32_t sum           = 0;
#pragma unroll
    for (uint32_t k = 0; k < PER; ++k)
        if (base + k < keys)
            sum += hist[leafSlot(base + k)];
    uint32_t all;
    uint32_t off = sortBlockExclusiveScanN<LEAF_THREADS>(sum, all, scanLds);
#pragma unroll
    for (uint32_t k = 0; k < PER; ++k)
        if (base + k < keys)
        {
            const uint32_t v         = hist[leafSlot(base + k)];
            hist[leafSlot(base + k)] = off;
            off += v;
        }
    __syncthreads();

#pragma unroll
    for (int k = 0; k < LEAF_ITEMS; ++k)
        if (threadIdx.x + k * LEAF_THREADS < cnt)
            out[src + hist[leafSlot(key[k])] + rank[k]] = rec[k];
    __syncthreads();
}

template <typename T>
static __global__ __launch_bounds__(LEAF_THREADS) void kLeafCellOrder(const uint64_t* __restrict__ chunkList, uint32_t first,
                                                                const uint64_t* __restrict__ totals, LeafOrderParams p,
                                                                const uint32_t* __restrict__ nodeKey,
                                                                const int32_t* __restrict__ parent,
                                                                const uint32_t* __restrict__ count,
                                                                const uint32_t* __restrict__ sortedStart,
                                                                const SortedPoint<T>* __restrict__ bucketed,
                                                                const uint32_t* __restrict__ perm,
                                                                SortedPoint<T>* __restrict__ out, uint64_t* stamp)
{
    __shared__ LeafOrderLds lds;
    stampStart(stamp);
    const uint32_t chunk = first + blockIdx.x;
    if (chunk >= *totals >> 32)
        return;  // the whole workgroup: the grid is an upper bound
    leafCellOrderChunk<T>(chunkList[chunk], leafOrderView(p), nodeKey, parent, count, sortedStart, bucketed, perm,
                          out, lds);
}

// packed (tiles << 32 | inputs) per segment, so one scan yields both prefix sums
struct SegmentIn
{
    const uint32_t* segCount;
    __device__ uint64_t operator()(uint64_t s) const
    {
        uint64_t c = segCount[s];
        return (((c + TILE - 1) / TILE) << 32) | c;
    }
};

struct SegmentOut
{
    uint32_t* segTile;
    uint32_t* segInput;
    __device__ void operator()(uint64_t s, uint64_t prefix, uint64_t) const
    {
        segTile[s]  = static_cast<uint32_t>(prefix >> 32);
        segInput[s] = static_cast<uint32_t>(prefix);
    }
};

__device__ __forceinline__ void tileListOf(uint64_t s, const uint32_t* __restrict__ segCount,
                                           const uint32_t* __restrict__ segTile, uint32_t* __restrict__ tileList)
{
    uint32_t tiles = (segCount[s] + TILE - 1) / TILE;
    uint32_t first = segTile[s];
    for (uint32_t t = 0; t < tiles; ++t)
        tileList[first + t] = static_cast<uint32_t>(s);
}

// Single cloud: the child slots of all internal nodes (8 k + slot, k in id order), one scan.
// Item: chunks of a leaf child (high half; kLeafCellOrder) and its points (low half), so that the
// prefix is its data offset (A4: blocks in parent-id order, children in slot order).
struct ChildSlots
{
    const uint32_t* internal;  // ids of the internal nodes, ascending
    const uint8_t* flags;
    const int32_t* children;
    const uint32_t* nodeCount;
    __device__ __forceinline__ int32_t child(uint64_t s) const
    {
        return children[8 * static_cast<uint64_t>(internal[s >> 3]) + (s & 7)];
    }
};

struct LeafSlotIn
{
    ChildSlots cs;
    __device__ uint64_t operator()(uint64_t s) const
    {
        const int32_t c = cs.child(s);
        if (c < 0 || (cs.flags[c] & NODE_INTERNAL))
            return 0;
        const uint32_t n = cs.nodeCount[c];
        return (static_cast<uint64_t>((n + LEAF_CHUNK - 1) / LEAF_CHUNK) << 32) | n;
    }
};

struct LeafSlotOut
{
    ChildSlots cs;
    uint64_t* dataIdx;
    uint64_t* chunkList;  // chunk number << 32 | leaf id
    __device__ void operator()(uint64_t s, uint64_t prefix, uint64_t v) const
    {
        if (v == 0)
            return;
        const uint32_t c = static_cast<uint32_t>(cs.child(s));
        dataIdx[c]       = static_cast<uint32_t>(prefix);
        for (uint32_t k = 0; k < (v >> 32); ++k)
            chunkList[(prefix >> 32) + k] = (static_cast<uint64_t>(k) << 32) | c;
    }
};

// Input segments of one level: the child slots of its internal nodes (cs.internal is the level's part
// of the list), scanned as (tiles << 32 | inputs).
struct LevelSegmentIn
{
    ChildSlots cs;
    const uint32_t* pointCount;
    uint32_t tile;  // inputs per tile
    __device__ uint64_t operator()(uint64_t s) const
    {
        const int32_t c  = cs.child(s);
        const uint64_t n = c >= 0 ? pointCount[c] : 0u;
        return (((n + tile - 1) / tile) << 32) | n;
    }
};

struct LevelSegmentOut
{
    ChildSlots cs;
    const uint32_t* sortedStart;
    const uint32_t* stage;
    uint32_t *segCount, *segSrc, *segTile, *segInput;
    __device__ void operator()(uint64_t s, uint64_t prefix, uint64_t v) const
    {
        const int32_t c = cs.child(s);
        segCount[s]     = static_cast<uint32_t>(v);
        segSrc[s]       = c < 0 ? 0u : (cs.flags[c] & NODE_INTERNAL) ? stage[c] : sortedStart[c];
        segTile[s]      = static_cast<uint32_t>(prefix >> 32);
        segInput[s]     = static_cast<uint32_t>(prefix);
    }
};

// Per-cell state of the accumulation, by dense index: no winner, no colour sum, no points. Arrays that
// the colour mode does not use are null.
struct CellState
{
    uint64_t* win;
    uint64_t* color;
    uint32_t* cellCnt;
    __device__ __forceinline__ void reset(uint64_t c) const
    {
        if (win)
            win[c] = ~0ull;
        if (color)
            color[c] = 0;
        if (cellCnt)
            cellCnt[c] = 0;
    }
};

// Before a level's first pass: the griddings of its nodes, the segment of every tile (a search per
// tile, all of them in flight; a thread per segment wrote a large child's thousands of entries by
// itself, 71 us of a 5.1M-point build) and a clear bitmap. nodes = 0: only the bitmap and the cells (a later
// step of the same level). For a small level also the state of as many cells as it has inputs (it has no
// more, and no more than `reset`, the ones that the cell arrays hold), which spares it kClearCompact.
__device__ __forceinline__ void levelPrepare(uint32_t nodes, const SubsampleParams& sp,
                                             const uint32_t* __restrict__ internal,
                                             const uint32_t* __restrict__ nodeKey, NodeGrid* __restrict__ nodeGrid,
                                             const uint32_t* segTile, uint64_t segTotal,
                                             uint32_t* __restrict__ tileList, uint64_t words,
                                             uint32_t* __restrict__ bitmap, const CellState& cells, uint32_t reset)
{
    for (uint64_t k = globalThread(); k < nodes; k += globalStride())
        nodeGrid[k] = nodeGridOf(internal[k], nodeKey[internal[k]], sp.levelOffset, sp.levelGrid, sp.level, sp.depth,
                                 sp.cubicMin, sp.sideHalf, sp.side, sp.g, sp.seed);
    const uint32_t tiles = nodes ? static_cast<uint32_t>(segTotal >> 32) : 0u;
    for (uint64_t t = globalThread(); t < tiles; t += globalStride())
    {
        // the last segment that starts at or before t; segments without tiles start where the next does
        uint32_t lo = 0, hi = 8 * nodes;
        while (hi - lo > 1)
        {
            const uint32_t mid = (lo + hi) >> 1;
            if (segTile[mid] <= t)
                lo = mid;
            else
                hi = mid;
        }
        tileList[t] = lo;
    }
    for (uint64_t w = globalThread(); w < words; w += globalStride())
        bitmap[w] = 0;
    if (reset)
    {
        const uint32_t inputs = static_cast<uint32_t>(segTotal), most = inputs < reset ? inputs : reset;
        for (uint64_t c = globalThread(); c < most; c += globalStride())
            cells.reset(c);
    }
}

static __global__ __launch_bounds__(BLOCK) void kLevelPrepare(uint32_t nodes, SubsampleParams sp,
                                                        const uint32_t* __restrict__ internal,
                                                        const uint32_t* __restrict__ nodeKey,
                                                        NodeGrid* __restrict__ nodeGrid,
                                                        const uint32_t* __restrict__ segTile,
                                                        const uint64_t* __restrict__ segTotal,
                                                        uint32_t* __restrict__ tileList, uint64_t words,
                                                        uint32_t* __restrict__ bitmap, CellState cells, uint32_t reset,
                                                        uint64_t* stamp)
{
    stampStart(stamp);
    levelPrepare(nodes, sp, internal, nodeKey, nodeGrid, segTile, *segTotal, tileList, words, bitmap, cells, reset);
}

// Levels of up to START_NODES nodes: the segment scan and kLevelPrepare in one launch. Every workgroup
// scans the (at most SCAN_TILE) segments into its LDS, so none waits for another; the first one writes
// them out.
constexpr uint32_t START_NODES = SCAN_TILE / 8;
static_assert(BLOCK == SCAN_THREADS, "kLevelStart scans with one workgroup's threads");

static __global__ __launch_bounds__(BLOCK) void kLevelStart(uint32_t nodes, SubsampleParams sp, LevelSegmentIn in,
                                                      LevelSegmentOut out, const uint32_t* __restrict__ nodeKey,
                                                      NodeGrid* __restrict__ nodeGrid, uint64_t* __restrict__ segTotal,
                                                      uint32_t* __restrict__ tileList, uint64_t words,
                                                      uint32_t* __restrict__ bitmap, CellState cells, uint32_t reset,
                                                      uint64_t* stamp)
{
    __shared__ uint64_t lds[SCAN_ITEMS * SCAN_WAVES];
    __shared__ uint32_t segTile[SCAN_TILE];
    stampStart(stamp);
    const uint32_t segments = 8 * nodes;
    uint64_t v[SCAN_ITEMS], pre[SCAN_ITEMS];
    loadTile<uint64_t>(in, 0, segments, v);
    const uint64_t total = tileExclusiveScan(v, pre, lds);
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k)
        segTile[k * SCAN_THREADS + threadIdx.x] = static_cast<uint32_t>(pre[k] >> 32);
    __syncthreads();
    if (blockIdx.x == 0)
    {
        storeTile<uint64_t>(out, 0, segments, v, pre, 0);
        if (threadIdx.x == 0)
            *segTotal = total;
    }
    levelPrepare(nodes, sp, in.cs.internal, nodeKey, nodeGrid, segTile, total, tileList, words, bitmap, cells, reset);
}

// Tiles that one launch takes: a launch holds fewer than 2^32 work-items, kScatterPayload's 256 for each of
// up to four parts of a tile.
constexpr uint32_t LAUNCH_TILES = 1u << 21;

// The tiles of a batch of a level's nodes, from *lo (null: 0) to *hi, without the `skip` first ones (of
// earlier launches): as many of them as one launch takes.
struct TileRange
{
    const uint32_t* lo;
    const uint32_t* hi;
    uint32_t skip;
    __device__ __forceinline__ uint32_t first() const { return (lo ? *lo : 0u) + skip; }
    __device__ __forceinline__ uint32_t count() const
    {
        const uint32_t from = first(), to = *hi;
        return to <= from ? 0u : to - from < LAUNCH_TILES ? to - from : LAUNCH_TILES;
    }
};

// Clock stamps of a subsampling step, then one after the last step.
enum StepStamp : uint32_t
{
    ST_BEGIN,
    ST_INSERT_BEGIN,
    ST_INSERT_END,
    ST_EMIT_BEGIN,
    ST_STAMPS
};

// One step of the subsampling (a batch of a level's nodes), with the sizes that only the device
// knows: the output cursor before and after it and its occupied cells.
struct StepSizes
{
    const uint64_t* cursor;  // N + points subsampled before this step
    uint64_t* next;          // the same after it
    const uint32_t* cells;   // occupied cells
    uint64_t capacity;       // E
    // false: the points do not fit the output (A14); nothing of this step or a later one is written
    __device__ __forceinline__ bool fits() const { return *cursor + *cells <= capacity; }
    // the cells to work on (the cell arrays hold no more than the output has room for)
    __device__ uint64_t operator()() const { return fits() ? *cells : 0u; }
};

constexpr uint64_t CURSOR_FULL = 1ull << 62;

// Identifies the input of this thread: tile -> segment -> (node k, input position, input index q). Large
// tiles are read in parts of TILE inputs; `tile` then counts the parts.
struct InputRef
{
    uint32_t seg, local, k, pos, q;
    bool valid;
};

__device__ __forceinline__ InputRef inputOf(uint32_t tile, const uint32_t* tileList, const uint32_t* segTile,
                                            const uint32_t* segCount, const uint32_t* segSrc,
                                            const uint32_t* segInput, uint32_t parts = 1)
{
    InputRef r;
    r.seg   = tileList[tile / parts];
    r.local = (tile - segTile[r.seg] * parts) * TILE + threadIdx.x;
    r.valid = r.local < segCount[r.seg];
    r.k     = r.seg >> 3;
    r.pos   = segSrc[r.seg] + r.local;
    r.q     = segInput[r.seg] + r.local;
    return r;
}

// Evaluate, part 1 (rp_subsample_evaluation.cuh:37-203, fp_subsample_evaluation.cuh:22-110):
// the cell of every input point in its node's grid; marks the cell occupied.
template <typename T>
__device__ __forceinline__ void markTile(uint32_t tile, uint32_t nodeBase, uint64_t wordsPerNode,
                                         const uint32_t* __restrict__ tileList, const uint32_t* __restrict__ segTile,
                                         const uint32_t* __restrict__ segCount, const uint32_t* __restrict__ segSrc,
                                         const uint32_t* __restrict__ segInput, const NodeGrid* __restrict__ nodeGrid,
                                         const PointStore<T>& ps, CellOrder order, uint32_t* __restrict__ bitmap,
                                         uint32_t* __restrict__ cellOf, uint32_t* __restrict__ err)
{
    // All lanes take part in the wave-level merge of bit sets bound for the same bitmap word.
    InputRef in   = inputOf(tile, tileList, segTile, segCount, segSrc, segInput);
    bool valid    = in.valid;
    uint32_t cell = ~0u;
    if (valid)
    {
        const NodeGrid ng = nodeGrid[in.k];
        T px, py, pz;
        ps.xyz(in.pos, px, py, pz);
        uint32_t ix, iy, iz;
        gridCoords(static_cast<double>(px), static_cast<double>(py), static_cast<double>(pz), ng.grid, ix, iy, iz);
        const uint32_t gs = ng.grid.gridSize;
        if (ix >= gs || iy >= gs || iz >= gs)
        {
            atomicOr(err, ERR_OUTSIDE);  // skipped by the later passes; the build reports the error
            cellOf[in.q] = ~0u;
            valid        = false;
        }
        else
        {
            cell         = cellIndex(ix, iy, iz, gs, order);
            cellOf[in.q] = cell;
        }
    }
    const uint64_t word = valid ? (in.k - nodeBase) * wordsPerNode + (cell >> 5) : ~0ull - threadIdx.x;
    const WaveRun run   = waveRun(word);
    const uint32_t bits = runScan<uint32_t>(valid ? 1u << (cell & 31) : 0u, run,
                                            [](uint32_t x, uint32_t y) { return x | y; });
    if (valid && run.lane == run.end)
        atomicOr(bitmap + word, bits);
}

template <typename T>
static __global__ __launch_bounds__(TILE) void kMark(TileRange range, uint32_t nodeBase, uint64_t wordsPerNode,
                                               const uint32_t* __restrict__ tileList,
                                               const uint32_t* __restrict__ segTile,
                                               const uint32_t* __restrict__ segCount,
                                               const uint32_t* __restrict__ segSrc,
                                               const uint32_t* __restrict__ segInput,
                                               const NodeGrid* __restrict__ nodeGrid, PointStore<T> ps, CellOrder order,
                                               uint32_t* __restrict__ bitmap, uint32_t* __restrict__ cellOf,
                                               uint32_t* __restrict__ err, uint64_t* stamp)
{
    stampStart(stamp);
    // consecutive tiles share bitmap words: runs of them per XCD
    const uint32_t t = xcdRunItem(blockIdx.x, XCD_TILE_RUN);
    if (t >= range.count())
        return;
    markTile<T>(range.first() + t, nodeBase, wordsPerNode, tileList, segTile, segCount, segSrc, segInput, nodeGrid, ps,
                order, bitmap, cellOf, err);
}

// Levels of large builds: tiles of LARGE_TILE inputs, combined in LDS before anything goes to memory.
//
// What bounds the passes over the inputs there is the number of their atomics: the XCDs' L2s are not
// coherent with each other, so every global atomic is carried out in memory, some 20 requests per ns on
// the whole chip whatever their kind (measured from 5.1M to 119.7M points), and a level's inputs come in
// the order of their children's grids, in which the points of one cell are mostly close together but not
// consecutive. So a tile first combines its points per bitmap word (kMarkLarge) and per cell
// (kAccumulateLarge) in a hash table in LDS. Of the tiles that meet in a cell the one whose bit was set
// first owns it: kMarkLarge takes the old bits from its atomics and flags the cell index of every other
// tile's inputs (NOT_OWNED). The owner stores the cell's state without reading it, so it needs no reset,
// and kAccumulateRest then adds the flagged inputs with atomics. Mark + accumulate (+ reset of the cells):
//   25.8M points, intra-cell   478 + 984 + 82 -> 468 + 560 + 119 us
//   119.7M, distance-weighted  2122 + 3150 + 87 -> 1930 + 1798 + 623 us
//   5.1M, inter-cell           143 + 345 -> 144 + 185 + 51 us
//   1.5M, no filter            54 + 66 -> 77 + 68 + 27 us
// so from LARGE_POINTS on (below, a level has too few tiles to hide their barriers and one launch more; whole
// builds with / without, intra-cell and weighted: 2M points 791 / 770 and 1366 / 1323 us, 3.2M 958 / 973 and
// 1539 / 1528, 4M 1136 / 1164, 8M 1753 / 1886 and 2969 / 3050), on the levels whose children can have
// LARGE_CHILD points each: a tile holds inputs of one child, and one that is nearly empty clears its table for
// a few of them. 8M points at threshold 20, a dozen inputs a child: 17.7 ms with large tiles, 15.3 without;
// threshold 60: 10.6 / 9.3; threshold 1000, about 200 a child: 4.05 / 4.15. (512 instead of 256: alike.)
constexpr uint32_t LARGE_POINTS = 3u << 20;
constexpr uint32_t LARGE_CHILD  = 256;
constexpr int LARGE_THREADS     = 256;
constexpr int LARGE_ITEMS       = 4;  // per thread
constexpr uint32_t LARGE_TILE   = LARGE_THREADS * LARGE_ITEMS;
constexpr uint32_t NOT_OWNED    = 1u << 31;  // cell and dense indices are below

// Hash table in LDS of the at most LARGE_TILE distinct keys of a tile: key << 32 | the input that put it
// there, whose number is also that of the key's values. Open addressing from a multiplicative hash: the
// keys come in runs of consecutive ones, which would pile up in consecutive slots (5.1M points, rows in
// pencils: accumulating them took 1380 instead of 182 us). The size is a compromise between probes and workgroups
// per CU.
constexpr uint32_t TABLE_SLOTS          = LARGE_TILE * 3 / 2;
constexpr unsigned long long TABLE_FREE = ~0ull;

// The input that put `key` into the table; `input` itself if it is the first one with it.
__device__ __forceinline__ uint32_t tableInput(unsigned long long* table, uint32_t key, uint32_t input)
{
    uint32_t s                   = __umulhi(key * 2654435769u, TABLE_SLOTS);
    const unsigned long long own = (static_cast<unsigned long long>(key) << 32) | input;
    for (;;)  // ends: there are fewer keys than slots
    {
        const unsigned long long was = atomicCAS(table + s, TABLE_FREE, own);
        if (was == TABLE_FREE)
            return input;
        if (was >> 32 == key)
            return static_cast<uint32_t>(was);
        s = s + 1 < TABLE_SLOTS ? s + 1 : 0;
    }
}

// The inputs of a workgroup's tile: LARGE_ITEMS per thread, a wave's inputs of one item consecutive.
struct LargeTile
{
    uint32_t k, pos, q, count;  // node of the level, position and index of the first input, inputs
    __device__ __forceinline__ uint32_t at(int item) const { return LARGE_THREADS * item + threadIdx.x; }
    __device__ __forceinline__ bool has(int item) const { return at(item) < count; }
};

__device__ __forceinline__ LargeTile largeTile(uint32_t tile, const uint32_t* tileList, const uint32_t* segTile,
                                               const uint32_t* segCount, const uint32_t* segSrc,
                                               const uint32_t* segInput)
{
    const uint32_t seg   = tileList[tile];
    const uint32_t first = (tile - segTile[seg]) * LARGE_TILE;
    const uint32_t left  = segCount[seg] - first;
    return LargeTile{seg >> 3, segSrc[seg] + first, segInput[seg] + first, left < LARGE_TILE ? left : LARGE_TILE};
}

template <typename T>
static __global__ __launch_bounds__(LARGE_THREADS) void kMarkLarge(TileRange range, uint32_t nodeBase, uint64_t wordsPerNode,
                                                    const uint32_t* __restrict__ tileList,
                                                    const uint32_t* __restrict__ segTile,
                                                    const uint32_t* __restrict__ segCount,
                                                    const uint32_t* __restrict__ segSrc,
                                                    const uint32_t* __restrict__ segInput,
                                                    const NodeGrid* __restrict__ nodeGrid, PointStore<T> ps,
                                                    CellOrder order, uint32_t* __restrict__ bitmap,
                                                    uint32_t* __restrict__ cellOf, uint32_t* __restrict__ err,
                                                    uint64_t* stamp)
{
    __shared__ unsigned long long table[TABLE_SLOTS];
    __shared__ uint32_t bits[LARGE_TILE];
    stampStart(stamp);
    // consecutive tiles share bitmap words: runs of them per XCD
    const uint32_t t = xcdRunItem(blockIdx.x, XCD_TILE_RUN * TILE / LARGE_TILE);
    if (t >= range.count())
        return;  // the whole workgroup
    const LargeTile in  = largeTile(range.first() + t, tileList, segTile, segCount, segSrc, segInput);
    const Gridding grid = nodeGrid[in.k].grid;
    T px[LARGE_ITEMS], py[LARGE_ITEMS], pz[LARGE_ITEMS];
#pragma unroll
    for (int i = 0; i < LARGE_ITEMS; ++i)
        if (in.has(i))
            ps.xyz(in.pos + in.at(i), px[i], py[i], pz[i]);
    for (uint32_t s = threadIdx.x; s < TABLE_SLOTS; s += LARGE_THREADS)
        table[s] = TABLE_FREE;
    for (uint32_t s = threadIdx.x; s < LARGE_TILE; s += LARGE_THREADS)
        bits[s] = 0;
    __syncthreads();

    uint32_t cell[LARGE_ITEMS], slot[LARGE_ITEMS];
    bool created[LARGE_ITEMS];
#pragma unroll
    for (int i = 0; i < LARGE_ITEMS; ++i)
    {
        cell[i] = ~0u;
        if (in.has(i))
        {
            uint32_t ix, iy, iz;
            gridCoords(static_cast<double>(px[i]), static_cast<double>(py[i]), static_cast<double>(pz[i]), grid, ix,
                       iy, iz);
            const uint32_t gs = grid.gridSize;
            if (ix >= gs || iy >= gs || iz >= gs)
                atomicOr(err, ERR_OUTSIDE);  // skipped by the later passes; the build reports the error
            else
                cell[i] = cellIndex(ix, iy, iz, gs, order);
        }
        // one insertion per run of lanes in the same word; all lanes take part
        const bool valid  = cell[i] != ~0u;
        const WaveRun run = waveRun(valid ? cell[i] >> 5 : ~0ull - threadIdx.x);
        slot[i]           = 0;
        if (valid && run.lane == run.start)
            slot[i] = tableInput(table, cell[i] >> 5, in.at(i));
        slot[i]    = __shfl(slot[i], run.start, 64);
        created[i] = valid && slot[i] == in.at(i);
        if (valid)
            atomicOr(bits + slot[i], 1u << (cell[i] & 31));
    }
    __syncthreads();
    uint32_t* words = bitmap + (in.k - nodeBase) * wordsPerNode;
    uint32_t old[LARGE_ITEMS];
#pragma unroll
    for (int i = 0; i < LARGE_ITEMS; ++i)
        if (created[i])
            old[i] = atomicOr(words + (cell[i] >> 5), bits[slot[i]]);
#pragma unroll
    for (int i = 0; i < LARGE_ITEMS; ++i)
        if (created[i])
            bits[slot[i]] &= ~old[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < LARGE_ITEMS; ++i)
        if (in.has(i))
        {
            const bool owned = cell[i] == ~0u || ((bits[slot[i]] >> (cell[i] & 31)) & 1u) != 0;
            cellOf[in.q + in.at(i)] = owned ? cell[i] : cell[i] | NOT_OWNED;
        }
}

struct PopcountIn
{
    const uint32_t* bitmap;
    __device__ uint32_t operator()(uint64_t w) const { return __popc(bitmap[w]); }
};

// dense index of a set cell: exclusive popcount prefix of its word + set bits below it
__device__ __forceinline__ uint32_t cellRank(const uint32_t* bitmap, const uint32_t* prefix, uint64_t word,
                                             uint32_t bit)
{
    return prefix[word] + __popc(bitmap[word] & ((1u << bit) - 1u));
}

// Per node of the batch: subsample size (occupied cells) and staging position.
__device__ __forceinline__ void batchNodeOf(uint64_t kl, uint32_t nodeBase, uint64_t wordsPerNode,
                                            const NodeGrid* __restrict__ nodeGrid,
                                            const uint32_t* __restrict__ prefix, uint32_t cursor,
                                            uint32_t* __restrict__ pointCount, uint32_t* __restrict__ stage)
{
    const uint32_t b = prefix[kl * wordsPerNode], e = prefix[(kl + 1) * wordsPerNode];
    uint32_t id    = nodeGrid[nodeBase + kl].id;
    pointCount[id] = e - b;
    stage[id]      = cursor + b;
}

// the state of a large level's cells
static __global__ __launch_bounds__(BLOCK) void kClearCompact(StepSizes step, CellState cells)
{
    const uint64_t count = step();
    for (uint64_t c = globalThread(); c < count; c += globalStride())
        cells.reset(c);
}

// Large levels, the popcount scan's first pass: occupied cells per tile of SCAN_TILE words and per
// workgroup's range of tiles.
static __global__ __launch_bounds__(SCAN_THREADS) void kWordReduce(const uint32_t* __restrict__ bitmap, uint64_t words,
                                                            uint32_t* __restrict__ tileSums,
                                                            uint32_t* __restrict__ rangeSums)
{
    __shared__ uint32_t lds[SCAN_WAVES];
    uint64_t first, last;
    tileRange(scanTiles(words), first, last);
    uint32_t range = 0;
    for (uint64_t tile = first; tile < last; ++tile)
    {
        uint32_t v[SCAN_ITEMS], s = 0;
        loadTile<uint32_t>(PopcountIn{bitmap}, tile * SCAN_TILE, words, v);
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k)
            s += v[k];
        const uint32_t sum = __syncthreads_or(s != 0) ? blockSum(s, lds) : 0u;
        if (threadIdx.x == 0)
            tileSums[tile] = sum;
        range += sum;
    }
    if (threadIdx.x == 0)
        rangeSums[blockIdx.x] = range;
}

// Second pass: the prefix of every word in the tiles that hold any occupied cell, and of the words of the
// others that are read (emptyWordPrefixes). The nodes' cells lie on surfaces, so most tiles (a slab of four
// cell layers of a 128^3 grid) are empty: not read here, and next to nothing written.
static __global__ __launch_bounds__(SCAN_THREADS) void kWordPrefix(const uint32_t* __restrict__ bitmap, uint64_t words,
                                                            uint64_t wordsPerNode,
                                                            const uint32_t* __restrict__ tileSums,
                                                            const uint32_t* __restrict__ rangeSums,
                                                            uint32_t* __restrict__ prefix)
{
    __shared__ uint32_t lds[SCAN_ITEMS * SCAN_WAVES];
    uint64_t first, last;
    tileRange(scanTiles(words), first, last);
    uint32_t carry = sumBefore(rangeSums, lds);
    for (uint64_t tile = first; tile < last; ++tile)
    {
        const uint64_t base = tile * SCAN_TILE;
        const uint32_t sum  = tileSums[tile];
        if (sum == 0)
        {
            const uint64_t end = base + SCAN_TILE < words ? base + SCAN_TILE : words;
            emptyWordPrefixes(base, end, wordsPerNode, threadIdx.x, SCAN_THREADS, [=](uint64_t w) { prefix[w] = carry; });
            continue;
        }
        uint32_t v[SCAN_ITEMS], pre[SCAN_ITEMS];
        loadTile<uint32_t>(PopcountIn{bitmap}, base, words, v);
        (void)tileExclusiveScan(v, pre, lds);
        storeTile<uint32_t>(ExclusiveToArray{prefix}, base, words, v, pre, carry);
        carry += sum;
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0)
        prefix[words] = carry;
}

// Evaluate, part 2: winner (A7/A8: atomicMin of rank << 32 | input position, rank = point index
// for the implicit method or the keyed bijective hash of it for the explicit one), the packed
// colour sum of the input records (intra-cell, and the per-cell sums the inter-cell filter is
// built from), and per-cell point counts + each point's rank in its cell (weighted filter).
template <typename T, uint32_t MODE, bool RANDOM>
__device__ __forceinline__ void accumulateTile(uint32_t tile, uint32_t nodeBase, uint64_t wordsPerNode,
                                               const uint32_t* __restrict__ tileList,
                                               const uint32_t* __restrict__ segTile,
                                               const uint32_t* __restrict__ segCount,
                                               const uint32_t* __restrict__ segSrc,
                                               const uint32_t* __restrict__ segInput,
                                               const NodeGrid* __restrict__ nodeGrid,
                                               const uint32_t* __restrict__ bitmap,
                                               const uint32_t* __restrict__ prefix, uint32_t* __restrict__ cellOf,
                                               const PointStore<T>& ps, uint64_t* __restrict__ win,
                                               uint64_t* __restrict__ color, uint32_t* __restrict__ cellCnt,
                                               uint32_t* __restrict__ cellKey, uint32_t* __restrict__ cellNode,
                                               uint32_t* __restrict__ rankOf)
{
    // All lanes take part: runs of lanes in the same cell make one atomic per run.
    InputRef in         = inputOf(tile, tileList, segTile, segCount, segSrc, segInput);
    const uint32_t cell = in.valid ? cellOf[in.q] : ~0u;
    const bool valid    = cell != ~0u;  // an invalid cell: the point lay outside its node's grid
    uint32_t c          = 0;
    if (valid)
    {
        const uint64_t word = (in.k - nodeBase) * wordsPerNode + (cell >> 5);
        c                   = cellRank(bitmap, prefix, word, cell & 31);
    }
    const WaveRun run = waveRun(valid ? c : ~0ull - threadIdx.x);
    if (valid && run.lane == run.start)
    {
        cellKey[c]  = cell;
        cellNode[c] = in.k - nodeBase;
    }
    if (MODE == COLOR_INTER_WEIGHTED)
    {
        // the winner is taken from the cell's payload run in the emit; the input's cell index is
        // replaced by the cell's dense index (the payload scatter reads the cell back from cellKey)
        uint32_t base = 0;
        if (valid && run.lane == run.end)
            base = atomicAdd(cellCnt + c, static_cast<uint32_t>(run.end - run.start + 1));
        base = __shfl(base, run.end, 64);
        if (valid)
        {
            cellOf[in.q] = c;
            rankOf[in.q] = base + static_cast<uint32_t>(run.lane - run.start);
        }
        return;
    }
    uint64_t key = ~0ull, col = 0;
    if (valid)
    {
        const uint32_t idx  = ps.index(in.pos);
        const uint32_t rank = RANDOM ? fmix32(idx ^ nodeGrid[in.k].salt) : idx;
        key                 = (static_cast<uint64_t>(rank) << 32) | in.pos;
        if (MODE == COLOR_INTRA || MODE == COLOR_INTER)
            col = ps.packed(in.pos);
    }
    key = runScan<uint64_t>(key, run, [](uint64_t x, uint64_t y) { return x < y ? x : y; });
    if (MODE == COLOR_INTRA || MODE == COLOR_INTER)
        col = runScan<uint64_t>(col, run, [](uint64_t x, uint64_t y) { return x + y; });
    if (valid && run.lane == run.end)
    {
        atomicMin(reinterpret_cast<unsigned long long*>(win + c), static_cast<unsigned long long>(key));
        if (MODE == COLOR_INTRA || MODE == COLOR_INTER)
            atomicAdd(reinterpret_cast<unsigned long long*>(color + c), static_cast<unsigned long long>(col));
    }
}

// Subsampled points of an internal node and all internal nodes below it (a leaf's: zero).
__device__ __forceinline__ void subtreeOf(uint32_t id, const uint8_t* __restrict__ flags,
                                          const int32_t* __restrict__ children, const uint32_t* pointCount,
                                          uint32_t* subtree)
{
    if (!(flags[id] & NODE_INTERNAL))
        return;
    uint32_t s = pointCount[id];
    for (int k = 0; k < 8; ++k)
    {
        const int32_t c = children[8 * static_cast<uint64_t>(id) + k];
        if (c >= 0)
            s += subtree[c];
    }
    subtree[id] = s;
}

// The nodes' subsample sizes, subtree sums and the next step's cursor go with it (one thread per node).
__device__ __forceinline__ bool accumulateNodes(const StepSizes& step, uint32_t nodeBase, uint32_t nodes,
                                                uint64_t wordsPerNode, const NodeGrid* __restrict__ nodeGrid,
                                                const uint32_t* __restrict__ prefix, uint32_t* __restrict__ pointCount,
                                                uint32_t* __restrict__ stage, uint32_t* __restrict__ subtree,
                                                const uint8_t* __restrict__ flags,
                                                const int32_t* __restrict__ children, uint32_t* __restrict__ err)
{
    const bool fits       = step.fits();
    const uint64_t cursor = *step.cursor;
    if (globalThread() == 0)
    {
        *step.next = fits ? cursor + *step.cells : CURSOR_FULL;
        if (!fits)
            atomicOr(err, ERR_OVERFLOW);
    }
    for (uint64_t kl = globalThread(); kl < nodes; kl += globalStride())
    {
        const uint32_t id = nodeGrid[nodeBase + kl].id;
        if (fits)
            batchNodeOf(kl, nodeBase, wordsPerNode, nodeGrid, prefix, static_cast<uint32_t>(cursor), pointCount, stage);
        else
            pointCount[id] = 0;  // no input of a later step
        subtreeOf(id, flags, children, pointCount, subtree);  // of the levels below: complete
    }
    return fits;
}

template <typename T, uint32_t MODE, bool RANDOM>
static __global__ __launch_bounds__(TILE) void kAccumulate(TileRange range, StepSizes step, uint32_t nodeBase,
                                                     uint32_t nodes, uint64_t wordsPerNode,
                                                     const uint32_t* __restrict__ tileList,
                                                     const uint32_t* __restrict__ segTile,
                                                     const uint32_t* __restrict__ segCount,
                                                     const uint32_t* __restrict__ segSrc,
                                                     const uint32_t* __restrict__ segInput,
                                                     const NodeGrid* __restrict__ nodeGrid,
                                                     const uint32_t* __restrict__ bitmap,
                                                     const uint32_t* __restrict__ prefix,
                                                     uint32_t* __restrict__ cellOf, PointStore<T> ps,
                                                     uint64_t* __restrict__ win,
                                                     uint64_t* __restrict__ color, uint32_t* __restrict__ cellCnt,
                                                     uint32_t* __restrict__ cellKey, uint32_t* __restrict__ cellNode,
                                                     uint32_t* __restrict__ rankOf, uint32_t* __restrict__ pointCount,
                                                     uint32_t* __restrict__ stage, uint32_t* __restrict__ subtree,
                                                     const uint8_t* __restrict__ flags,
                                                     const int32_t* __restrict__ children, uint32_t* __restrict__ err)
{
    if (!accumulateNodes(step, nodeBase, nodes, wordsPerNode, nodeGrid, prefix, pointCount, stage, subtree, flags,
                         children, err))
        return;
    if (blockIdx.x < range.count())
        accumulateTile<T, MODE, RANDOM>(range.first() + blockIdx.x, nodeBase, wordsPerNode, tileList, segTile,
                                        segCount, segSrc, segInput, nodeGrid, bitmap, prefix, cellOf, ps, win, color,
                                        cellCnt, cellKey, cellNode, rankOf);
}

// A large tile's points per cell: the cells that the tile owns get their state from it.
template <uint32_t MODE>
struct CellTable
{
    static constexpr bool WEIGHTED = MODE == COLOR_INTER_WEIGHTED;
    static constexpr bool COLOR    = MODE == COLOR_INTRA || MODE == COLOR_INTER;
    unsigned long long cells[TABLE_SLOTS];
    unsigned long long color[COLOR ? LARGE_TILE : 0];
    uint32_t value[LARGE_TILE];  // least rank; points
};

template <typename T, uint32_t MODE, bool RANDOM>
static __global__ __launch_bounds__(LARGE_THREADS) void kAccumulateLarge(
        TileRange range, StepSizes step, uint32_t nodeBase, uint32_t nodes, uint64_t wordsPerNode,
        const uint32_t* __restrict__ tileList, const uint32_t* __restrict__ segTile,
        const uint32_t* __restrict__ segCount, const uint32_t* __restrict__ segSrc,
        const uint32_t* __restrict__ segInput, const NodeGrid* __restrict__ nodeGrid,
        const uint32_t* __restrict__ bitmap, const uint32_t* __restrict__ prefix, uint32_t* __restrict__ cellOf,
        PointStore<T> ps, uint64_t* __restrict__ win, uint64_t* __restrict__ color, uint32_t* __restrict__ cellCnt,
        uint32_t* __restrict__ cellKey, uint32_t* __restrict__ cellNode, uint32_t* __restrict__ rankOf,
        uint32_t* __restrict__ pointCount, uint32_t* __restrict__ stage, uint32_t* __restrict__ subtree,
        const uint8_t* __restrict__ flags, const int32_t* __restrict__ children, uint32_t* __restrict__ err)
{
    using Table = CellTable<MODE>;
    __shared__ Table table;
    if (!accumulateNodes(step, nodeBase, nodes, wordsPerNode, nodeGrid, prefix, pointCount, stage, subtree, flags,
                         children, err))
        return;
    if (blockIdx.x >= range.count())
        return;  // the whole workgroup
    const LargeTile in  = largeTile(range.first() + blockIdx.x, tileList, segTile, segCount, segSrc, segInput);
    const uint32_t kl   = in.k - nodeBase;
    const uint64_t base = kl * wordsPerNode;
    uint32_t cell[LARGE_ITEMS], c[LARGE_ITEMS], idx[LARGE_ITEMS];
    uint64_t col[LARGE_ITEMS];
#pragma unroll
    for (int i = 0; i < LARGE_ITEMS; ++i)
    {
        cell[i] = in.has(i) ? cellOf[in.q + in.at(i)] : ~0u;
        if (!Table::WEIGHTED && in.has(i))
        {
            idx[i] = ps.index(in.pos + in.at(i));
            if (Table::COLOR)
                col[i] = ps.packed(in.pos + in.at(i));
        }
    }
#pragma unroll
    for (int i = 0; i < LARGE_ITEMS; ++i)
        if ((cell[i] & NOT_OWNED) == 0)
            c[i] = cellRank(bitmap, prefix, base + (cell[i] >> 5), cell[i] & 31);
    for (uint32_t s = threadIdx.x; s < TABLE_SLOTS; s += LARGE_THREADS)
        table.cells[s] = TABLE_FREE;
    for (uint32_t s = threadIdx.x; s < LARGE_TILE; s += LARGE_THREADS)
    {
        table.value[s] = Table::WEIGHTED ? 0u : ~0u;
        if (Table::COLOR)
            table.color[s] = 0;
    }
    const uint32_t salt = RANDOM && !Table::WEIGHTED ? nodeGrid[in.k].salt : 0u;
    __syncthreads();
    uint32_t slot[LARGE_ITEMS], rank[LARGE_ITEMS];
    bool created[LARGE_ITEMS];
#pragma unroll
    for (int i = 0; i < LARGE_ITEMS; ++i)
    {
        created[i] = false;
        if (cell[i] & NOT_OWNED)
            continue;
        slot[i]    = tableInput(table.cells, c[i], in.at(i));
        created[i] = slot[i] == in.at(i);
        if (Table::WEIGHTED)
        {
            // the winner is taken from the cell's payload run in the emit; the input's cell index is
            // replaced by the cell's dense index (the payload scatter reads the cell back from cellKey)
            cellOf[in.q + in.at(i)] = c[i];
            rankOf[in.q + in.at(i)] = atomicAdd(table.value + slot[i], 1u);
            continue;
        }
        rank[i] = RANDOM ? fmix32(idx[i] ^ salt) : idx[i];
        atomicMin(table.value + slot[i], rank[i]);
        if (Table::COLOR)
            atomicAdd(table.color + slot[i], static_cast<unsigned long long>(col[i]));
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < LARGE_ITEMS; ++i)
    {
        if (created[i])
        {
            cellKey[c[i]]  = cell[i];
            cellNode[c[i]] = kl;
            if (Table::WEIGHTED)
                cellCnt[c[i]] = table.value[slot[i]];
            if (Table::COLOR)
                color[c[i]] = table.color[slot[i]];
        }
        // the winner itself: no two points have the same rank
        if (!Table::WEIGHTED && (cell[i] & NOT_OWNED) == 0 && table.value[slot[i]] == rank[i])
            win[c[i]] = (static_cast<uint64_t>(rank[i]) << 32) | (in.pos + in.at(i));
    }
}

// The inputs in cells that another tile owns, after kAccumulateLarge: one atomic per run of lanes.
template <typename T, uint32_t MODE, bool RANDOM>
static __global__ __launch_bounds__(LARGE_THREADS) void kAccumulateRest(
        TileRange range, StepSizes step, uint32_t nodeBase, uint64_t wordsPerNode,
        const uint32_t* __restrict__ tileList, const uint32_t* __restrict__ segTile,
        const uint32_t* __restrict__ segCount, const uint32_t* __restrict__ segSrc,
        const uint32_t* __restrict__ segInput, const NodeGrid* __restrict__ nodeGrid,
        const uint32_t* __restrict__ bitmap, const uint32_t* __restrict__ prefix, uint32_t* __restrict__ cellOf,
        PointStore<T> ps, uint64_t* __restrict__ win, uint64_t* __restrict__ color, uint32_t* __restrict__ cellCnt,
        uint32_t* __restrict__ rankOf)
{
    if (!step.fits() || blockIdx.x >= range.count())
        return;
    const LargeTile in  = largeTile(range.first() + blockIdx.x, tileList, segTile, segCount, segSrc, segInput);
    const uint64_t base = (in.k - nodeBase) * wordsPerNode;
    uint32_t cells[LARGE_ITEMS];
#pragma unroll
    for (int i = 0; i < LARGE_ITEMS; ++i)
        cells[i] = in.has(i) ? cellOf[in.q + in.at(i)] : ~0u;
#pragma unroll
    for (int i = 0; i < LARGE_ITEMS; ++i)
    {
        const bool rest = (cells[i] & NOT_OWNED) != 0 && cells[i] != ~0u;
        if (!__any(rest))
            continue;  // the whole wave
        const uint32_t cell = cells[i] & ~NOT_OWNED;
        const uint32_t c    = rest ? cellRank(bitmap, prefix, base + (cell >> 5), cell & 31) : 0u;
        const WaveRun run   = waveRun(rest ? c : ~0ull - threadIdx.x);
        const bool last     = rest && run.lane == run.end;
        if (MODE == COLOR_INTER_WEIGHTED)
        {
            uint32_t first = 0;
            if (last)
                first = atomicAdd(cellCnt + c, static_cast<uint32_t>(run.end - run.start + 1));
            first = __shfl(first, run.end, 64);
            if (rest)
            {
                cellOf[in.q + in.at(i)] = c;
                rankOf[in.q + in.at(i)] = first + static_cast<uint32_t>(run.lane - run.start);
            }
            continue;
        }
        uint64_t key = ~0ull, col = 0;
        if (rest)
        {
            const uint32_t idx  = ps.index(in.pos + in.at(i));
            const uint32_t rank = RANDOM ? fmix32(idx ^ nodeGrid[in.k].salt) : idx;
            key                 = (static_cast<uint64_t>(rank) << 32) | (in.pos + in.at(i));
            if (MODE == COLOR_INTRA || MODE == COLOR_INTER)
                col = ps.packed(in.pos + in.at(i));
        }
        key = runScan<uint64_t>(key, run, [](uint64_t x, uint64_t y) { return x < y ? x : y; });
        if (MODE == COLOR_INTRA || MODE == COLOR_INTER)
            col = runScan<uint64_t>(col, run, [](uint64_t x, uint64_t y) { return x + y; });
        if (last)
        {
            atomicMin(reinterpret_cast<unsigned long long*>(win + c), static_cast<unsigned long long>(key));
            if (MODE == COLOR_INTRA || MODE == COLOR_INTER)
                atomicAdd(reinterpret_cast<unsigned long long*>(color + c), static_cast<unsigned long long>(col));
        }
    }
}

// exclusive prefix into an array, with the total behind it
struct ExclusiveWithTotal
{
    uint32_t* dst;
    const uint32_t* n;
    __device__ void operator()(uint64_t i, uint32_t prefix, uint32_t v) const
    {
        dst[i] = prefix;
        if (i + 1 == *n)
            dst[i + 1] = prefix + v;
    }
};

// Per-point data of the weighted filter, in cell order so that a cell's points are one contiguous
// run (cellStart[cell] + arrival rank), in two arrays:
//   WeightPayload: the point's offset from its own cell's centre, (p - centre) rounded to float,
//     and its colour r | g << 8 | b << 16 with the cell's x coordinate mod 4 in bits 24-25 (a
//     neighbour's x differs from the selecting cell's by -1, 0 or 1, which x mod 4 identifies).
//     16 bytes: the select's loop reads one record per lane from lines that differ between lanes,
//     and every load instruction costs the memory pipeline a pass per line touched.
//   winner key: rank << 32 | source position, the rank being the point index (implicit method) or
//     its hash (explicit). Ranks are bijective, so the minimum key of a cell names its winner.
struct alignas(16) WeightPayload
{
    float ox, oy, oz;
    uint32_t rgbx;
};
static_assert(sizeof(WeightPayload) == 16, "weighted payload is one 16-byte load");

// Centre of cell (ix, iy, iz) of a node grid, in the select's expression order (min + i t + t / 2).
__device__ __forceinline__ void cellCentre(const Gridding& g, uint32_t ix, uint32_t iy, uint32_t iz, double& x,
                                           double& y, double& z)
{
    const double t = g.bbSize / g.gridSize;
    x              = g.minX + ix * t + (t * 0.5);
    y              = g.minY + iy * t + (t * 0.5);
    z              = g.minZ + iz * t + (t * 0.5);
}

template <typename T, bool RANDOM>
__device__ __forceinline__ void scatterPayloadTile(uint32_t tile, uint32_t g, const uint32_t* __restrict__ tileList,
                                                   const uint32_t* __restrict__ segTile,
                                                   const uint32_t* __restrict__ segCount,
                                                   const uint32_t* __restrict__ segSrc,
                                                   const uint32_t* __restrict__ segInput,
                                                   const NodeGrid* __restrict__ nodeGrid,
                                                   const uint32_t* __restrict__ cellKey,
                                                   const uint32_t* __restrict__ rankOf,
                                                   const uint32_t* __restrict__ cellStart,
                                                   const uint32_t* __restrict__ cellOf, const PointStore<T>& ps,
                                                   WeightPayload* __restrict__ payload, uint64_t* __restrict__ winKey,
                                                   uint32_t parts = 1)
{
    InputRef in = inputOf(tile, tileList, segTile, segCount, segSrc, segInput, parts);
    if (!in.valid)
        return;
    const uint32_t c = cellOf[in.q];  // the dense index kAccumulate left there
    if (c == ~0u)
        return;
    const uint32_t cell = cellKey[c];
    const NodeGrid ng   = nodeGrid[in.k];
    uint32_t ix, iy, iz;
    cellCoords(cell, g, ix, iy, iz);
    double cx, cy, cz;
    cellCentre(ng.grid, ix, iy, iz, cx, cy, cz);
    T px, py, pz;
    ps.xyz(in.pos, px, py, pz);
    WeightPayload pl;
    pl.ox   = static_cast<float>(static_cast<double>(px) - cx);
    pl.oy   = static_cast<float>(static_cast<double>(py) - cy);
    pl.oz   = static_cast<float>(static_cast<double>(pz) - cz);
    pl.rgbx = ps.rgb(in.pos) | ((ix & 3u) << 24);
    const uint32_t idx  = ps.index(in.pos);
    const uint32_t rank = RANDOM ? fmix32(idx ^ ng.salt) : idx;
    const uint32_t slot = cellStart[c] + rankOf[in.q];
    payload[slot]       = pl;
    winKey[slot]        = (static_cast<uint64_t>(rank) << 32) | in.pos;
}

template <typename T, bool RANDOM>
static __global__ __launch_bounds__(TILE) void kScatterPayload(TileRange range, StepSizes step, uint32_t g,
                                                         const uint32_t* __restrict__ tileList,
                                                         const uint32_t* __restrict__ segTile,
                                                         const uint32_t* __restrict__ segCount,
                                                         const uint32_t* __restrict__ segSrc,
                                                         const uint32_t* __restrict__ segInput,
                                                         const NodeGrid* __restrict__ nodeGrid,
                                                         const uint32_t* __restrict__ cellKey,
                                                         const uint32_t* __restrict__ rankOf,
                                                         const uint32_t* __restrict__ cellStart,
                                                         const uint32_t* __restrict__ cellOf, PointStore<T> ps,
                                                         WeightPayload* __restrict__ payload,
                                                         uint64_t* __restrict__ winKey, uint32_t parts,
                                                         uint64_t* stamp)
{
    stampStart(stamp);
    if (!step.fits())
        return;
    // consecutive tiles store to neighbouring payload slots: runs of them per XCD
    const uint32_t t = xcdRunItem(blockIdx.x, XCD_TILE_RUN);
    if (t < range.count() * parts)
        scatterPayloadTile<T, RANDOM>(range.first() * parts + t, g, tileList, segTile, segCount, segSrc, segInput, nodeGrid,
                                      cellKey, rankOf, cellStart, cellOf, ps, payload, winKey, parts);
}

// Select (rp_subsampling.cuh:70-321, fp_subsampling.cuh:30-306): one point per occupied
// cell, written to staging at its dense index (node by node, cells ascending). The point keeps the
// winner's position; the colour is the winner's (no filter), the decoded intra
// sum, or the decoded sum of the per-cell sums over the 3x3x3 neighbourhood (inter; equal to the
// reference's per-point scatter into occupied neighbours because integer sums commute). The
// neighbourhood is walked as 9 x-rows: the occupied cells among x-1..x+1 of one row have
// consecutive dense indices, so each row is one contiguous run of per-cell sums.
template <typename T, uint32_t MODE>
__device__ __forceinline__ void emitCell(uint32_t c, uint64_t wordsPerNode, uint32_t cursor, uint32_t g,
                                         const uint32_t* __restrict__ bitmap,
                                         const uint32_t* __restrict__ prefix, const uint32_t* __restrict__ cellKey,
                                         const uint32_t* __restrict__ cellNode, const uint64_t* __restrict__ win,
                                         const uint64_t* __restrict__ color, const PointStore<T>& ps)
{
    {
        uint64_t sum = 0;  // packed colours

        if (MODE == COLOR_INTRA)
            sum = color[c];
        else if (MODE == COLOR_INTER)
        {
            const uint64_t words = cellNode[c] * wordsPerNode;
            uint32_t cx, cy, cz;
            cellCoords(cellKey[c], g, cx, cy, cz);
            const uint32_t x0 = cx > 0 ? cx - 1 : 0;
            const uint32_t x1 = cx + 1 < g ? cx + 1 : cx;
            const uint32_t span = x1 - x0 + 1;
            const CellRows rows(cy, cz, g);
            const uint32_t *nodeBits = bitmap + words, *nodePrefix = prefix + words;
#pragma unroll
            for (int r = 0; r < 9; ++r)
            {
                if (!rows.has(r))
                    continue;
                const RowRun run = rowRun(nodeBits, nodePrefix, rows.start(r) + x0, span);
                // at most 3 occupied cells (x - 1 .. x + 1): predicated loads, no loop, so the
                // rows' loads are all in flight together
                const uint32_t n = run.count, first = run.first;
                if (n > 0)
                    sum += color[first];
                if (n > 1)
                    sum += color[first + 1];
                if (n > 2)
                    sum += color[first + 2];
            }
        }
        const uint32_t wpos = static_cast<uint32_t>(win[c] & 0xFFFFFFFFull);
        const uint32_t st   = cursor - ps.N + c;  // staging index
        if (MODE == COLOR_NONE)
            ps.staged.rgb[st] = ps.rgb(wpos);
        else
        {
            uint16_t r, g, b;
            decodeColors(sum, r, g, b);
            ps.staged.packed[st] = encodeColors(r, g, b);
        }
        ps.stLut[st] = ps.index(wpos);
        T* d         = ps.stPts + 3 * static_cast<uint64_t>(st);
        ps.xyz(wpos, d[0], d[1], d[2]);
    }
}

template <typename T, uint32_t MODE>
static __global__ __launch_bounds__(BLOCK) void kEmit(StepSizes step, uint64_t wordsPerNode, uint32_t g,
                                                const uint32_t* __restrict__ bitmap,
                                                const uint32_t* __restrict__ prefix,
                                                const uint32_t* __restrict__ cellKey,
                                                const uint32_t* __restrict__ cellNode,
                                                const uint64_t* __restrict__ win, const uint64_t* __restrict__ color,
                                                PointStore<T> ps, uint64_t* insertEnd, uint64_t* stamp)
{
    stampStart(insertEnd);
    stampStart(stamp);
    if (!step.fits())
        return;
    const uint32_t cells = *step.cells, cursor = static_cast<uint32_t>(*step.cursor);
    for (uint64_t ci = globalThread(); ci < cells; ci += globalStride())
        emitCell<T, MODE>(static_cast<uint32_t>(ci), wordsPerNode, cursor, g, bitmap, prefix, cellKey, cellNode, win, color,
                          ps);
}

// Select with the distance-weighted inter-cell filter (kernel_inter_cell_filtering.cuh:109-194,
// weighted decode rp_subsampling.cuh:222-230): the gathered average over the points of the 3x3x3
// neighbourhood, with the weight of a point p for this cell c
//   res = float(sqrt(|centre(c) - p|^2) / diag);  w = expf(-(res * res) * 10)
// and colour u16(sum c w / sum w). One thread per cell; the winner is the minimum key of the
// cell's own run, its exact coordinates and index read back through the key's source position.
// The neighbourhood is walked as 9 x-rows, each one contiguous run of payloads. With the point in
// neighbour cell m = c + d (d in {-1, 0, 1}^3) and its offset o from m's centre,
//   centre(c) - p = -d t - o,
// evaluated in float, and w = 2^(|centre(c) - p|^2 * (-10 log2(e) / diag^2)), which is the same
// function as the reference's expression. The float evaluation moves a weight by a few parts in
// 10^6, so a channel can differ by one where the average lies that close to an integer, the
// same tolerance the float sums' order dependence already needs (the reference adds with
// atomics). WEIGHT_LOADS records per step, their loads in flight before any is weighed.
constexpr uint32_t WEIGHT_LOADS = 4;
constexpr uint32_t WEIGHT_LDS   = 9 * BLOCK;  // run bounds of a workgroup's cells

template <typename T>
__device__ __forceinline__ void emitWeightedCell(uint32_t c, uint32_t nodeBase, uint64_t wordsPerNode,
                                                 uint32_t cursor, uint32_t g, const NodeGrid* __restrict__ nodeGrid,
                                                 const uint32_t* __restrict__ bitmap,
                                                 const uint32_t* __restrict__ prefix,
                                                 const uint32_t* __restrict__ cellKey,
                                                 const uint32_t* __restrict__ cellNode,
                                                 const uint32_t* __restrict__ cellStart,
                                                 const WeightPayload* __restrict__ payload,
                                                 const uint64_t* __restrict__ winKey, const PointStore<T>& ps,
                                                 uint2* lds)
{
    const uint32_t kl    = cellNode[c];
    const float tf       = nodeGrid[nodeBase + kl].cell;
    const float kexp     = nodeGrid[nodeBase + kl].weight;
    const uint64_t words = kl * wordsPerNode;
    uint32_t cx, cy, cz;
    cellCoords(cellKey[c], g, cx, cy, cz);
    const uint32_t x0 = cx > 0 ? cx - 1 : 0;
    const uint32_t x1 = cx + 1 < g ? cx + 1 : cx;
    const uint32_t span = x1 - x0 + 1;
    const CellRows rows(cy, cz, g);
    const uint32_t *nodeBits = bitmap + words, *nodePrefix = prefix + words;

    // first dense index and number of occupied cells of every row
    uint32_t first[9], count[9];
#pragma unroll
    for (int r = 0; r < 9; ++r)
    {
        count[r] = 0;
        first[r] = 0;
        if (!rows.has(r))
            continue;
        const RowRun run = rowRun(nodeBits, nodePrefix, rows.start(r) + x0, span);
        count[r]         = run.count;
        first[r]         = run.first;
    }
    // the payload runs of the non-empty rows, in order, through LDS: the loop below takes them by number
    uint32_t lo[9], hi[9];
#pragma unroll
    for (int r = 0; r < 9; ++r)
    {
        lo[r] = count[r] ? cellStart[first[r]] : 0;
        hi[r] = count[r] ? cellStart[first[r] + count[r]] : 0;
    }
    uint32_t points = 0, runs = 0;
    uint64_t steps  = 0;  // d.y + 1 and d.z + 1 of every run, two bits each
#pragma unroll
    for (int r = 0; r < 9; ++r)
        if (hi[r] > lo[r])
        {
            lds[runs * BLOCK + threadIdx.x] = make_uint2(lo[r], hi[r]);
            steps |= static_cast<uint64_t>(r / 3 | (r % 3) << 2) << (4 * runs);
            points += hi[r] - lo[r];
            ++runs;
        }

    // the winner: minimum key of the cell's own run
    uint64_t best = ~0ull;
    for (uint32_t q = cellStart[c], e = cellStart[c + 1]; q < e; ++q)
    {
        const uint64_t k = winKey[q];
        best             = k < best ? k : best;
    }
    const uint32_t wpos = static_cast<uint32_t>(best);
    T bx, by, bz;
    ps.xyz(wpos, bx, by, bz);
    const uint32_t bestIdx = ps.index(wpos);

    const uint32_t cxm = (cx + 3u) & 3u;  // (c.x - 1) mod 4: d.x = ((m.x - cxm) & 3) - 1
    float acc[4]       = {0.f, 0.f, 0.f, 0.f};
    // payloads as 16-byte vectors (they stay in registers under conditional loads)
    const uint4* pv = reinterpret_cast<const uint4*>(payload);
    auto weigh      = [&](const uint4& pl, float uyc, float uzc) {
        const int32_t dx = static_cast<int32_t>(((pl.w >> 24) + 4u - cxm) & 3u) - 1;
        const float ux   = __builtin_fmaf(-static_cast<float>(dx), tf, -__uint_as_float(pl.x));
        const float uy   = uyc - __uint_as_float(pl.y);
        const float uz   = uzc - __uint_as_float(pl.z);
        float d2         = ux * ux;
        d2               = __builtin_fmaf(uy, uy, d2);
        d2               = __builtin_fmaf(uz, uz, d2);
        const float w    = __builtin_amdgcn_exp2f(d2 * kexp);
        acc[0]           = __builtin_fmaf(static_cast<float>(pl.w & 0xFF), w, acc[0]);
        acc[1]           = __builtin_fmaf(static_cast<float>((pl.w >> 8) & 0xFF), w, acc[1]);
        acc[2]           = __builtin_fmaf(static_cast<float>((pl.w >> 16) & 0xFF), w, acc[2]);
        acc[3] += w;
    };
    // Every lane walks its own runs one after the other, WEIGHT_LOADS payloads in flight: a wave then
    // takes as many steps as its fullest neighbourhood has points, and not in every one of the nine rows
    // as many as the fullest of that row (119.7M points: 75 payload loads a wave -> 45, 11.1 -> 10.8 ms; two
    // or three in flight 11.5 ms). Lanes that are all well inside a run take its next payloads without
    // looking for its end: the last lanes around a cell that holds a good part of the cloud walk nothing else
    // (three quarters of 5M points in one cell: 842 -> 705 ms, row by row 744; 119.7M points 30.9 / 30.4 ms).
    uint32_t run = 0, q = 0, e = 0;
    float uyc = 0.f, uzc = 0.f;
    while (points > 0)
    {
        uint4 pl[WEIGHT_LOADS];
        if (__all(e - q >= WEIGHT_LOADS))
        {
#pragma unroll
            for (uint32_t k = 0; k < WEIGHT_LOADS; ++k)
                pl[k] = pv[q + k];
#pragma unroll
            for (uint32_t k = 0; k < WEIGHT_LOADS; ++k)
                weigh(pl[k], uyc, uzc);
            q += WEIGHT_LOADS;
            points -= WEIGHT_LOADS;
            continue;
        }
        float uy[WEIGHT_LOADS], uz[WEIGHT_LOADS];
#pragma unroll
        for (uint32_t k = 0; k < WEIGHT_LOADS; ++k)
            if (k < points)
            {
                if (q == e)
                {
                    const uint2 range = lds[run * BLOCK + threadIdx.x];
                    const uint32_t d  = static_cast<uint32_t>(steps >> (4 * run));
                    q                 = range.x;
                    e                 = range.y;
                    uyc               = (1.f - static_cast<float>(d & 3u)) * tf;         // -d.y t
                    uzc               = (1.f - static_cast<float>((d >> 2) & 3u)) * tf;  // -d.z t
                    ++run;
                }
                pl[k] = pv[q++];
                uy[k] = uyc;
                uz[k] = uzc;
            }
#pragma unroll
        for (uint32_t k = 0; k < WEIGHT_LOADS; ++k)
            if (k < points)
                weigh(pl[k], uy[k], uz[k]);
        points -= points < WEIGHT_LOADS ? points : WEIGHT_LOADS;
    }
    // the colour (averages of 8-bit channels: at most 255); the record itself is quantised from
    // the staged coordinates by the final placement (kPermute)
    const uint32_t cr = static_cast<uint16_t>(acc[0] / acc[3]);
    const uint32_t cg = static_cast<uint16_t>(acc[1] / acc[3]);
    const uint32_t cb = static_cast<uint16_t>(acc[2] / acc[3]);
    const uint32_t st = cursor - ps.N + c;  // staging index
    ps.stLut[st] = bestIdx;
    ps.staged.rgb[st] = (cr & 0xFF) | ((cg & 0xFF) << 8) | ((cb & 0xFF) << 16);
    T* d         = ps.stPts + 3 * static_cast<uint64_t>(st);
    d[0]         = bx;
    d[1]         = by;
    d[2]         = bz;
}

template <typename T>
static __global__ __launch_bounds__(BLOCK) void kEmitWeighted(StepSizes step, uint32_t nodeBase, uint64_t wordsPerNode,
                                                        uint32_t g,
                                                        const NodeGrid* __restrict__ nodeGrid,
                                                        const uint32_t* __restrict__ bitmap,
                                                        const uint32_t* __restrict__ prefix,
                                                        const uint32_t* __restrict__ cellKey,
                                                        const uint32_t* __restrict__ cellNode,
                                                        const uint32_t* __restrict__ cellStart,
                                                        const WeightPayload* __restrict__ payload,
                                                        const uint64_t* __restrict__ winKey, PointStore<T> ps,
                                                        uint64_t* stamp)
{
    __shared__ uint2 lds[WEIGHT_LDS];
    stampStart(stamp);
    if (!step.fits())
        return;
    // each XCD takes runs of EMIT_CHUNK consecutive cell blocks
    const uint64_t c = static_cast<uint64_t>(xcdRunItem(blockIdx.x, EMIT_CHUNK)) * BLOCK + threadIdx.x;
    if (c < *step.cells)
        emitWeightedCell<T>(static_cast<uint32_t>(c), nodeBase, wordsPerNode, static_cast<uint32_t>(*step.cursor),
                            g, nodeGrid, bitmap, prefix, cellKey, cellNode, cellStart, payload, winKey, ps, lds);
}

// DFS post-order placement (A6, kernel_helpers.cuh:55-59): subtree sums of subsample sizes
// bottom-up (with the levels), then region starts: an internal node's data follows its children's
// subtrees: dataIdx = N + regionStart + sum of its children's subtree sizes.
__device__ __forceinline__ void regionOf(uint32_t id, uint32_t root, uint32_t N, const uint8_t* __restrict__ flags,
                                         const int32_t* __restrict__ children, const uint32_t* __restrict__ subtree,
                                         uint32_t* __restrict__ region, uint64_t* __restrict__ dataIdx)
{
    if (!(flags[id] & NODE_INTERNAL))
        return;
    uint32_t r = (id == root) ? 0u : region[id];
    for (int k = 0; k < 8; ++k)
    {
        const int32_t c = children[8 * static_cast<uint64_t>(id) + k];
        if (c >= 0)
        {
            region[c] = r;
            r += subtree[c];
        }
    }
    dataIdx[id] = static_cast<uint64_t>(N) + r;
}

// Placement of the subsampled records: the staged records of an internal node are one contiguous
// range, and so is its final range [dataIdx, dataIdx + pointCount), so every (node, chunk of
// PLACE_CHUNK records) work item is a contiguous copy. A workgroup takes a chunk in steps that wait for
// their loads: 4096 records a chunk were 16 of them (50K points 13.4 -> 7.2 us, 1.5M 22 -> 13.8, 25.8M
// 353 -> 327).
constexpr uint32_t PLACE_CHUNK = 1024;

// Single cloud: every internal node of the list on its own, its region from the subtrees of the
// lower-slot siblings on its way up. No level waits for another (one workgroup going down level by
// level took 105 us for 6600 nodes). Its chunks go to the work list in no particular order.
static __global__ __launch_bounds__(64) void kPlaceNodes(const uint32_t* __restrict__ list, uint32_t nodes, uint32_t N,
                                                   const int32_t* __restrict__ parent,
                                                   const int32_t* __restrict__ children,
                                                   const uint32_t* __restrict__ pointCount,
                                                   const uint32_t* __restrict__ subtree, uint64_t* __restrict__ dataIdx,
                                                   uint64_t* __restrict__ chunkList, uint32_t* __restrict__ chunks,
                                                   uint64_t* stamp)
{
    stampStart(stamp);
    for (uint64_t j = globalThread(); j < nodes; j += globalStride())
    {
        const uint32_t id = list[j];
        uint32_t before   = subtree[id] - pointCount[id];  // its children's subtrees
        int32_t cur       = static_cast<int32_t>(id);
        for (int32_t p = parent[cur]; p >= 0; cur = p, p = parent[cur])
        {
            int32_t c[8];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                c[k] = children[8 * static_cast<uint64_t>(p) + k];
            bool lower = true;  // slots before cur's
#pragma unroll
            for (int k = 0; k < 8; ++k)
            {
                lower = lower && c[k] != cur;
                if (lower && c[k] >= 0)
                    before += subtree[c[k]];
            }
        }
        dataIdx[id]       = static_cast<uint64_t>(N) + before;
        const uint32_t n  = (pointCount[id] + PLACE_CHUNK - 1) / PLACE_CHUNK;
        const uint32_t at = atomicAdd(chunks, n);
        for (uint32_t k = 0; k < n; ++k)
            chunkList[at + k] = (static_cast<uint64_t>(k) << 32) | id;
    }
}

// chunks of an internal node's placement
struct PlacedChunksIn
{
    const uint8_t* flags;
    const uint32_t* pointCount;
    __device__ uint32_t operator()(uint64_t i) const
    {
        return (flags[i] & NODE_INTERNAL) ? (pointCount[i] + PLACE_CHUNK - 1) / PLACE_CHUNK : 0u;
    }
};

template <typename T>
__device__ __forceinline__ void permuteChunk(uint64_t entry, uint32_t N, const uint32_t* __restrict__ stage,
                                             const uint64_t* __restrict__ dataIdx,
                                             const uint32_t* __restrict__ pointCount,
                                             const uint32_t* __restrict__ stLut, const T* __restrict__ stPts,
                                             const StagedColors& staged, const Gridding& cubic, double sx, double sy, double sz,
                                             uint32_t* __restrict__ lut, OutRecord* __restrict__ out, OutStage& lds)
{
    const uint32_t id    = static_cast<uint32_t>(entry);
    const uint32_t first = static_cast<uint32_t>(entry >> 32) * PLACE_CHUNK;
    const uint32_t total = pointCount[id];
    const uint32_t cnt   = total - first < PLACE_CHUNK ? total - first : PLACE_CHUNK;
    const uint64_t src   = static_cast<uint64_t>(stage[id]) - N + first;  // staging index of the chunk
    const uint64_t dst   = dataIdx[id] + first;
    const uint32_t lane  = threadIdx.x & 63;
    for (uint32_t base = threadIdx.x - lane; base < cnt; base += BLOCK)
    {
        const uint32_t count = cnt - base < 64 ? cnt - base : 64u;
        OutRecord r{};
        if (lane < count)
        {
            const uint64_t s     = src + base + lane;
            lut[dst + base + lane] = stLut[s];
            const T* q           = stPts + 3 * s;
            r                    = quantizePoint(q[0], q[1], q[2], staged.rgb ? staged.rgb[s] : 0u, cubic, sx, sy, sz);
            if (staged.packed)
            {
                const uint64_t c = staged.packed[s];
                r.r              = static_cast<uint16_t>(c >> 46);
                r.g              = static_cast<uint16_t>(c >> 28);
                r.b              = static_cast<uint16_t>(c >> 10);
            }
        }
        storeRecords(out + dst + base, r, count, lds);
    }
}

template <typename T>
static __global__ __launch_bounds__(BLOCK) void kPermute(const uint64_t* __restrict__ chunkList,
                                                   const uint32_t* __restrict__ chunks, uint32_t N,
                                                   const uint32_t* __restrict__ stage,
                                                   const uint64_t* __restrict__ dataIdx,
                                                   const uint32_t* __restrict__ pointCount,
                                                   const uint32_t* __restrict__ stLut,
                                                   const T* __restrict__ stPts, StagedColors staged, Gridding cubic,
                                                   double sx, double sy, double sz, uint32_t* __restrict__ lut,
                                                   OutRecord* __restrict__ out)
{
    __shared__ OutStage lds[BLOCK / 64];
    const uint32_t all = *chunks;
    for (uint32_t c = blockIdx.x; c < all; c += gridDim.x)
        permuteChunk<T>(chunkList[c], N, stage, dataIdx, pointCount, stLut, stPts, staged, cubic, sx, sy, sz, lut, out,
                        lds[threadIdx.x >> 6]);
}

}  // namespace oc
