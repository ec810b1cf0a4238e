// Level-batched LOD octree build on one MI355X (gfx950). See builder.h for the phase overview.
//
// Data layout in HBM (per session):
//   cloud          N x S bytes, packed AoS records (15 or 27 bytes), read twice (bucket
//                  histogram, bucket scatter)
//   bucketed       N sorted-point records (32 bytes for double clouds, 20 for float) grouped by
//                  coarse bucket, plus a u16 fine code per point
//   sorted         the same records in level-0 Morton order: every node is one contiguous range;
//                  the leaves' points are read from here by the subsampling
//   count          D x u32 dense count pyramid; after the merge its level-0 part maps cell -> leaf
//   occupancy, id base  a bit per dense cell, a u32 per 32 cells: dense cell -> sparse id
//   nodes (SoA)    key, dense count, pointCount, dataIdx (u64), parent, children[8], flags, ...
//   output region  E records: lut (u32 point index), out (18-byte record). [0, N) holds the leaves,
//                  [N, N + I) the subsampled points in DFS post-order
//   staging        subsampled points in level order (index, coordinates, colour), read by the
//                  next level; their records go to the output region at the end
#include "builder.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <stdexcept>
#include <string>

#include "device_common.h"
#include "host_staging.h"
#include "kernels_chunking.h"
#include "kernels_sort.h"
#include "kernels_subsample.h"
#include "scan.h"

namespace oc {

#define OC_HIP_CHECK(expr)                                                                                             \
    do                                                                                                                 \
    {                                                                                                                  \
        hipError_t e_ = (expr);                                                                                        \
        if (e_ != hipSuccess)                                                                                          \
            throw std::runtime_error(std::string(#expr) + " failed: " + hipGetErrorString(e_));                      \
    } while (0)

#define OC_LAUNCH_CHECK() OC_HIP_CHECK(hipGetLastError())

// ------------------------------------------------------------------------------------------------
// Device arena
// ------------------------------------------------------------------------------------------------

static std::atomic<size_t> gAllocated{0};
static std::atomic<size_t> gPeak{0};

DeviceBuffer::~DeviceBuffer()
{
    release();
}

void DeviceBuffer::release()
{
    if (itsPtr)
    {
        (void)hipFree(itsPtr);
        gAllocated -= itsBytes;
    }
    itsPtr   = nullptr;
    itsBytes = 0;
}

void DeviceBuffer::ensure(size_t bytes)
{
    if (bytes <= itsBytes)
        return;
    release();
    size_t rounded = (bytes + 255) & ~size_t(255);
    void* p        = nullptr;
    hipError_t e   = hipMalloc(&p, rounded);
    if (e != hipSuccess)
        throw std::runtime_error("hipMalloc of " + std::to_string(rounded) + " bytes failed: " + hipGetErrorString(e));
    itsPtr   = p;
    itsBytes = rounded;
    size_t now = (gAllocated += rounded);
    size_t peak = gPeak.load();
    while (now > peak && !gPeak.compare_exchange_weak(peak, now))
    {
    }
}

size_t DeviceBuffer::totalAllocated()
{
    return gAllocated.load();
}

size_t DeviceBuffer::peakAllocated()
{
    return gPeak.load();
}

// ------------------------------------------------------------------------------------------------
// Kernels
// ------------------------------------------------------------------------------------------------

// ------------------------------------------------------------------------------------------------
// Host orchestration
// ------------------------------------------------------------------------------------------------

// Bytes of bitmap + prefix the nodes of one subsampling batch may use.
static constexpr uint64_t kBitmapBudget = 6ull << 30;

// Bitmap words up to which a level's cells are reset with its bitmap, one per input (a launch less: 2M points
// at grids 256 / 64 904 us, 922 with a launch of its own). On larger levels there are many more inputs than
// cells; up to 3M points it makes no more than 2 % there, either way.
static constexpr uint64_t RESET_INPUTS_WORDS = 1u << 20;

// Points, and children of a level's nodes, from which the host reads a level's tiles and inputs back to size
// its launches (subsampleLevels). Points: 4M 1168 us with readbacks, 1129 without; 8M 1779 / 1747; 30M 5191
// / 5250, the weighted filter 9382 / 9545; 14M to 20M alike. Children (4M points, threshold 20, g = 8, 800K
// children on the lowest level): 10.7 ms with them, 11.3 without; 1M points 3.01 / 3.13; from 4096 children
// on instead of 131072 alike.
static constexpr uint32_t READ_INPUTS_POINTS   = 1u << 24;
static constexpr uint32_t READ_INPUTS_CHILDREN = 1u << 17;

// Points from which the arrays of a level's inputs and cells are sized by what the host reads back, as each
// level turns out (a readback more per step), instead of by the most that they can be: those bounds take up
// to 8 % of a build's memory (40M points, grids 64 / 32: 10.6 GB instead of 9.8), which matters where a
// build takes a good part of the card's 288 GB and costs nothing to speak of there.
static constexpr uint32_t EXACT_ARRAYS_POINTS = 1u << 27;
static_assert(EXACT_ARRAYS_POINTS >= READ_INPUTS_POINTS, "their levels' inputs are read back");

// words of the host mailbox
enum MailSlot
{
    MAIL_SEQ,
    MAIL_ERROR,
    MAIL_NODES,
    MAIL_INTERNAL,
    MAIL_USED,
    MAIL_LEVEL = 8,                        // first node of every level
    MAIL_INNER = MAIL_LEVEL + MAX_LEVELS,  // first internal node of every level
    MAIL_TICKS = MAIL_INNER + MAX_LEVELS,  // stage durations
    MAIL_STEPS = MAIL_TICKS + 7,           // tiles and inputs before a level's steps and after the last of them
    MAIL_TOTAL = MAIL_STEPS + 63,          // and of the whole level
    MAIL_WORDS
};
constexpr uint32_t PUBLISHED_STEPS = MAIL_TOTAL - MAIL_STEPS - 1;

static uint32_t octreeDepth(uint32_t grid)  // tools.cu:63-88
{
    for (uint32_t d = 1; d <= 9; ++d)
        if (grid == (1u << d))
            return d;
    return 0;
}

OctreeBuilder::OctreeBuilder(int device) : itsDevice(device)
{
    OC_HIP_CHECK(hipSetDevice(itsDevice));
    OC_HIP_CHECK(hipStreamCreateWithFlags(&itsStream, hipStreamNonBlocking));
    OC_HIP_CHECK(hipStreamCreateWithFlags(&itsCopyStream, hipStreamNonBlocking));
    OC_HIP_CHECK(hipEventCreateWithFlags(&itsBuiltEvent, hipEventDisableTiming));
    OC_HIP_CHECK(hipEventCreateWithFlags(&itsCopiedEvent, hipEventDisableTiming));
    OC_HIP_CHECK(hipEventCreateWithFlags(&itsUploadedEvent, hipEventDisableTiming));
    OC_HIP_CHECK(hipDeviceGetAttribute(&itsClockRate, hipDeviceAttributeWallClockRate, itsDevice));
    OC_HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&itsMailbox), MAIL_WORDS * sizeof(uint64_t), hipHostMallocCoherent));
    std::fill(itsMailbox, itsMailbox + MAIL_WORDS, 0);
}

OctreeBuilder::OctreeBuilder(int device, const CloudInfo& cloud, const ProcessingInfo& proc,
                             const uint8_t* hostCloud, const uint8_t* deviceCloud)
    : OctreeBuilder(device)
{
    setup(cloud, proc, hostCloud, deviceCloud);
}

static uint64_t coordinateBytes(const CloudInfo& c)
{
    return c.cloudType == CLOUD_FLOAT_UINT8_T ? 12 : 24;
}

static uint64_t sortedPointBytes(const CloudInfo& c)
{
    return c.cloudType == CLOUD_FLOAT_UINT8_T ? sizeof(SortedPoint<float>) : sizeof(SortedPoint<double>);
}

void OctreeBuilder::setup(const CloudInfo& cloud, const ProcessingInfo& proc, const uint8_t* hostCloud,
                          const uint8_t* deviceCloud)
{
    OC_HIP_CHECK(hipSetDevice(itsDevice));
    itsReady = false;
    itsBuilt = false;
    itsCloud = cloud;
    itsProc  = proc;
    itsDepth = octreeDepth(proc.chunkingGrid);
    itsDense = 0;
    for (uint32_t l = 0; l <= itsDepth; ++l)
    {
        uint32_t g          = proc.chunkingGrid >> l;
        itsLevelGrid[l]     = g;
        itsLevelOffset[l]   = itsDense;
        itsLevelNodes[l]    = g * g * g;
        itsDense += g * g * g;
    }
    itsCoarse  = coarseLevel(itsDepth);
    itsBuckets = (proc.chunkingGrid >> itsCoarse) * (proc.chunkingGrid >> itsCoarse) * (proc.chunkingGrid >> itsCoarse);
    itsColorMode = proc.useIntraCellAvg ? COLOR_INTRA
                                        : (proc.useInterCellAvg ? (proc.useWeightingFunction ? COLOR_INTER_WEIGHTED
                                                                                            : COLOR_INTER)
                                                                : COLOR_NONE);
    itsE = static_cast<uint64_t>(static_cast<float>(cloud.pointAmount) * proc.outputFactor);  // point_cloud.cuh:24

    const uint64_t cloudBytes = static_cast<uint64_t>(cloud.pointAmount) * cloud.dataStride;
    if (deviceCloud)
    {
        itsCloudDevice = deviceCloud;
    }
    else
    {
        itsCloudOwned.ensure(cloudBytes);
        upload(itsCloudOwned.get(), hostCloud, cloudBytes);
        OC_HIP_CHECK(hipEventRecord(itsUploadedEvent, itsStream));
        itsCloudDevice = itsCloudOwned.as<uint8_t>();
    }

    // Fixed-size state: the dense pyramid, the node key/count arrays (bounded by min(D, levels*N))
    // and the output region.
    itsCount.ensure(sizeof(uint32_t) * static_cast<uint64_t>(itsDense));
    itsIdBase.ensure(sizeof(uint32_t) * ((static_cast<uint64_t>(itsDense) + 31) / 32));
    itsOccupancy.ensure(sizeof(uint32_t) * ((static_cast<uint64_t>(itsDense) + 31) / 32));
    const uint64_t mBound = nodeBound();
    // The previous build's snapshot copies may still read the node keys and counts, the LUT and
    // the output: growing one of them frees it, so those copies are waited for first. (The other
    // arrays a snapshot reads are grown by the merge, after its stream has waited for the copies
    // and the host has read the node count back.)
    if (itsSnapshotPending && (sizeof(uint32_t) * mBound > itsNodeKey.capacity() ||
                               sizeof(uint32_t) * mBound > itsNodeCount.capacity() ||
                               sizeof(uint32_t) * itsE > itsLut.capacity() ||
                               sizeof(OutRecord) * itsE > itsOut.capacity()))
        waitSnapshot();
    itsNodeKey.ensure(sizeof(uint32_t) * mBound);
    itsNodeCount.ensure(sizeof(uint32_t) * mBound);
    itsLut.ensure(sizeof(uint32_t) * itsE);
    itsOut.ensure(sizeof(OutRecord) * itsE);
    const uint64_t coordBytes  = coordinateBytes(cloud);
    const uint64_t sortedBytes = sortedPointBytes(cloud);
    const uint64_t stagedCap   = std::max<uint64_t>(1, itsE - cloud.pointAmount);
    itsSorted.ensure(sortedBytes * cloud.pointAmount);
    itsBucketed.ensure(sortedBytes * cloud.pointAmount);
    itsFineCode.ensure(sizeof(uint16_t) * cloud.pointAmount);
    itsPerm.ensure(sizeof(uint32_t) * cloud.pointAmount);
    itsBucketCount.ensure(sizeof(uint32_t) * (itsBuckets + 1));
    itsBucketStart.ensure(sizeof(uint32_t) * (itsBuckets + 1));
    itsBucketCursor.ensure(sizeof(uint32_t) * (itsBuckets + 1));
    itsBucketList.ensure(sizeof(uint32_t) * itsBuckets);
    itsStLut.ensure(sizeof(uint32_t) * stagedCap);
    itsStPts.ensure(coordBytes * stagedCap);
    itsStColor.ensure(sizeof(OutRecord) * stagedCap);  // what the footprint charges a staged point
    itsScalars.ensure(sizeof(uint64_t) * SC_COUNT);
    // The output starts zeroed (the tail past N + I stays zero, A15). The fill goes on the copy
    // stream, behind the previous build's snapshot copies that still read the output; the build
    // waits for that stream before its first write to anything a snapshot reads (generate).
    OC_HIP_CHECK(hipMemsetAsync(itsOut.get(), 0, sizeof(OutRecord) * itsE, itsCopyStream));
    OC_HIP_CHECK(hipEventRecord(itsCopiedEvent, itsCopyStream));
    itsSnapshotPending = true;
    // the caller's cloud buffer is borrowed until this returns: wait for the upload only
    if (!deviceCloud)
        OC_HIP_CHECK(hipEventSynchronize(itsUploadedEvent));
    itsReady = true;
}

std::vector<DeviceBuffer*> OctreeBuilder::arena()
{
    return {&itsCloudOwned,  &itsCount,       &itsIdBase,       &itsOccupancy,
            &itsNodeKey,     &itsNodeCount,   &itsNodePoints,
            &itsNodeData,    &itsNodeParent,  &itsNodeChild,     &itsNodeFlags,    &itsNodeSorted,
            &itsNodeStage,   &itsNodeSub,     &itsBucketed,     &itsSorted,      &itsFineCode,
            &itsPerm,
            &itsBucketCount, &itsBucketStart, &itsBucketCursor,  &itsBucketList,  &itsLut,          &itsOut,
            &itsStLut,       &itsStPts,       &itsStColor,       &itsInternalList, &itsSegCount,    &itsSegSrc,
            &itsSegTile,     &itsSegInput,    &itsNodeGrid,      &itsTileList,     &itsBitmap,      &itsPrefix,
            &itsCursors,     &itsStamps,      &itsWin,         &itsColor,         &itsCellCnt,      &itsCellStart,   &itsCellKey,
            &itsCellNode,    &itsCellOf,      &itsRankOf,        &itsPayload,      &itsScalars,
            &itsScanScratch, &itsLeafList,   &itsSplitChunks,   &itsSplitHist};
}

uint64_t OctreeBuilder::arenaBytes() const
{
    uint64_t total = 0;
    for (DeviceBuffer* b : const_cast<OctreeBuilder*>(this)->arena())
        total += b->capacity();
    return total;
}

void OctreeBuilder::releaseArena()
{
    OC_HIP_CHECK(hipStreamSynchronize(itsCopyStream));
    itsSnapshotPending = false;
    OC_HIP_CHECK(hipStreamSynchronize(itsStream));
    for (DeviceBuffer* b : arena())
        b->release();
    itsReady = false;
    itsBuilt = false;
}

uint64_t OctreeBuilder::estimateFootprint(const CloudInfo& cloud, const ProcessingInfo& proc, bool hostCloud)
{
    const uint32_t depth = octreeDepth(proc.chunkingGrid);
    uint64_t dense       = 0;
    for (uint32_t l = 0; l <= depth; ++l)
    {
        const uint64_t g = proc.chunkingGrid >> l;
        dense += g * g * g;
    }
    const uint64_t n      = cloud.pointAmount;
    const uint64_t e      = static_cast<uint64_t>(static_cast<float>(cloud.pointAmount) * proc.outputFactor);
    const uint64_t staged = e > n ? e - n : 1;
    const uint64_t mBound = std::min<uint64_t>(dense, (depth + 1) * n);
    uint64_t bytes        = hostCloud ? n * cloud.dataStride : 0;
    bytes += 8 * dense + 4 * ((dense + 31) / 32);          // count pyramid; occupancy bits and id bases (at most a word a cell)
    bytes += 8 * mBound + 77 * mBound + n / 1024;           // node keys / counts, node arrays, leaf chunks
    bytes += 22 * e;                                        // lut + output records
    bytes += (2 * sortedPointBytes(cloud) + 2 + 4) * n;     // bucketed, sorted, fine codes, permutation
    if (n > FINE_SPLIT)                                     // split buckets of the fine sort
        bytes += (2 * n / FINE_SPLIT + 1) * (8 + 4ull * MAX_FINE_CELLS);
    bytes += (4 + 18 + coordinateBytes(cloud)) * staged;     // staging
    bytes += 8 * (staged / 4096 + 1);                       // placement work list (the rest of it from the staging)
    if (proc.useInterCellAvg && proc.useWeightingFunction && !proc.useIntraCellAvg)
        bytes += 4 * staged;                                // staged colours of the weighted filter
    // per-level work: inputs (cell, then its dense index; rank; payload), at most N and with it E, and cells
    // (winner, colour sum, count, start, key, node), at most as many as are staged; the occupancy bitmaps
    // and their prefix
    const uint64_t wordsPerNode = (rowsPerNode(proc.subsamplingGrid) * proc.subsamplingGrid + 31) / 32;
    const uint64_t levelNodes   = std::min<uint64_t>(mBound, n / std::max<uint32_t>(1, proc.mergingThreshold) + 8);
    bytes += (8 + sizeof(WeightPayload) + sizeof(uint64_t)) * e + 32 * staged;
    bytes += std::min<uint64_t>(kBitmapBudget, 8 * wordsPerNode * levelNodes);
    return bytes;
}

OctreeBuilder::~OctreeBuilder()
{
    if (itsCopyStream)
    {
        (void)hipStreamSynchronize(itsCopyStream);
        (void)hipStreamDestroy(itsCopyStream);
    }
    if (itsStream)
    {
        (void)hipStreamSynchronize(itsStream);
        (void)hipStreamDestroy(itsStream);
    }
    if (itsBuiltEvent)
        (void)hipEventDestroy(itsBuiltEvent);
    if (itsCopiedEvent)
        (void)hipEventDestroy(itsCopiedEvent);
    if (itsUploadedEvent)
        (void)hipEventDestroy(itsUploadedEvent);
    if (itsMailbox)
        (void)hipHostFree(itsMailbox);
}

// The sizes after the merge, to the host mailbox: the nodes, the error flags, the internal nodes,
// and the first node and first internal node of every level. The values first, then (after a
// system-scope release) the sequence number the host waits for.
__global__ __launch_bounds__(64) void kPublishMerge(const uint64_t* __restrict__ sc, const uint32_t* __restrict__ internal,
                                                    uint32_t levels, uint64_t* box, uint64_t seq)
{
    const uint32_t l     = threadIdx.x;
    const uint32_t inner = static_cast<uint32_t>(sc[SC_INTERNAL]);
    auto post            = [&](uint32_t at, uint64_t v) {
        __hip_atomic_store(box + at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    };
    if (l < levels)
    {
        const uint32_t start = reinterpret_cast<const uint32_t*>(sc + SC_LEVEL_START)[l];
        uint32_t a = 0, b = inner;  // the first internal node at or after the level's first node
        while (a < b)
        {
            const uint32_t mid = a + (b - a) / 2;
            if (internal[mid] < start)
                a = mid + 1;
            else
                b = mid;
        }
        post(MAIL_LEVEL + l, start);
        post(MAIL_INNER + l, a);
    }
    if (l == 0)
    {
        post(MAIL_NODES, sc[SC_M]);
        post(MAIL_ERROR, sc[SC_ERROR]);
        post(MAIL_INTERNAL, inner);
    }
    __threadfence_system();
    __syncthreads();
    if (l == 0)
        __hip_atomic_store(box + MAIL_SEQ, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// (tiles << 32 | inputs) of a level before its step `first` and the PUBLISHED_STEPS after it, a step being
// stepNodes of the level's `nodes`; past the last one, and behind them (MAIL_TOTAL): all of the level.
// segTile, segInput: the segment scan.
__global__ __launch_bounds__(64) void kPublishSteps(const uint64_t* __restrict__ segTotal,
                                                    const uint32_t* __restrict__ segTile,
                                                    const uint32_t* __restrict__ segInput, uint32_t nodes,
                                                    uint32_t stepNodes, uint32_t first, uint64_t* box, uint64_t seq)
{
    const uint64_t node = (static_cast<uint64_t>(first) + threadIdx.x) * stepNodes;
    const uint64_t v    = threadIdx.x <= PUBLISHED_STEPS && node < nodes
                                  ? (static_cast<uint64_t>(segTile[8 * node]) << 32) | segInput[8 * node]
                                  : *segTotal;
    __hip_atomic_store(box + MAIL_STEPS + threadIdx.x, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_store(box + MAIL_SEQ, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The cells that a step works on.
__global__ void kPublishCells(StepSizes step, uint64_t* box, uint64_t seq)
{
    if (threadIdx.x != 0)
        return;
    __hip_atomic_store(box + MAIL_USED, step(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(box + MAIL_SEQ, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The end of a build: the error flags, the used output records (the last cursor) and the stage
// durations from the clock stamps, in clock ticks.
__global__ __launch_bounds__(64) void kPublishEnd(const uint64_t* __restrict__ sc, const uint64_t* __restrict__ cursors,
                                                  const uint64_t* __restrict__ stamps, uint32_t steps, uint64_t* box,
                                                  uint64_t seq)
{
    const uint64_t now = wall_clock64();
    if (threadIdx.x != 0)
        return;
    auto post = [&](uint32_t at, uint64_t v) {
        __hip_atomic_store(box + at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    };
    const uint64_t start = sc[SC_STAMP], merge = sc[SC_STAMP + 1], dist = sc[SC_STAMP + 2];
    const uint64_t levels = steps ? stamps[ST_BEGIN] : now;
    uint64_t insert = 0, emit = 0;
    for (uint32_t i = 0; i < steps; ++i)
    {
        const uint64_t* st = stamps + ST_STAMPS * i;
        insert += st[ST_INSERT_END] - st[ST_INSERT_BEGIN];
        emit += st[ST_STAMPS + ST_BEGIN] - st[ST_EMIT_BEGIN];
    }
    const uint64_t ticks[7] = {merge - start, dist - merge, levels - dist, now - levels, now - start, insert, emit};
    for (uint32_t k = 0; k < 7; ++k)
        post(MAIL_TICKS + k, ticks[k]);
    post(MAIL_ERROR, sc[SC_ERROR]);
    post(MAIL_USED, cursors[steps]);
    __hip_atomic_store(box + MAIL_SEQ, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Sizes the host needs from the device. The stream is drained up to the publish: the
// host spins on the mailbox for up to 2 ms (the common case: the value is ready within microseconds
// of the last kernel) and then falls back to a blocking synchronisation, which also reports a
// failed kernel instead of waiting forever.
void OctreeBuilder::waitMailbox(uint64_t seq)
{
    const auto start = std::chrono::steady_clock::now();
    while (__atomic_load_n(itsMailbox + MAIL_SEQ, __ATOMIC_ACQUIRE) != seq)
    {
        __builtin_ia32_pause();
        if (std::chrono::steady_clock::now() - start > std::chrono::milliseconds(2))
        {
            OC_HIP_CHECK(hipStreamSynchronize(itsStream));
            if (__atomic_load_n(itsMailbox + MAIL_SEQ, __ATOMIC_ACQUIRE) != seq)
                throw std::runtime_error("device value was not published");
            break;
        }
    }
}

void OctreeBuilder::generate()
{
    OC_HIP_CHECK(hipSetDevice(itsDevice));
    if (!itsReady)
        throw std::runtime_error("the builder has not been set up for a cloud");
    itsBuilt = false;
    if (itsCloud.cloudType == CLOUD_FLOAT_UINT8_T)
        generateTyped<float>();
    else
        generateTyped<double>();
    itsBuilt = true;
}

template <typename T>
void OctreeBuilder::generateTyped()
{
    countPoints<T>();  // writes nothing a snapshot reads, so it overlaps the previous one's copies
    progress();
    waitForSnapshotOnStream();
    mergeLevels();
    progress();
    distributePoints<T>();
    progress();
    subsampleLevels<T>();
    placeInternalNodes();
    const uint64_t seq = ++itsMailSeq;
    kPublishEnd<<<1, 64, 0, itsStream>>>(itsScalars.as<uint64_t>(), itsCursors.as<uint64_t>(),
                                         itsStamps.as<uint64_t>(), itsSteps, itsMailbox, seq);
    OC_LAUNCH_CHECK();
    waitMailbox(seq);

    const uint64_t err = itsMailbox[MAIL_ERROR];
    if (err & ERR_OVERFLOW)  // A14
        throw std::runtime_error("the subsampled points exceed the estimated output size (N + I > E); "
                                 "raise the output factor");
    if (err & ERR_OUTSIDE)
        throw std::runtime_error("a point lies outside the cubic bounding box");
    itsUsed = itsMailbox[MAIL_USED];
    itsTimings.assign(7, 0.f);
    for (uint32_t k = 0; k < 7; ++k)
        itsTimings[k] = static_cast<float>(static_cast<double>(itsMailbox[MAIL_TICKS + k]) / itsClockRate);
}

template <typename T>
void OctreeBuilder::countPoints()
{
    uint64_t* sc       = itsScalars.as<uint64_t>();
    const uint32_t n   = itsCloud.pointAmount;
    const uint32_t nb  = itsBuckets;
    uint32_t* bucketCount  = itsBucketCount.as<uint32_t>();
    uint32_t* bucketStart  = itsBucketStart.as<uint32_t>();
    uint32_t* bucketCursor = itsBucketCursor.as<uint32_t>();
    const Gridding g = gridding(itsCloud.bbMin[0], itsCloud.bbMin[1], itsCloud.bbMin[2],
                                itsCloud.bbMax[0] - itsCloud.bbMin[0], itsProc.chunkingGrid);
    itsScanScratch.ensure(sizeof(uint64_t) * scanTiles(nb));
    uint32_t* occ         = itsOccupancy.as<uint32_t>();
    const uint64_t words  = (static_cast<uint64_t>(itsDense) + 31) / 32;
    const uint64_t counts = itsLevelOffset[itsCoarse];  // read for empty cells from here on
    kBuildInit<<<gridFor(std::max<uint64_t>({nb, words, itsDense - counts}), 2048), BLOCK, 0, itsStream>>>(
            sc, bucketCount, nb + 1, occ, words, itsCount.as<uint32_t>(), counts, itsDense);
    OC_LAUNCH_CHECK();

    // four rounds of records per workgroup until the chip is full, then sixteen: every workgroup adds its
    // histogram to the global one at the end (5.1M points: 35 us, with four rounds 49)
    const unsigned histBlocks = static_cast<unsigned>(std::min<uint64_t>(
            2048, std::max<uint64_t>((static_cast<uint64_t>(n) + 8191) / 8192,
                                     std::min<uint64_t>(COMPUTE_UNITS, (static_cast<uint64_t>(n) + 2047) / 2048))));
    kBucketHist<T><<<histBlocks, HIST_THREADS, 0, itsStream>>>(itsCloudDevice, n, itsCloud.dataStride, g,
                                                               3 * itsCoarse, nb, bucketCount,
                                                               reinterpret_cast<uint32_t*>(sc + SC_ERROR));
    OC_LAUNCH_CHECK();
    // buckets above FINE_SPLIT points, a chunk per workgroup (at most 2 n / FINE_SPLIT chunks)
    const uint64_t chunkBound = 2ull * n / FINE_SPLIT + 1;
    itsSplitChunks.ensure(sizeof(uint64_t) * chunkBound);
    const uint64_t* totals = sc + SC_BUCKETS;
    scanExclusive<uint64_t>(nb, BucketIn{bucketCount},
                            BucketTablesOut{bucketStart, bucketCursor, itsBucketList.as<uint32_t>(),
                                            itsSplitChunks.as<uint64_t>(), nb},
                            itsScanScratch.as<uint64_t>(), sc + SC_BUCKETS, itsStream);
    OC_LAUNCH_CHECK();
    auto scatter = [&](auto kernel, uint32_t items) {
        const uint64_t chunk = static_cast<uint64_t>(SCATTER_THREADS) * items;
        kernel<<<static_cast<unsigned>((n + chunk - 1) / chunk), SCATTER_THREADS, 0, itsStream>>>(
                itsCloudDevice, n, itsCloud.dataStride, g, 3 * itsCoarse, nb, bucketCursor,
                itsBucketed.as<SortedPoint<T>>(), itsFineCode.as<uint16_t>());
        OC_LAUNCH_CHECK();
    };
    if (n <= SCATTER_ONE_POINTS)
        scatter(kBucketScatter<T, 1>, 1);
    else if (n <= SCATTER_TWO_POINTS)
        scatter(kBucketScatter<T, 2>, 2);
    else
        scatter(kBucketScatter<T, LARGE_STAGE_ITEMS<T>>, LARGE_STAGE_ITEMS<T>);
    FineSortParams fp{};
    fp.lc         = itsCoarse;
    fp.bucketGrid = itsProc.chunkingGrid >> itsCoarse;
    for (uint32_t l = 0; l <= itsDepth; ++l)
    {
        fp.levelOffset[l] = itsLevelOffset[l];
        fp.levelGrid[l]   = itsLevelGrid[l];
    }
    auto fineSort = [&](auto kernel, uint32_t perUnit) {
        kernel<<<std::min<uint32_t>(nb, perUnit * COMPUTE_UNITS), SORT_THREADS, 0, itsStream>>>(
                itsFineCode.as<uint16_t>(), bucketStart, itsBucketList.as<uint32_t>(), totals,
                reinterpret_cast<uint32_t*>(sc + SC_NEXT_BUCKET), fp, itsCount.as<uint32_t>(),
                itsPerm.as<uint32_t>(), occ);
        OC_LAUNCH_CHECK();
    };
    if (itsCoarse < MAX_COARSE_LEVEL)
        fineSort(kFineSort<SMALL_FINE_CELLS>, 2);
    else
        fineSort(kFineSort<MAX_FINE_CELLS>, 1);
    if (n > FINE_SPLIT)
    {
        itsSplitHist.ensure(sizeof(uint32_t) * MAX_FINE_CELLS * chunkBound);
        const unsigned grid = static_cast<unsigned>((chunkBound + XCD_COUNT - 1) / XCD_COUNT * XCD_COUNT);
        kFineChunkHist<<<grid, SORT_THREADS, 0, itsStream>>>(itsFineCode.as<uint16_t>(), bucketStart,
                                                             itsSplitChunks.as<uint64_t>(), totals, fp.lc,
                                                             itsSplitHist.as<uint32_t>());
        OC_LAUNCH_CHECK();
        kFineSplitScan<<<grid, SORT_THREADS, 0, itsStream>>>(bucketStart, itsSplitChunks.as<uint64_t>(), totals,
                                                             fp, itsCount.as<uint32_t>(), itsSplitHist.as<uint32_t>(),
                                                             occ);
        OC_LAUNCH_CHECK();
        kFineChunkPerm<<<grid, SORT_THREADS, 0, itsStream>>>(itsFineCode.as<uint16_t>(), bucketStart,
                                                             itsSplitChunks.as<uint64_t>(), totals, fp.lc,
                                                             itsSplitHist.as<uint32_t>(), itsPerm.as<uint32_t>());
        OC_LAUNCH_CHECK();
    }
}

LevelParams OctreeBuilder::levelParams() const
{
    LevelParams lp{};
    for (uint32_t l = 0; l <= itsDepth; ++l)
    {
        lp.offset[l] = itsLevelOffset[l];
        lp.grid[l]   = itsLevelGrid[l];
    }
    lp.depth     = itsDepth;
    lp.threshold = itsProc.mergingThreshold;
    return lp;
}

void OctreeBuilder::mergeLevels()
{
    uint64_t* sc    = itsScalars.as<uint64_t>();
    uint32_t* count = itsCount.as<uint32_t>();
    LevelOffsets lo{};
    for (uint32_t l = 0; l <= itsDepth; ++l)
        lo.offset[l] = itsLevelOffset[l];
    lo.levels = itsDepth + 1;
    // levels 0..coarse come from the fine sort: counts and occupancy bits of the levels above, sparse ids
    // (A2) + node keys / counts
    // + first id of every level by a scan over the bitmap's words, and the list of internal nodes
    uint32_t* occ         = itsOccupancy.as<uint32_t>();
    uint32_t* levelStart  = reinterpret_cast<uint32_t*>(sc + SC_LEVEL_START);
    uint32_t* nodes       = reinterpret_cast<uint32_t*>(sc + SC_M);
    const uint64_t words  = (static_cast<uint64_t>(itsDense) + 31) / 32;
    // at most N / threshold internal nodes on a level (they hold disjoint point sets), and at most
    // as many as nodes above level 0
    uint64_t inner = 0;
    for (uint32_t l = 1; l <= itsDepth; ++l)
        inner += std::min<uint64_t>(std::min<uint64_t>(itsLevelNodes[l], itsCloud.pointAmount),
                                    itsCloud.pointAmount / std::max<uint32_t>(1, itsProc.mergingThreshold));
    itsInternalList.ensure(sizeof(uint32_t) * std::max<uint64_t>(1, inner));
    itsScanScratch.ensure(sizeof(uint64_t) * SCAN_GRID);
    uint32_t* sums = itsScanScratch.as<uint32_t>();
    const unsigned wordGrid = static_cast<unsigned>(std::min<uint64_t>(scanTiles(words), SCAN_GRID));
    kOccupancy<<<wordGrid, SCAN_THREADS, 0, itsStream>>>(occ, count, itsDense, lo, itsCoarse,
                                                         itsProc.chunkingGrid, sums, sc + SC_STAMP + 1);
    OC_LAUNCH_CHECK();
    const IdTables ids{occ, count, itsIdBase.as<uint32_t>(), itsNodeKey.as<uint32_t>(),
                       itsNodeCount.as<uint32_t>(), levelStart, lo};
    kOccupiedIds<<<wordGrid, SCAN_THREADS, 0, itsStream>>>(ids, words, sums, nodes);
    OC_LAUNCH_CHECK();
    uint32_t* internal = itsInternalList.as<uint32_t>();
    scanExclusive<uint32_t>(DeviceCount{nodes, levelStart + 1}, nodeBound(),
                            InternalNodeIn{itsNodeCount.as<uint32_t>(), levelStart, itsProc.mergingThreshold},
                            InternalNodeOut{internal, levelStart}, sums, reinterpret_cast<uint32_t*>(sc + SC_INTERNAL),
                            itsStream);
    OC_LAUNCH_CHECK();
    const uint64_t seq = ++itsMailSeq;
    kPublishMerge<<<1, 64, 0, itsStream>>>(sc, internal, itsDepth + 1, itsMailbox, seq);
    OC_LAUNCH_CHECK();
    waitMailbox(seq);
    if (itsMailbox[MAIL_ERROR] & ERR_OUTSIDE)
        throw std::runtime_error("a point lies outside the cubic bounding box");
    itsM = static_cast<uint32_t>(itsMailbox[MAIL_NODES]);
    for (uint32_t l = 0; l <= itsDepth; ++l)
    {
        itsLevelStart[l] = static_cast<uint32_t>(itsMailbox[MAIL_LEVEL + l]);
        itsInner[l]      = static_cast<uint32_t>(itsMailbox[MAIL_INNER + l]);
    }
    itsLevelStart[itsDepth + 1] = itsM;
    itsInner[itsDepth + 1]      = static_cast<uint32_t>(itsMailbox[MAIL_INTERNAL]);
    if (itsM == 0)
        throw std::runtime_error("the cloud has no points inside the bounding box");

    const uint64_t m = itsM;
    itsNodePoints.ensure(sizeof(uint32_t) * m);
    itsNodeData.ensure(sizeof(uint64_t) * m);
    itsNodeParent.ensure(sizeof(int32_t) * m);
    itsNodeChild.ensure(sizeof(int32_t) * 8 * m);
    itsNodeFlags.ensure(m);
    itsNodeSorted.ensure(sizeof(uint32_t) * m);
    itsNodeStage.ensure(sizeof(uint32_t) * m);
    itsNodeSub.ensure(sizeof(uint32_t) * m);
    itsCursors.ensure(sizeof(uint64_t) * (planSteps() + 1));
    itsStamps.ensure(sizeof(uint64_t) * (ST_STAMPS * itsSteps + 1));
    kNodeLinks<<<gridFor(m), BLOCK, 0, itsStream>>>(
            itsM, levelParams(), itsNodeKey.as<uint32_t>(), itsNodeCount.as<uint32_t>(),
            IdMap{occ, itsIdBase.as<uint32_t>()}, itsNodePoints.as<uint32_t>(), itsNodeData.as<uint64_t>(),
            itsNodeParent.as<int32_t>(), itsNodeChild.as<int32_t>(), itsNodeFlags.as<uint8_t>(),
            itsNodeSub.as<uint32_t>(), itsCoarse, itsBucketStart.as<uint32_t>(), itsNodeSorted.as<uint32_t>(), count,
            itsCursors.as<uint64_t>(), itsCloud.pointAmount);
    OC_LAUNCH_CHECK();
}

uint64_t OctreeBuilder::nodeBound() const
{
    return std::min<uint64_t>(itsDense, static_cast<uint64_t>(itsDepth + 1) * itsCloud.pointAmount);
}

ChildSlots OctreeBuilder::childSlots(uint32_t firstInternal) const
{
    return ChildSlots{itsInternalList.as<uint32_t>() + firstInternal, itsNodeFlags.as<uint8_t>(),
                      itsNodeChild.as<int32_t>(), itsNodeCount.as<uint32_t>()};
}

// Leaf data blocks (A4) and leaf chunks.
LeafOrderParams OctreeBuilder::leafTables()
{
    uint64_t* sc             = itsScalars.as<uint64_t>();
    const uint32_t nodes     = itsInner[itsDepth + 1];
    const double cubicSize   = itsCloud.bbMax[0] - itsCloud.bbMin[0];  // metadata.cuh:66-69
    LeafOrderParams p{};
    for (int a = 0; a < 3; ++a)
        p.cubicMin[a] = itsCloud.bbMin[a];
    for (uint32_t l = 0; l <= itsDepth; ++l)
    {
        p.side[l]     = cubicSize / std::pow(2.0, static_cast<double>(itsDepth - l));  // rp_subsampling.cu:17-18
        p.sideHalf[l] = p.side[l] / 2.0;
    }
    p.lp                = levelParams();
    p.g                 = itsProc.subsamplingGrid;
    p.order             = cellOrderOf(itsColorMode, p.g);
    const uint32_t h    = p.g > 1 ? p.g / 2 : 1;  // cells per axis of a leaf's octant, as kLeafCellOrder
    const uint64_t keys = rowsPerNode(h) * ((h + 31) / 32);
    while (((keys - 1) >> p.keyShift) >= LEAF_KEYS)
        ++p.keyShift;
    if (nodes == 0)
        return p;
    const uint64_t slots = 8ull * nodes;
    // one list for the leaf chunks here and the placement chunks at the end
    itsLeafList.ensure(sizeof(uint64_t) * std::max<uint64_t>(leafChunkBound(), placeChunkBound()));
    const ChildSlots cs = childSlots(0);
    scanExclusive<uint64_t>(slots, LeafSlotIn{cs},
                            LeafSlotOut{cs, itsNodeData.as<uint64_t>(), itsLeafList.as<uint64_t>()},
                            itsScanScratch.as<uint64_t>(), sc + SC_LEAF_TOTAL, itsStream);
    OC_LAUNCH_CHECK();
    return p;
}

// chunks of leaves: at most N / LEAF_CHUNK plus one per leaf, and a leaf is a child of an internal node
uint64_t OctreeBuilder::leafChunkBound() const
{
    return itsCloud.pointAmount / LEAF_CHUNK + std::min<uint64_t>(8ull * itsInner[itsDepth + 1], itsM);
}

uint64_t OctreeBuilder::placeChunkBound() const
{
    return (itsE - itsCloud.pointAmount) / PLACE_CHUNK + itsInner[itsDepth + 1];
}

// The host's copy of the totals before the steps of a level from step `first` on (kPublishSteps).
const uint64_t* OctreeBuilder::readSteps(const uint64_t* total, uint32_t nodes, uint32_t stepNodes, uint32_t first)
{
    const uint64_t seq = ++itsMailSeq;
    kPublishSteps<<<1, 64, 0, itsStream>>>(total, itsSegTile.as<uint32_t>(), itsSegInput.as<uint32_t>(), nodes, stepNodes,
                                           first, itsMailbox, seq);
    OC_LAUNCH_CHECK();
    waitMailbox(seq);
    return itsMailbox + MAIL_STEPS;
}

template <typename T>
void OctreeBuilder::distributePoints()
{
    const Gridding g = gridding(itsCloud.bbMin[0], itsCloud.bbMin[1], itsCloud.bbMin[2],
                                itsCloud.bbMax[0] - itsCloud.bbMin[0], itsProc.chunkingGrid);
    // octree_chunking.cu:108-112
    double sx = 1.0 / itsCloud.scale[0], sy = 1.0 / itsCloud.scale[1], sz = 1.0 / itsCloud.scale[2];
    const LeafOrderParams p = leafTables();
    uint64_t* stamp         = itsScalars.as<uint64_t>() + SC_STAMP + 2;
    // the records move to the sorted cloud: leaf and cell order when there are internal nodes and
    // more than one cell to a node's grid, plain Morton order otherwise; then the leaf data blocks are
    // copied from it
    const uint32_t n = itsCloud.pointAmount;
    if (itsInner[itsDepth + 1] > 0 && p.g >= 2)
    {
        uint64_t chunks = leafChunkBound();
        if (std::min<uint64_t>(8ull * itsInner[itsDepth + 1], itsM) >= READ_INPUTS_CHILDREN)
            chunks = readSteps(itsScalars.as<uint64_t>() + SC_LEAF_TOTAL, 0, 0, 0)[0] >> 32;
        for (uint64_t first = 0; first == 0 || first < chunks; first += LEAF_LAUNCH_CHUNKS)
        {
            const uint64_t some = std::min<uint64_t>(chunks - first, LEAF_LAUNCH_CHUNKS);
            kLeafCellOrder<T><<<static_cast<unsigned>(std::max<uint64_t>(1, some)), LEAF_THREADS, 0, itsStream>>>(
                    itsLeafList.as<uint64_t>(), static_cast<uint32_t>(first),
                    itsScalars.as<uint64_t>() + SC_LEAF_TOTAL, p, itsNodeKey.as<uint32_t>(),
                    itsNodeParent.as<int32_t>(), itsNodeCount.as<uint32_t>(), itsNodeSorted.as<uint32_t>(),
                    itsBucketed.as<SortedPoint<T>>(), itsPerm.as<uint32_t>(), itsSorted.as<SortedPoint<T>>(),
                    first == 0 ? stamp : nullptr);
        }
    }
    else
        kGatherSorted<T><<<gatherGrid(n), BLOCK, 0, itsStream>>>(itsBucketed.as<SortedPoint<T>>(),
                                                                     itsPerm.as<uint32_t>(), n,
                                                                     itsSorted.as<SortedPoint<T>>(), stamp);
    OC_LAUNCH_CHECK();
    kDistributeSorted<T><<<gridFor(n, 16384), BLOCK, 0, itsStream>>>(
            itsSorted.as<SortedPoint<T>>(), n, g, itsCount.as<uint32_t>(), itsNodeSorted.as<uint32_t>(),
            itsNodeData.as<uint64_t>(), itsLut.as<uint32_t>(), itsOut.as<OutRecord>(), sx, sy, sz);
    OC_LAUNCH_CHECK();
}

StagedColors OctreeBuilder::stagedColors() const
{
    const bool packed = packedColors(itsColorMode);
    return StagedColors{packed ? nullptr : itsStColor.as<uint32_t>(), packed ? itsStColor.as<uint64_t>() : nullptr};
}

// Nodes of one subsampling step: their bitmaps and prefixes fit kBitmapBudget.
uint32_t OctreeBuilder::stepNodes() const
{
    const uint64_t words = (rowsPerNode(itsProc.subsamplingGrid) * itsProc.subsamplingGrid + 31) / 32;
    return static_cast<uint32_t>(std::max<uint64_t>(1, kBitmapBudget / (2 * sizeof(uint32_t) * words)));
}

// Subsampling steps of the build (batches of a level's nodes).
uint32_t OctreeBuilder::planSteps()
{
    itsSteps = 0;
    for (uint32_t l = 1; l <= itsDepth; ++l)
        itsSteps += (itsInner[l + 1] - itsInner[l] + stepNodes() - 1) / stepNodes();
    return itsSteps;
}

// The levels bottom-up, a step per batch of a level's nodes. The merge has told the host the internal
// nodes of every level; inputs, tiles, occupied cells and the output cursor stay on the device, the
// launches are sized by bounds (a level's inputs are distinct points, so there are at most N of them,
// and no more cells than inputs; only children that there are can have tiles), and a step that does not fit
// the output leaves itself and the later ones without work. So the host waits for nothing: with two
// readbacks a level, each of which drains the GPU for ~15 us, small builds spent a third of their time
// waiting. From READ_INPUTS_POINTS points or READ_INPUTS_CHILDREN children on, one readback a level costs
// less than the empty workgroups (a 120M-point bound is 470K of them, ~30 us a launch, three or four
// launches a level), and a level of several steps reads the sizes of each: the level's bound would be
// launched again for every step. Grids that stride over
// the work instead were slower on large levels (payload scatter 3.9 -> 4.9 ms, emit 11.0 -> 11.9 ms at
// 119.7M points): workgroups drift apart and no longer share cache lines while they are in L2.
template <typename T>
void OctreeBuilder::subsampleLevels()
{
    uint64_t* sc     = itsScalars.as<uint64_t>();
    uint32_t* err    = reinterpret_cast<uint32_t*>(sc + SC_ERROR);
    const uint32_t N = itsCloud.pointAmount;
    const uint32_t g = itsProc.subsamplingGrid;
    const double cubicSize   = itsCloud.bbMax[0] - itsCloud.bbMin[0];  // metadata.cuh:66-69
    const uint64_t cellsPerNode = rowsPerNode(g) * g;
    const uint64_t wordsPerNode = (cellsPerNode + 31) / 32;
    const uint32_t batchNodes   = stepNodes();
    const bool packed   = packedColors(itsColorMode);
    const bool weighted = itsColorMode == COLOR_INTER_WEIGHTED;
    PointStore<T> ps{};
    ps.sorted = itsSorted.as<SortedPoint<T>>();
    ps.stLut  = itsStLut.as<uint32_t>();
    ps.stPts  = itsStPts.as<T>();
    ps.staged = stagedColors();
    ps.N      = N;

    SubsampleParams sp{};
    for (int a = 0; a < 3; ++a)
        sp.cubicMin[a] = itsCloud.bbMin[a];
    for (uint32_t L = 0; L <= itsDepth; ++L)
        sp.sideHalf[L] = (cubicSize / std::pow(2.0, static_cast<double>(itsDepth - L))) / 2.0;
    sp.depth = itsDepth;
    sp.g     = g;
    sp.seed  = itsProc.seed;

    // sizes over all levels
    uint32_t levelMost = 0;
    for (uint32_t l = 1; l <= itsDepth; ++l)
        levelMost = std::max(levelMost, itsInner[l + 1] - itsInner[l]);
    uint64_t* cursors = itsCursors.as<uint64_t>();
    if (levelMost == 0)
        return;
    const uint64_t segMost  = 8ull * levelMost;
    const uint64_t wordMost = std::min(levelMost, batchNodes) * wordsPerNode;
    itsSegCount.ensure(sizeof(uint32_t) * segMost);
    itsSegSrc.ensure(sizeof(uint32_t) * segMost);
    itsSegTile.ensure(sizeof(uint32_t) * segMost);
    itsSegInput.ensure(sizeof(uint32_t) * segMost);
    itsNodeGrid.ensure(sizeof(NodeGrid) * levelMost);
    itsTileList.ensure(sizeof(uint32_t) * (N / TILE + segMost));
    itsBitmap.ensure(sizeof(uint32_t) * wordMost);
    itsPrefix.ensure(sizeof(uint32_t) * (wordMost + 1));
    itsScanScratch.ensure(sizeof(uint64_t) * SCAN_GRID + sizeof(uint32_t) * scanTiles(wordMost));  // range, tile sums
    // Arrays for the inputs of a level and for the cells of a step. A step that fits the output (no other one
    // touches the cells' arrays) has no more cells than are staged.
    const uint32_t cellCap = static_cast<uint32_t>(std::min<uint64_t>(N, std::max<uint64_t>(1, itsE - N)));
    const bool exactArrays = N >= EXACT_ARRAYS_POINTS;
    uint64_t *winKey = nullptr, *win = nullptr, *color = nullptr;
    uint32_t* cellCnt = nullptr;
    auto sizeInputs   = [&](uint64_t inputs) {
        itsCellOf.ensure(sizeof(uint32_t) * inputs);
        if (weighted)
        {
            itsRankOf.ensure(sizeof(uint32_t) * inputs);
            itsPayload.ensure((sizeof(WeightPayload) + sizeof(uint64_t)) * inputs);  // payloads, then winner keys
            winKey = reinterpret_cast<uint64_t*>(itsPayload.as<uint8_t>() + sizeof(WeightPayload) * inputs);
        }
    };
    auto sizeCells = [&](uint64_t cells) {
        itsCellKey.ensure(sizeof(uint32_t) * cells);
        itsCellNode.ensure(sizeof(uint32_t) * cells);
        if (weighted)  // takes its winners from the payload keys
        {
            itsCellCnt.ensure(sizeof(uint32_t) * cells);
            itsCellStart.ensure(sizeof(uint32_t) * (cells + 1));
            cellCnt = itsCellCnt.as<uint32_t>();
        }
        else
        {
            itsWin.ensure(sizeof(uint64_t) * cells);
            win = itsWin.as<uint64_t>();
        }
        if (packed)
        {
            itsColor.ensure(sizeof(uint64_t) * cells);
            color = itsColor.as<uint64_t>();
        }
    };
    if (!exactArrays)
    {
        sizeInputs(N);
        sizeCells(cellCap);
    }
    uint32_t* bitmap  = itsBitmap.as<uint32_t>();
    uint32_t* prefix  = itsPrefix.as<uint32_t>();
    uint32_t stepAt = 0;
    for (uint32_t l = 1; l <= itsDepth; ++l)
    {
        const uint32_t K = itsInner[l + 1] - itsInner[l];
        if (K == 0)
            continue;
        // the segments that can hold inputs: children of the level's nodes
        const uint64_t children = std::min<uint64_t>(8ull * K, itsLevelStart[l] - itsLevelStart[l - 1]);
        // tiles combined in LDS, where there are enough points for them and the flag bit is free
        const bool large = N >= LARGE_POINTS && N / children >= LARGE_CHILD && N < NOT_OWNED &&
                           32 * wordsPerNode < NOT_OWNED;
        const uint32_t tileInputs  = large ? LARGE_TILE : TILE;
        const int tileThreads      = large ? LARGE_THREADS : static_cast<int>(TILE);
        const ChildSlots cs        = childSlots(itsInner[l]);
        NodeGrid* nodeGrid         = itsNodeGrid.as<NodeGrid>();
        const LevelSegmentIn segIn{cs, itsNodePoints.as<uint32_t>(), tileInputs};
        const LevelSegmentOut segOut{cs, itsNodeSorted.as<uint32_t>(), itsNodeStage.as<uint32_t>(),
                                     itsSegCount.as<uint32_t>(), itsSegSrc.as<uint32_t>(), itsSegTile.as<uint32_t>(),
                                     itsSegInput.as<uint32_t>()};
        const bool readBack     = N >= READ_INPUTS_POINTS || K > batchNodes || children >= READ_INPUTS_CHILDREN;
        // in one launch with the level's other preparations, when it is one step sized without a readback
        const bool oneLaunch = K <= START_NODES && !readBack;
        if (!oneLaunch)
        {
            scanExclusive<uint64_t>(8ull * K, segIn, segOut, itsScanScratch.as<uint64_t>(), sc + SC_SEG_TOTAL, itsStream);
            OC_LAUNCH_CHECK();
        }
        const uint32_t parts    = tileInputs / TILE;
        const uint64_t* totals  = nullptr;  // read back, from step stepAt - firstStep on
        const uint32_t firstStep = stepAt;
        sp.level       = l;
        sp.levelOffset = itsLevelOffset[l];
        sp.levelGrid   = itsLevelGrid[l];
        sp.side        = cubicSize / std::pow(2.0, static_cast<double>(itsDepth - l));  // rp_subsampling.cu:17-18

        for (uint32_t k0 = 0; k0 < K; k0 += batchNodes)
        {
            const uint32_t k1 = std::min<uint32_t>(K, k0 + batchNodes);
            const uint32_t Kb = k1 - k0;
            const uint64_t words = static_cast<uint64_t>(Kb) * wordsPerNode;
            uint64_t inputMost = N, tileMost = N / tileInputs + std::min<uint64_t>(children, 8ull * Kb);
            if (readBack)
            {
                const uint32_t at = (stepAt - firstStep) % PUBLISHED_STEPS;
                if (at == 0)
                    totals = readSteps(sc + SC_SEG_TOTAL, K, batchNodes, stepAt - firstStep);
                if (exactArrays && k0 == 0)
                    sizeInputs(std::max<uint32_t>(1, static_cast<uint32_t>(itsMailbox[MAIL_TOTAL])));
                inputMost = static_cast<uint32_t>(totals[at + 1] - totals[at]);
                tileMost  = (totals[at + 1] >> 32) - (totals[at] >> 32);
            }
            const uint64_t cellMost = std::min<uint64_t>({inputMost, 32 * words, cellCap});
            const uint32_t* tilesLo = k0 > 0 ? itsSegTile.as<uint32_t>() + 8ull * k0 : nullptr;
            const uint32_t* tilesHi = k1 < K ? itsSegTile.as<uint32_t>() + 8ull * k1
                                             : reinterpret_cast<uint32_t*>(sc + SC_SEG_TOTAL) + 1;
            // launch(tiles, workgroups, first launch) until all tiles of the step are taken
            auto overTiles = [&](auto launch) {
                for (uint64_t skip = 0; skip == 0 || skip < tileMost; skip += LAUNCH_TILES)
                {
                    const uint64_t some = std::max<uint64_t>(1, std::min<uint64_t>(tileMost - skip, LAUNCH_TILES));
                    launch(TileRange{tilesLo, tilesHi, static_cast<uint32_t>(skip)},
                           xcdRunGrid(some, XCD_TILE_RUN / parts), skip == 0);
                    OC_LAUNCH_CHECK();
                }
            };
            const StepSizes step{cursors + stepAt, cursors + stepAt + 1, prefix + words, itsE};
            uint64_t* stamps = itsStamps.as<uint64_t>() + ST_STAMPS * stepAt;
            ++stepAt;

            const bool resetInputs = !exactArrays && !large && words <= RESET_INPUTS_WORDS;
            const uint32_t reset   = resetInputs ? cellCap : 0;
            const unsigned prepareGrid = gridFor(std::max<uint64_t>(words, inputMost / TILE), 16384);
            if (oneLaunch)
                kLevelStart<<<std::min(prepareGrid, 2048u), BLOCK, 0, itsStream>>>(
                        K, sp, segIn, segOut, itsNodeKey.as<uint32_t>(), nodeGrid, sc + SC_SEG_TOTAL,
                        itsTileList.as<uint32_t>(), words, bitmap, CellState{win, color, cellCnt}, reset,
                        stamps + ST_BEGIN);
            else
                kLevelPrepare<<<prepareGrid, BLOCK, 0, itsStream>>>(
                        k0 == 0 ? K : 0, sp, cs.internal, itsNodeKey.as<uint32_t>(), nodeGrid, itsSegTile.as<uint32_t>(),
                        sc + SC_SEG_TOTAL, itsTileList.as<uint32_t>(), words, bitmap, CellState{win, color, cellCnt},
                        reset, stamps + ST_BEGIN);
            OC_LAUNCH_CHECK();
            auto mark = [&](auto kernel) {
                overTiles([&](const TileRange& tiles, uint32_t grid, bool begin) {
                    kernel<<<grid, tileThreads, 0, itsStream>>>(
                            tiles, k0, wordsPerNode, itsTileList.as<uint32_t>(), itsSegTile.as<uint32_t>(),
                            itsSegCount.as<uint32_t>(), itsSegSrc.as<uint32_t>(), itsSegInput.as<uint32_t>(), nodeGrid,
                            ps, cellOrderOf(itsColorMode, g), bitmap, itsCellOf.as<uint32_t>(), err,
                            begin ? stamps + ST_INSERT_BEGIN : nullptr);
                });
            };
            mark(large ? kMarkLarge<T> : kMark<T>);
            const uint64_t wordTiles = scanTiles(words);
            uint32_t* rangeSums      = itsScanScratch.as<uint32_t>();
            if (wordTiles <= SCAN_DIRECT_TILES)
                scanExclusive<uint32_t>(words, PopcountIn{bitmap}, ExclusiveToArray{prefix}, rangeSums, prefix + words,
                                        itsStream);
            else
            {
                const unsigned grid = static_cast<unsigned>(std::min<uint64_t>(wordTiles, SCAN_GRID));
                uint32_t* tileSums  = rangeSums + 2 * SCAN_GRID;
                kWordReduce<<<grid, SCAN_THREADS, 0, itsStream>>>(bitmap, words, tileSums, rangeSums);
                kWordPrefix<<<grid, SCAN_THREADS, 0, itsStream>>>(bitmap, words, wordsPerNode, tileSums, rangeSums,
                                                                  prefix);
            }
            OC_LAUNCH_CHECK();
            if (exactArrays)
            {
                const uint64_t seq = ++itsMailSeq;
                kPublishCells<<<1, 64, 0, itsStream>>>(step, itsMailbox, seq);
                OC_LAUNCH_CHECK();
                waitMailbox(seq);
                sizeCells(std::max<uint64_t>(1, itsMailbox[MAIL_USED]));
            }
            if (!large && !resetInputs)
            {
                kClearCompact<<<gridFor(cellMost, 16384), BLOCK, 0, itsStream>>>(step, CellState{win, color, cellCnt});
                OC_LAUNCH_CHECK();
            }

            auto accumulate = [&](auto kernel) {
                overTiles([&](const TileRange& tiles, uint32_t grid, bool begin) {
                    kernel<<<grid, tileThreads, 0, itsStream>>>(
                            tiles, step, k0, begin ? Kb : 0, wordsPerNode, itsTileList.as<uint32_t>(),
                            itsSegTile.as<uint32_t>(), itsSegCount.as<uint32_t>(), itsSegSrc.as<uint32_t>(),
                            itsSegInput.as<uint32_t>(), nodeGrid, bitmap, prefix, itsCellOf.as<uint32_t>(), ps, win,
                            color, cellCnt, itsCellKey.as<uint32_t>(), itsCellNode.as<uint32_t>(),
                            weighted ? itsRankOf.as<uint32_t>() : nullptr, itsNodePoints.as<uint32_t>(),
                            itsNodeStage.as<uint32_t>(), itsNodeSub.as<uint32_t>(), itsNodeFlags.as<uint8_t>(),
                            itsNodeChild.as<int32_t>(), err);
                });
            };
            auto rest = [&](auto kernel) {
                overTiles([&](const TileRange& tiles, uint32_t grid, bool) {
                    kernel<<<grid, tileThreads, 0, itsStream>>>(
                            tiles, step, k0, wordsPerNode, itsTileList.as<uint32_t>(), itsSegTile.as<uint32_t>(),
                            itsSegCount.as<uint32_t>(), itsSegSrc.as<uint32_t>(), itsSegInput.as<uint32_t>(), nodeGrid,
                            bitmap, prefix, itsCellOf.as<uint32_t>(), ps, win, color, cellCnt,
                            weighted ? itsRankOf.as<uint32_t>() : nullptr);
                });
            };
            auto accumulateMode = [&](auto mode, auto random) {
                constexpr uint32_t M = decltype(mode)::value;
                constexpr bool R     = decltype(random)::value;
                accumulate(large ? kAccumulateLarge<T, M, R> : kAccumulate<T, M, R>);
                if (large)
                    rest(kAccumulateRest<T, M, R>);
            };
            auto accumulateAll = [&](auto mode) {
                if (itsProc.useRandomSubsampling)
                    accumulateMode(mode, std::true_type{});
                else
                    accumulateMode(mode, std::false_type{});
            };
            const bool random = itsProc.useRandomSubsampling;
            switch (itsColorMode)
            {
            case COLOR_NONE: accumulateAll(std::integral_constant<uint32_t, COLOR_NONE>{}); break;
            case COLOR_INTRA: accumulateAll(std::integral_constant<uint32_t, COLOR_INTRA>{}); break;
            case COLOR_INTER: accumulateAll(std::integral_constant<uint32_t, COLOR_INTER>{}); break;
            default: accumulateAll(std::integral_constant<uint32_t, COLOR_INTER_WEIGHTED>{}); break;
            }

            if (weighted)
            {
                scanExclusive<uint32_t>(step, cellMost, ArrayIn{cellCnt},
                                        ExclusiveWithTotal{itsCellStart.as<uint32_t>(), step.cells},
                                        itsScanScratch.as<uint32_t>(), static_cast<uint32_t*>(nullptr), itsStream);
                OC_LAUNCH_CHECK();
                auto scatter = [&](auto kernel) {
                    overTiles([&](const TileRange& tiles, uint32_t grid, bool begin) {
                        kernel<<<grid * parts, TILE, 0, itsStream>>>(
                                tiles, step, g, itsTileList.as<uint32_t>(), itsSegTile.as<uint32_t>(),
                                itsSegCount.as<uint32_t>(), itsSegSrc.as<uint32_t>(), itsSegInput.as<uint32_t>(),
                                nodeGrid, itsCellKey.as<uint32_t>(), itsRankOf.as<uint32_t>(),
                                itsCellStart.as<uint32_t>(), itsCellOf.as<uint32_t>(), ps,
                                itsPayload.as<WeightPayload>(), winKey, parts, begin ? stamps + ST_INSERT_END : nullptr);
                    });
                };
                scatter(random ? kScatterPayload<T, true> : kScatterPayload<T, false>);
            }

            if (weighted)
                kEmitWeighted<T><<<xcdRunGrid(std::max<uint64_t>(1, (cellMost + BLOCK - 1) / BLOCK), EMIT_CHUNK), BLOCK, 0, itsStream>>>(
                        step, k0, wordsPerNode, g, nodeGrid, bitmap, prefix, itsCellKey.as<uint32_t>(),
                        itsCellNode.as<uint32_t>(), itsCellStart.as<uint32_t>(), itsPayload.as<WeightPayload>(), winKey,
                        ps, stamps + ST_EMIT_BEGIN);
            else
            {
                auto emit = [&](auto kernel) {
                    kernel<<<gridFor(cellMost), BLOCK, 0, itsStream>>>(
                            step, wordsPerNode, g, bitmap, prefix, itsCellKey.as<uint32_t>(),
                            itsCellNode.as<uint32_t>(), win, color, ps, stamps + ST_INSERT_END, stamps + ST_EMIT_BEGIN);
                };
                switch (itsColorMode)
                {
                case COLOR_NONE: emit(kEmit<T, COLOR_NONE>); break;
                case COLOR_INTRA: emit(kEmit<T, COLOR_INTRA>); break;
                default: emit(kEmit<T, COLOR_INTER>); break;
                }
            }
            OC_LAUNCH_CHECK();
        }
        progress();
    }
}

void OctreeBuilder::placeInternalNodes()
{
    const uint32_t N     = itsCloud.pointAmount;
    const uint32_t nodes = itsInner[itsDepth + 1];
    if (nodes == 0)
        return;
    const uint32_t* list = itsInternalList.as<uint32_t>();
    // (internal node, chunk) work items; the leaf chunk list is free again after the distribution
    uint32_t* chunks = reinterpret_cast<uint32_t*>(itsScalars.as<uint64_t>() + SC_TABLE_TOTAL);  // zero so far
    kPlaceNodes<<<std::min<uint32_t>((nodes + 63) / 64, 4096), 64, 0, itsStream>>>(
            list, nodes, N, itsNodeParent.as<int32_t>(), itsNodeChild.as<int32_t>(), itsNodePoints.as<uint32_t>(),
            itsNodeSub.as<uint32_t>(), itsNodeData.as<uint64_t>(), itsLeafList.as<uint64_t>(), chunks, itsStamps.as<uint64_t>() + ST_STAMPS * itsSteps);
    OC_LAUNCH_CHECK();
    const Gridding cubic = gridding(itsCloud.bbMin[0], itsCloud.bbMin[1], itsCloud.bbMin[2],
                                    itsCloud.bbMax[0] - itsCloud.bbMin[0], itsProc.chunkingGrid);
    const double sx = 1.0 / itsCloud.scale[0], sy = 1.0 / itsCloud.scale[1], sz = 1.0 / itsCloud.scale[2];
    const unsigned grid = static_cast<unsigned>(std::min<uint64_t>(placeChunkBound(), 1u << 20));
    if (itsCloud.cloudType == CLOUD_FLOAT_UINT8_T)
        kPermute<float><<<grid, BLOCK, 0, itsStream>>>(
                itsLeafList.as<uint64_t>(), chunks, N, itsNodeStage.as<uint32_t>(), itsNodeData.as<uint64_t>(),
                itsNodePoints.as<uint32_t>(), itsStLut.as<uint32_t>(),
                itsStPts.as<float>(), stagedColors(), cubic, sx, sy, sz, itsLut.as<uint32_t>(), itsOut.as<OutRecord>());
    else
        kPermute<double><<<grid, BLOCK, 0, itsStream>>>(
                itsLeafList.as<uint64_t>(), chunks, N, itsNodeStage.as<uint32_t>(), itsNodeData.as<uint64_t>(),
                itsNodePoints.as<uint32_t>(), itsStLut.as<uint32_t>(),
                itsStPts.as<double>(), stagedColors(), cubic, sx, sy, sz, itsLut.as<uint32_t>(), itsOut.as<OutRecord>());
    OC_LAUNCH_CHECK();
}

// Copies go through the builder's own stream, so slots of a build service copy concurrently.
void OctreeBuilder::copyNodes(HostOctree& o) const
{
    if (!itsBuilt)
        throw std::runtime_error("the octree has not been generated");
    const uint64_t m = itsM;
    o.denseKey.resize(m);
    o.count.resize(m);
    o.pointCount.resize(m);
    o.dataIdx.resize(m);
    o.parent.resize(m);
    o.children.resize(8 * m);
    o.flags.resize(m);
    auto copy = [&](void* dst, const void* src, uint64_t bytes) {
        OC_HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, itsStream));
    };
    copy(o.denseKey.data(), itsNodeKey.get(), 4 * m);
    copy(o.count.data(), itsNodeCount.get(), 4 * m);
    copy(o.pointCount.data(), itsNodePoints.get(), 4 * m);
    copy(o.dataIdx.data(), itsNodeData.get(), 8 * m);
    copy(o.parent.data(), itsNodeParent.get(), 4 * m);
    copy(o.children.data(), itsNodeChild.get(), 32 * m);
    copy(o.flags.data(), itsNodeFlags.get(), m);
    OC_HIP_CHECK(hipStreamSynchronize(itsStream));
}

void OctreeBuilder::progress()
{
    if (itsProgress)
        itsProgress();
}

bool OctreeBuilder::snapshotDone()
{
    const hipError_t e = hipEventQuery(itsCopiedEvent);
    if (e == hipErrorNotReady)
        return false;
    OC_HIP_CHECK(e);
    return true;
}

void OctreeBuilder::drainCopies() noexcept
{
    (void)hipStreamSynchronize(itsCopyStream);
    (void)hipGetLastError();
}

std::unique_ptr<SlotBuilder> makeSlotBuilder(int device)
{
    return std::make_unique<OctreeBuilder>(device);
}

uint64_t slotFootprint(const CloudInfo& cloud, const ProcessingInfo& proc, bool hostCloud)
{
    return OctreeBuilder::estimateFootprint(cloud, proc, hostCloud);
}

void OctreeBuilder::waitForSnapshotOnStream()
{
    if (itsSnapshotPending)
    {
        OC_HIP_CHECK(hipStreamWaitEvent(itsStream, itsCopiedEvent, 0));
        itsSnapshotPending = false;
    }
}

void OctreeBuilder::copySnapshot(uint8_t* dst) const
{
    auto* self = const_cast<OctreeBuilder*>(this);
    self->snapshotAsync(dst);
    self->waitSnapshot();
}

void OctreeBuilder::waitSnapshot()
{
    OC_HIP_CHECK(hipEventSynchronize(itsCopiedEvent));
}

void OctreeBuilder::snapshotAsync(uint8_t* dst)
{
    if (!itsBuilt)
        throw std::runtime_error("the octree has not been generated");
    const SnapshotLayout l(itsM, itsUsed);
    const uint64_t m = itsM;
    OC_HIP_CHECK(hipEventRecord(itsBuiltEvent, itsStream));
    OC_HIP_CHECK(hipStreamWaitEvent(itsCopyStream, itsBuiltEvent, 0));
    auto copy = [&](uint64_t offset, const void* src, uint64_t bytes) {
        if (bytes)
            OC_HIP_CHECK(hipMemcpyAsync(dst + offset, src, bytes, hipMemcpyDeviceToHost, itsCopyStream));
    };
    copy(l.dataIdx, itsNodeData.get(), 8 * m);
    copy(l.denseKey, itsNodeKey.get(), 4 * m);
    copy(l.count, itsNodeCount.get(), 4 * m);
    copy(l.pointCount, itsNodePoints.get(), 4 * m);
    copy(l.parent, itsNodeParent.get(), 4 * m);
    copy(l.children, itsNodeChild.get(), 32 * m);
    copy(l.flags, itsNodeFlags.get(), m);
    copy(l.lut, itsLut.get(), 4 * itsUsed);
    copy(l.out, itsOut.get(), sizeof(OutRecord) * itsUsed);
    OC_HIP_CHECK(hipEventRecord(itsCopiedEvent, itsCopyStream));
    itsSnapshotPending = true;
}

// Device to host, synchronous; large copies into pageable memory are staged (host_staging.h).
void OctreeBuilder::download(void* dst, const void* src, uint64_t bytes) const
{
    OC_HIP_CHECK(hipSetDevice(itsDevice));
    downloadStaged(dst, src, bytes, itsStream);
}

// Host to device on the builder's stream; large copies from pageable memory are staged and have
// left the host memory when this returns (host_staging.h).
void OctreeBuilder::upload(void* dst, const void* src, uint64_t bytes)
{
    const HostSegment seg{dst, src, bytes};
    uploadSegments(&seg, 1, itsStream);
}

void OctreeBuilder::copyLut(uint32_t* dst, uint64_t count) const
{
    if (count > itsE)
        throw std::runtime_error("copy beyond the output capacity");
    download(dst, itsLut.get(), 4 * count);
}

void OctreeBuilder::copyOutputRange(uint8_t* dst, uint64_t first, uint64_t count) const
{
    if (first + count > itsE)
        throw std::runtime_error("copy beyond the output capacity");
    download(dst, itsOut.as<OutRecord>() + first, sizeof(OutRecord) * count);
}

}  // namespace oc
