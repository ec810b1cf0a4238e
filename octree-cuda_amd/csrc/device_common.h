// Device-side helpers shared by the builder's kernels: record decoding, the cell mapping, packed
// colours, quantisation and the explicit-random ranking.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "types.h"

namespace oc {

// Unaligned load of the three coordinates of a packed AoS record (the reference reads them through
// a #pragma pack(1) Vector3, metadata.cuh:13-19). gfx950 serves unaligned dword loads directly.
template <typename T>
__device__ __forceinline__ void loadXYZ(const uint8_t* rec, double& x, double& y, double& z)
{
    T v[3];
    __builtin_memcpy(v, rec, sizeof(v));
    x = static_cast<double>(v[0]);
    y = static_cast<double>(v[1]);
    z = static_cast<double>(v[2]);
}

// Packed records staged through LDS: a wave reads the lines of 64 consecutive records as aligned
// 16-byte words, the next ones while it works on these, and every lane takes its record out of the
// wave's own part of LDS; no workgroup barrier. Histogram of 119.7M 27-byte records: 602 us, 5.3 TB/s of
// their lines (loaded from their places 638 us; a workgroup's records staged between two barriers 1280);
// of 25M records of 15 to 32 bytes within 2 % either way. Strides above STAGE_STRIDE are loaded from
// their places.
constexpr uint32_t STAGE_STRIDE = 32;
constexpr int STAGE_LOADS       = 3;  // words per lane, at most

struct RecordStage
{
    uint4 word[64 * STAGE_STRIDE / 16 + 1];  // the first record may start inside a word
};

struct RecordWords
{
    uint4 w[STAGE_LOADS];
    uint32_t skip;  // bytes of the first word before the first record
};

// The words of records [first, first + count), count <= 64 and stride <= STAGE_STRIDE. Only words that
// hold a byte of these records are read, so no other page is touched.
__device__ __forceinline__ RecordWords loadRecords(const uint8_t* cloud, uint64_t first, uint32_t count, uint32_t stride)
{
    RecordWords r;
    const uint64_t begin = reinterpret_cast<uint64_t>(cloud) + first * stride;
    r.skip               = static_cast<uint32_t>(begin & 15);
    const uint4* src     = reinterpret_cast<const uint4*>(begin - r.skip);
    const uint32_t words = count ? (r.skip + count * stride + 15) / 16 : 0u;
    const uint32_t lane  = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < STAGE_LOADS; ++k)
        if (lane + 64 * k < words)
            r.w[k] = src[lane + 64 * k];
    return r;
}

// The words into the wave's stage.
__device__ __forceinline__ void putRecords(const RecordWords& r, uint32_t count, uint32_t stride, RecordStage& stage)
{
    const uint32_t words = count ? (r.skip + count * stride + 15) / 16 : 0u;
    const uint32_t lane  = threadIdx.x & 63;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int k = 0; k < STAGE_LOADS; ++k)
        if (lane + 64 * k < words)
            stage.word[lane + 64 * k] = r.w[k];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Coordinates of the record at byte offset `at` of a stage.
template <typename T>
__device__ __forceinline__ void stagedXYZ(const RecordStage& stage, uint32_t at, double& x, double& y, double& z)
{
    constexpr int WORDS = 3 * sizeof(T) / 4;
    const uint32_t* src = reinterpret_cast<const uint32_t*>(stage.word) + (at >> 2);
    uint32_t w[WORDS + 1], v[WORDS];
#pragma unroll
    for (int k = 0; k <= WORDS; ++k)
        w[k] = src[k];  // the last one is in the stage: at most the record's colour and its word
#pragma unroll
    for (int k = 0; k < WORDS; ++k)
        v[k] = __builtin_amdgcn_alignbyte(w[k + 1], w[k], at & 3);
    T c[3];
    __builtin_memcpy(c, v, sizeof(c));
    x = static_cast<double>(c[0]);
    y = static_cast<double>(c[1]);
    z = static_cast<double>(c[2]);
}

// body(x, y, z) for the coordinates of every record of a cloud, in a grid of workgroups of THREADS;
// stages: one RecordStage per wave, in LDS.
template <typename T, int THREADS, typename Body>
__device__ __forceinline__ void forRecords(const uint8_t* cloud, uint32_t n, uint32_t stride, RecordStage* stages, Body body)
{
    const uint64_t step = static_cast<uint64_t>(gridDim.x) * THREADS;
    if (stride > STAGE_STRIDE)
    {
        for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * THREADS + threadIdx.x; i < n; i += step)
        {
            double x, y, z;
            loadXYZ<T>(cloud + i * stride, x, y, z);
            body(x, y, z);
        }
        return;
    }
    RecordStage& stage  = stages[threadIdx.x >> 6];
    const uint32_t lane = threadIdx.x & 63;
    auto countAt        = [n](uint64_t first) { return first < n ? (n - first < 64 ? static_cast<uint32_t>(n - first) : 64u) : 0u; };
    uint64_t first      = static_cast<uint64_t>(blockIdx.x) * THREADS + (threadIdx.x & ~63u);
    uint32_t count      = countAt(first);
    RecordWords words   = loadRecords(cloud, first, count, stride);
    while (count)
    {
        putRecords(words, count, stride, stage);
        const uint32_t at   = words.skip + lane * stride;
        const uint32_t more = countAt(first + step);
        words               = loadRecords(cloud, first + step, more, stride);
        if (lane < count)
        {
            double x, y, z;
            stagedXYZ<T>(stage, at, x, y, z);
            body(x, y, z);
        }
        first += step;
        count = more;
    }
}

// Cell coordinates of a point in a grid, with the reference's exact expression order
// (kernel_helpers.cuh:11-25): t = bbSize / G; u = (p - min) / t; clamp to G - 1 with fmin;
// truncate to int64, then reinterpret as uint64. Returned in 32 bits: a coordinate outside the grid is
// any value >= G.
//
// Four divisions and three 64-bit conversions are ~150 instructions (without them, 25.8M points: kMark
// 506 -> 478 us, kDistributeSorted 278 -> 257; 119.7M: kDistributeSorted 1421 -> 1357). The product q = (p - min) * inv has three roundings where u has two, so
// |u - q| <= 2^-50 |q| < 2^-30 for |q| < 2^20: unless q lies within 2^-30 of a whole number, u and q
// truncate (and clamp) alike. A wave takes the divisions only where one of its points lies that close
// to a cell face, far outside, or is not a number.
__device__ __forceinline__ void gridCoords(double px, double py, double pz, const Gridding& g, uint32_t& ix,
                                           uint32_t& iy, uint32_t& iz)
{
    constexpr double NEAR = 1.0 / (1u << 30), FAR = 1u << 20;
    const double top = g.gridSize - 1.0;
    const double dx = px - g.minX, dy = py - g.minY, dz = pz - g.minZ;
    const double qx = dx * g.inv, qy = dy * g.inv, qz = dz * g.inv;
    const double fx = qx - floor(qx), fy = qy - floor(qy), fz = qz - floor(qz);
    // the sum is not below FAR where any of them is not a number
    if (fabs(qx) + fabs(qy) + fabs(qz) < FAR && fmin(fmin(fx, fy), fz) > NEAR && fmax(fmax(fx, fy), fz) < 1.0 - NEAR)
    {
        ix = static_cast<uint32_t>(static_cast<int32_t>(fmin(qx, top)));
        iy = static_cast<uint32_t>(static_cast<int32_t>(fmin(qy, top)));
        iz = static_cast<uint32_t>(static_cast<int32_t>(fmin(qz, top)));
        return;
    }
    const double t = g.bbSize / g.gridSize;
    auto coord     = [&](double d) {
        const uint64_t i = static_cast<uint64_t>(static_cast<int64_t>(fmin(d / t, top)));
        return i < g.gridSize ? static_cast<uint32_t>(i) : ~0u;
    };
    ix = coord(dx);
    iy = coord(dy);
    iz = coord(dz);
}

// Packed colour (kernel_helpers.cuh:49-53): 18-bit r, g, b fields and a 10-bit count; sums wrap
// exactly like the reference's uint64 atomics.
__device__ __forceinline__ uint64_t encodeColors(uint16_t r, uint16_t g, uint16_t b)
{
    return (static_cast<uint64_t>(r) << 46) | (static_cast<uint64_t>(g) << 28) | (static_cast<uint64_t>(b) << 10) |
           1ull;
}

// rp_subsampling.cuh:123-129; a zero amount (count == 0 mod 1024) decodes to 0 instead of dividing
// by zero.
__device__ __forceinline__ void decodeColors(uint64_t e, uint16_t& r, uint16_t& g, uint16_t& b)
{
    uint32_t amount = static_cast<uint32_t>(e & 0x3FF);
    if (amount == 0)
    {
        r = g = b = 0;
        return;
    }
    r = static_cast<uint16_t>(static_cast<uint32_t>((e >> 46) & 0xFFFF) / amount);
    g = static_cast<uint16_t>(static_cast<uint32_t>((e >> 28) & 0xFFFF) / amount);
    b = static_cast<uint16_t>(static_cast<uint32_t>((e >> 10) & 0xFFFF) / amount);
}

// Explicit random subsampling ranks the points of a node with MurmurHash3's 32-bit finalizer
// (a bijection, so no ties) keyed by a per-node salt from the SplitMix64 finalizer; the winner of
// a cell is the point of minimum rank. Identical on host and device.
__host__ __device__ __forceinline__ uint64_t splitmix64Mix(uint64_t z)
{
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

__host__ __device__ __forceinline__ uint32_t fmix32(uint32_t h)
{
    h ^= h >> 16;
    h *= 0x85EBCA6BU;
    h ^= h >> 13;
    h *= 0xC2B2AE35U;
    h ^= h >> 16;
    return h;
}

__host__ __device__ __forceinline__ uint32_t nodeSalt(uint64_t seed, uint32_t nodeKey)
{
    return static_cast<uint32_t>(
            splitmix64Mix(seed + 0x9E3779B97F4A7C15ULL * (static_cast<uint64_t>(nodeKey) + 1)) >> 32);
}

// Output record of a point (point_distributing.cuh:62-74): int32(floor((p - cubicMin) * (1 / scale)))
// per axis with the reciprocal taken on the host (octree_chunking.cu:108-112); rgb packs r | g << 8
// | b << 16.
__device__ __forceinline__ OutRecord quantizePoint(double x, double y, double z, uint32_t rgb, const Gridding& g,
                                                   double sx, double sy, double sz)
{
    OutRecord o;
    o.x = static_cast<int32_t>(floor((x - g.minX) * sx));
    o.y = static_cast<int32_t>(floor((y - g.minY) * sy));
    o.z = static_cast<int32_t>(floor((z - g.minZ) * sz));
    o.r = static_cast<uint16_t>(rgb & 0xFF);
    o.g = static_cast<uint16_t>((rgb >> 8) & 0xFF);
    o.b = static_cast<uint16_t>((rgb >> 16) & 0xFF);
    return o;
}

__device__ __forceinline__ void storeRecord(OutRecord* dst, const OutRecord& r)
{
    __builtin_memcpy(dst, &r, sizeof(OutRecord));
}

// Output records of a wave, put in place through LDS: stored by their own lanes they are 18 bytes apart,
// and each of the five stores of a lane touches the same ten lines again.
struct OutStage
{
    uint32_t word[64 * sizeof(OutRecord) / 4 + 1];
};

// Lane i's record to dst[i], i < count <= 64, dst at an even address: every lane writes its record at its
// place of the wave's stage (as four words and a half, whichever comes first at its alignment), then the
// wave stores consecutive words. All lanes of the wave take part.
__device__ __forceinline__ void storeRecords(OutRecord* dst, const OutRecord& r, uint32_t count, OutStage& stage)
{
    const uint32_t lane  = threadIdx.x & 63;
    const uint64_t begin = reinterpret_cast<uint64_t>(dst);
    const uint32_t skip  = static_cast<uint32_t>(begin & 2);
    const uint32_t end   = skip + count * static_cast<uint32_t>(sizeof(OutRecord));
    uint16_t* halves     = reinterpret_cast<uint16_t*>(stage.word);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane < count)
    {
        const uint32_t at   = skip + lane * static_cast<uint32_t>(sizeof(OutRecord));
        const bool half     = (at & 2) != 0;  // the record starts with the second half of a word
        const uint32_t v[5] = {static_cast<uint32_t>(r.x), static_cast<uint32_t>(r.y), static_cast<uint32_t>(r.z),
                               r.r | (static_cast<uint32_t>(r.g) << 16), r.b};
        uint32_t* w         = stage.word + ((at + 2) >> 2);
#pragma unroll
        for (int k = 0; k < 4; ++k)
            w[k] = half ? __builtin_amdgcn_alignbyte(v[k + 1], v[k], 2) : v[k];
        halves[(at >> 1) + (half ? 0 : 8)] = static_cast<uint16_t>(half ? v[0] : v[4]);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    uint32_t* out = reinterpret_cast<uint32_t*>(begin - skip);
#pragma unroll
    for (int k = 0; k < 5; ++k)
    {
        const uint32_t i = lane + 64 * k;
        if (4 * i >= skip && 4 * i + 4 <= end)
            out[i] = stage.word[i];
    }
    if (count && lane == 0)  // halves of words that other records share
    {
        if (skip)
            reinterpret_cast<uint16_t*>(out)[1] = halves[1];
        if (end & 2)
            reinterpret_cast<uint16_t*>(out)[(end >> 1) - 1] = halves[(end >> 1) - 1];
    }
}

// Wave-level runs: consecutive lanes holding equal keys (inputs arrive spatially sorted, so lanes
// often share a bitmap word or a cell). Every lane must take part; a lane without work passes a key
// of its own. start / end are the first and last lane of the lane's run.
__device__ __forceinline__ uint64_t shflUp64(uint64_t v, int delta)
{
    const uint32_t lo = __shfl_up(static_cast<uint32_t>(v), delta, 64);
    const uint32_t hi = __shfl_up(static_cast<uint32_t>(v >> 32), delta, 64);
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

struct WaveRun
{
    int lane, start, end;
};

__device__ __forceinline__ WaveRun waveRun(uint64_t key)
{
    WaveRun r;
    r.lane                 = static_cast<int>(threadIdx.x & 63);
    const uint64_t prev    = shflUp64(key, 1);
    const bool head        = r.lane == 0 || prev != key;
    const uint64_t heads   = __ballot(head);
    const uint64_t upToMe  = (r.lane == 63) ? ~0ull : ((2ull << r.lane) - 1);
    r.start                = 63 - __clzll(heads & upToMe);
    const uint64_t after   = heads & ~upToMe;
    r.end                  = after ? (__ffsll(static_cast<long long>(after)) - 2) : 63;
    return r;
}

// Inclusive scan with op over the lanes of each run (log-step, limited to the run).
template <typename V, typename Op>
__device__ __forceinline__ V runScan(V v, const WaveRun& r, Op op)
{
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
    {
        const V n = static_cast<V>(shflUp64(static_cast<uint64_t>(v), o));
        if (r.lane - o >= r.start)
            v = op(v, n);
    }
    return v;
}

// Bit interleaving for coordinates below 2^10 (part1by2 / compact1by2).
__host__ __device__ __forceinline__ uint32_t spread3(uint32_t v)
{
    v &= 0x000003FFu;
    v = (v ^ (v << 16)) & 0xFF0000FFu;
    v = (v ^ (v << 8)) & 0x0300F00Fu;
    v = (v ^ (v << 4)) & 0x030C30C3u;
    v = (v ^ (v << 2)) & 0x09249249u;
    return v;
}

__host__ __device__ __forceinline__ uint32_t compact3(uint32_t v)
{
    v &= 0x09249249u;
    v = (v ^ (v >> 2)) & 0x030C30C3u;
    v = (v ^ (v >> 4)) & 0x0300F00Fu;
    v = (v ^ (v >> 8)) & 0xFF0000FFu;
    v = (v ^ (v >> 16)) & 0x000003FFu;
    return v;
}

// Morton code whose 3-bit groups are child slots (x -> 4, y -> 2, z -> 1).
__host__ __device__ __forceinline__ uint32_t morton3(uint32_t x, uint32_t y, uint32_t z)
{
    return (spread3(x) << 2) | (spread3(y) << 1) | spread3(z);
}

// The device's constant-rate clock at the start of a kernel, for the stage timings: events would put a
// packet of their own, with a wait, between the kernels (24 of them took ~60 us of a 50K-point build).
__device__ __forceinline__ void stampStart(uint64_t* stamp)
{
    if (stamp && blockIdx.x == 0 && threadIdx.x == 0)
        *stamp = wall_clock64();
}

// grid-stride helpers
__device__ __forceinline__ uint64_t globalThread()
{
    return static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
}

__device__ __forceinline__ uint64_t globalStride()
{
    return static_cast<uint64_t>(gridDim.x) * blockDim.x;
}

}  // namespace oc
