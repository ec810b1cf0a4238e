// Bounding box of a device-resident cloud: the caller-side step of the reference CLI
// (calculateRealBB, src/boundingbox.h:10-33: per-axis fmin / fmax of the coordinates widened to
// double) as a two-pass min/max reduction, and calculateCubicBB (:35-52) on the host.
#include "bounds.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "device_common.h"
#include "types.h"

namespace oc {

namespace {

// Bound by HBM (40M 15-byte records 108 us, 5.6 TB/s), a small cloud by the launches. In one launch, whose last
// workgroup reduced the others' results, every workgroup's release to the device cost more than the second
// launch (~6 us, mostly under the first one's enqueueing): 1M 15-byte records 37 us a call instead of 19, 10M
// 59 / 37, 40M 170 / 120; records staged through LDS or 512 threads a workgroup gained nothing there.
constexpr int BB_THREADS = 256;
constexpr int BB_BLOCKS  = 1024;

__device__ __forceinline__ void waveMinMax(double v[6])
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
    {
#pragma unroll
        for (int a = 0; a < 3; ++a)
        {
            v[a]     = fmin(v[a], __shfl_xor(v[a], o, 64));
            v[3 + a] = fmax(v[3 + a], __shfl_xor(v[3 + a], o, 64));
        }
    }
}

// Minima and maxima of the workgroup, complete in thread 0.
__device__ __forceinline__ void blockMinMax(double v[6])
{
    __shared__ double lds[BB_THREADS / 64][6];
    waveMinMax(v);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 6; ++k)
            lds[w][k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int i = 1; i < BB_THREADS / 64; ++i)
            for (int a = 0; a < 3; ++a)
            {
                v[a]     = fmin(v[a], lds[i][a]);
                v[3 + a] = fmax(v[3 + a], lds[i][3 + a]);
            }
}

__device__ __forceinline__ void include(double v[6], double x, double y, double z)
{
    v[0] = fmin(v[0], x);
    v[1] = fmin(v[1], y);
    v[2] = fmin(v[2], z);
    v[3] = fmax(v[3], x);
    v[4] = fmax(v[4], y);
    v[5] = fmax(v[5], z);
}

// Device memory of one reduction: the workgroups' minima and maxima, and the final ones.
struct BoundsScratch
{
    double partial[6 * BB_BLOCKS];
    double result[6];
};

// Minima and maxima of each workgroup.
template <typename T>
__global__ __launch_bounds__(BB_THREADS) void kBoundsPartial(const uint8_t* __restrict__ cloud, uint32_t n,
                                                             uint32_t stride, BoundsScratch* __restrict__ scratch)
{
    double v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for (uint64_t i = globalThread(); i < n; i += globalStride())
    {
        double x, y, z;
        loadXYZ<T>(cloud + i * stride, x, y, z);
        include(v, x, y, z);
    }
    blockMinMax(v);
    if (threadIdx.x == 0)
        for (int k = 0; k < 6; ++k)
            scratch->partial[6 * blockIdx.x + k] = v[k];
}

// The final ones, from those of `blocks` workgroups. box: null, or a coherent host mailbox of 6 values and a
// sequence number, so that the caller needs no copy.
__global__ __launch_bounds__(BB_THREADS) void kBoundsFinal(BoundsScratch* scratch, uint32_t blocks, uint64_t* box,
                                                           uint64_t seq)
{
    double v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for (uint32_t b = threadIdx.x; b < blocks; b += BB_THREADS)
        for (int a = 0; a < 3; ++a)
        {
            v[a]     = fmin(v[a], scratch->partial[6 * b + a]);
            v[3 + a] = fmax(v[3 + a], scratch->partial[6 * b + 3 + a]);
        }
    blockMinMax(v);
    if (threadIdx.x != 0)
        return;
    for (int k = 0; k < 6; ++k)
        if (box)
            __hip_atomic_store(box + k, static_cast<uint64_t>(__double_as_longlong(v[k])), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_SYSTEM);
        else
            scratch->result[k] = v[k];
    if (box)
        __hip_atomic_store(box + 6, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

void check(hipError_t e, const char* what)
{
    if (e != hipSuccess)
        throw std::runtime_error(std::string(what) + " failed: " + hipGetErrorString(e));
}

void checkCloud(const uint8_t* deviceCloud, uint32_t n, uint32_t stride, uint8_t cloudType)
{
    if (!deviceCloud || n == 0)
        throw std::runtime_error("the cloud is empty");
    if (cloudType > 1 || stride < (cloudType == 0 ? 12u : 24u))
        throw std::runtime_error("invalid cloud type or stride");
}

void launchBounds(const uint8_t* cloud, uint32_t n, uint32_t stride, uint8_t cloudType, BoundsScratch* scratch,
                  uint64_t* box, uint64_t seq, hipStream_t stream)
{
    const uint32_t blocks =
            static_cast<uint32_t>(std::min<uint64_t>(BB_BLOCKS, (static_cast<uint64_t>(n) + BB_THREADS - 1) / BB_THREADS));
    if (cloudType == CLOUD_FLOAT_UINT8_T)
        kBoundsPartial<float><<<blocks, BB_THREADS, 0, stream>>>(cloud, n, stride, scratch);
    else
        kBoundsPartial<double><<<blocks, BB_THREADS, 0, stream>>>(cloud, n, stride, scratch);
    kBoundsFinal<<<1, BB_THREADS, 0, stream>>>(scratch, blocks, box, seq);
}

// What one reduction uses: a stream of its own, scratch memory and a mailbox. A call takes one from the
// device's pool and gives it back, so calls on several threads run side by side as before, and a call
// alone creates nothing (200K points: 18 us, of 73 with a stream, an allocation and a copy of its own).
struct BoundsContext
{
    hipStream_t stream     = nullptr;
    BoundsScratch* scratch = nullptr;
    uint64_t* box          = nullptr;
    uint64_t seq           = 0;
    BoundsContext()        = default;
    BoundsContext(const BoundsContext&) = delete;
    BoundsContext& operator=(const BoundsContext&) = delete;
    ~BoundsContext()
    {
        if (stream)
        {
            (void)hipStreamSynchronize(stream);
            (void)hipStreamDestroy(stream);
        }
        if (scratch)
            (void)hipFree(scratch);
        if (box)
            (void)hipHostFree(box);
    }
    void create()
    {
        check(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking), "hipStreamCreate");
        check(hipMalloc(&scratch, sizeof(BoundsScratch)), "hipMalloc of the bounding-box scratch");
        check(hipHostMalloc(reinterpret_cast<void**>(&box), 7 * sizeof(uint64_t), hipHostMallocCoherent),
              "hipHostMalloc of the bounding-box mailbox");
        std::fill(box, box + 7, 0);
    }
};

constexpr int MAX_DEVICES         = 64;
constexpr size_t CONTEXTS_KEPT    = 4;  // idle ones per device
std::mutex gContextMutex;
std::mutex gScratchMutex[MAX_DEVICES];
BoundsScratch* gScratchPtr[MAX_DEVICES] = {};

// idle contexts of every device; kept until the process ends (the runtime may be gone by the time
// static objects are destroyed, so they are not freed then)
std::vector<std::unique_ptr<BoundsContext>>* idleContexts()
{
    static auto* pools = new std::vector<std::unique_ptr<BoundsContext>>[MAX_DEVICES];
    return pools;
}

}  // namespace

// The scratch of the allocation-free variant, one per device. In host code this name only stands for
// the object; its device address comes from hipGetSymbolAddress, once per device.
static __device__ __align__(256) BoundsScratch scratch;
static_assert(sizeof(BoundsScratch) == 49200, "the documented size of the static scratch");

void realBoundingBox(const uint8_t* deviceCloud, uint32_t n, uint32_t stride, uint8_t cloudType, int device,
                     double real[6])
{
    checkCloud(deviceCloud, n, stride, cloudType);
    check(hipSetDevice(device), "hipSetDevice");  // (refuses a device that does not exist)
    const size_t pool = static_cast<size_t>(device) % MAX_DEVICES;
    std::unique_ptr<BoundsContext> ctx;
    {
        std::lock_guard<std::mutex> lock(gContextMutex);
        auto& idle = idleContexts()[pool];
        if (device < MAX_DEVICES && !idle.empty())
        {
            ctx = std::move(idle.back());
            idle.pop_back();
        }
    }
    if (!ctx)
    {
        ctx = std::make_unique<BoundsContext>();
        ctx->create();
    }
    // on an error the context goes, its stream drained
    const uint64_t seq = ++ctx->seq;
    launchBounds(deviceCloud, n, stride, cloudType, ctx->scratch, ctx->box, seq, ctx->stream);
    check(hipGetLastError(), "bounding box reduction");
    const auto start = std::chrono::steady_clock::now();
    while (__atomic_load_n(ctx->box + 6, __ATOMIC_ACQUIRE) != seq)
    {
        __builtin_ia32_pause();
        if (std::chrono::steady_clock::now() - start > std::chrono::milliseconds(2))
        {
            check(hipStreamSynchronize(ctx->stream), "bounding box reduction");
            if (__atomic_load_n(ctx->box + 6, __ATOMIC_ACQUIRE) != seq)
                throw std::runtime_error("the bounding box was not published");
        }
    }
    std::memcpy(real, ctx->box, 6 * sizeof(double));
    std::lock_guard<std::mutex> lock(gContextMutex);
    auto& idle = idleContexts()[pool];
    if (device < MAX_DEVICES && idle.size() < CONTEXTS_KEPT)
        idle.push_back(std::move(ctx));
}

void realBoundingBoxNoAlloc(const uint8_t* deviceCloud, uint32_t n, uint32_t stride, uint8_t cloudType, int device,
                            double real[6])
{
    checkCloud(deviceCloud, n, stride, cloudType);
    if (device < 0 || device >= MAX_DEVICES)
        throw std::runtime_error("device " + std::to_string(device) + " is out of range");
    // one call per device at a time: every call on a device shares its scratch
    std::lock_guard<std::mutex> lock(gScratchMutex[device]);
    check(hipSetDevice(device), "hipSetDevice");
    if (!gScratchPtr[device])
    {
        void* p = nullptr;
        check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress of the bounding-box scratch");
        gScratchPtr[device] = static_cast<BoundsScratch*>(p);
    }
    // the null stream: creating a stream would allocate runtime resources
    launchBounds(deviceCloud, n, stride, cloudType, gScratchPtr[device], nullptr, 0, nullptr);
    check(hipGetLastError(), "bounding box reduction launch");
    check(hipMemcpy(real, gScratchPtr[device]->result, sizeof(double) * 6, hipMemcpyDeviceToHost), "bounding box copy");
}

void cubicBoundingBox(const double real[6], double cubic[6])  // src/boundingbox.h:35-52
{
    const double dimX = real[3] - real[0];
    const double dimY = real[4] - real[1];
    const double dimZ = real[5] - real[2];
    const double side = std::fmax(std::fmax(dimX, dimY), dimZ);
    cubic[0]          = real[0] - ((side - dimX) / 2.0f);
    cubic[1]          = real[1] - ((side - dimY) / 2.0f);
    cubic[2]          = real[2] - ((side - dimZ) / 2.0f);
    cubic[3]          = cubic[0] + side;
    cubic[4]          = cubic[1] + side;
    cubic[5]          = cubic[2] + side;
}

}  // namespace oc
