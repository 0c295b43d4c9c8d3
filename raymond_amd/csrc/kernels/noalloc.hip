// Allocation-free closest-hit batches: rm_trace_closest_noalloc.
//
// For callers that cannot allocate device memory (code under HIP graph
// capture, tight serving loops): the caller passes device arrays for the
// rays and the hits, and the intermediate state lives in `scratch`, a
// fixed array of this library in device memory.  Each GPU holds its own
// copy of the array until the process ends; host code reaches it only
// through the address hipGetSymbolAddress returns for that GPU, taken once
// when the device is created.  Every call on a GPU shares that copy, so
// calls that overlap on one GPU race.
//
// The trace kernel reads the caller's rays and writes the caller's hits.
// `scratch` holds the persistent scheduler's counters, which a batch of more
// than one 64-ray batch per wave uses and a kernel clears first (no memset
// node), and a copy of the rays for callers whose hit arrays overlap them.
// Without the two copies to and from columns that every call made, 100003
// rays over 82k triangles take 83 to 85 us instead of 99 to 107; what is left
// is the longest ray's chain of steps.
#include <hip/hip_runtime.h>

#include "../host/core.h"
#include "noalloc_api.h"
#include "trace_api.h"

namespace rm {

constexpr size_t kNoAllocHeadWords = kFetchWords;
static __device__ __align__(256) uint32_t scratch[kNoAllocHeadWords + 8 * (size_t)kNoAllocMaxRays];

void noalloc_init(rm_device* dev) {
    void* ptr = nullptr;
    RM_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    RM_REQUIRE(ptr != nullptr, "no device address for the allocation-free scratch array");
    dev->noalloc_scratch = static_cast<uint32_t*>(ptr);
}

__global__ void noalloc_clear_kernel(uint32_t* s) { s[threadIdx.x] = 0u; }

__global__ void noalloc_copy_kernel(const float4* __restrict__ rays, uint32_t n, float4* __restrict__ copy) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < 2u * n) copy[i] = rays[i];
}

static bool overlap(const void* a, size_t na, const void* b, size_t nb) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return x < y + nb && y < x + na;
}

void trace_closest_noalloc(rm_scene* sc, const float* rays, uint32_t n, float* t, uint32_t* inst, uint32_t* prim,
                           float* bary, hipStream_t stream) {
    RM_REQUIRE(sc->accel_built, "acceleration structure not built");
    RM_REQUIRE(n <= kNoAllocMaxRays, "rm_trace_closest_noalloc takes at most " + std::to_string(kNoAllocMaxRays) +
                                         " rays per call (got " + std::to_string(n) + ")");
    RM_REQUIRE((reinterpret_cast<uintptr_t>(rays) & 15u) == 0 && (reinterpret_cast<uintptr_t>(bary) & 7u) == 0,
               "rays must be 16-byte and bary 8-byte aligned device arrays");
    uint32_t* s = sc->dev->noalloc_scratch;
    RM_REQUIRE(s != nullptr, "allocation-free scratch array not set up on this device");
    if (n == 0) return;
    hipStream_t st = stream ? stream : sc->dev->stream;
    ClosestArgs a{};
    a.nodes = sc->d_nodes.as<Bvh8Node>();
    a.tlas = sc->two_level ? sc->d_tlas.as<TlasInstance>() : nullptr;
    a.root2l = sc->root2l;
    a.tris = sc->d_tris.as<BvhTri>();
    a.count = n;
    a.fetch = s;
    a.rays = reinterpret_cast<const float4*>(rays);
    a.bary = reinterpret_cast<float2*>(bary);
    a.hits.t = t;
    a.hits.inst = inst;
    a.hits.prim = prim;
    a.spill = sc->d_spill.as<uint2>();
    a.counters = nullptr;
    const size_t nr = (size_t)n * 32, nh = (size_t)n * 4;
    if (overlap(rays, nr, t, nh) || overlap(rays, nr, inst, nh) || overlap(rays, nr, prim, nh) ||
        overlap(rays, nr, bary, 2 * nh)) {
        float4* copy = reinterpret_cast<float4*>(s + kNoAllocHeadWords);
        hipLaunchKernelGGL(noalloc_copy_kernel, dim3((2 * n + 255) / 256), dim3(256), 0, st, a.rays, n, copy);
        RM_HIP(hipGetLastError());
        a.rays = copy;
    }
    const int tblocks = sc->dev->props.multiProcessorCount * sc->dev->trace_blocks_per_cu;
    if ((n + kTraceBlock - 1) / kTraceBlock > (uint32_t)trace_closest_blocks(sc->two_level, tblocks)) {
        hipLaunchKernelGGL(noalloc_clear_kernel, dim3(1), dim3(kFetchWords), 0, st, s);
        RM_HIP(hipGetLastError());
    }
    RM_HIP(launch_trace_closest(a, tblocks, false, st));
}

}  // namespace rm
