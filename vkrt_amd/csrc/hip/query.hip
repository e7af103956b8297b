// Ray queries for caller-supplied rays: closest hits and occlusion, on host
// arrays and on device memory.
#include <algorithm>

#include "dev_traverse.h"
#include "mrt_internal.hpp"

namespace mrt {

// Where a query writes; null arrays are left out.
struct QueryOut {
    uint32_t *mesh, *prim;
    float *t, *bary;
    uint32_t* visibility;  // of an occlusion query
};

// One ray per lane, with lanes refilled as in kExtend. A wavefront takes runs of
// 64 rays: its own, then every run a whole grid of wavefronts further on, so
// nothing is claimed and nothing is cleared before a launch. A traversal waits on
// its node loads, so it wants the six wavefronts per SIMD that the registers
// and LDS stacks allow: 2^22 random rays at 1,048,820 triangles take 1.30 ms
// (3.2 Grays/s); one wavefront per SIMD without refill took 6.0 ms.
template <bool ANY, bool ALPHA>
__global__ __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(ALPHA ? 4 : 6))) void kQuery(
    SceneView sv, const float4* rays, uint32_t n, uint32_t keyBase, QueryOut out, uint32_t* gstack, uint32_t* dropped) {
    __shared__ uint2 lds[kLdsStackEntries];
    TraversalStack st(lds, gstack);
    const uint32_t lane = threadIdx.x & 63u, stride = gridDim.x * kTraceBlock;
    const uint64_t lanesBelow = (1ull << lane) - 1ull;
    uint32_t run = (blockIdx.x * kTraceBlock + threadIdx.x) & ~63u, next = run, end = min(run + 64u, n);
    uint32_t rayId = kNoRay, alphaKey = 0u;
    float tmin = 0.0f;
    TraversalRay r;
    ClosestState cs;
    closestBegin(cs, st, 0.0f);
    auto finish = [&](uint32_t i, const Hit& h) {
        if (ANY) {
            out.visibility[i] = classifyOccluder(sv, h.tri);
            return;
        }
        const bool hit = h.tri != kNoHit && h.tri < sv.triCount;
        const uint32_t mesh = hit ? sv.triMesh[h.tri] : VKRT_INVALID_INDEX;
        out.mesh[i] = mesh;
        out.prim[i] = hit ? h.tri - sv.meshTriBase[mesh] : VKRT_INVALID_INDEX;
        if (out.t) out.t[i] = hit ? h.t : 0.0f;
        if (out.bary) {
            out.bary[2 * (size_t)i] = hit ? h.u : 0.0f;
            out.bary[2 * (size_t)i + 1] = hit ? h.v : 0.0f;
        }
    };
    while (true) {
        const uint64_t idleMask = __ballot(rayId == kNoRay);
        const uint32_t idle = (uint32_t)__popcll(idleMask);
        if (idle >= kRefillLanes && run < n) {
            const uint32_t i = next + (uint32_t)__popcll(idleMask & lanesBelow);
            if (rayId == kNoRay && i < end) {
                const float4 a = rays[2 * (size_t)i], b = rays[2 * (size_t)i + 1];
                tmin = a.w;
                r = makeTraversalRay(xyz(a), xyz(b));
                // no tree: a miss at once. The frames' test against the scene's box is left
                // out: it is for intervals ahead of the origin and unit directions
                if (sv.nodeCount != 0u) {
                    // a query ray has no path: its index is its key
                    if (ALPHA) alphaKey = alphaRayKey(alphaSalt(0u, 0ull, 0u, 3u), keyBase + i);
                    closestBegin(cs, st, b.w);
                    rayId = i;
                } else {
                    finish(i, Hit{0.0f, kNoHit, 0.0f, 0.0f});
                }
            }
            next = min(next + idle, end);
            if (next >= end) {  // n <= 2^30, so the next run's index does not wrap
                run += stride;
                next = run;
                end = min(run + 64u, n);
            }
        }
        if (rayId != kNoRay) {
            const bool more = ANY ? anyStep<ALPHA>(sv, r, tmin, cs, st, alphaKey)
                                  : closestStep<ALPHA, ALPHA>(sv, r, tmin, cs, st, alphaKey);
            if (!more) {
                finish(rayId, cs.h);
                rayId = kNoRay;
            }
        }
        if (run >= n && __ballot(rayId != kNoRay) == 0ull) break;
    }
    if (dropped && st.dropped) atomicAdd(dropped, st.dropped);
}

// Queries n rays in device memory; maxBlocks: how many blocks `stack` has room for.
template <bool ANY>
static void launchQuery(mrt_context* ctx, const float4* rays, uint32_t n, uint32_t keyBase, const QueryOut& out,
                        uint32_t* stack, uint32_t maxBlocks, uint32_t* dropped) {
    const SceneView sv = ctx->view();
    const bool alpha = sv.triAlpha != nullptr;
    // the blocks that are resident at once, or one wavefront per 64 rays
    const uint32_t resident = (uint32_t)std::max(1, ctx->cuCount) * (alpha ? 4u : 6u);
    const uint32_t blocks = std::min(std::min(resident, maxBlocks), (n + kTraceBlock - 1u) / kTraceBlock);
    if (alpha)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(kQuery<ANY, true>), dim3(blocks), dim3(kTraceBlock), 0, ctx->stream, sv, rays,
                           n, keyBase, out, stack, dropped);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(kQuery<ANY, false>), dim3(blocks), dim3(kTraceBlock), 0, ctx->stream, sv,
                           rays, n, keyBase, out, stack, dropped);
}

}  // namespace mrt

using namespace mrt;

// A tree of more levels than the build follows refers to nodes that were never
// written. Frames refuse far shallower ones (setupFrame).
bool mrt::traceable(const mrt_context* ctx) {
    if (ctx->triCount == 0u || ctx->bvhComplete) return true;
    setError("BVH deeper than the build supports");
    return false;
}

// Host queries go through device buffers of the context in pieces of at most
// kQueryPiece rays (32 bytes in and 20 out per ray: 54 MB), which stay for the next call.
constexpr size_t kQueryPiece = 1u << 20;

template <bool ANY>
static int runQuery(mrt_context* ctx, const float* rays, size_t count, const QueryOut& host) {
    if (!check(hipSetDevice(ctx->device), "hipSetDevice") || !traceable(ctx)) return -2;
    if (!ensureTraversalScratch(ctx)) return -3;
    if (count > 0xFFFFFFFFull / 2) {
        setError("too many rays");
        return -1;
    }
    hipStream_t s = ctx->stream;
    const size_t piece = std::min(count, kQueryPiece);
    if (!ctx->queryRays.reserve(2 * piece) || !ctx->queryOut.reserve((ANY ? 1 : 5) * piece)) return -3;
    for (size_t begin = 0; begin < count; begin += piece) {
        const uint32_t n = (uint32_t)std::min(piece, count - begin);
        uint32_t* o = ctx->queryOut.ptr;
        QueryOut dev{};
        if (ANY)
            dev.visibility = o;
        else
            dev = QueryOut{o, o + n, reinterpret_cast<float*>(o + 2 * (size_t)n), reinterpret_cast<float*>(o + 3 * (size_t)n),
                           nullptr};
        if (!check(hipMemcpyAsync(ctx->queryRays.ptr, rays + 8 * begin, (size_t)n * 8 * sizeof(float),
                                  hipMemcpyHostToDevice, s),
                   "upload rays"))
            return -4;
        launchQuery<ANY>(ctx, ctx->queryRays.ptr, n, (uint32_t)begin, dev, ctx->traversalStack.ptr, ctx->traceGrid,
                         nullptr);
        auto read = [&](void* dst, const void* src, size_t words) {
            return !dst || check(hipMemcpyAsync(dst, src, words * 4u, hipMemcpyDeviceToHost, s), "read hits");
        };
        bool ok = check(hipGetLastError(), "trace query");
        if (ANY)
            ok = ok && read(host.visibility + begin, dev.visibility, n);
        else
            ok = ok && read(host.mesh + begin, dev.mesh, n) && read(host.prim + begin, dev.prim, n) &&
                 read(host.t ? host.t + begin : nullptr, dev.t, n) &&
                 read(host.bary ? host.bary + 2 * begin : nullptr, dev.bary, 2 * (size_t)n);
        if (!check(hipStreamSynchronize(s), "trace query") || !ok) return -4;
    }
    return 0;
}

// ------------------------------------------------------ allocation-free --
// The allocation-free ray query uses the context's traversal stacks when it
// has them (from the first frame or host query). Before that it has one fixed
// device array: a header whose word 0 counts dropped traversal-stack pushes,
// then the global traversal stacks of a grid of kNoAllocBlocks blocks
// (kTraceBlock lanes x kGlobalStackWords words each): 64 + 256 * 256 * 232 words,
// about 61 MB, held on every device the library runs on until the process ends.
constexpr uint32_t kNoAllocBlocks = 256;
constexpr size_t kNoAllocHeaderWords = 64;
constexpr size_t kNoAllocScratchWords =
    kNoAllocHeaderWords + (size_t)kNoAllocBlocks * kTraceBlock * (size_t)kGlobalStackWords;
static __device__ __align__(256) uint32_t scratch[kNoAllocScratchWords];

// Device address of scratch on the current device; called once per context
// at creation with its device current (the array's name is not a device
// address in host code).
bool mrt::noAllocScratchInit(mrt_context* ctx) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
        (void)hipGetLastError();
        ctx->noAllocScratch = nullptr;
        return false;
    }
    ctx->noAllocScratch = static_cast<uint32_t*>(p);
    return true;
}

__global__ void kClearWords(uint32_t* p, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

extern "C" int mrt_trace_rays_noalloc(mrt_context* ctx, const float* deviceRays, size_t count, uint32_t* deviceMesh,
                                      uint32_t* devicePrim, float* deviceT, float* deviceBary) {
    if (!ctx || !deviceRays || !deviceMesh || !devicePrim) return -1;
    if (count > MRT_NOALLOC_MAX_RAYS) {
        setError("allocation-free ray query: more rays than its maximum of 2^30 per call");
        return -1;
    }
    if (!ctx->noAllocScratch) {
        setError("allocation-free ray query: no device address for its scratch array");
        return -2;
    }
    if (!check(hipSetDevice(ctx->device), "hipSetDevice") || !traceable(ctx)) return -2;
    if (count == 0) return 0;
    hipStream_t s = ctx->stream;
    const bool own = ctx->traceGrid != 0u && ctx->traversalStack.ptr &&
                     ctx->traversalStack.capacity >= (size_t)ctx->traceGrid * kTraceBlock * kGlobalStackWords;
    uint32_t* stack = own ? ctx->traversalStack.ptr : ctx->noAllocScratch + kNoAllocHeaderWords;
    // What the count holds: pushes beyond the stack, which a tree of few enough levels cannot
    // make, and traversals cut off at their visit limit, which a tree of no more nodes and
    // leaves than that cannot reach. Where neither can be there is nothing to clear and read
    const bool counted = ctx->bvhMaxDepth * (kBvhWidth - 1u) + 1u > (uint32_t)(kLdsStack + kGlobalStack) ||
                         ctx->nodes.count + ctx->tris.count > kMaxTraversalSteps;
    if (counted)
        hipLaunchKernelGGL(kClearWords, dim3(1), dim3((uint32_t)kNoAllocHeaderWords), 0, s, ctx->noAllocScratch,
                           (uint32_t)kNoAllocHeaderWords);
    launchQuery<false>(ctx, reinterpret_cast<const float4*>(deviceRays), (uint32_t)count, 0u,
                       QueryOut{deviceMesh, devicePrim, deviceT, deviceBary, nullptr}, stack,
                       own ? ctx->traceGrid : kNoAllocBlocks, counted ? ctx->noAllocScratch : nullptr);
    if (!check(hipGetLastError(), "allocation-free ray query launch") ||
        !check(hipStreamSynchronize(s), "allocation-free ray query"))
        return -4;
    uint32_t dropped = 0;
    if (counted &&
        !check(hipMemcpy(&dropped, ctx->noAllocScratch, sizeof(dropped), hipMemcpyDeviceToHost), "read counter"))
        return -4;
    if (dropped) {
        setError("traversal stack overflow or visit limit");
        return -5;
    }
    return 0;
}

extern "C" int mrt_trace_rays(mrt_context* ctx, const float* rays, size_t count, uint32_t* outMesh, uint32_t* outPrim,
                              float* outT, float* outBary) {
    if (!ctx || !rays || !outMesh || !outPrim) return -1;
    return runQuery<false>(ctx, rays, count, QueryOut{outMesh, outPrim, outT, outBary, nullptr});
}

extern "C" int mrt_trace_shadow_rays(mrt_context* ctx, const float* rays, size_t count, uint32_t* outVisibility) {
    if (!ctx || !rays || !outVisibility) return -1;
    return runQuery<true>(ctx, rays, count, QueryOut{nullptr, nullptr, nullptr, nullptr, outVisibility});
}
