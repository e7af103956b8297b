// On-GPU BVH build for gfx950, replacing the driver-built BLAS/TLAS of the
// reference (src/core/render/accel/blas.c:222-262, tlas.c:535-559).
//
//  1. per-triangle bounds and the centroid bounds of the scene
//  2. 63-bit Morton codes (21 bits per axis) of triangle centroids
//  3. radix sort of (code, triangle) pairs (rocPRIM)
//  4. binary tree by parallel locally-ordered clustering over the Morton order
//     (PLOC, Meister and Bittner, TVCG 2018): every cluster finds the
//     neighbour within kPlocRadius positions whose merged box has the least
//     surface area, mutual nearest neighbours merge, survivors are compacted;
//     repeated until one cluster remains. This refines the LBVH order into a
//     tree of surface-area-heuristic quality.
//  5. top-down collapse into 8-wide nodes: a node is opened greedily by
//     splitting its largest-area child until eight children remain; subtrees
//     of at most leafMax triangles (kLeafMaxTris, or kLeafMaxTrisLarge for
//     scenes above kLargeScene triangles) become leaves whose triangles are
//     written contiguously (depth-first order) as 48-byte records; child
//     boxes are quantised to 8 bits per plane, conservatively
#include <cstring>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_select.hpp>

#include <algorithm>
#include <chrono>
#include <vector>

#include "mrt_internal.hpp"

namespace mrt {

constexpr int kB = 256;

struct Aabb {
    float lo[3], hi[3];
};

__device__ __forceinline__ uint32_t floatToOrdered(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float orderedToFloat(uint32_t u) {
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// World-space triangles from the packed vertices and the meshes' transforms:
// the arithmetic (and rounding) of the host's worldPoint, so that they are the
// triangles an exported scene shows. Moving a mesh then sends 64 bytes per mesh
// instead of re-packing and sending the scene.
__global__ __launch_bounds__(kB) void kPlaceTriangles(const ShaderVertex* vertices, const uint32_t* indices,
                                                     const MeshInfo* meshes, const uint32_t* triMesh,
                                                     const uint32_t* meshTriBase, const float* transforms, uint32_t n,
                                                     float* worldTris) {
    const uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= n) return;
    const uint32_t mi = triMesh[i];
    const MeshInfo& mesh = meshes[mi];
    const float* m = transforms + (size_t)mi * 16u;
    const uint32_t* tri = indices + mesh.indexBase + (size_t)(i - meshTriBase[mi]) * 3u;
    for (int c = 0; c < 3; c++) {
        uint32_t vi = tri[c];
        if (vi >= mesh.vertexCount) vi = 0u;
        const float* v = vertices[mesh.vertexBase + vi].position;
        const float x = v[0], y = v[1], z = v[2];
        for (int r = 0; r < 3; r++)
            worldTris[(size_t)i * 9u + 3u * c + r] = (m[r] * x) + (m[4 + r] * y) + (m[8 + r] * z) + m[12 + r];
    }
}

// per-triangle box, centroid bounds reduced into ordered-int min/max. At most
// kBoundsBlocks blocks: the six atomics that end a block all meet on one line, and one
// block per 256 triangles made them the kernel (384,004 triangles: 108 us, now 40 us).
constexpr uint32_t kBoundsBlocks = 512;
__global__ __launch_bounds__(kB) void kTriBounds(const float* tris9, uint32_t n, Aabb* boxes, uint32_t* centroidBounds) {
    float c[3] = {INFINITY, INFINITY, INFINITY}, C[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t i = blockIdx.x * kB + threadIdx.x; i < n; i += gridDim.x * kB) {
        const float* t = tris9 + (size_t)i * 9u;
        Aabb b;
        for (int a = 0; a < 3; a++) {
            b.lo[a] = fminf(fminf(t[a], t[3 + a]), t[6 + a]);
            b.hi[a] = fmaxf(fmaxf(t[a], t[3 + a]), t[6 + a]);
            float m = 0.5f * (b.lo[a] + b.hi[a]);
            c[a] = fminf(c[a], m);
            C[a] = fmaxf(C[a], m);
        }
        boxes[i] = b;
    }
    __shared__ uint32_t red[6][kB];
    for (int a = 0; a < 3; a++) {
        red[a][threadIdx.x] = floatToOrdered(c[a]);
        red[3 + a][threadIdx.x] = floatToOrdered(C[a]);
    }
    __syncthreads();
    for (int s = kB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            for (int a = 0; a < 3; a++) {
                red[a][threadIdx.x] = min(red[a][threadIdx.x], red[a][threadIdx.x + s]);
                red[3 + a][threadIdx.x] = max(red[3 + a][threadIdx.x], red[3 + a][threadIdx.x + s]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        for (int a = 0; a < 3; a++) {
            atomicMin(&centroidBounds[a], red[a][0]);
            atomicMax(&centroidBounds[3 + a], red[3 + a][0]);
        }
    }
}

__device__ __forceinline__ uint64_t spread21(uint64_t v) {
    v &= 0x1fffffull;
    v = (v | (v << 32)) & 0x1f00000000ffffull;
    v = (v | (v << 16)) & 0x1f0000ff0000ffull;
    v = (v | (v << 8)) & 0x100f00f00f00f00full;
    v = (v | (v << 4)) & 0x10c30c30c30c30c3ull;
    v = (v | (v << 2)) & 0x1249249249249249ull;
    return v;
}

__global__ __launch_bounds__(kB) void kMorton(const Aabb* boxes, uint32_t n, const uint32_t* centroidBounds,
                                             uint64_t* keys, uint32_t* values) {
    uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= n) return;
    uint64_t code = 0;
    for (int a = 0; a < 3; a++) {
        float lo = orderedToFloat(centroidBounds[a]);
        float hi = orderedToFloat(centroidBounds[3 + a]);
        float ext = hi - lo;
        float m = 0.5f * (boxes[i].lo[a] + boxes[i].hi[a]);
        float t = ext > 0.0f ? (m - lo) / ext : 0.5f;
        uint64_t q = (uint64_t)fminf(fmaxf(t * 2097152.0f, 0.0f), 2097151.0f);
        code |= spread21(q) << (2 - a);
    }
    keys[i] = code;
    values[i] = i;
}

__device__ __forceinline__ float halfArea(const Aabb& b) {
    float dx = fmaxf(b.hi[0] - b.lo[0], 0.0f), dy = fmaxf(b.hi[1] - b.lo[1], 0.0f), dz = fmaxf(b.hi[2] - b.lo[2], 0.0f);
    return dx * dy + dy * dz + dz * dx;
}

// Quantisation of one axis of a node: the smallest power-of-two step with
// which 255 steps from the node's lower plane reach its upper plane, checked
// with the decode arithmetic of the traversal (fmaf(q, step, origin)).
__device__ uint32_t nodeExponent(float lo, float hi) {
    float ext = hi - lo;
    int e = 1;
    if (ext > 0.0f) {
        int ex;
        frexpf(ext / 255.0f, &ex);  // ext/255 = m * 2^ex, m in [0.5, 1): 2^ex >= ext/255
        e = min(max(ex + 127, 1), 254);
    }
    while (e < 254 && fmaf(255.0f, __uint_as_float((uint32_t)e << 23), lo) < hi) e++;
    return (uint32_t)e;
}
// Lower and upper plane codes of a child interval [clo, chi] inside the node:
// the exact planes origin + q * step (step a power of two, so q * step is
// exact and the sum is exact in double precision) satisfy lo <= clo and
// hi >= chi, with no rounding in between: the traversal folds the decode into
// its slab distances and never rounds a plane on its own.
__device__ void quantizePlanes(float origin, float step, float clo, float chi, uint32_t& qlo, uint32_t& qhi) {
    float a = floorf((clo - origin) / step), b = ceilf((chi - origin) / step);
    int l = (int)fminf(fmaxf(a, 0.0f), 255.0f), h = (int)fminf(fmaxf(b, 0.0f), 255.0f);
    while (l > 0 && (double)l * (double)step + (double)origin > (double)clo) l--;
    while (h < 255 && (double)h * (double)step + (double)origin < (double)chi) h++;
    qlo = (uint32_t)l;
    qhi = (uint32_t)h;
}

// ---------------------------------------------------------------- PLOC --
// Neighbourhood searched for each cluster's nearest neighbour. With one
// triangle per leaf, radii of 4, 8, 12 and 16 gave 7.97, 8.02, 8.12 and 8.39
// node visits per ray on the 1080p spectral workload (12.60, 12.57, 12.52
// and 13.01 on the 20.8M-triangle one) and 4 traced fastest on both.
constexpr int kPlocRadius = 4;

__device__ __forceinline__ Aabb merge(const Aabb& a, const Aabb& b) {
    Aabb m;
    for (int k = 0; k < 3; k++) {
        m.lo[k] = fminf(a.lo[k], b.lo[k]);
        m.hi[k] = fmaxf(a.hi[k], b.hi[k]);
    }
    return m;
}

// Leaf i is sorted triangle i; nodes n.. are created by merges.
__global__ __launch_bounds__(kB) void kPlocInit(const Aabb* triBoxes, const uint32_t* sortedTri, uint32_t n,
                                               Aabb* boxes, uint32_t* counts, uint32_t* clusters) {
    uint32_t i = blockIdx.x * kB + threadIdx.x;
    if (i >= n) return;
    boxes[i] = triBoxes[sortedTri[i]];
    counts[i] = 1u;
    clusters[i] = i;
}

// Pairs are ordered by (merged surface area, lower index, higher index), so the
// globally smallest pair is always a mutual nearest-neighbour pair and every
// pass merges at least once.
__device__ __forceinline__ bool pairBefore(float c0, int i, int j0, float c1, int j1) {
    if (c0 != c1) return c0 < c1;
    int a0 = min(i, j0), b0 = max(i, j0), a1 = min(i, j1), b1 = max(i, j1);
    return a0 != a1 ? a0 < a1 : b0 < b1;
}

__global__ __launch_bounds__(kB) void kPlocNearest(const uint32_t* clusters, uint32_t m, const Aabb* boxes, int* nn) {
    __shared__ Aabb tile[kB + 2 * kPlocRadius];
    const int b0 = (int)(blockIdx.x * kB);
    for (int t = threadIdx.x; t < kB + 2 * kPlocRadius; t += kB) {
        int g = b0 - kPlocRadius + t;
        if (g >= 0 && g < (int)m) tile[t] = boxes[clusters[g]];
    }
    __syncthreads();
    const int i = b0 + (int)threadIdx.x;
    if (i >= (int)m) return;
    const Aabb a = tile[threadIdx.x + kPlocRadius];
    float best = INFINITY;
    int bj = -1;
    for (int k = -kPlocRadius; k <= kPlocRadius; k++) {
        int j = i + k;
        if (k == 0 || j < 0 || j >= (int)m) continue;
        float c = halfArea(merge(a, tile[threadIdx.x + kPlocRadius + k]));
        if (bj < 0 || pairBefore(c, i, j, best, bj)) {
            best = c;
            bj = j;
        }
    }
    nn[i] = bj;
}

__global__ __launch_bounds__(kB) void kPlocMerge(uint32_t* clusters, uint32_t m, const int* nn, Aabb* boxes,
                                                uint32_t* counts, int2* children, uint32_t n, uint32_t* nodeCounter,
                                                uint8_t* keep) {
    const int i = (int)(blockIdx.x * kB + threadIdx.x);
    if (i >= (int)m) return;
    const int j = nn[i];
    const bool mutual = j >= 0 && nn[j] == i;
    if (mutual && i < j) {
        const uint32_t a = clusters[i], b = clusters[j];
        const uint32_t id = atomicAdd(nodeCounter, 1u);
        children[id - n] = make_int2((int)a, (int)b);
        boxes[id] = merge(boxes[a], boxes[b]);
        counts[id] = counts[a] + counts[b];
        clusters[i] = id;
    }
    keep[i] = (mutual && i > j) ? 0u : 1u;
}

// The last passes in one workgroup: once kPlocSmall clusters are left, a pass
// is a microsecond of work and its launches, compaction and the wait for its
// count were some 65 us. The pairs and their order are those of the passes above.
constexpr int kPlocSmall = 2048;
constexpr int kPlocThreads = 1024;
__global__ __launch_bounds__(kPlocThreads) void kPlocFinish(uint32_t* clusters, uint32_t mBegin, Aabb* boxes,
                                                           uint32_t* counts, int2* children, uint32_t n,
                                                           uint32_t* nodeCounter, uint32_t* left) {
    __shared__ Aabb box[kPlocSmall];
    __shared__ uint32_t id[kPlocSmall], cnt[kPlocSmall];
    __shared__ int nn[kPlocSmall];
    __shared__ uint32_t waveKept[kPlocThreads / 64], nodeNext;
    const int t = (int)threadIdx.x, lane = t & 63, wave = t >> 6;
    int m = (int)mBegin;
    for (int i = t; i < m; i += kPlocThreads) {
        id[i] = clusters[i];
        box[i] = boxes[id[i]];
        cnt[i] = counts[id[i]];
    }
    if (t == 0) nodeNext = *nodeCounter;
    __syncthreads();
    while (m > 1) {
        for (int i = t; i < m; i += kPlocThreads) {
            const Aabb a = box[i];
            float best = INFINITY;
            int bj = -1;
            for (int k = -kPlocRadius; k <= kPlocRadius; k++) {
                const int j = i + k;
                if (k == 0 || j < 0 || j >= m) continue;
                const float c = halfArea(merge(a, box[j]));
                if (bj < 0 || pairBefore(c, i, j, best, bj)) {
                    best = c;
                    bj = j;
                }
            }
            nn[i] = bj;
        }
        __syncthreads();
        // clusters 2t and 2t + 1, so that the survivors keep their order
        Aabb b[2];
        uint32_t newId[2], newCnt[2], kept = 0;
        bool keep[2];
        for (int e = 0; e < 2; e++) {
            const int i = 2 * t + e, j = i < m ? nn[i] : -1;
            const bool mutual = j >= 0 && nn[j] == i;
            keep[e] = i < m && !(mutual && i > j);
            if (!keep[e]) continue;
            kept++;
            b[e] = box[i];
            newId[e] = id[i];
            newCnt[e] = cnt[i];
            if (mutual) {
                newId[e] = atomicAdd(&nodeNext, 1u);
                b[e] = merge(b[e], box[j]);
                newCnt[e] += cnt[j];
                children[newId[e] - n] = make_int2((int)id[i], (int)id[j]);
                boxes[newId[e]] = b[e];
                counts[newId[e]] = newCnt[e];
            }
        }
        uint32_t before = kept;  // inclusive sum over the wave
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t v = (uint32_t)__shfl_up((int)before, off);
            if (lane >= off) before += v;
        }
        if (lane == 63) waveKept[wave] = before;
        before -= kept;
        __syncthreads();
        uint32_t total = 0;
        for (int w = 0; w < kPlocThreads / 64; w++) {
            if (w < wave) before += waveKept[w];
            total += waveKept[w];
        }
        for (int e = 0; e < 2; e++) {
            if (!keep[e]) continue;
            id[before] = newId[e];
            box[before] = b[e];
            cnt[before] = newCnt[e];
            before++;
        }
        __syncthreads();
        if ((int)total >= m) break;  // no progress (uniform): the host reports it
        m = (int)total;
    }
    if (t == 0) {
        clusters[0] = id[0];
        *left = (uint32_t)m;
    }
}

// ------------------------------------------------------------- collapse --
struct CollapseItem {
    uint32_t node;   // binary node: leaf (< n) or merged node (>= n)
    uint32_t wide;   // wide node slot to fill
    uint32_t first;  // first triangle slot of the subtree in leaf order
    uint32_t pad;
};

__device__ __forceinline__ void writeTriangle(const float* tris9, uint32_t t, TriRecord* out) {
    const float* p = tris9 + (size_t)t * 9u;
    TriRecord r;
    r.v0 = make_float4(p[0], p[1], p[2], __uint_as_float(t));
    r.v1 = make_float4(p[3], p[4], p[5], 0.0f);
    r.v2 = make_float4(p[6], p[7], p[8], 0.0f);
    *out = r;
}

// One level of the collapse: eight lanes per wide node, lane k holding child k
// and opening it when it is the largest box among the eight (the lowest lane
// among equals). A lane per node kept its children in indexed arrays, which
// live in scratch memory, and read them one after the other.
__global__ __launch_bounds__(kB) void kCollapse(const CollapseItem* in, const uint32_t* inCount, CollapseItem* out,
                                               uint32_t* outCount, uint32_t* nodeAlloc, uint32_t n,
                                               const int2* children, const uint32_t* counts, const Aabb* boxes,
                                               const uint32_t* sortedTri, const float* tris9, TriRecord* triOut,
                                               BvhNode* nodes, uint32_t nodeCapacity, uint32_t* overflow,
                                               uint32_t leafMax) {
    const uint32_t items = *inCount;
    const int k = (int)(threadIdx.x & 7u);
    // whole groups of eight lanes go round together; a wave leaves with its last group
    for (uint32_t w = (blockIdx.x * kB + threadIdx.x) >> 3; __ballot(w < items) != 0ull; w += gridDim.x * (kB / 8)) {
        const bool live = w < items;
        const CollapseItem it = live ? in[w] : CollapseItem{0u, 0u, 0u, 0u};
        uint32_t slot = it.node, first = it.first, count = 1u;  // child k, once k < cnt
        Aabb b{};
        int cnt = 0;
        if (live) {
            cnt = 1;  // a tiny scene's root may be a leaf
            if (it.node >= n && counts[it.node] > leafMax) {
                cnt = 2;
                const int2 c = children[it.node - n];
                if (k == 1) first = it.first + counts[c.x];
                slot = (uint32_t)(k == 1 ? c.y : c.x);
            }
            if (k < cnt) {
                count = counts[slot];
                b = boxes[slot];
            }
        }
        while (true) {
            // the largest child that has too many triangles for a leaf
            float area = k < cnt && cnt < kBvhWidth && count > leafMax ? halfArea(b) : -1.0f;
            if (!(area == area)) area = -1.0f;  // not a number: never opened
            int best = k;
            float bestArea = area;
            for (int off = 1; off < 8; off <<= 1) {
                const float oa = __shfl_xor(bestArea, off);
                const int ob = __shfl_xor(best, off);
                if (oa > bestArea || (oa == bestArea && ob < best)) {
                    bestArea = oa;
                    best = ob;
                }
            }
            const bool open = bestArea > -1.0f;
            if (__ballot(open) == 0ull) break;
            int2 c2 = make_int2(0, 0);
            uint32_t f2 = 0u;
            if (open && k == best) {
                c2 = children[slot - n];
                f2 = first + counts[c2.x];
                slot = (uint32_t)c2.x;
            }
            const int lane = (int)(threadIdx.x & 63u), from = (lane & ~7) | best;
            const int right = __shfl(c2.y, from);
            const uint32_t rightFirst = (uint32_t)__shfl((int)f2, from);
            if (open && k == cnt) {
                slot = (uint32_t)right;
                first = rightFirst;
            }
            if (open && (k == best || k == cnt)) {
                count = counts[slot];
                b = boxes[slot];
            }
            if (open) cnt++;
        }
        const bool child = k < cnt;
        uint32_t ref = kEmptyRef;
        if (child && count <= leafMax) {
            // the subtree's triangles, depth first, into [first, first + count)
            uint32_t stack[kLeafMaxTrisLarge];
            int sp = 0;
            uint32_t written = 0;
            stack[sp++] = slot;
            while (sp > 0) {
                uint32_t x = stack[--sp];
                if (x < n) {
                    writeTriangle(tris9, sortedTri[x], &triOut[first + written]);
                    written++;
                } else {
                    int2 c = children[x - n];
                    stack[sp++] = (uint32_t)c.y;
                    stack[sp++] = (uint32_t)c.x;
                }
            }
            ref = kLeafBit | ((count - 1u) << 27) | first;
        }
        // slots of the inner children in the node array and the next frontier, one atomic per wave
        const bool inner = child && count > leafMax;
        const unsigned long long mask = __ballot(inner);
        const int lane = (int)(threadIdx.x & 63u);
        uint32_t base = 0, outBase = 0;
        if (mask != 0ull && lane == __ffsll(mask) - 1) {
            base = atomicAdd(nodeAlloc, (uint32_t)__popcll(mask));
            outBase = atomicAdd(outCount, (uint32_t)__popcll(mask));
        }
        if (mask != 0ull) {
            base = (uint32_t)__shfl((int)base, __ffsll(mask) - 1);
            outBase = (uint32_t)__shfl((int)outBase, __ffsll(mask) - 1);
        }
        if (inner) {
            const uint32_t rank = (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
            if (base + rank < nodeCapacity) {
                ref = base + rank;
                out[outBase + rank] = CollapseItem{slot, ref, first, 0u};
            } else {
                atomicAdd(overflow, 1u);
            }
        }
        // the node: its own box, and lane k's plane codes in byte k of each row
        Aabb P{};
        if (live) P = boxes[it.node];
        uint32_t e[3], plane[6];
        for (int a = 0; a < 3; a++) {
            e[a] = nodeExponent(P.lo[a], P.hi[a]);
            uint32_t ql = 0u, qh = 0u;
            if (child) quantizePlanes(P.lo[a], __uint_as_float(e[a] << 23), b.lo[a], b.hi[a], ql, qh);
            plane[a] = ql << ((k & 3) * 8);
            plane[3 + a] = qh << ((k & 3) * 8);
        }
        for (int q = 0; q < 6; q++) {
            plane[q] |= (uint32_t)__shfl_xor((int)plane[q], 1);
            plane[q] |= (uint32_t)__shfl_xor((int)plane[q], 2);
        }
        if (live) {
            BvhNode& node = nodes[it.wide];
            node.child[k] = ref;
            if ((k & 3) == 0) {
                for (int a = 0; a < 3; a++) {
                    node.qlo[a * 2 + (k >> 2)] = plane[a];
                    node.qhi[a * 2 + (k >> 2)] = plane[3 + a];
                }
            }
            if (k == 0) {
                node.ox = P.lo[0];
                node.oy = P.lo[1];
                node.oz = P.lo[2];
                node.packed = e[0] | (e[1] << 8) | (e[2] << 16) | ((uint32_t)cnt << 24);
            }
        }
    }
}

// levels[l]: nodes of level l of the collapse (level 0 is the root). A tree of more
// levels than this is left unfinished, and nothing may traverse it (bvhComplete).
constexpr uint32_t kMaxLevels = 4100;
constexpr uint32_t kLevelBatch = 4;  // levels launched between two looks of the host
__global__ void kInitCollapse(CollapseItem* items, uint32_t* counts, uint32_t* levels, const uint32_t* root) {
    for (uint32_t i = threadIdx.x; i < kMaxLevels + 2u; i += blockDim.x) levels[i] = i == 0u ? 1u : 0u;
    if (threadIdx.x == 0u) {
        items[0] = CollapseItem{*root, 0u, 0u, 0u};
        counts[0] = 1u;  // wide nodes allocated
        counts[1] = 0u;  // overflow
    }
}

__global__ void kInitBuild(uint32_t* centroidBounds, uint32_t* nodeCounter, uint32_t n) {
    if (threadIdx.x < 6u) centroidBounds[threadIdx.x] = threadIdx.x < 3u ? 0xffffffffu : 0u;
    if (threadIdx.x == 0u) *nodeCounter = n;
}

static uint32_t blocks(size_t n) { return (uint32_t)((n + kB - 1) / kB); }

}  // namespace mrt

using namespace mrt;

extern "C" int mrt_build_bvh(mrt_context* ctx, mrt_bvh_stats* stats) {
    if (!ctx) return -1;
    if (!check(hipSetDevice(ctx->device), "hipSetDevice")) return -2;
    hipStream_t s = ctx->stream;
    uint32_t n = ctx->triCount;
    if (stats) memset(stats, 0, sizeof(*stats));
    if (n == 0) {
        ctx->nodes.count = 0;
        ctx->tris.count = 0;
        ctx->bvhMaxDepth = 0;
        ctx->bvhComplete = true;
        return 0;
    }
    hipEventRecord(ctx->evStage[0], s);
    const size_t binNodes = (size_t)2 * n - 1;
    const size_t wideCap = n;  // every wide node but the root is a distinct binary node with more than one triangle
    if (!ctx->nodes.reserve(wideCap) || !ctx->tris.reserve(n)) return -3;
    // everything else in one allocation, which the context keeps for the next build while
    // it is at most kKeepScratch bytes (some 1.9M triangles)
    constexpr size_t kKeepScratch = 256u << 20;
    size_t sortBytes = 0, selectBytes = 0;
    rocprim::radix_sort_pairs(nullptr, sortBytes, (uint64_t*)nullptr, (uint64_t*)nullptr, (uint32_t*)nullptr,
                              (uint32_t*)nullptr, n, 0, 63, s);
    rocprim::select(nullptr, selectBytes, (uint32_t*)nullptr, (uint8_t*)nullptr, (uint32_t*)nullptr, (uint32_t*)nullptr,
                    (size_t)n, s);
    size_t bytes = 0;
    auto take = [&](size_t size) {
        const size_t at = bytes;
        bytes += (size + 255u) & ~(size_t)255u;
        return at;
    };
    const size_t aBoxes = take(binNodes * sizeof(Aabb)), aNodeCounts = take(binNodes * 4u), aValsSorted = take(n * 4u),
                 aChildren = take(n * sizeof(int2)), aClusters0 = take(n * 4u), aClusters1 = take(n * 4u),
                 aSmall = take(64u), aLevels = take((kMaxLevels + 2u) * 4u),
                 aTemp = take(std::max<size_t>(std::max(sortBytes, selectBytes), 1));
    // needed until the tree stands, then the collapse's frontiers take their place
    const size_t aShared = bytes;
    const size_t aTriBoxes = take(n * sizeof(Aabb)), aKeys = take(n * 8u), aKeysSorted = take(n * 8u),
                 aVals = take(n * 4u), aNn = take(n * 4u), aKeep = take(n);
    const size_t aFront0 = aShared;
    bytes = std::max(bytes, aShared + 2u * ((wideCap * sizeof(CollapseItem) + 255u) & ~(size_t)255u));
    const size_t aFront1 = aShared + ((wideCap * sizeof(CollapseItem) + 255u) & ~(size_t)255u);
    if (!ctx->buildScratch.reserve(bytes)) return -3;
    uint8_t* base = ctx->buildScratch.ptr;
    Aabb *boxes = (Aabb*)(base + aBoxes), *triBoxes = (Aabb*)(base + aTriBoxes);
    uint32_t *nodeCounts = (uint32_t*)(base + aNodeCounts), *valsSorted = (uint32_t*)(base + aValsSorted),
             *vals = (uint32_t*)(base + aVals), *small = (uint32_t*)(base + aSmall), *levels = (uint32_t*)(base + aLevels);
    uint32_t* clusters[2] = {(uint32_t*)(base + aClusters0), (uint32_t*)(base + aClusters1)};
    uint64_t *keys = (uint64_t*)(base + aKeys), *keysSorted = (uint64_t*)(base + aKeysSorted);
    int2* children = (int2*)(base + aChildren);
    int* nn = (int*)(base + aNn);
    uint8_t* keep = base + aKeep;
    CollapseItem* front[2] = {(CollapseItem*)(base + aFront0), (CollapseItem*)(base + aFront1)};
    void* temp = base + aTemp;
    uint32_t *cb = small, *nodeCounter = small + 6, *selected = small + 7, *counts = small + 8;
    auto cleanup = [&]() {
        if (ctx->buildScratch.capacity > kKeepScratch) ctx->buildScratch.release();
    };
    // 1-3: bounds, Morton codes, sort
    hipLaunchKernelGGL(kInitBuild, dim3(1), dim3(64), 0, s, cb, nodeCounter, n);
    hipLaunchKernelGGL(kTriBounds, dim3(std::min(blocks(n), kBoundsBlocks)), dim3(kB), 0, s, ctx->worldTris.ptr, n,
                       triBoxes, cb);
    hipLaunchKernelGGL(kMorton, dim3(blocks(n)), dim3(kB), 0, s, triBoxes, n, cb, keys, vals);
    rocprim::radix_sort_pairs(temp, sortBytes, keys, keysSorted, vals, valsSorted, n, 0, 63, s);

    // 4: PLOC
    hipLaunchKernelGGL(kPlocInit, dim3(blocks(n)), dim3(kB), 0, s, triBoxes, valsSorted, n, boxes, nodeCounts,
                       clusters[0]);
    uint32_t m = n;
    int cur = 0;
    uint32_t passes = 0;
    while (m > 1) {
        const bool last = m <= (uint32_t)kPlocSmall;
        if (last) {
            hipLaunchKernelGGL(kPlocFinish, dim3(1), dim3(kPlocThreads), 0, s, clusters[cur], m, boxes, nodeCounts,
                               children, n, nodeCounter, selected);
        } else {
            hipLaunchKernelGGL(kPlocNearest, dim3(blocks(m)), dim3(kB), 0, s, clusters[cur], m, boxes, nn);
            hipLaunchKernelGGL(kPlocMerge, dim3(blocks(m)), dim3(kB), 0, s, clusters[cur], m, nn, boxes, nodeCounts,
                               children, n, nodeCounter, keep);
            size_t tempBytes = selectBytes;
            rocprim::select(temp, tempBytes, clusters[cur], keep, clusters[1 - cur], selected, (size_t)m, s);
            cur = 1 - cur;
        }
        uint32_t next = 0;
        if (!check(hipMemcpyAsync(&next, selected, sizeof(uint32_t), hipMemcpyDeviceToHost, s), "ploc count") ||
            !check(hipStreamSynchronize(s), "ploc sync")) {
            cleanup();
            return -4;
        }
        passes++;
        if (next >= m || passes > 100000u || (last && next != 1u)) {  // every pass merges at least one pair
            cleanup();
            setError("BVH clustering made no progress");
            return -5;
        }
        m = next;
    }

    // the root cluster's box, padded outward by 1e-5 of its size and coordinates
    // so that rounding in the rays' slab test can never reject a ray that
    // reaches a triangle
    Aabb rb{};
    {
        uint32_t root = 0;
        if (!check(hipMemcpyAsync(&root, clusters[cur], sizeof(root), hipMemcpyDeviceToHost, s), "root") ||
            !check(hipStreamSynchronize(s), "root sync") ||
            !check(hipMemcpy(&rb, boxes + root, sizeof(rb), hipMemcpyDeviceToHost), "root box")) {
            cleanup();
            return -4;
        }
        for (int a = 0; a < 3; a++) {
            const float ext = rb.hi[a] - rb.lo[a];
            const bool finite = std::isfinite(rb.lo[a]) && std::isfinite(rb.hi[a]) && ext >= 0.0f;
            ctx->sceneBoxLo[a] = finite ? rb.lo[a] - 1e-5f * (fabsf(rb.lo[a]) + ext) - 1e-30f : -INFINITY;
            ctx->sceneBoxHi[a] = finite ? rb.hi[a] + 1e-5f * (fabsf(rb.hi[a]) + ext) + 1e-30f : INFINITY;
        }
    }

    // 5: collapse into 8-wide nodes, writing triangle records in leaf order. A level's
    // length is read by the next level's launch; the host looks after every few levels
    hipLaunchKernelGGL(kInitCollapse, dim3(1), dim3(kB), 0, s, front[0], counts, levels, clusters[cur]);
    uint32_t depth = 0, launched = 0, hostCounts[2] = {1, 0}, lengths[kLevelBatch + 1];
    uint64_t bound = 1;  // of a level's length
    static_assert(kMaxLevels % kLevelBatch == 0, "levels are launched in whole batches");
    int fc = 0;
    while (launched < kMaxLevels) {
        for (uint32_t l = 0; l < kLevelBatch; l++) {
            const uint32_t grid = std::min(blocks((size_t)bound * 8u), 8192u);
            hipLaunchKernelGGL(kCollapse, dim3(grid), dim3(kB), 0, s, front[fc], levels + launched, front[1 - fc],
                               levels + launched + 1u, counts, n, children, nodeCounts, boxes, valsSorted,
                               ctx->worldTris.ptr, ctx->tris.ptr, ctx->nodes.ptr, (uint32_t)wideCap, counts + 1,
                               n > kLargeScene ? kLeafMaxTrisLarge : kLeafMaxTris);
            fc = 1 - fc;
            launched++;
            bound = std::min<uint64_t>(bound * 8u, n);
        }
        if (!check(hipMemcpyAsync(lengths, levels + launched - kLevelBatch, (kLevelBatch + 1u) * 4u, hipMemcpyDeviceToHost, s),
                   "collapse") ||
            !check(hipMemcpyAsync(hostCounts, counts, sizeof(hostCounts), hipMemcpyDeviceToHost, s), "collapse") ||
            !check(hipStreamSynchronize(s), "collapse sync")) {
            cleanup();
            return -4;
        }
        for (uint32_t l = 0; l < kLevelBatch; l++) depth += lengths[l] != 0u;
        if (lengths[kLevelBatch] == 0u) break;
    }
    hipEventRecord(ctx->evStage[1], s);
    hipStreamSynchronize(s);
    cleanup();
    if (hostCounts[1] != 0) {
        setError("BVH collapse exceeded node capacity");
        return -5;
    }
    ctx->nodes.count = hostCounts[0];
    ctx->tris.count = n;
    ctx->bvhMaxDepth = depth;
    ctx->bvhComplete = lengths[kLevelBatch] == 0u;
    float ms = 0.0f;
    hipEventElapsedTime(&ms, ctx->evStage[0], ctx->evStage[1]);
    if (stats) {
        stats->buildMs = ms;
        stats->nodeCount = hostCounts[0];
        stats->leafTriangles = n;
        stats->maxDepth = depth;
        for (int a = 0; a < 3; a++) {
            stats->boxMin[a] = rb.lo[a];
            stats->boxMax[a] = rb.hi[a];
        }
    }
    return check(hipGetLastError(), "bvh build") ? 0 : -4;
}

extern "C" int mrt_place_triangles(mrt_context* ctx, const float* transforms, uint32_t meshCount) {
    if (!ctx || (meshCount && !transforms)) return -1;
    if (!check(hipSetDevice(ctx->device), "hipSetDevice")) return -2;
    const uint32_t n = ctx->triCount;
    if (meshCount != ctx->meshes.count || meshCount != ctx->meshTriBase.count) {
        setError("mrt_place_triangles: mesh count differs from the uploaded geometry");
        return -1;
    }
    if (!ctx->worldTris.reserve((size_t)n * 9u) || !ctx->meshTransforms.upload(transforms, (size_t)meshCount * 16u, ctx->stream))
        return -3;
    ctx->worldTris.count = (size_t)n * 9u;
    if (n > 0)
        hipLaunchKernelGGL(kPlaceTriangles, dim3(blocks(n)), dim3(kB), 0, ctx->stream, ctx->vertices.ptr,
                           ctx->indices.ptr, ctx->meshes.ptr, ctx->triMesh.ptr, ctx->meshTriBase.ptr,
                           ctx->meshTransforms.ptr, n, ctx->worldTris.ptr);
    ctx->shadeTrisDirty = true;
    return check(hipGetLastError(), "place triangles") && check(hipStreamSynchronize(ctx->stream), "place triangles") ? 0 : -4;
}
