// BVH8 builder on the GPU: the tree host/bvh_build.cpp builds (32-bin SAH
// over the three axes, collapse to 8-wide nodes by dynamic programming,
// octant slots, conservative 8-bit boxes), from the same expressions in the
// same precision, so both builders choose the same splits and write the same
// nodes.  They differ in three places, none of which a hit depends on:
//   * a range whose centroids coincide halves by position, and phase 1 leaves
//     records in the order of its atomics: which triangles go where then
//     differs from the host's tree, above kBig also from run to run;
//   * the exponent's ceil(log2(x)) is exact here and rounded on the host;
//   * centroids less than about 1e-37 apart give an infinite bin scale, whose
//     conversion to an integer differs between the processors.
//
// The host builder takes 0.84 s for 1.3M triangles (16 threads, upload
// included); this one takes 5.4 ms: 0.9 phase 1, 0.6 phase 2, 1.3 phase 3,
// 1.5 phase 5, the rest set-up, allocation and the gaps between its 100
// launches.  Phases 1 and 5 wait on memory and launches, phases 2 and 3 on
// their own split arithmetic.
// Triangles are 32-byte records (bounds, id) that partitions move, so every
// pass reads them in order:
//   1. ranges above kBig records: level by level, several workgroups per
//      range (bins through global atomics, bounds as one partial union each);
//   2. ranges of kSmall+1..kBig records: one workgroup builds a range down
//      to kSmall records, bins in LDS, with its own stack of ranges;
//   3. ranges of at most kSmall = 64 records: one wave builds the whole
//      subtree, one record per lane, all ranges of a level at a time.  Bins
//      would be mostly empty there: each lane scores the split after its own
//      record's bin against the records of its range instead, which visits
//      exactly the splits that separate records (the split after an empty
//      bin equals one of those, and the host keeps the first).  The wave
//      then fills its subtree's collapse costs;
//   4. collapse costs above the small subtrees, deepest level first;
//   5. BVH8 nodes level by level in the host builder's breadth-first order:
//      child lists and slots, a scan of the counts, then boxes, triangles
//      and the next level.
// A split at triangle position m names its children: 2 m - 1 and 2 m.  Split
// positions are unique within a tree, so no node counter is shared.
#include <algorithm>

#include "bvh_build_api.h"

namespace rm {

namespace {

constexpr int kBins = 32;
constexpr uint32_t kSmall = 64;
// One workgroup's chain of splits (12-15 us each) bounds small builds: 4096
// instead of 1024 here took 1516 against 881 us for 4096 triangles, and 1.03
// against 0.61 ms in phase 2 for 1.3M.
constexpr uint32_t kBig = 1024;
constexpr uint32_t kChunk = 4096;    // records of one workgroup in phase 1
constexpr uint32_t kRecBlocks = 1024;  // workgroups that write the records
constexpr uint32_t kMaxLevels = 96;  // phase 1 levels; deeper input goes to the host builder
constexpr uint32_t kBvhLevels = 64;  // BVH8 levels
constexpr int kBlock = 256;
constexpr int kBinWords = 3 * kBins * 7;  // bounds (6) and count per bin and axis

constexpr double kCostNode = 1.0;  // as in the host builder
constexpr double kCostTri = 0.6;

struct alignas(16) Rec {
    float lx, ly, lz;
    uint32_t id;
    float hx, hy, hz;
    uint32_t pad;
};

struct alignas(16) Node2 {
    float lo[3];
    int32_t left;  // -1: leaf; the right child is left + 1
    float hi[3];
    uint32_t first;
    uint32_t count, depth, pad0, pad1;
};

// Bounds of records and of their centroids.
struct Bounds {
    float v[12];  // box lo, box hi, centroid lo, centroid hi
};

// A range of phase 1.  Its bounds are the union of the partial bounds that
// the workgroups of its parent's partition wrote for its side.
struct BigRange {
    uint32_t begin, end, node, depth, chunk0;
    uint32_t part0, parts, side;  // those workgroups
    Bounds bounds;                // written by the range's first bins workgroup
    // the chosen split
    int axis, split;
    float clo, k;
    uint32_t left_count;
    uint32_t cursor[2];  // records written left and right so far
    int child[2];        // index of the child in the next level's ranges, or -1
};

struct Range {
    uint32_t begin, end, node, depth, buf;
};

struct Counters2 {
    uint32_t big[kMaxLevels + 1];     // ranges of each phase-1 level
    uint32_t chunks[kMaxLevels + 1];  // workgroups of each phase-1 level
    uint32_t mid, small, upper, max_depth;
    uint32_t nonfinite, bad_quant;
    uint32_t level_base[kBvhLevels + 1], level_count[kBvhLevels + 1], tri_base[kBvhLevels + 1];
};

struct BuildArgs {
    const float* vertices;
    const uint32_t* indices;
    const BvhSource* sources;
    uint32_t num_sources, n, max_leaf;
    Rec* rec[2];
    Node2* nodes;
    float* cost;        // 8 per node
    uint64_t* how;      // 8 bytes per node
    uint32_t* order;    // triangle ids in leaf order
    BigRange* big[2];
    uint2* chunk_map[2];  // (range, part) of each workgroup
    Bounds* partial[2];   // [workgroup][side]
    uint32_t* bins;     // kBinWords per phase-1 range
    Range* mid;
    Range* small;
    uint32_t* upper;    // nodes split in phases 1 and 2
    Counters2* c;
    // phase 5
    uint32_t* pend[2];
    uint32_t* slots;    // 8 per pending node: child | leaf << 31, or ~0
    uint32_t* counts;   // per pending node: internal children | triangles << 8
    uint2* tile_sums;
    Bvh8Node* out_nodes;
    BvhTri* out_tris;
};

__device__ inline uint32_t enc(float f) {
    const uint32_t u = __float_as_uint(f);
    return u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
}
__device__ inline float dec(uint32_t e) {
    return __uint_as_float(e ^ ((uint32_t)((int32_t)~e >> 31) | 0x80000000u));
}
constexpr uint32_t kEncPosInf = 0xff800000u;  // enc(+inf): an empty lower bound
constexpr uint32_t kEncNegInf = 0x007fffffu;  // enc(-inf): an empty upper bound

struct Box3 {
    float lo[3], hi[3];
    __device__ void clear() {
#pragma unroll
        for (int a = 0; a < 3; a++) {
            lo[a] = __builtin_huge_valf();
            hi[a] = -__builtin_huge_valf();
        }
    }
    __device__ double area() const {
        const double dx = fmax(0.0, (double)hi[0] - (double)lo[0]);
        const double dy = fmax(0.0, (double)hi[1] - (double)lo[1]);
        const double dz = fmax(0.0, (double)hi[2] - (double)lo[2]);
        return 2.0 * (dx * dy + dy * dz + dz * dx);
    }
};

__device__ inline float bin_scale(float ext) { return (float)kBins * (1.0f - 1e-6f) / ext; }
__device__ inline int bin_of(float c, float clo, float k) {
    const int b = (int)((c - clo) * k);
    return min(max(b, 0), kBins - 1);
}
__device__ inline double split_cost(const Box3& l, uint32_t lc, const Box3& r, uint32_t rc, double parent_area) {
    return 1.0 + (l.area() * lc + r.area() * rc) / fmax(parent_area, 1e-30);
}
__device__ inline float center(float lo, float hi) { return 0.5f * (lo + hi); }

__device__ inline const BvhSource& source_of(const BuildArgs& a, uint32_t tri) {
    uint32_t lo = 0, hi = a.num_sources;
    while (hi - lo > 1) {
        const uint32_t m = (lo + hi) / 2;
        if (a.sources[m].first <= tri) lo = m;
        else hi = m;
    }
    return a.sources[lo];
}
__device__ inline void triangle(const BuildArgs& a, const BvhSource& s, uint32_t face, vec3 v[3]) {
    const uint32_t* ix = a.indices + 3 * ((size_t)s.face_offset + face);
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const float* p = a.vertices + 3 * ((size_t)s.vertex_offset + ix[j]);
        const vec3 q(p[0], p[1], p[2]);
        v[j] = s.transformed ? s.transform.point(q) : q;
    }
}

__device__ inline float wave_min(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o));
    return v;
}
__device__ inline float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

__device__ inline void grow(Box3& box, Box3& cbox, const Rec& r) {
    const float lo[3] = {r.lx, r.ly, r.lz}, hi[3] = {r.hx, r.hy, r.hz};
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float c = center(lo[k], hi[k]);
        box.lo[k] = fminf(box.lo[k], lo[k]);
        box.hi[k] = fmaxf(box.hi[k], hi[k]);
        cbox.lo[k] = fminf(cbox.lo[k], c);
        cbox.hi[k] = fmaxf(cbox.hi[k], c);
    }
}
__device__ inline void wave_reduce(Box3& b) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
        b.lo[k] = wave_min(b.lo[k]);
        b.hi[k] = wave_max(b.hi[k]);
    }
}

// Union over the workgroup, in every thread (kBlock threads; `part` is one
// entry per wave).
__device__ inline void block_reduce(Box3& box, Box3& cbox, Bounds* part) {
    wave_reduce(box);
    wave_reduce(cbox);
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x & 63;
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            part[wave].v[k] = box.lo[k];
            part[wave].v[3 + k] = box.hi[k];
            part[wave].v[6 + k] = cbox.lo[k];
            part[wave].v[9 + k] = cbox.hi[k];
        }
    }
    __syncthreads();
    for (int w = 0; w < kBlock / 64; w++) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            box.lo[k] = fminf(box.lo[k], part[w].v[k]);
            box.hi[k] = fmaxf(box.hi[k], part[w].v[3 + k]);
            cbox.lo[k] = fminf(cbox.lo[k], part[w].v[6 + k]);
            cbox.hi[k] = fmaxf(cbox.hi[k], part[w].v[9 + k]);
        }
    }
}
__device__ inline Bounds bounds_of(const Box3& box, const Box3& cbox) {
    Bounds b;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        b.v[k] = box.lo[k];
        b.v[3 + k] = box.hi[k];
        b.v[6 + k] = cbox.lo[k];
        b.v[9 + k] = cbox.hi[k];
    }
    return b;
}
__device__ inline void grow(Box3& box, Box3& cbox, const Bounds& b) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
        box.lo[k] = fminf(box.lo[k], b.v[k]);
        box.hi[k] = fmaxf(box.hi[k], b.v[3 + k]);
        cbox.lo[k] = fminf(cbox.lo[k], b.v[6 + k]);
        cbox.hi[k] = fmaxf(cbox.hi[k], b.v[9 + k]);
    }
}

// ---------------------------------------------------------------------------
// Set-up

__host__ __device__ inline uint32_t rec_blocks(uint32_t n) {
    const uint32_t b = (n + kBlock - 1) / kBlock;
    return b < kRecBlocks ? b : kRecBlocks;
}

__global__ void init_kernel(BuildArgs a, uint32_t big_ranges) {
    const uint32_t stride = gridDim.x * blockDim.x, t0 = blockIdx.x * blockDim.x + threadIdx.x;
    for (size_t i = t0; i < (size_t)big_ranges * kBinWords; i += stride) {
        const uint32_t k = (uint32_t)(i % 7);
        a.bins[i] = k == 6 ? 0u : (k < 3 ? kEncPosInf : kEncNegInf);
    }
    const uint32_t words = sizeof(Counters2) / 4;
    for (uint32_t i = t0; i < words; i += stride) reinterpret_cast<uint32_t*>(a.c)[i] = 0u;
    const uint32_t chunks = (a.n + kChunk - 1) / kChunk;
    if (a.n > kBig)
        for (uint32_t i = t0; i < chunks; i += stride) a.chunk_map[0][i] = make_uint2(0u, i);
    if (t0 == 0) {
        BigRange r{};
        r.end = a.n;
        r.parts = rec_blocks(a.n);
        a.big[0][0] = r;
    }
}

// Records of all triangles, the partial bounds of the root, and the root's
// list entry (after init_kernel).  Partial bounds instead of atomics: at 1.3M
// triangles one atomic per wave and bound took 2.6 ms on two cache lines.
__global__ __launch_bounds__(kBlock) void records_kernel(BuildArgs a) {
    __shared__ Bounds part[kBlock / 64];
    Box3 box, cbox;
    box.clear();
    cbox.clear();
    bool finite = true;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < a.n; i += gridDim.x * kBlock) {
        const BvhSource& s = source_of(a, i);
        vec3 v[3];
        triangle(a, s, i - s.first, v);
        Rec r;
        r.lx = fminf(fminf(v[0].x, v[1].x), v[2].x);
        r.ly = fminf(fminf(v[0].y, v[1].y), v[2].y);
        r.lz = fminf(fminf(v[0].z, v[1].z), v[2].z);
        r.hx = fmaxf(fmaxf(v[0].x, v[1].x), v[2].x);
        r.hy = fmaxf(fmaxf(v[0].y, v[1].y), v[2].y);
        r.hz = fmaxf(fmaxf(v[0].z, v[1].z), v[2].z);
        r.id = i;
        r.pad = 0;
        // centroids enter the bins as 0.5 (lo + hi), which can overflow
        finite = finite && all_finite(v[0]) && all_finite(v[1]) && all_finite(v[2]) && isfinite_(r.lx + r.hx) &&
                 isfinite_(r.ly + r.hy) && isfinite_(r.lz + r.hz);
        a.rec[0][i] = r;
        grow(box, cbox, r);
    }
    if (__ballot(!finite) && (threadIdx.x & 63) == 0) a.c->nonfinite = 1u;
    block_reduce(box, cbox, part);
    if (threadIdx.x == 0) a.partial[0][2 * (size_t)blockIdx.x] = bounds_of(box, cbox);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const Range r{0u, a.n, 0u, 0u, 0u};
        if (a.n > kBig) {
            a.c->big[0] = 1u;
            a.c->chunks[0] = (a.n + kChunk - 1) / kChunk;
        } else if (a.n > kSmall) {
            a.mid[0] = r;
            a.c->mid = 1u;
        } else {
            a.small[0] = r;
            a.c->small = 1u;
        }
    }
}

// ---------------------------------------------------------------------------
// Split selection over filled bins, by one wave (lane b % 32 holds bin b).
// Bins are 7 words: ordered lo, ordered hi, count.

struct Split {
    int axis, bin;  // axis -1: coincident centroids
    uint32_t left;
};

__device__ inline Split choose_split(const uint32_t* bins, const float* clo, const float* chi, double parent_area) {
    const int b = threadIdx.x & (kBins - 1);
    Split out{-1, -1, 0u};
    double best = __builtin_huge_val();
    for (int a = 0; a < 3; a++) {
        if (!(chi[a] - clo[a] > 0.0f)) continue;
        const uint32_t* w = bins + (a * kBins + b) * 7;
        Box3 l, r;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            l.lo[k] = r.lo[k] = dec(w[k]);
            l.hi[k] = r.hi[k] = dec(w[3 + k]);
        }
        uint32_t lc = w[6], rc = w[6];
#pragma unroll
        for (int o = 1; o < kBins; o <<= 1) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const float x = __shfl_up(l.lo[k], o, kBins), y = __shfl_up(l.hi[k], o, kBins);
                const float z = __shfl_down(r.lo[k], o, kBins), q = __shfl_down(r.hi[k], o, kBins);
                if (b >= o) {
                    l.lo[k] = fminf(l.lo[k], x);
                    l.hi[k] = fmaxf(l.hi[k], y);
                }
                if (b + o < kBins) {
                    r.lo[k] = fminf(r.lo[k], z);
                    r.hi[k] = fmaxf(r.hi[k], q);
                }
            }
            const uint32_t x = __shfl_up(lc, o, kBins), y = __shfl_down(rc, o, kBins);
            if (b >= o) lc += x;
            if (b + o < kBins) rc += y;
        }
        // the right side of the split after bin b starts at bin b + 1
        Box3 rr;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            rr.lo[k] = __shfl_down(r.lo[k], 1, kBins);
            rr.hi[k] = __shfl_down(r.hi[k], 1, kBins);
        }
        const uint32_t rrc = __shfl_down(rc, 1, kBins);
        double cost = __builtin_huge_val();
        if (b < kBins - 1 && lc != 0u && rrc != 0u) cost = split_cost(l, lc, rr, rrc, parent_area);
        int at = b;
        uint32_t left = lc;
#pragma unroll
        for (int o = kBins / 2; o > 0; o >>= 1) {
            const double c2 = __shfl_xor(cost, o, kBins);
            const int a2 = __shfl_xor(at, o, kBins);
            const uint32_t l2 = __shfl_xor(left, o, kBins);
            if (c2 < cost || (c2 == cost && a2 < at)) {
                cost = c2;
                at = a2;
                left = l2;
            }
        }
        if (cost < best) {
            best = cost;
            out.axis = a;
            out.bin = at;
            out.left = left;
        }
    }
    return out;
}

__device__ inline void add_to_bins(uint32_t* bins, const Rec& r, const float* clo, const float* k) {
    const float lo[3] = {r.lx, r.ly, r.lz}, hi[3] = {r.hx, r.hy, r.hz};
    const uint32_t e[6] = {enc(r.lx), enc(r.ly), enc(r.lz), enc(r.hx), enc(r.hy), enc(r.hz)};
#pragma unroll
    for (int a = 0; a < 3; a++) {
        if (k[a] == 0.0f) continue;
        uint32_t* w = bins + (a * kBins + bin_of(center(lo[a], hi[a]), clo[a], k[a])) * 7;
#pragma unroll
        for (int j = 0; j < 3; j++) {
            atomicMin(w + j, e[j]);
            atomicMax(w + 3 + j, e[3 + j]);
        }
        atomicAdd(w + 6, 1u);
    }
}
__device__ inline void bin_scales(const float* clo, const float* chi, float* k) {
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float ext = chi[a] - clo[a];
        k[a] = ext > 0.0f ? bin_scale(ext) : 0.0f;
    }
}
__device__ inline void clear_bins(uint32_t* bins) {
    for (int i = threadIdx.x; i < kBinWords; i += (int)blockDim.x)
        bins[i] = i % 7 == 6 ? 0u : (i % 7 < 3 ? kEncPosInf : kEncNegInf);
}
__device__ inline bool goes_left(const Rec& r, uint32_t pos, int axis, int bin, float clo, float k, uint32_t left) {
    if (axis < 0) return pos < left;  // coincident centroids: the first half
    const float lo = axis == 0 ? r.lx : (axis == 1 ? r.ly : r.lz);
    const float hi = axis == 0 ? r.hx : (axis == 1 ? r.hy : r.hz);
    return bin_of(center(lo, hi), clo, k) <= bin;
}

// ---------------------------------------------------------------------------
// Phase 1: ranges above kBig

__global__ __launch_bounds__(kBlock) void big_bins_kernel(BuildArgs a, uint32_t level) {
    if (blockIdx.x >= a.c->chunks[level]) return;
    __shared__ uint32_t bins[kBinWords];
    __shared__ Bounds part[kBlock / 64];
    clear_bins(bins);
    const uint2 cm = a.chunk_map[level & 1][blockIdx.x];
    BigRange& r = a.big[level & 1][cm.x];
    Box3 box, cbox;
    box.clear();
    cbox.clear();
    for (uint32_t i = threadIdx.x; i < r.parts; i += kBlock)
        grow(box, cbox, a.partial[level & 1][2 * (size_t)(r.part0 + i) + r.side]);
    block_reduce(box, cbox, part);
    if (cm.y == 0u && threadIdx.x == 0) r.bounds = bounds_of(box, cbox);
    float k[3];
    bin_scales(cbox.lo, cbox.hi, k);
    const uint32_t b0 = r.begin + cm.y * kChunk, b1 = min(r.end, b0 + kChunk);
    const Rec* src = a.rec[level & 1];
    for (uint32_t i = b0 + threadIdx.x; i < b1; i += kBlock) add_to_bins(bins, src[i], cbox.lo, k);
    __syncthreads();
    uint32_t* g = a.bins + (size_t)cm.x * kBinWords;
    for (int i = threadIdx.x; i < kBinWords; i += kBlock) {
        const int w = i % 7;
        if (bins[i - w + 6] == 0u) continue;
        if (w == 6) atomicAdd(g + i, bins[i]);
        else if (w < 3) atomicMin(g + i, bins[i]);
        else atomicMax(g + i, bins[i]);
    }
}

__device__ inline void write_node(const BuildArgs& a, uint32_t node, const Box3& box, int32_t left, uint32_t first,
                                  uint32_t count, uint32_t depth) {
    Node2 n;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        n.lo[k] = box.lo[k];
        n.hi[k] = box.hi[k];
    }
    n.left = left;
    n.first = first;
    n.count = count;
    n.depth = depth;
    n.pad0 = n.pad1 = 0u;
    a.nodes[node] = n;
}

// One wave per range.
__global__ __launch_bounds__(64) void big_split_kernel(BuildArgs a, uint32_t level) {
    const uint32_t count = a.c->big[level];
    for (uint32_t j = blockIdx.x; j < count; j += gridDim.x) {
        BigRange& r = a.big[level & 1][j];
        uint32_t* bins = a.bins + (size_t)j * kBinWords;
        Box3 box;
        float clo[3], chi[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            box.lo[k] = r.bounds.v[k];
            box.hi[k] = r.bounds.v[3 + k];
            clo[k] = r.bounds.v[6 + k];
            chi[k] = r.bounds.v[9 + k];
        }
        const uint32_t n = r.end - r.begin;
        Split s = choose_split(bins, clo, chi, box.area());
        if (s.axis < 0) s.left = n / 2;
        __syncthreads();
        clear_bins(bins);
        if (threadIdx.x == 0) {
            float k[3];
            bin_scales(clo, chi, k);
            r.axis = s.axis;
            r.split = s.bin;
            r.clo = s.axis < 0 ? 0.0f : (s.axis == 0 ? clo[0] : (s.axis == 1 ? clo[1] : clo[2]));
            r.k = s.axis < 0 ? 0.0f : (s.axis == 0 ? k[0] : (s.axis == 1 ? k[1] : k[2]));
            r.left_count = s.left;
            r.cursor[0] = r.cursor[1] = 0u;
            const uint32_t mid = r.begin + s.left;
            const uint32_t left = 2u * mid - 1u;
            write_node(a, r.node, box, (int32_t)left, r.begin, n, r.depth);
            a.upper[atomicAdd(&a.c->upper, 1u)] = r.node;
            atomicMax(&a.c->max_depth, r.depth);
            for (int side = 0; side < 2; side++) {
                Range ch;
                ch.begin = side ? mid : r.begin;
                ch.end = side ? r.end : mid;
                ch.node = left + side;
                ch.depth = r.depth + 1u;
                ch.buf = (level + 1u) & 1u;
                const uint32_t m = ch.end - ch.begin;
                int at = -1;
                if (m > kBig) {
                    at = (int)atomicAdd(&a.c->big[level + 1], 1u);
                    const uint32_t parts = (m + kChunk - 1) / kChunk;
                    const uint32_t c0 = atomicAdd(&a.c->chunks[level + 1], parts);
                    BigRange& d = a.big[ch.buf][at];
                    d.begin = ch.begin;
                    d.end = ch.end;
                    d.node = ch.node;
                    d.depth = ch.depth;
                    d.part0 = r.chunk0;
                    d.parts = (n + kChunk - 1) / kChunk;
                    d.side = (uint32_t)side;
                    d.chunk0 = c0;
                    for (uint32_t p = 0; p < parts; p++) a.chunk_map[ch.buf][c0 + p] = make_uint2((uint32_t)at, p);
                } else if (m > kSmall) {
                    a.mid[atomicAdd(&a.c->mid, 1u)] = ch;
                } else {
                    a.small[atomicAdd(&a.c->small, 1u)] = ch;
                }
                r.child[side] = at;
            }
        }
        __syncthreads();
    }
}

// Moves a workgroup's records to their side of the range in the other buffer
// and writes its partial bounds of children that stay in phase 1.
__global__ __launch_bounds__(kBlock) void big_partition_kernel(BuildArgs a, uint32_t level) {
    if (blockIdx.x >= a.c->chunks[level]) return;
    constexpr int kPer = kChunk / kBlock;
    __shared__ uint32_t wave_left[kBlock / 64], wave_right[kBlock / 64], base[2];
    __shared__ Bounds part[2][kBlock / 64];
    const uint2 cm = a.chunk_map[level & 1][blockIdx.x];
    BigRange& r = a.big[level & 1][cm.x];
    const uint32_t b0 = r.begin + cm.y * kChunk, b1 = min(r.end, b0 + kChunk);
    const Rec* src = a.rec[level & 1];
    Rec* dst = a.rec[(level + 1) & 1];
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x & 63;
    const unsigned long long lt = (1ull << lane) - 1ull;
    uint32_t flags = 0, nl = 0, nr = 0;
#pragma unroll 4
    for (int t = 0; t < kPer; t++) {
        const uint32_t i = b0 + t * kBlock + threadIdx.x;
        const bool in = i < b1;
        bool l = false;
        if (in) l = goes_left(src[i], i - r.begin, r.axis, r.split, r.clo, r.k, r.left_count);
        flags |= (uint32_t)l << t;
        nl += (uint32_t)__popcll(__ballot(in && l));
        nr += (uint32_t)__popcll(__ballot(in && !l));
    }
    if (lane == 0) {
        wave_left[wave] = nl;
        wave_right[wave] = nr;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t l = 0, q = 0;
        for (int w = 0; w < kBlock / 64; w++) {
            const uint32_t x = wave_left[w], y = wave_right[w];
            wave_left[w] = l;
            wave_right[w] = q;
            l += x;
            q += y;
        }
        base[0] = r.begin + (l ? atomicAdd(&r.cursor[0], l) : 0u);
        base[1] = r.begin + r.left_count + (q ? atomicAdd(&r.cursor[1], q) : 0u);
    }
    __syncthreads();
    uint32_t lpos = base[0] + wave_left[wave], rpos = base[1] + wave_right[wave];
    Box3 box[2], cbox[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
        box[s].clear();
        cbox[s].clear();
    }
    for (int t = 0; t < kPer; t++) {
        const uint32_t i = b0 + t * kBlock + threadIdx.x;
        const bool in = i < b1;
        const bool l = (flags >> t) & 1u;
        const unsigned long long ml = __ballot(in && l), mr = __ballot(in && !l);
        if (in) {
            const Rec rec = src[i];
            dst[l ? lpos + (uint32_t)__popcll(ml & lt) : rpos + (uint32_t)__popcll(mr & lt)] = rec;
            if (l) grow(box[0], cbox[0], rec);
            else grow(box[1], cbox[1], rec);
        }
        lpos += (uint32_t)__popcll(ml);
        rpos += (uint32_t)__popcll(mr);
    }
#pragma unroll
    for (int s = 0; s < 2; s++) {
        if (r.child[s] < 0) continue;
        block_reduce(box[s], cbox[s], part[s]);
        if (threadIdx.x == 0)
            a.partial[(level + 1) & 1][2 * (size_t)blockIdx.x + s] = bounds_of(box[s], cbox[s]);
    }
}

// ---------------------------------------------------------------------------
// Phase 2: one workgroup per range of kSmall+1..kBig records

constexpr uint32_t kListed = 64;  // list entries a workgroup gathers before it claims room for them

__global__ __launch_bounds__(kBlock) void mid_kernel(BuildArgs a) {
    __shared__ uint32_t bins[kBinWords];
    __shared__ Bounds part[kBlock / 64];
    __shared__ Range stack[32], listed[kListed];
    __shared__ uint32_t upper[kListed];
    __shared__ uint32_t wave_left[kBlock / 64];
    __shared__ uint32_t num_listed, num_upper, at[2];
    __shared__ int sp;
    __shared__ Split split;
    const uint32_t count = a.c->mid;
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x & 63;
    const unsigned long long lt = (1ull << lane) - 1ull;
    for (uint32_t e = blockIdx.x; e < count; e += gridDim.x) {
        if (threadIdx.x == 0) {
            stack[0] = a.mid[e];
            sp = 1;
            num_listed = num_upper = 0u;
        }
        __syncthreads();
        while (sp > 0) {
            const Range r = stack[sp - 1];
            const Rec* src = a.rec[r.buf];
            Rec* dst = a.rec[r.buf ^ 1u];
            const uint32_t n = r.end - r.begin;
            // bounds
            Box3 box, cbox;
            box.clear();
            cbox.clear();
            for (uint32_t i = r.begin + threadIdx.x; i < r.end; i += kBlock) grow(box, cbox, src[i]);
            clear_bins(bins);
            block_reduce(box, cbox, part);
            float k[3];
            bin_scales(cbox.lo, cbox.hi, k);
            for (uint32_t i = r.begin + threadIdx.x; i < r.end; i += kBlock) add_to_bins(bins, src[i], cbox.lo, k);
            __syncthreads();
            if (wave == 0) {
                Split s = choose_split(bins, cbox.lo, cbox.hi, box.area());
                if (s.axis < 0) s.left = n / 2;
                if (lane == 0) split = s;
            }
            __syncthreads();
            const Split s = split;
            const float clo = s.axis <= 0 ? cbox.lo[0] : (s.axis == 1 ? cbox.lo[1] : cbox.lo[2]);
            const float sk = s.axis <= 0 ? k[0] : (s.axis == 1 ? k[1] : k[2]);
            // stable partition: each wave takes a contiguous share of the range
            const uint32_t share = ((n + kBlock - 1) / kBlock) * 64u;
            const uint32_t w0 = min(r.end, r.begin + wave * share), w1 = min(r.end, w0 + share);
            uint32_t nl = 0;
            for (uint32_t i = w0; i < w1; i += 64u) {
                const bool in = i + lane < w1;
                const bool l = in && goes_left(src[i + lane], i + lane - r.begin, s.axis, s.bin, clo, sk, s.left);
                nl += (uint32_t)__popcll(__ballot(l));
            }
            if (lane == 0) wave_left[wave] = nl;
            __syncthreads();
            uint32_t before = 0;
            for (uint32_t w = 0; w < wave; w++) before += wave_left[w];
            uint32_t lpos = r.begin + before, rpos = r.begin + s.left + (w0 - r.begin) - before;
            for (uint32_t i = w0; i < w1; i += 64u) {
                const bool in = i + lane < w1;
                bool l = false;
                Rec rec;
                if (in) {
                    rec = src[i + lane];
                    l = goes_left(rec, i + lane - r.begin, s.axis, s.bin, clo, sk, s.left);
                }
                const unsigned long long ml = __ballot(in && l), mr = __ballot(in && !l);
                if (in) dst[l ? lpos + (uint32_t)__popcll(ml & lt) : rpos + (uint32_t)__popcll(mr & lt)] = rec;
                lpos += (uint32_t)__popcll(ml);
                rpos += (uint32_t)__popcll(mr);
            }
            if (threadIdx.x == 0) {
                const uint32_t mid = r.begin + s.left, left = 2u * mid - 1u;
                write_node(a, r.node, box, (int32_t)left, r.begin, n, r.depth);
                upper[num_upper++] = r.node;
                sp--;
                Range c[2] = {{r.begin, mid, left, r.depth + 1u, r.buf ^ 1u},
                              {mid, r.end, left + 1u, r.depth + 1u, r.buf ^ 1u}};
                // the larger child below the smaller: the stack stays within log2(kBig) entries
                const int big = (mid - r.begin) >= (r.end - mid) ? 0 : 1;
                for (int q = 0; q < 2; q++) {
                    const Range& ch = c[q == 0 ? big : 1 - big];
                    if (ch.end - ch.begin > kSmall) stack[sp++] = ch;
                    else listed[num_listed++] = ch;
                }
                atomicMax(&a.c->max_depth, r.depth);
            }
            __syncthreads();
            if (num_listed >= kListed - 1u || num_upper >= kListed || sp == 0) {
                const uint32_t m = num_listed, u = num_upper;
                if (threadIdx.x == 0) {
                    at[0] = atomicAdd(&a.c->small, m);
                    at[1] = atomicAdd(&a.c->upper, u);
                }
                __syncthreads();
                if (threadIdx.x < m) a.small[at[0] + threadIdx.x] = listed[threadIdx.x];
                if (threadIdx.x < u) a.upper[at[1] + threadIdx.x] = upper[threadIdx.x];
                __syncthreads();
                if (threadIdx.x == 0) num_listed = num_upper = 0u;
                __syncthreads();
            }
        }
        __syncthreads();  // every thread has left the loop before the next range resets the stack
    }
}

// ---------------------------------------------------------------------------
// Collapse costs (host/bvh_build.cpp, Collapse::run): c[i - 1] is the least
// cost of the subtree over at most i slots of its parent.

__device__ inline void collapse_leaf(double area, uint32_t count, float* c, uint64_t& how) {
    const float v = (float)(area * kCostTri * count);
#pragma unroll
    for (int i = 0; i < 8; i++) c[i] = v;
    how = 0;
}
__device__ inline void collapse_node(double area, uint32_t count, uint32_t max_leaf, const float* cl, const float* cr,
                                     float* c, uint64_t& how) {
    double dist[9];
    uint32_t dk[9];
#pragma unroll
    for (int i = 2; i <= 8; i++) {
        double d = __builtin_huge_val();
        uint32_t at = 1;
#pragma unroll
        for (int k = 1; k < i; k++) {
            const double v = (double)cl[k - 1] + (double)cr[i - k - 1];
            if (v < d) {
                d = v;
                at = (uint32_t)k;
            }
        }
        dist[i] = d;
        dk[i] = at;
    }
    const double internal = area * kCostNode + dist[8];
    const double leaf = count <= max_leaf ? area * kCostTri * count : __builtin_huge_val();
    c[0] = (float)fmin(internal, leaf);
    uint64_t h = count <= max_leaf && leaf <= internal ? 0 : 1;
#pragma unroll
    for (int i = 2; i <= 8; i++) {
        if (dist[i] < (double)c[i - 2]) {
            c[i - 1] = (float)dist[i];
            h |= (uint64_t)dk[i] << (8 * (i - 1));
        } else {
            c[i - 1] = c[i - 2];
        }
    }
    how = h;
}
__device__ inline void load8(const float* p, float* c) {
    const float4 x = reinterpret_cast<const float4*>(p)[0], y = reinterpret_cast<const float4*>(p)[1];
    c[0] = x.x; c[1] = x.y; c[2] = x.z; c[3] = x.w;
    c[4] = y.x; c[5] = y.y; c[6] = y.z; c[7] = y.w;
}
__device__ inline void store8(float* p, const float* c) {
    reinterpret_cast<float4*>(p)[0] = make_float4(c[0], c[1], c[2], c[3]);
    reinterpret_cast<float4*>(p)[1] = make_float4(c[4], c[5], c[6], c[7]);
}

__device__ inline double node_area(const Node2& nd) {
    Box3 b;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        b.lo[k] = nd.lo[k];
        b.hi[k] = nd.hi[k];
    }
    return b.area();
}

// Phase 4: nodes split in phases 1 and 2 at `depth` (deeper ones are done).
__global__ __launch_bounds__(kBlock) void collapse_kernel(BuildArgs a, uint32_t depth) {
    const uint32_t count = a.c->upper;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < count; i += gridDim.x * kBlock) {
        const uint32_t node = a.upper[i];
        const Node2 nd = a.nodes[node];
        if (nd.depth != depth) continue;
        float cl[8], cr[8], c[8];
        uint64_t how;
        load8(a.cost + 8 * (size_t)nd.left, cl);
        load8(a.cost + 8 * (size_t)(nd.left + 1), cr);
        collapse_node(node_area(nd), nd.count, a.max_leaf, cl, cr, c, how);
        store8(a.cost + 8 * (size_t)node, c);
        a.how[node] = how;
    }
}

// ---------------------------------------------------------------------------
// Phase 3: one wave per range of at most 64 records

constexpr int kLocal = 2 * (int)kSmall;  // nodes of a small subtree

__global__ __launch_bounds__(64) void small_kernel(BuildArgs a) {
    __shared__ float rec[6][kSmall];
    __shared__ uint32_t ids[kSmall], bin3[kSmall], keys[kSmall];
    __shared__ double costs[kSmall];
    __shared__ float nbox[6][kLocal];
    __shared__ uint8_t nleft[kLocal], nfirst[kLocal], ncount[kLocal], ndepth[kLocal];
    __shared__ alignas(16) float ncost[kLocal][8];
    const int lane = threadIdx.x;
    const unsigned long long lt = (1ull << lane) - 1ull;
    const uint32_t ranges = a.c->small;
    for (uint32_t e = blockIdx.x; e < ranges; e += gridDim.x) {
        const Range range = a.small[e];
        const int m = (int)(range.end - range.begin);
        if (lane < m) {
            const Rec r = a.rec[range.buf][range.begin + lane];
            rec[0][lane] = r.lx;
            rec[1][lane] = r.ly;
            rec[2][lane] = r.lz;
            rec[3][lane] = r.hx;
            rec[4][lane] = r.hy;
            rec[5][lane] = r.hz;
            ids[lane] = r.id;
        }
        int s = 0, t = m;   // the lane's range
        int node = 0, depth = 0;
        bool done = lane >= m;
        int nodes = 1;
        if (lane == 0) {
            nfirst[0] = 0;
            ncount[0] = (uint8_t)m;
            ndepth[0] = 0;
        }
        __syncthreads();
        while (__any(!done)) {
            const int len = done ? 0 : t - s;
            int longest = len;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) longest = max(longest, __shfl_xor(longest, o));
            // bounds of the range
            Box3 box, cbox;
            box.clear();
            cbox.clear();
            for (int q = 0; q < longest; q++) {
                if (q >= len) continue;
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    const float lo = rec[k][s + q], hi = rec[3 + k][s + q], c = center(lo, hi);
                    box.lo[k] = fminf(box.lo[k], lo);
                    box.hi[k] = fmaxf(box.hi[k], hi);
                    cbox.lo[k] = fminf(cbox.lo[k], c);
                    cbox.hi[k] = fmaxf(cbox.hi[k], c);
                }
            }
            if (!done && lane == s) {
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    nbox[k][node] = box.lo[k];
                    nbox[3 + k][node] = box.hi[k];
                }
                nleft[node] = 0;
            }
            if (len == 1) done = true;
            // bins of the lane's record
            int b[3] = {0, 0, 0};
            bool valid[3] = {false, false, false};
            if (!done) {
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    const float ext = cbox.hi[k] - cbox.lo[k];
                    valid[k] = ext > 0.0f;
                    if (valid[k]) b[k] = bin_of(center(rec[k][lane], rec[3 + k][lane]), cbox.lo[k], bin_scale(ext));
                }
                bin3[lane] = (uint32_t)b[0] | ((uint32_t)b[1] << 8) | ((uint32_t)b[2] << 16);
            }
            __syncthreads();
            // cost of the split after the lane's bin, per axis
            const int live = done ? 0 : len;
            double best = __builtin_huge_val();
            uint32_t key = 0xffffffffu;
            const double parent = box.area();
            Box3 l[3], r[3];
            uint32_t lc[3] = {0u, 0u, 0u};
#pragma unroll
            for (int ax = 0; ax < 3; ax++) {
                l[ax].clear();
                r[ax].clear();
            }
            for (int q = 0; q < longest; q++) {
                if (q >= live) continue;
                const int j = s + q;
                const uint32_t bj = bin3[j];
                float lo[3], hi[3];
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    lo[k] = rec[k][j];
                    hi[k] = rec[3 + k][j];
                }
#pragma unroll
                for (int ax = 0; ax < 3; ax++) {
                    const bool left = (int)((bj >> (8 * ax)) & 0xffu) <= b[ax];
                    lc[ax] += left ? 1u : 0u;
#pragma unroll
                    for (int k = 0; k < 3; k++) {
                        l[ax].lo[k] = fminf(l[ax].lo[k], left ? lo[k] : __builtin_huge_valf());
                        l[ax].hi[k] = fmaxf(l[ax].hi[k], left ? hi[k] : -__builtin_huge_valf());
                        r[ax].lo[k] = fminf(r[ax].lo[k], left ? __builtin_huge_valf() : lo[k]);
                        r[ax].hi[k] = fmaxf(r[ax].hi[k], left ? -__builtin_huge_valf() : hi[k]);
                    }
                }
            }
#pragma unroll
            for (int ax = 0; ax < 3; ax++) {
                const uint32_t rc = (uint32_t)live - lc[ax];
                if (valid[ax] && rc != 0u) {
                    const double c = split_cost(l[ax], lc[ax], r[ax], rc, parent);
                    if (c < best) {
                        best = c;
                        key = (uint32_t)(ax * kBins + b[ax]);
                    }
                }
            }
            costs[lane] = best;
            keys[lane] = key;
            __syncthreads();
            // the range's first least split (axis, then bin)
            for (int q = 0; q < longest; q++) {
                if (q >= live) continue;
                const double c = costs[s + q];
                const uint32_t kk = keys[s + q];
                if (c < best || (c == best && kk < key)) {
                    best = c;
                    key = kk;
                }
            }
            const bool none = key == 0xffffffffu;
            if (!done && (uint32_t)len <= a.max_leaf && (none || (double)len <= best)) done = true;
            // partition the split ranges
            const bool splitting = !done;
            bool left = false;
            if (splitting) {
                const int ax = (int)(key / kBins), bin = (int)(key % kBins);
                left = none ? (lane - s) < len / 2 : (ax == 0 ? b[0] : (ax == 1 ? b[1] : b[2])) <= bin;
            }
            const unsigned long long lm = __ballot(splitting && left);
            const unsigned long long leaders = __ballot(splitting && lane == s);
            const unsigned long long seg = len >= 64 ? ~0ull : ((1ull << len) - 1ull) << (s & 63);
            const int nl = __popcll(lm & seg);
            float mv[6];
            uint32_t mid = 0;
            int to = lane;
            if (splitting) {
                to = left ? s + __popcll(lm & seg & lt) : s + nl + __popcll(~lm & seg & lt);
#pragma unroll
                for (int k = 0; k < 6; k++) mv[k] = rec[k][lane];
                mid = ids[lane];
            }
            __syncthreads();
            if (splitting) {
#pragma unroll
                for (int k = 0; k < 6; k++) rec[k][to] = mv[k];
                ids[to] = mid;
                const int child = nodes + 2 * __popcll(leaders & ((1ull << s) - 1ull));
                if (lane == s) {
                    nleft[node] = (uint8_t)child;
                    nfirst[child] = (uint8_t)s;
                    ncount[child] = (uint8_t)nl;
                    nfirst[child + 1] = (uint8_t)(s + nl);
                    ncount[child + 1] = (uint8_t)(len - nl);
                    ndepth[child] = ndepth[child + 1] = (uint8_t)(depth + 1);
                }
                depth++;
                if (lane < s + nl) {
                    t = s + nl;
                    node = child;
                } else {
                    s = s + nl;
                    node = child + 1;
                }
            }
            nodes += 2 * __popcll(leaders);
            __syncthreads();
        }
        // collapse costs, deepest nodes first
        int deepest = depth;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) deepest = max(deepest, __shfl_xor(deepest, o));
        for (int d = deepest; d >= 0; d--) {
            for (int i = lane; i < nodes; i += 64) {
                if (ndepth[i] != d) continue;
                Box3 box;
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    box.lo[k] = nbox[k][i];
                    box.hi[k] = nbox[3 + k][i];
                }
                const uint32_t cnt = ncount[i];
                const uint32_t l = nleft[i];
                float c[8];
                uint64_t how;
                if (l == 0u) {
                    collapse_leaf(box.area(), cnt, c, how);
                } else {
                    float cl[8], cr[8];
                    load8(ncost[l], cl);
                    load8(ncost[l + 1], cr);
                    collapse_node(box.area(), cnt, a.max_leaf, cl, cr, c, how);
                }
                store8(ncost[i], c);
                // global ids: the range's node, or 2 split - 1 and 2 split
                auto gid = [&](uint32_t local, uint32_t right) {
                    return 2u * (range.begin + nfirst[local] + (right ? 0u : (uint32_t)ncount[local])) - (right ? 0u : 1u);
                };
                const uint32_t g = i == 0 ? range.node : gid((uint32_t)i, (uint32_t)((i & 1) == 0));
                write_node(a, g, box, l == 0u ? -1 : (int32_t)gid(l, 0u), range.begin + nfirst[i], cnt,
                           range.depth + (uint32_t)d);
                store8(a.cost + 8 * (size_t)g, c);
                a.how[g] = how;
            }
            __syncthreads();
        }
        if (lane < m) a.order[range.begin + lane] = ids[lane];
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Phase 5: BVH8 nodes, one level at a time

constexpr uint32_t kLeafBit = 0x80000000u;

__global__ void bvh8_root_kernel(BuildArgs a) {
    if (threadIdx.x == 0) {
        a.pend[0][0] = 0u;
        a.c->level_count[0] = 1u;
    }
}

__device__ inline uint32_t group_min_u32(uint32_t v) {
#pragma unroll
    for (int o = 4; o > 0; o >>= 1) v = min(v, (uint32_t)__shfl_xor(v, o, 8));
    return v;
}

// Children and their slots for each pending node, and the tile's counts.
__global__ __launch_bounds__(kBlock) void bvh8_children_kernel(BuildArgs a, uint32_t level) {
    __shared__ uint32_t ch[kBlock][9];    // children (| leaf bit); padded rows
    __shared__ uint32_t todo[kBlock][8];  // node << 4 | slots to spread it over
    __shared__ uint8_t nch[kBlock];
    __shared__ uint32_t sum[2];
    const uint32_t count = a.c->level_count[level];
    const uint32_t tiles = (count + kBlock - 1) / kBlock;
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const uint32_t p = tile * kBlock + threadIdx.x;
        if (threadIdx.x < 2) sum[threadIdx.x] = 0u;
        if (p < count) {
            const uint32_t node = a.pend[level & 1][p];
            const int32_t root_left = a.nodes[node].left;
            int nc = 0, n = 0;
            if (root_left < 0 || (node == 0u && (a.how[0] & 0xffu) == 0u)) {
                ch[threadIdx.x][nc++] = node | kLeafBit;
            } else {
                // the node's own 8 slots: the best split of 8 between its children
                float cl[8], cr[8];
                load8(a.cost + 8 * (size_t)root_left, cl);
                load8(a.cost + 8 * (size_t)(root_left + 1), cr);
                uint32_t best_k = 1;
                double best = __builtin_huge_val();
#pragma unroll
                for (int k = 1; k < 8; k++) {
                    const double v = (double)cl[k - 1] + (double)cr[8 - k - 1];
                    if (v < best) {
                        best = v;
                        best_k = (uint32_t)k;
                    }
                }
                // entries: right child below the left, so the left comes out first
                uint2 stack_top;
                todo[threadIdx.x][n++] = ((uint32_t)root_left + 1u) * 8u + (8u - best_k - 1u);
                stack_top = make_uint2((uint32_t)root_left, best_k);
                for (;;) {
                    uint32_t cur = stack_top.x, i = stack_top.y;
                    const uint64_t how = a.how[cur];
                    while (i > 1u && ((how >> (8u * (i - 1u))) & 0xffu) == 0u) i--;
                    if (i == 1u) {
                        const bool leaf = a.nodes[cur].left < 0 || (how & 0xffu) == 0u;
                        ch[threadIdx.x][nc++] = cur | (leaf ? kLeafBit : 0u);
                        if (n == 0) break;
                        const uint32_t w = todo[threadIdx.x][--n];
                        stack_top = make_uint2(w / 8u, w % 8u + 1u);
                    } else {
                        const uint32_t k = (uint32_t)((how >> (8u * (i - 1u))) & 0xffu);
                        const uint32_t l = (uint32_t)a.nodes[cur].left;
                        todo[threadIdx.x][n++] = (l + 1u) * 8u + (i - k - 1u);
                        stack_top = make_uint2(l, k);
                    }
                }
            }
            nch[threadIdx.x] = (uint8_t)nc;
        }
        __syncthreads();
        // eight lanes per node, lane = child
        const int c = threadIdx.x & 7;
        for (uint32_t g = threadIdx.x / 8; g < kBlock; g += kBlock / 8) {
            const uint32_t q = tile * kBlock + g;
            if (q >= count) break;  // uniform over the eight lanes
            const int nc = nch[g];
            const bool mine = c < nc;
            const uint32_t child = mine ? ch[g][c] : 0xffffffffu;
            Node2 nd;
            Box3 box;
            box.clear();
            uint32_t tris = 0;
            if (mine) {
                nd = a.nodes[child & ~kLeafBit];
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    box.lo[k] = nd.lo[k];
                    box.hi[k] = nd.hi[k];
                }
                if (child & kLeafBit) tris = nd.count;
            }
            double cc[3];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                float lo = box.lo[k], hi = box.hi[k];
#pragma unroll
                for (int o = 4; o > 0; o >>= 1) {
                    lo = fminf(lo, __shfl_xor(lo, o, 8));
                    hi = fmaxf(hi, __shfl_xor(hi, o, 8));
                }
                const double pc = 0.5 * ((double)lo + (double)hi);
                cc[k] = 0.5 * ((double)box.lo[k] + (double)box.hi[k]) - pc;
            }
            // greedy: the least (v, child, slot) of the pairs still open
            uint32_t free_slots = 0xffu;
            int my_slot = mine ? -1 : 8;
            for (int round = 0; round < nc; round++) {
                double v = __builtin_huge_val();
                uint32_t id = 0xffffffffu;
                if (my_slot < 0) {
#pragma unroll
                    for (int s = 0; s < 8; s++) {
                        double x = 0.0;
#pragma unroll
                        for (int k = 0; k < 3; k++) x -= cc[k] * (((s >> k) & 1) ? 1.0 : -1.0);
                        if (((free_slots >> s) & 1u) && (id == 0xffffffffu || x < v)) {
                            v = x;
                            id = (uint32_t)(c * 8 + s);
                        }
                    }
                }
#pragma unroll
                for (int o = 4; o > 0; o >>= 1) {
                    const double v2 = __shfl_xor(v, o, 8);
                    const uint32_t i2 = __shfl_xor(id, o, 8);
                    if (i2 != 0xffffffffu && (id == 0xffffffffu || v2 < v || (v2 == v && i2 < id))) {
                        v = v2;
                        id = i2;
                    }
                }
                if ((int)(id / 8u) == c && my_slot < 0) my_slot = (int)(id % 8u);
                free_slots &= ~(1u << (id % 8u));
            }
            // slot order: lane s takes the child whose slot is s
            uint32_t out = 0xffffffffu, internal = 0, total = tris;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int sl = __shfl(my_slot, j, 8);
                const uint32_t cj = __shfl(child, j, 8);
                if (sl == c) out = cj;
            }
            internal = mine && !(child & kLeafBit) ? 1u : 0u;
#pragma unroll
            for (int o = 4; o > 0; o >>= 1) {
                internal += __shfl_xor(internal, o, 8);
                total += __shfl_xor(total, o, 8);
            }
            a.slots[8 * (size_t)q + c] = out;
            if (c == 0) {
                a.counts[q] = internal | (total << 8);
                atomicAdd(&sum[0], internal);
                atomicAdd(&sum[1], total);
            }
        }
        __syncthreads();
        if (threadIdx.x == 0) a.tile_sums[tile] = make_uint2(sum[0], sum[1]);
        __syncthreads();
    }
}

// One workgroup: exclusive prefix of the tile counts, and the next level.
__global__ __launch_bounds__(1024) void bvh8_scan_kernel(BuildArgs a, uint32_t level) {
    __shared__ uint2 s[1024];
    __shared__ uint2 carry;
    const uint32_t count = a.c->level_count[level];
    const uint32_t tiles = (count + kBlock - 1) / kBlock;
    if (threadIdx.x == 0) carry = make_uint2(0u, 0u);
    __syncthreads();
    for (uint32_t t0 = 0; t0 < tiles; t0 += 1024u) {
        const uint32_t t = t0 + threadIdx.x;
        const uint2 own = t < tiles ? a.tile_sums[t] : make_uint2(0u, 0u);
        s[threadIdx.x] = own;
        __syncthreads();
        for (uint32_t o = 1; o < 1024u; o <<= 1) {
            const uint2 add = threadIdx.x >= o ? s[threadIdx.x - o] : make_uint2(0u, 0u);
            __syncthreads();
            s[threadIdx.x].x += add.x;
            s[threadIdx.x].y += add.y;
            __syncthreads();
        }
        const uint2 inc = s[threadIdx.x], c0 = carry;
        if (t < tiles) a.tile_sums[t] = make_uint2(c0.x + inc.x - own.x, c0.y + inc.y - own.y);
        __syncthreads();
        if (threadIdx.x == 1023) carry = make_uint2(c0.x + inc.x, c0.y + inc.y);
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        a.c->level_base[level + 1] = a.c->level_base[level] + count;
        a.c->level_count[level + 1] = carry.x;
        a.c->tri_base[level + 1] = a.c->tri_base[level] + carry.y;
    }
}

__device__ inline float next_below(float x) {
    const uint32_t u = __float_as_uint(x);
    if ((u & 0x7fffffffu) == 0u) return __uint_as_float(0x80000001u);
    return __uint_as_float(u & 0x80000000u ? u + 1u : u - 1u);
}
// ceil(log2(x)) for x > 0
__device__ inline int ceil_log2(double x) {
    int e;
    const double m = frexp(x, &e);
    return m == 0.5 ? e - 1 : e;
}

__global__ __launch_bounds__(kBlock) void bvh8_emit_kernel(BuildArgs a, uint32_t level) {
    __shared__ uint2 scan[kBlock];
    const uint32_t count = a.c->level_count[level];
    const uint32_t tiles = (count + kBlock - 1) / kBlock;
    const uint32_t base = a.c->level_base[level], next_base = base + count, tri0 = a.c->tri_base[level];
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const uint32_t p = tile * kBlock + threadIdx.x;
        const uint32_t w = p < count ? a.counts[p] : 0u;
        const uint2 own = make_uint2(w & 0xffu, w >> 8);
        scan[threadIdx.x] = own;
        __syncthreads();
        for (uint32_t o = 1; o < (uint32_t)kBlock; o <<= 1) {
            const uint2 add = threadIdx.x >= o ? scan[threadIdx.x - o] : make_uint2(0u, 0u);
            __syncthreads();
            scan[threadIdx.x].x += add.x;
            scan[threadIdx.x].y += add.y;
            __syncthreads();
        }
        const uint2 inc = scan[threadIdx.x], ts = a.tile_sums[tile];
        __syncthreads();
        scan[threadIdx.x] = make_uint2(ts.x + inc.x - own.x, ts.y + inc.y - own.y);
        __syncthreads();
        // eight lanes per node, lane = slot
        const int c = threadIdx.x & 7;
        for (uint32_t g = threadIdx.x / 8; g < kBlock; g += kBlock / 8) {
            const uint32_t q = tile * kBlock + g;
            if (q >= count) break;  // uniform over the eight lanes
            const uint32_t child = a.slots[8 * (size_t)q + c];
            const bool used = child != 0xffffffffu;
            const bool leaf = used && (child & kLeafBit);
            Node2 nd;
            Box3 box, all;
            box.clear();
            if (used) {
                nd = a.nodes[child & ~kLeafBit];
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    box.lo[k] = nd.lo[k];
                    box.hi[k] = nd.hi[k];
                }
            }
            all = box;
#pragma unroll
            for (int k = 0; k < 3; k++)
#pragma unroll
                for (int o = 4; o > 0; o >>= 1) {
                    all.lo[k] = fminf(all.lo[k], __shfl_xor(all.lo[k], o, 8));
                    all.hi[k] = fmaxf(all.hi[k], __shfl_xor(all.hi[k], o, 8));
                }
            // quantisation (host/bvh_build.cpp, quantise): per axis the
            // smallest exponent whose decoded boxes strictly enclose the
            // exact ones
            float org[3];
            uint32_t e8[3], qlo8[3], qhi8[3];
            bool failed = false;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const float po = next_below(all.lo[k]);
                org[k] = po;
                const double ext = (double)all.hi[k] - (double)po;
                int ee = 1;
                if (ext > 0.0) {
                    ee = ceil_log2(ext / 255.0) + 127;
                    ee = max(1, min(254, ee));
                }
                uint32_t lo_q = 0, hi_q = 0;
                for (;; ee++) {
                    if (ee > 254) {
                        failed = true;
                        break;
                    }
                    const float scale = exp_scale((uint8_t)ee);
                    bool ok = true;
                    if (used) {
                        const double rlo = ((double)box.lo[k] - (double)po) / (double)scale;
                        const double rhi = ((double)box.hi[k] - (double)po) / (double)scale;
                        // clamped before the conversion: the host's int is within [0, 255] too
                        int ql = (int)fmax(0.0, fmin(255.0, floor(rlo)));
                        int qh = (int)fmax(0.0, fmin(255.0, ceil(rhi)));
                        while (ql > 0 && decode_q(po, (uint8_t)ql, scale) >= box.lo[k]) ql--;
                        while (qh < 255 && decode_q(po, (uint8_t)qh, scale) <= box.hi[k]) qh++;
                        ok = !(decode_q(po, (uint8_t)ql, scale) >= box.lo[k] ||
                               decode_q(po, (uint8_t)qh, scale) <= box.hi[k]);
                        lo_q = (uint32_t)ql;
                        hi_q = (uint32_t)qh;
                    }
                    if (group_min_u32(ok ? 1u : 0u) == 1u) break;
                }
                e8[k] = (uint32_t)min(ee, 254);
                qlo8[k] = used ? lo_q : 0u;
                qhi8[k] = used ? hi_q : 0u;
            }
            // ranks of internal children and triangle offsets, in slot order
            uint32_t cnt = leaf ? nd.count : 0u, inner = used && !leaf ? 1u : 0u;
            uint32_t tri_off = cnt, rank = inner;
#pragma unroll
            for (int o = 1; o < 8; o <<= 1) {
                const uint32_t x = __shfl_up(tri_off, o, 8), y = __shfl_up(rank, o, 8);
                if (c >= o) {
                    tri_off += x;
                    rank += y;
                }
            }
            tri_off -= cnt;
            rank -= inner;
            uint32_t meta = 0;
            if (used) meta = leaf ? ((((1u << cnt) - 1u) << 5) | tri_off) : ((1u << 5) | (24u + (uint32_t)c));
            const uint2 at = scan[g];
            const uint32_t child_base = next_base + at.x, tri_base = tri0 + at.y;
            // bytes of the eight lanes into words: lane j < 4 of each word half
            uint32_t imask = inner << c;
            uint32_t words[7] = {meta, qlo8[0], qlo8[1], qlo8[2], qhi8[0], qhi8[1], qhi8[2]};
#pragma unroll
            for (int o = 4; o > 0; o >>= 1) imask |= __shfl_xor(imask, o, 8);
            uint64_t packed[7];
#pragma unroll
            for (int j = 0; j < 7; j++) {
                uint64_t v = (uint64_t)words[j] << (8 * c);
#pragma unroll
                for (int o = 4; o > 0; o >>= 1) v |= __shfl_xor(v, o, 8);
                packed[j] = v;
            }
            uint4* np = reinterpret_cast<uint4*>(a.out_nodes + base + q);
            if (c == 0)
                np[0] = make_uint4(__float_as_uint(org[0]), __float_as_uint(org[1]), __float_as_uint(org[2]),
                                   e8[0] | (e8[1] << 8) | (e8[2] << 16) | (imask << 24));
            if (c == 1) np[1] = make_uint4(child_base, tri_base, (uint32_t)packed[0], (uint32_t)(packed[0] >> 32));
            if (c == 2)
                np[2] = make_uint4((uint32_t)packed[1], (uint32_t)(packed[1] >> 32), (uint32_t)packed[2],
                                   (uint32_t)(packed[2] >> 32));
            if (c == 3)
                np[3] = make_uint4((uint32_t)packed[3], (uint32_t)(packed[3] >> 32), (uint32_t)packed[4],
                                   (uint32_t)(packed[4] >> 32));
            if (c == 4)
                np[4] = make_uint4((uint32_t)packed[5], (uint32_t)(packed[5] >> 32), (uint32_t)packed[6],
                                   (uint32_t)(packed[6] >> 32));
            if (c == 5 && failed) a.c->bad_quant = 1u;
            if (used && !leaf) {
                a.pend[(level + 1) & 1][at.x + rank] = child;
            } else if (leaf) {
                // leaf triangles in id order, so that the array does not
                // depend on the order the partitions left them in
                uint32_t id[3];
#pragma unroll
                for (uint32_t j = 0; j < 3; j++) id[j] = j < cnt ? a.order[nd.first + j] : 0xffffffffu;
                auto sw = [&](int x, int y) {
                    const uint32_t lo = min(id[x], id[y]), hi = max(id[x], id[y]);
                    id[x] = lo;
                    id[y] = hi;
                };
                sw(0, 1);
                sw(1, 2);
                sw(0, 1);
                for (uint32_t j = 0; j < cnt; j++) {
                    const uint32_t ti = j == 0 ? id[0] : (j == 1 ? id[1] : id[2]);
                    const BvhSource& s = source_of(a, ti);
                    vec3 v[3];
                    triangle(a, s, ti - s.first, v);
                    float4* tp = reinterpret_cast<float4*>(a.out_tris + tri_base + tri_off + j);
                    tp[0] = make_float4(v[0].x, v[0].y, v[0].z, __uint_as_float(s.inst));
                    tp[1] = make_float4(v[1].x, v[1].y, v[1].z, __uint_as_float(ti - s.first));
                    tp[2] = make_float4(v[2].x, v[2].y, v[2].z, 0.0f);
                }
            }
        }
        __syncthreads();
    }
}

// Scratch layout: every array 256-byte aligned.
struct Layout {
    size_t off = 0;
    size_t take(size_t bytes) {
        const size_t at = off;
        off += (bytes + 255) & ~(size_t)255;
        return at;
    }
};

uint32_t big_capacity(uint32_t n) { return n / kBig + 2; }
uint32_t chunk_capacity(uint32_t n) { return n / kChunk + n / kBig + 4; }

size_t lay_out(uint32_t n, char* p, BuildArgs* a) {
    Layout l;
    const size_t n2 = 2 * (size_t)n;
    size_t rec[2], big[2], map[2], pend[2], partial[2];
    for (size_t& x : rec) x = l.take(n * sizeof(Rec));
    const size_t nodes = l.take(n2 * sizeof(Node2)), cost = l.take(n2 * 32), how = l.take(n2 * 8),
                 order = l.take((size_t)n * 4);
    for (size_t& x : big) x = l.take(big_capacity(n) * sizeof(BigRange));
    for (size_t& x : map) x = l.take(chunk_capacity(n) * sizeof(uint2));
    for (size_t& x : partial) x = l.take(2 * (size_t)std::max(chunk_capacity(n), kRecBlocks) * sizeof(Bounds));
    const size_t bins = l.take((size_t)big_capacity(n) * kBinWords * 4), mid = l.take((n / kSmall + 2) * sizeof(Range)),
                 small = l.take(((size_t)n + 1) * sizeof(Range)), upper = l.take(((size_t)n + 1) * 4),
                 c = l.take(sizeof(Counters2));
    for (size_t& x : pend) x = l.take(((size_t)n + 1) * 4);
    const size_t slots = l.take(((size_t)n + 1) * 32), counts = l.take(((size_t)n + 1) * 4),
                 sums = l.take((n / kBlock + 2) * sizeof(uint2));
    if (a) {
        for (int k = 0; k < 2; k++) {
            a->rec[k] = reinterpret_cast<Rec*>(p + rec[k]);
            a->big[k] = reinterpret_cast<BigRange*>(p + big[k]);
            a->chunk_map[k] = reinterpret_cast<uint2*>(p + map[k]);
            a->pend[k] = reinterpret_cast<uint32_t*>(p + pend[k]);
            a->partial[k] = reinterpret_cast<Bounds*>(p + partial[k]);
        }
        a->nodes = reinterpret_cast<Node2*>(p + nodes);
        a->cost = reinterpret_cast<float*>(p + cost);
        a->how = reinterpret_cast<uint64_t*>(p + how);
        a->order = reinterpret_cast<uint32_t*>(p + order);
        a->bins = reinterpret_cast<uint32_t*>(p + bins);
        a->mid = reinterpret_cast<Range*>(p + mid);
        a->small = reinterpret_cast<Range*>(p + small);
        a->upper = reinterpret_cast<uint32_t*>(p + upper);
        a->c = reinterpret_cast<Counters2*>(p + c);
        a->slots = reinterpret_cast<uint32_t*>(p + slots);
        a->counts = reinterpret_cast<uint32_t*>(p + counts);
        a->tile_sums = reinterpret_cast<uint2*>(p + sums);
    }
    return l.off;
}

}  // namespace

size_t bvh_device_scratch_bytes(uint32_t n) { return lay_out(n, nullptr, nullptr); }

#define BVH_TRY(expr)                        \
    do {                                     \
        const hipError_t e_ = (expr);        \
        if (e_ != hipSuccess) return e_;     \
    } while (0)

hipError_t bvh_device_build(const float* vertices, const uint32_t* indices, const BvhSource* sources,
                            uint32_t num_sources, uint32_t n, uint32_t max_leaf, void* scratch, Bvh8Node* nodes,
                            BvhTri* tris, uint32_t* num_nodes, uint32_t* depth, BvhDeviceStatus* status,
                            hipStream_t st) {
    BuildArgs a{};
    lay_out(n, static_cast<char*>(scratch), &a);
    a.vertices = vertices;
    a.indices = indices;
    a.sources = sources;
    a.num_sources = num_sources;
    a.n = n;
    a.max_leaf = max_leaf;
    a.out_nodes = nodes;
    a.out_tris = tris;
    *status = kBvhBuilt;

    Counters2 c;
    auto read = [&]() -> hipError_t {
        BVH_TRY(hipGetLastError());
        BVH_TRY(hipMemcpyAsync(&c, a.c, sizeof(c), hipMemcpyDeviceToHost, st));
        return hipStreamSynchronize(st);
    };
    hipLaunchKernelGGL(init_kernel, dim3(256), dim3(256), 0, st, a, big_capacity(n));
    hipLaunchKernelGGL(records_kernel, dim3(rec_blocks(n)), dim3(kBlock), 0, st, a);
    // phase 1: about log2(n / kBig) levels for ordinary scenes
    uint32_t done = 0;
    if (n > kBig) {
        uint32_t round = 4;
        for (uint32_t m = n / kBig; m > 0; m >>= 1) round++;
        const uint32_t max_chunks = chunk_capacity(n), ranges = big_capacity(n);
        for (;;) {
            const uint32_t end = std::min(done + round, kMaxLevels - 1);
            for (; done < end; done++) {
                hipLaunchKernelGGL(big_bins_kernel, dim3(max_chunks), dim3(kBlock), 0, st, a, done);
                hipLaunchKernelGGL(big_split_kernel, dim3(ranges), dim3(64), 0, st, a, done);
                hipLaunchKernelGGL(big_partition_kernel, dim3(max_chunks), dim3(kBlock), 0, st, a, done);
            }
            BVH_TRY(read());
            if (c.nonfinite || (c.big[done] != 0u && done >= kMaxLevels - 1)) {
                *status = kBvhUnsupported;
                return hipSuccess;
            }
            if (c.big[done] == 0u) break;
            round = 8;
        }
    }
    hipLaunchKernelGGL(mid_kernel, dim3(std::min<uint32_t>(n / kSmall + 1, 2048)), dim3(kBlock), 0, st, a);
    hipLaunchKernelGGL(small_kernel, dim3(std::min<uint32_t>(n / 8 + 1, 16384)), dim3(64), 0, st, a);
    BVH_TRY(read());
    if (c.nonfinite) {
        *status = kBvhUnsupported;
        return hipSuccess;
    }
    if (c.upper != 0u) {
        const uint32_t blocks = std::min<uint32_t>((c.upper + kBlock - 1) / kBlock, 1024);
        for (int d = (int)c.max_depth; d >= 0; d--)
            hipLaunchKernelGGL(collapse_kernel, dim3(blocks), dim3(kBlock), 0, st, a, (uint32_t)d);
    }
    hipLaunchKernelGGL(bvh8_root_kernel, dim3(1), dim3(64), 0, st, a);
    uint32_t level = 0;
    const uint32_t blocks = std::min<uint32_t>(n / (2 * kBlock) + 1, 2048);
    for (;;) {
        const uint32_t end = std::min(level + 12u, kBvhLevels);
        for (; level < end; level++) {
            hipLaunchKernelGGL(bvh8_children_kernel, dim3(blocks), dim3(kBlock), 0, st, a, level);
            hipLaunchKernelGGL(bvh8_scan_kernel, dim3(1), dim3(1024), 0, st, a, level);
            hipLaunchKernelGGL(bvh8_emit_kernel, dim3(blocks), dim3(kBlock), 0, st, a, level);
        }
        BVH_TRY(read());
        if (c.level_count[level] == 0u || level >= kBvhLevels) break;
    }
    if (c.bad_quant) {
        *status = kBvhQuantisation;
        return hipSuccess;
    }
    uint32_t levels = 0, total = 0;
    for (uint32_t l = 0; l < level && c.level_count[l] != 0u; l++) {
        levels = l + 1;
        total += c.level_count[l];
    }
    if (levels >= 60u) {  // the host builder's limit
        *status = kBvhTooDeep;
        return hipSuccess;
    }
    *num_nodes = total;
    *depth = levels;
    return hipSuccess;
}

}  // namespace rm
