// bvh_device.hip — BVH8 construction on the GPU (REINA_RT_BUILD_DEVICE), the
// replacement of the driver's BLAS/TLAS build (src/graphics/Blas.cpp:8-124,
// src/tools/vktools.cpp:460-596) for flattened scenes.
//
//   1. triangle boxes and centroids; scene box and centroid bounds
//   2. a binary BVH, top-down and breadth-first by the surface area heuristic:
//      - a task (a contiguous range of the triangle reference array with its
//        box and centroid bounds) of more than kSmall triangles is one
//        workgroup (of more than kBig, one per chunk of its range, the same
//        steps as separate launches): 32 bins per axis over the centroid bounds (counts and bin
//        boxes by LDS atomics), prefix and suffix sums over the bins with
//        the SAH cost area(L)·N(L) + area(R)·N(R) evaluated in FP64, the
//        cheapest split over the three axes, then a stable partition of the
//        range into the other of two reference buffers (block-wide scans of
//        the side flags) and the exact box and centroid bounds of both sides;
//        as the host builder, but every level in a few launches;
//      - a task of at most kSmall triangles is one wave, which builds its
//        whole subtree in registers: per range and axis a bitonic sort of the
//        centroids across the 64 lanes, prefix and suffix boxes by lane
//        shuffles, and the exact (unbinned) SAH split, FP64 cost.
//      A binary tree over positions [0, n) cuts each position boundary m
//      exactly once, so the internal node that splits its range at m gets the
//      id n + m - 1 and the leaf at position p the id p: ids are
//      deterministic without counters, and a child writes its id into its
//      parent when it splits. Nodes that cannot be split (all centroids equal)
//      are halved by position.
//   3. collapse to BVH8 level by level: a subtree of <= 3 triangles is a
//      leaf unless splitting it is cheaper by the SAH; a node opens its
//      largest-area internal child until it has 8 children, children take
//      octant slots as in the host builder, and node / triangle offsets come
//      from exclusive scans (this file's own), so the result is deterministic.
// The output has the host builder's format (Bvh8Node, leaf-ordered triangles,
// boxes padded outward by one ulp), so the traversal, the quantizer and the
// oracle's restatement apply unchanged.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <functional>
#include <string>
#include <vector>

#include "bvh_host.h"

namespace rt {
namespace {

constexpr uint32_t kLeafMax = 3;
constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr int kBins = 32;
constexpr uint32_t kSmall = 64;   // tasks of at most this many triangles: one wave each

__device__ __forceinline__ uint32_t ord_key(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_ord(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

struct Box6 {   // ordered-integer keys: lo (min), hi (max)
    uint32_t lo[3], hi[3];
};

// scene box (b) and centroid bounds (c)
struct SceneBounds {
    Box6 b, c;
    uint32_t nonfinite;   // k_flatten: some coordinate is infinite or NaN
};

__device__ __forceinline__ void tri_box(const float* w, float* lo, float* hi) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        lo[a] = fminf(fminf(w[a], w[3 + a]), w[6 + a]);
        hi[a] = fmaxf(fmaxf(w[a], w[3 + a]), w[6 + a]);
    }
}

__device__ __forceinline__ float half_area(float x0, float y0, float z0, float x1, float y1, float z1) {
    const float dx = x1 - x0, dy = y1 - y0, dz = z1 - z0;
    return dx * dy + dy * dz + dz * dx;
}

__device__ __forceinline__ float wave_min(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

// World-space triangles, world = ((c0 x + c1 y) + c2 z) + c3 in the host
// flattening's operation order, and the instance and primitive of every
// triangle; w may be null (only the ids). A thread finds its instance by
// bisection over the first-triangle ids (an instance without triangles shares
// its successor's id and is never the last one at or below g). It reads and
// writes ~100 bytes per triangle once: 14 us for 327,686 triangles, where the
// loop on the host and the upload of its result took 2.6 ms.
__global__ __launch_bounds__(256) void k_flatten(const InstanceRec* __restrict__ inst, uint32_t num_inst,
                                                 const float4* __restrict__ vertices,
                                                 const uint32_t* __restrict__ indices, uint32_t n,
                                                 float* __restrict__ w, uint32_t* __restrict__ tri_inst,
                                                 uint32_t* __restrict__ tri_prim, SceneBounds* sb) {
    const uint32_t g = blockIdx.x * 256u + threadIdx.x;
    if (g >= n) return;
    uint32_t a = 0, b = num_inst;   // inst[a].tri_base <= g; inst[b].tri_base > g
    while (b - a > 1) {
        const uint32_t m = (a + b) / 2;
        if (inst[m].tri_base <= g) a = m; else b = m;
    }
    const InstanceRec& r = inst[a];
    const uint32_t prim = g - r.tri_base;
    tri_inst[g] = a;
    tri_prim[g] = prim;
    if (!w) return;
    bool bad = false;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float4 v = vertices[indices[3ull * prim + r.index_offset + k]];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float o = ((r.c0[c] * v.x + r.c1[c] * v.y) + r.c2[c] * v.z) + r.c3[c];
            w[9ull * g + 3 * k + c] = o;
            bad |= !(fabsf(o) < INFINITY);
        }
    }
    if (bad) sb->nonfinite = 1;
}

// Triangle boxes (plo = lo.xyz, phi = hi.xyz), the identity reference order
// and the scene's box and centroid bounds. At most kPrepBlocks blocks, each
// adding its bounds with 12 atomics: one set per wave (61,000 atomics on 12
// words for 327,686 triangles) took 700 us.
constexpr uint32_t kPrepBlocks = 512;
__global__ __launch_bounds__(256) void k_prep(const float* __restrict__ wtri, uint32_t n, float4* __restrict__ plo,
                                              float4* __restrict__ phi, uint32_t* __restrict__ ref, SceneBounds* sb) {
    __shared__ float s_b[4][12];
    float v[12];
#pragma unroll
    for (int q = 0; q < 12; ++q) v[q] = (q % 6) < 3 ? INFINITY : -INFINITY;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) {
        float lo[3], hi[3];
        tri_box(wtri + 9ull * i, lo, hi);
        plo[i] = make_float4(lo[0], lo[1], lo[2], 0.0f);
        phi[i] = make_float4(hi[0], hi[1], hi[2], 0.0f);
        ref[i] = i;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const float c = 0.5f * lo[a] + 0.5f * hi[a];
            v[a] = fminf(v[a], lo[a]);
            v[3 + a] = fmaxf(v[3 + a], hi[a]);
            v[6 + a] = fminf(v[6 + a], c);
            v[9 + a] = fmaxf(v[9 + a], c);
        }
    }
#pragma unroll
    for (int q = 0; q < 12; ++q) {
        const float r = (q % 6) < 3 ? wave_min(v[q]) : wave_max(v[q]);
        if (__lane_id() == 0) s_b[threadIdx.x >> 6][q] = r;
    }
    __syncthreads();
    if (threadIdx.x < 6u) {
        const uint32_t q = threadIdx.x / 3u * 6u + threadIdx.x % 3u;   // lo of (b, c) axis a; hi is 3 further
        float lo = s_b[0][q], hi = s_b[0][q + 3];
        for (int w = 1; w < 4; ++w) { lo = fminf(lo, s_b[w][q]); hi = fmaxf(hi, s_b[w][q + 3]); }
        uint32_t* words = reinterpret_cast<uint32_t*>(sb);   // b.lo b.hi c.lo c.hi
        if (lo <= hi) {
            atomicMin(words + q, ord_key(lo));
            atomicMax(words + q + 3, ord_key(hi));
        }
    }
}

// ---- binary build --------------------------------------------------------------
struct BNode {
    uint32_t left, right;   // children; left = kNone for a triangle
    uint32_t count;         // triangles below
    uint32_t tri;           // triangle index (leaves)
    float lo[3], hi[3];
};

// A range [begin, begin + count) of reference buffer `buf` to split; its node
// id is known only once it splits, so it tells its parent then.
struct Task {
    uint32_t begin, count, parent, side;   // side: 0 left child, 1 right child
    uint32_t buf;
    uint32_t chunk0, nchunks, pad;   // big tasks: their chunks of the level
    float lo[3], hi[3];     // box
    float clo[3], chi[3];   // centroid bounds
};

struct SmallTask {
    uint32_t begin, count, parent, meta;   // meta: side | buf << 1
};

struct BuildCtl {
    uint32_t n_next;    // tasks appended for the next level
    uint32_t n_big;     // big tasks appended for the next level
    uint32_t n_chunks;  // chunks of those
    uint32_t pad;
    uint32_t n_small;   // small tasks appended
    uint32_t root;
};

// Tasks of more than kBig triangles are split by several workgroups, one per
// chunk of kChunk references. One workgroup per task left the GPU idle at the
// top of the tree: the 16 levels of 327,686 triangles took 25.0 ms, the first
// one alone a pass of 1,280 steps on one CU; now 1.3 ms in all.
constexpr uint32_t kChunk = 1024;
constexpr uint32_t kBig = 4096;
constexpr uint32_t kBinWords = 3 * kBins * 7;   // per axis and bin: count, box keys
// Shared state of a big task while its chunks work on it.
struct BigState {
    uint32_t bins[kBinWords];
    uint32_t side[2][12];      // exact bounds of both sides (ordered keys)
    int32_t axis, split;       // cheapest split: left = bins 0..split of `axis` (-1: halve by position)
    uint32_t nl, pad;          // triangles on the left
};

__device__ __forceinline__ void set_child(BNode* nodes, uint32_t parent, uint32_t side, uint32_t id, BuildCtl* ctl) {
    if (parent == kNone) ctl->root = id;
    else if (side == 0u) nodes[parent].left = id;
    else nodes[parent].right = id;
}

__device__ __forceinline__ void write_leaf(BNode* nodes, uint32_t pos, uint32_t tri, float4 lo, float4 hi) {
    BNode b;
    b.left = b.right = kNone;
    b.count = 1;
    b.tri = tri;
    b.lo[0] = lo.x; b.lo[1] = lo.y; b.lo[2] = lo.z;
    b.hi[0] = hi.x; b.hi[1] = hi.y; b.hi[2] = hi.z;
    nodes[pos] = b;
}

// Appends a child range as a task of the next level (> kSmall triangles; > kBig:
// a big task, whose index is returned) or a small task; a single triangle was
// already written as a leaf.
__device__ uint32_t emit_child(uint32_t begin, uint32_t count, uint32_t parent, uint32_t side, uint32_t buf,
                               const float* lo, const float* hi, const float* clo, const float* chi, Task* next,
                               Task* big, SmallTask* small, BuildCtl* ctl) {
    if (count < 2u) return kNone;
    if (count <= kSmall) {
        const uint32_t k = atomicAdd(&ctl->n_small, 1u);
        small[k] = SmallTask{begin, count, parent, side | (buf << 1)};
        return kNone;
    }
    Task t;
    t.begin = begin; t.count = count; t.parent = parent; t.side = side;
    t.buf = buf; t.chunk0 = t.nchunks = t.pad = 0u;
#pragma unroll
    for (int a = 0; a < 3; ++a) { t.lo[a] = lo[a]; t.hi[a] = hi[a]; t.clo[a] = clo[a]; t.chi[a] = chi[a]; }
    if (count > kBig) {
        const uint32_t k = atomicAdd(&ctl->n_big, 1u);
        t.nchunks = (count + kChunk - 1u) / kChunk;
        t.chunk0 = atomicAdd(&ctl->n_chunks, t.nchunks);
        big[k] = t;
        return k;
    }
    next[atomicAdd(&ctl->n_next, 1u)] = t;
    return kNone;
}

// ---- pieces of a split shared by the one-workgroup and the chunked kernels ----
struct BinScale {
    float sc[3];   // bins per unit of centroid, 0: no extent
};
__device__ __forceinline__ BinScale bin_scale(const Task& T) {
    BinScale b;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float ext = T.chi[a] - T.clo[a];
        b.sc[a] = ext > 0.0f ? (float)kBins / ext : 0.0f;
    }
    return b;
}
__device__ __forceinline__ int bin_of(float c, float clo, float sc) {
    const int k = (int)((c - clo) * sc);
    return min(max(k, 0), kBins - 1);
}

// Empty bins: s[(axis * kBins + bin) * 7] = {count, lo keys, hi keys}.
__device__ __forceinline__ uint32_t empty_bin_word(uint32_t k) {
    const uint32_t q = k % 7u;
    return q == 0u || q > 3u ? 0u : 0xFFFFFFFFu;
}

// Adds one triangle's box to the three axes' bins (LDS).
__device__ __forceinline__ void add_to_bins(uint32_t* s, const Task& T, const BinScale& bs, float4 lo, float4 hi) {
    const float b[6] = {lo.x, lo.y, lo.z, hi.x, hi.y, hi.z};
    uint32_t key[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) key[q] = ord_key(b[q]);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (bs.sc[a] == 0.0f) continue;
        uint32_t* w = s + (a * kBins + bin_of(0.5f * b[a] + 0.5f * b[3 + a], T.clo[a], bs.sc[a])) * 7;
        atomicAdd(w, 1u);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            atomicMin(w + 1 + q, key[q]);
            atomicMax(w + 4 + q, key[3 + q]);
        }
    }
}

// The cheapest split of axis a by one wave, lane = bin; cost (infinite: none) and bin in every lane.
__device__ __forceinline__ void best_split(const uint32_t* s, int a, bool extent, double& cost, int& k) {
    const uint32_t lane = __lane_id();
    const uint32_t* w = s + (a * kBins + (lane < (uint32_t)kBins ? lane : 0u)) * 7;
    const bool bin = lane < (uint32_t)kBins && extent;
    uint32_t cnt = bin ? w[0] : 0u;
    float lo[3], hi[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        lo[q] = (bin && cnt) ? key_ord(w[1 + q]) : INFINITY;
        hi[q] = (bin && cnt) ? key_ord(w[4 + q]) : -INFINITY;
    }
    uint32_t pc = cnt, qc = cnt;
    float plo_[3], phi_[3], qlo[3], qhi[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) { plo_[q] = qlo[q] = lo[q]; phi_[q] = qhi[q] = hi[q]; }
    for (int d = 1; d < kBins; d <<= 1) {   // prefix over bins 0..lane, suffix over lane..31
        const uint32_t uc = __shfl_up(pc, d), dc = __shfl_down(qc, d);
        float ul[3], uh[3], dl[3], dh[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            ul[q] = __shfl_up(plo_[q], d); uh[q] = __shfl_up(phi_[q], d);
            dl[q] = __shfl_down(qlo[q], d); dh[q] = __shfl_down(qhi[q], d);
        }
        if (lane >= (uint32_t)d) {
            pc += uc;
#pragma unroll
            for (int q = 0; q < 3; ++q) { plo_[q] = fminf(plo_[q], ul[q]); phi_[q] = fmaxf(phi_[q], uh[q]); }
        }
        if (lane + (uint32_t)d < (uint32_t)kBins) {
            qc += dc;
#pragma unroll
            for (int q = 0; q < 3; ++q) { qlo[q] = fminf(qlo[q], dl[q]); qhi[q] = fmaxf(qhi[q], dh[q]); }
        }
    }
    // split after bin `lane`: left = bins 0..lane, right = bins lane+1..31
    const uint32_t rc = __shfl_down(qc, 1);
    float rl[3], rh[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) { rl[q] = __shfl_down(qlo[q], 1); rh[q] = __shfl_down(qhi[q], 1); }
    cost = INFINITY;
    if (bin && lane + 1u < (uint32_t)kBins && pc > 0u && rc > 0u)
        cost = (double)half_area(plo_[0], plo_[1], plo_[2], phi_[0], phi_[1], phi_[2]) * (double)pc +
               (double)half_area(rl[0], rl[1], rl[2], rh[0], rh[1], rh[2]) * (double)rc;
    k = (int)lane;
    for (int o = 32; o > 0; o >>= 1) {   // argmin, ties to the lower bin
        const double oc = __shfl_xor(cost, o);
        const int ok = __shfl_xor(k, o);
        if (oc < cost || (oc == cost && ok < k)) { cost = oc; k = ok; }
    }
}

// Whether the i-th triangle of task T (box lo, hi) goes left.
__device__ __forceinline__ bool goes_left(const Task& T, const BinScale& bs, int axis, int split, uint32_t nl, uint32_t i,
                                          float4 lo, float4 hi) {
    if (axis < 0) return i < nl;
    const float c = 0.5f * (axis == 0 ? lo.x : axis == 1 ? lo.y : lo.z) +
                    0.5f * (axis == 0 ? hi.x : axis == 1 ? hi.y : hi.z);
    const float clo = axis == 0 ? T.clo[0] : axis == 1 ? T.clo[1] : T.clo[2];
    const float sc = axis == 0 ? bs.sc[0] : axis == 1 ? bs.sc[1] : bs.sc[2];
    return bin_of(c, clo, sc) <= split;
}

// Partitions references [first, last) of task T (256 threads) into dst: left
// ones from T.begin + offl on, right ones from T.begin + nl + offr on, in
// order; both sides' bounds go to s_side (LDS, ordered keys).
__device__ __forceinline__ void partition_range(const Task& T, const BinScale& bs, int axis, int split, uint32_t nl,
                                                uint32_t first, uint32_t last, uint32_t offl, uint32_t offr,
                                                const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                const float4* __restrict__ plo, const float4* __restrict__ phi,
                                                BNode* __restrict__ nodes, uint32_t* s_wl, uint32_t (*s_side)[12]) {
    const uint32_t tid = threadIdx.x, lane = __lane_id(), w = tid >> 6;
    const uint32_t nr = T.count - nl;
    float sb[2][12];
#pragma unroll
    for (int q = 0; q < 12; ++q) { sb[0][q] = sb[1][q] = (q % 6) < 3 ? INFINITY : -INFINITY; }
    for (uint32_t base = first; base < last; base += 256u) {
        const uint32_t i = base + tid;
        const bool valid = i < last;
        uint32_t t = 0;
        float4 lo = make_float4(0.0f, 0.0f, 0.0f, 0.0f), hi = lo;
        bool left = false;
        if (valid) {
            t = src[T.begin + i];
            lo = plo[t];
            hi = phi[t];
            left = goes_left(T, bs, axis, split, nl, i, lo, hi);
        }
        const uint64_t bal = __ballot(left);
        const uint32_t below = (uint32_t)__popcll(bal & ((1ull << lane) - 1ull));
        if (lane == 0) s_wl[w] = (uint32_t)__popcll(bal);
        __syncthreads();
        uint32_t wb = 0, tot = 0;
        for (uint32_t q = 0; q < 4; ++q) {
            if (q < w) wb += s_wl[q];
            tot += s_wl[q];
        }
        __syncthreads();
        if (valid) {
            const uint32_t rl = wb + below;
            const uint32_t pos = left ? T.begin + offl + rl : T.begin + nl + offr + (tid - rl);
            dst[pos] = t;
            if (left && nl == 1u) write_leaf(nodes, pos, t, lo, hi);
            if (!left && nr == 1u) write_leaf(nodes, pos, t, lo, hi);
            const int sd = left ? 0 : 1;
            const float b[6] = {lo.x, lo.y, lo.z, hi.x, hi.y, hi.z};
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const float c = 0.5f * b[q] + 0.5f * b[3 + q];
                sb[sd][q] = fminf(sb[sd][q], b[q]);
                sb[sd][3 + q] = fmaxf(sb[sd][3 + q], b[3 + q]);
                sb[sd][6 + q] = fminf(sb[sd][6 + q], c);
                sb[sd][9 + q] = fmaxf(sb[sd][9 + q], c);
            }
        }
        const uint32_t valid_n = min(256u, last - base);
        offl += tot;
        offr += valid_n - tot;
    }
#pragma unroll
    for (int sd = 0; sd < 2; ++sd) {
#pragma unroll
        for (int q = 0; q < 12; ++q) {
            const bool is_min = (q % 6) < 3;
            const float v = is_min ? wave_min(sb[sd][q]) : wave_max(sb[sd][q]);
            if (lane == 0) {   // also an infinity: a wave without triangles of this side changes nothing
                if (is_min) atomicMin(&s_side[sd][q], ord_key(v));
                else atomicMax(&s_side[sd][q], ord_key(v));
            }
        }
    }
}

__device__ __forceinline__ void write_split(const Task& T, uint32_t n, uint32_t nl, BNode* nodes, BuildCtl* ctl) {
    const uint32_t id = n + T.begin + nl - 1u;
    BNode b;
    b.left = nl == 1u ? T.begin : kNone;
    b.right = T.count - nl == 1u ? T.begin + nl : kNone;
    b.count = T.count;
    b.tri = kNone;
#pragma unroll
    for (int a = 0; a < 3; ++a) { b.lo[a] = T.lo[a]; b.hi[a] = T.hi[a]; }
    nodes[id] = b;
    set_child(nodes, T.parent, T.side, id, ctl);
}

// Child `sd` of a split task, its bounds from ordered keys.
__device__ __forceinline__ uint32_t emit_side(const Task& T, uint32_t n, uint32_t nl, uint32_t sd, const uint32_t* keys,
                                              Task* next, Task* big, SmallTask* small, BuildCtl* ctl) {
    float v[12];
    for (int q = 0; q < 12; ++q) v[q] = key_ord(keys[q]);
    return emit_child(sd ? T.begin + nl : T.begin, sd ? T.count - nl : nl, n + T.begin + nl - 1u, sd, T.buf ^ 1u, v, v + 3,
                      v + 6, v + 9, next, big, small, ctl);
}

__device__ __forceinline__ uint32_t empty_side_word(uint32_t q) { return q % 6u < 3u ? 0xFFFFFFFFu : 0u; }

// One workgroup per task of kSmall + 1 to kBig triangles: binned SAH split,
// stable partition into the other buffer, the node and its children.
__global__ __launch_bounds__(256) void k_split_tasks(const Task* __restrict__ tasks, uint32_t n,
                                                     const float4* __restrict__ plo, const float4* __restrict__ phi,
                                                     uint32_t* __restrict__ ref0, uint32_t* __restrict__ ref1,
                                                     BNode* __restrict__ nodes, Task* __restrict__ next,
                                                     SmallTask* __restrict__ small, BuildCtl* ctl) {
    __shared__ uint32_t s_bin[kBinWords];
    __shared__ double s_cost[3];
    __shared__ int s_split[3];
    __shared__ uint32_t s_wl[4];
    __shared__ uint32_t s_side[2][12];
    const Task T = tasks[blockIdx.x];
    const uint32_t tid = threadIdx.x, w = tid >> 6;
    const uint32_t* src = T.buf ? ref1 : ref0;
    uint32_t* dst = T.buf ? ref0 : ref1;
    const BinScale bs = bin_scale(T);
    for (uint32_t k = tid; k < kBinWords; k += 256u) s_bin[k] = empty_bin_word(k);
    if (tid < 24u) s_side[tid / 12u][tid % 12u] = empty_side_word(tid % 12u);
    __syncthreads();
    for (uint32_t i = tid; i < T.count; i += 256u) {
        const uint32_t t = src[T.begin + i];
        add_to_bins(s_bin, T, bs, plo[t], phi[t]);
    }
    __syncthreads();
    if (w < 3u) {
        double cost;
        int k;
        best_split(s_bin, (int)w, bs.sc[w] != 0.0f, cost, k);
        if (__lane_id() == 0) { s_cost[w] = cost; s_split[w] = k; }
    }
    __syncthreads();
    int axis = -1, split = 0;
    double best = INFINITY;
    for (int a = 0; a < 3; ++a)
        if (s_cost[a] < best) { best = s_cost[a]; axis = a; split = s_split[a]; }
    uint32_t nl = 0;
    if (axis >= 0) {
        for (int k = 0; k <= split; ++k) nl += s_bin[(axis * kBins + k) * 7];
    } else {
        nl = T.count / 2u;   // all centroids equal: halve by position
    }
    partition_range(T, bs, axis, split, nl, 0u, T.count, 0u, 0u, src, dst, plo, phi, nodes, s_wl, s_side);
    __syncthreads();
    if (tid == 0) {
        write_split(T, n, nl, nodes, ctl);
        emit_side(T, n, nl, 0u, s_side[0], next, nullptr, small, ctl);   // children of at most kBig: never big
        emit_side(T, n, nl, 1u, s_side[1], next, nullptr, small, ctl);
    }
}

// ---- tasks of more than kBig triangles: the same split by chunks ----------------
// Prepares the shared state and the chunk -> task map of a big task (256 threads).
__device__ __forceinline__ void init_big(BigState& B, const Task& T, uint32_t task, uint32_t* __restrict__ chunk_task) {
    for (uint32_t k = threadIdx.x; k < kBinWords; k += 256u) B.bins[k] = empty_bin_word(k);
    if (threadIdx.x < 24u) B.side[threadIdx.x / 12u][threadIdx.x % 12u] = empty_side_word(threadIdx.x % 12u);
    for (uint32_t k = threadIdx.x; k < T.nchunks; k += 256u) chunk_task[T.chunk0 + k] = task;
}

__global__ __launch_bounds__(256) void k_big_root(const Task* __restrict__ tasks, BigState* __restrict__ state,
                                                  uint32_t* __restrict__ chunk_task) {
    init_big(state[0], tasks[0], 0u, chunk_task);
}

// Bins of one chunk, merged into the task's.
__global__ __launch_bounds__(256) void k_big_bin(const Task* __restrict__ tasks, const uint32_t* __restrict__ chunk_task,
                                                 const float4* __restrict__ plo, const float4* __restrict__ phi,
                                                 const uint32_t* __restrict__ ref0, const uint32_t* __restrict__ ref1,
                                                 BigState* __restrict__ state) {
    __shared__ uint32_t s_bin[kBinWords];
    const uint32_t ti = chunk_task[blockIdx.x];
    const Task T = tasks[ti];
    const uint32_t* src = T.buf ? ref1 : ref0;
    const BinScale bs = bin_scale(T);
    for (uint32_t k = threadIdx.x; k < kBinWords; k += 256u) s_bin[k] = empty_bin_word(k);
    __syncthreads();
    const uint32_t first = (blockIdx.x - T.chunk0) * kChunk, last = min(first + kChunk, T.count);
    for (uint32_t i = first + threadIdx.x; i < last; i += 256u) {
        const uint32_t t = src[T.begin + i];
        add_to_bins(s_bin, T, bs, plo[t], phi[t]);
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < kBinWords; k += 256u) {
        const uint32_t v = s_bin[k], q = k % 7u;
        if (s_bin[k - q] == 0u) continue;   // an empty bin
        uint32_t* g = &state[ti].bins[k];
        if (q == 0u) atomicAdd(g, v);
        else if (q <= 3u) atomicMin(g, v);
        else atomicMax(g, v);
    }
}

// The cheapest split of each big task.
__global__ __launch_bounds__(256) void k_big_plan(const Task* __restrict__ tasks, BigState* __restrict__ state) {
    __shared__ double s_cost[3];
    __shared__ int s_split[3];
    BigState& B = state[blockIdx.x];
    const Task T = tasks[blockIdx.x];
    const BinScale bs = bin_scale(T);
    const uint32_t w = threadIdx.x >> 6;
    if (w < 3u) {
        double cost;
        int k;
        best_split(B.bins, (int)w, bs.sc[w] != 0.0f, cost, k);
        if (__lane_id() == 0) { s_cost[w] = cost; s_split[w] = k; }
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    int axis = -1, split = 0;
    double best = INFINITY;
    for (int a = 0; a < 3; ++a)
        if (s_cost[a] < best) { best = s_cost[a]; axis = a; split = s_split[a]; }
    uint32_t nl = T.count / 2u;
    if (axis >= 0) {
        nl = 0;
        for (int k = 0; k <= split; ++k) nl += B.bins[(axis * kBins + k) * 7];
    }
    B.axis = axis;
    B.split = split;
    B.nl = nl;
}

// Left triangles of each chunk.
__global__ __launch_bounds__(256) void k_big_count(const Task* __restrict__ tasks, const uint32_t* __restrict__ chunk_task,
                                                   const float4* __restrict__ plo, const float4* __restrict__ phi,
                                                   const uint32_t* __restrict__ ref0, const uint32_t* __restrict__ ref1,
                                                   const BigState* __restrict__ state, uint32_t* __restrict__ chunk_left) {
    __shared__ uint32_t s_w[4];
    const uint32_t ti = chunk_task[blockIdx.x];
    const Task T = tasks[ti];
    const uint32_t* src = T.buf ? ref1 : ref0;
    const BinScale bs = bin_scale(T);
    const int axis = state[ti].axis, split = state[ti].split;
    const uint32_t nl = state[ti].nl;
    const uint32_t first = (blockIdx.x - T.chunk0) * kChunk, last = min(first + kChunk, T.count);
    uint32_t c = 0;
    for (uint32_t base = first; base < last; base += 256u) {
        const uint32_t i = base + threadIdx.x;
        bool left = false;
        if (i < last) {
            const uint32_t t = src[T.begin + i];
            left = goes_left(T, bs, axis, split, nl, i, plo[t], phi[t]);
        }
        c += (uint32_t)__popcll(__ballot(left));
    }
    if (__lane_id() == 0) s_w[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) chunk_left[blockIdx.x] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

// Partition of each chunk: its place from the left counts of the chunks before it.
__global__ __launch_bounds__(256) void k_big_partition(const Task* __restrict__ tasks,
                                                       const uint32_t* __restrict__ chunk_task,
                                                       const float4* __restrict__ plo, const float4* __restrict__ phi,
                                                       uint32_t* __restrict__ ref0, uint32_t* __restrict__ ref1,
                                                       BigState* __restrict__ state,
                                                       const uint32_t* __restrict__ chunk_left,
                                                       BNode* __restrict__ nodes) {
    __shared__ uint32_t s_wl[4];
    __shared__ uint32_t s_side[2][12];
    const uint32_t ti = chunk_task[blockIdx.x];
    const Task T = tasks[ti];
    const uint32_t* src = T.buf ? ref1 : ref0;
    uint32_t* dst = T.buf ? ref0 : ref1;
    const BinScale bs = bin_scale(T);
    if (threadIdx.x < 24u) s_side[threadIdx.x / 12u][threadIdx.x % 12u] = empty_side_word(threadIdx.x % 12u);
    uint32_t before = 0;
    for (uint32_t k = T.chunk0 + threadIdx.x; k < blockIdx.x; k += 256u) before += chunk_left[k];
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o);
    if (__lane_id() == 0) s_wl[threadIdx.x >> 6] = before;
    __syncthreads();
    const uint32_t offl = s_wl[0] + s_wl[1] + s_wl[2] + s_wl[3];
    __syncthreads();
    const uint32_t first = (blockIdx.x - T.chunk0) * kChunk, last = min(first + kChunk, T.count);
    partition_range(T, bs, state[ti].axis, state[ti].split, state[ti].nl, first, last, offl, first - offl, src, dst, plo,
                    phi, nodes, s_wl, s_side);
    __syncthreads();
    if (threadIdx.x < 24u) {
        const uint32_t q = threadIdx.x % 12u, v = s_side[threadIdx.x / 12u][q];
        uint32_t* g = &state[ti].side[threadIdx.x / 12u][q];
        if (v != empty_side_word(q)) {
            if (q % 6u < 3u) atomicMin(g, v);
            else atomicMax(g, v);
        }
    }
}

// The node and the children of each big task; big children get their state and chunk map.
__global__ __launch_bounds__(256) void k_big_emit(const Task* __restrict__ tasks, const BigState* __restrict__ state,
                                                  uint32_t n, BNode* __restrict__ nodes, Task* __restrict__ next,
                                                  Task* __restrict__ big, BigState* __restrict__ big_state,
                                                  uint32_t* __restrict__ chunk_task, SmallTask* __restrict__ small,
                                                  BuildCtl* ctl) {
    __shared__ uint32_t s_child[2];
    __shared__ Task s_task[2];
    const Task T = tasks[blockIdx.x];
    const uint32_t nl = state[blockIdx.x].nl;
    if (threadIdx.x == 0) {
        write_split(T, n, nl, nodes, ctl);
        for (uint32_t sd = 0; sd < 2u; ++sd) {
            const uint32_t c = emit_side(T, n, nl, sd, state[blockIdx.x].side[sd], next, big, small, ctl);
            s_child[sd] = c;
            if (c != kNone) s_task[sd] = big[c];
        }
    }
    __syncthreads();
    for (uint32_t sd = 0; sd < 2u; ++sd)
        if (s_child[sd] != kNone) init_big(big_state[s_child[sd]], s_task[sd], s_child[sd], chunk_task);
}

// Lexicographic (key, payload) bitonic sort across lanes 0..width-1 (width a
// power of two), ascending. Integer keys: every pair has an order, so the
// lanes of a pair never keep the same entry. As floats, a NaN compares false
// either way and both lanes kept one entry of the two.
__device__ __forceinline__ void wave_sort(uint32_t& key, uint32_t& pay, uint32_t lane, uint32_t width) {
    for (uint32_t k = 2; k <= width; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            const uint32_t ok = __shfl_xor(key, (int)j);
            const uint32_t op = __shfl_xor(pay, (int)j);
            const bool other_less = ok < key || (ok == key && op < pay);
            const bool up = (lane & k) == 0u || k == width;
            const bool lower = (lane & j) == 0u;
            const bool take = (lower == up) ? other_less : !other_less;
            if (take) { key = ok; pay = op; }
        }
    }
}

// One wave per task of 2..kSmall triangles: the whole subtree by the exact
// SAH over centroid-sorted orders, lane i holding the triangle at position
// begin + i; pending ranges are a stack held one entry per lane.
__global__ __launch_bounds__(256) void k_small_tasks(const SmallTask* __restrict__ small, uint32_t nsmall, uint32_t n,
                                                     const float4* __restrict__ plo, const float4* __restrict__ phi,
                                                     const uint32_t* __restrict__ ref0,
                                                     const uint32_t* __restrict__ ref1, BNode* __restrict__ nodes,
                                                     BuildCtl* ctl) {
    const uint32_t ti = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (ti >= nsmall) return;   // whole waves only; no block barrier below
    const uint32_t lane = __lane_id();
    const SmallTask T = small[ti];
    const uint32_t* src = (T.meta >> 1) ? ref1 : ref0;
    uint32_t id = kNone;
    float4 lo = make_float4(INFINITY, INFINITY, INFINITY, 0.0f), hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f);
    if (lane < T.count) {
        id = src[T.begin + lane];
        lo = plo[id];
        hi = phi[id];
    }
    // stack entry k lives in lane k: (r0, size, parent, side)
    uint32_t s_r0 = 0, s_sz = 0, s_par = 0, s_side = 0;
    if (lane == 0) { s_r0 = 0; s_sz = T.count; s_par = T.parent; s_side = T.meta & 1u; }
    int sp = 1;
    while (sp > 0) {
        --sp;
        const uint32_t r0 = __shfl(s_r0, sp), sz = __shfl(s_sz, sp), par = __shfl(s_par, sp), side = __shfl(s_side, sp);
        const bool in = lane >= r0 && lane < r0 + sz;
        // the sort, scans and reductions below run over `width` lanes only: a tree of 64
        // triangles has 63 ranges, half of them of 2 (width 64 for all of them: 2.1 ms for
        // 327,686 triangles, now 0.94 ms)
        const uint32_t width = sz <= 2u ? 2u : 1u << (32 - __builtin_clz(sz - 1u));
        float box[6];   // the node's box, from the first axis's scan
        double best = INFINITY;
        uint32_t best_k = 0, best_perm = min(r0 + lane, 63u);
        for (int a = 0; a < 3; ++a) {
            const float la = a == 0 ? lo.x : a == 1 ? lo.y : lo.z, ha = a == 0 ? hi.x : a == 1 ? hi.y : hi.z;
            // lane k < sz starts with the range's k-th triangle, in lane r0 + k
            const uint32_t from0 = min(r0 + lane, 63u);
            // (+ 0: both zeros have one key)
            uint32_t key = ord_key(__shfl(0.5f * la + 0.5f * ha, (int)from0) + 0.0f);
            if (lane >= sz) key = 0xFFFFFFFFu;
            uint32_t pay = from0;
            if (lane >= sz) pay = 64u + lane;   // after every triangle, whatever its key
            wave_sort(key, pay, lane, width);
            if (lane >= sz) pay = lane;
            // lane k (< sz) now holds the k-th range triangle in centroid order
            float l3[3] = {__shfl(lo.x, (int)pay), __shfl(lo.y, (int)pay), __shfl(lo.z, (int)pay)};
            float h3[3] = {__shfl(hi.x, (int)pay), __shfl(hi.y, (int)pay), __shfl(hi.z, (int)pay)};
            const bool mine = lane < sz;
            float pl[3], ph[3], ql[3], qh[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                pl[q] = ql[q] = mine ? l3[q] : INFINITY;
                ph[q] = qh[q] = mine ? h3[q] : -INFINITY;
            }
            for (int d = 1; d < (int)width; d <<= 1) {
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const float ul = __shfl_up(pl[q], d), uh = __shfl_up(ph[q], d);
                    const float dl = __shfl_down(ql[q], d), dh = __shfl_down(qh[q], d);
                    if (lane >= (uint32_t)d) { pl[q] = fminf(pl[q], ul); ph[q] = fmaxf(ph[q], uh); }
                    if (lane + (uint32_t)d < width) { ql[q] = fminf(ql[q], dl); qh[q] = fmaxf(qh[q], dh); }
                }
            }
            if (a == 0) {
#pragma unroll
                for (int q = 0; q < 3; ++q) { box[q] = __shfl(ql[q], 0); box[3 + q] = __shfl(qh[q], 0); }
            }
            float rl[3], rh[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) { rl[q] = __shfl_down(ql[q], 1); rh[q] = __shfl_down(qh[q], 1); }
            // split after sorted position `lane`: left = 0..lane, right = lane+1..sz-1
            double cost = INFINITY;
            if (lane + 1u < sz)
                cost = (double)half_area(pl[0], pl[1], pl[2], ph[0], ph[1], ph[2]) * (double)(lane + 1u) +
                       (double)half_area(rl[0], rl[1], rl[2], rh[0], rh[1], rh[2]) * (double)(sz - lane - 1u);
            uint32_t k = lane;
            for (int o = (int)width >> 1; o > 0; o >>= 1) {
                const double oc = __shfl_xor(cost, o);
                const uint32_t okk = __shfl_xor(k, o);
                if (oc < cost || (oc == cost && okk < k)) { cost = oc; k = okk; }
            }
            cost = __shfl(cost, 0);   // lanes 0..width-1 agree; the others follow
            k = __shfl(k, 0);
            if (cost < best) {   // ties keep the lower axis
                best = cost;
                best_k = k;
                best_perm = pay;
            }
        }
        // reorder the range: position r0 + k takes the k-th triangle of the best
        // order (best_perm holds the lane it came from); every lane takes part
        // in each shuffle, so no source lane is inactive
        const uint32_t sel = __shfl(best_perm, (int)(in ? lane - r0 : lane));
        const uint32_t from = in ? sel : lane;
        const uint32_t nid = __shfl(id, (int)from);
        const float4 nlo = make_float4(__shfl(lo.x, (int)from), __shfl(lo.y, (int)from), __shfl(lo.z, (int)from), 0.0f);
        const float4 nhi = make_float4(__shfl(hi.x, (int)from), __shfl(hi.y, (int)from), __shfl(hi.z, (int)from), 0.0f);
        id = nid;
        lo = nlo;
        hi = nhi;
        // no split has a finite cost (a box area overflows or is not a number): halve by
        // position, as the larger tasks do; one triangle at a time would nest 63 deep
        if (!(best < (double)INFINITY)) best_k = sz / 2u - 1u;
        const uint32_t nl = best_k + 1u, nr = sz - nl;
        const uint32_t node = n + T.begin + r0 + nl - 1u;
        if (nl == 1u && lane == r0) write_leaf(nodes, T.begin + r0, id, lo, hi);
        if (nr == 1u && lane == r0 + nl) write_leaf(nodes, T.begin + r0 + nl, id, lo, hi);
        if (lane == 0) {
            BNode b;
            b.left = nl == 1u ? T.begin + r0 : kNone;
            b.right = nr == 1u ? T.begin + r0 + nl : kNone;
            b.count = sz;
            b.tri = kNone;
            b.lo[0] = box[0]; b.lo[1] = box[1]; b.lo[2] = box[2];
            b.hi[0] = box[3]; b.hi[1] = box[4]; b.hi[2] = box[5];
            nodes[node] = b;
            set_child(nodes, par, side, node, ctl);
        }
        // push right, then left (the left range is split next)
        if (nr >= 2u) {
            if (lane == (uint32_t)sp) { s_r0 = r0 + nl; s_sz = nr; s_par = node; s_side = 1u; }
            ++sp;
        }
        if (nl >= 2u) {
            if (lane == (uint32_t)sp) { s_r0 = r0; s_sz = nl; s_par = node; s_side = 0u; }
            ++sp;
        }
    }
}

// ---- collapse to BVH8 ---------------------------------------------------------
struct Item {
    uint32_t bnode, out;
};

__device__ __forceinline__ float area_f(const BNode& b) {
    const float dx = b.hi[0] - b.lo[0], dy = b.hi[1] - b.lo[1], dz = b.hi[2] - b.lo[2];
    return dx * dy + dy * dz + dz * dx;
}

// SAH-optimal collapse (Ylitie, Karras and Laine, "Efficient incoherent ray
// traversal on GPUs through compressed wide BVHs", HPG 2017): for every
// binary node, C[i-1] is the least surface-area cost of its subtree spread
// over i child slots of a BVH8 node (i = 1..8), computed bottom-up:
//   C(x, 1) = min(leaf: A x kCollapseTriCost x count (count <= kLeafMax),
//                 node: A x kCollapseNodeCost + D(x, 8))
//   C(x, i) = min(C(x, i - 1), D(x, i)),  D(x, i) = min_k C(l, k) + C(r, i - k).
// k[i-1] keeps the left child's slots of D(x, i) when that is the minimum
// (0: C(x, i) = C(x, i - 1)); split8 is the argmin of D(x, 8), the 8 slots of
// x's own BVH8 node. A triangle (id < n) is a leaf of cost A x kCollapseTriCost.
struct DpRec {
    float c[8];
    uint8_t k[8];
    uint8_t leaf, split8, pad0, pad1;
};

__device__ __forceinline__ float dp_cost(const BNode* nodes, const DpRec* dp, uint32_t n, uint32_t id, int slots) {
    return id < n ? area_f(nodes[id]) * kCollapseTriCost : dp[id - n].c[slots - 1];
}

// Parent of every binary node (the root's stays kNone) and cleared arrival counters.
__global__ void k_parents(const BNode* __restrict__ nodes, uint32_t n, uint32_t* __restrict__ parent,
                          uint32_t* __restrict__ arrive) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1u) return;
    const uint32_t x = n + i;
    parent[nodes[x].left] = x;
    parent[nodes[x].right] = x;
    arrive[i] = 0u;
}

// The record of a node from its children's costs for 1..8 slots.
__device__ __forceinline__ DpRec dp_node(const BNode& b, const float (&cl)[8], const float (&cr)[8]) {
    DpRec r;
    float dist[8];
    uint8_t dk[8];
    dist[0] = INFINITY;
    dk[0] = 0;
#pragma unroll
    for (int j = 2; j <= 8; ++j) {
        float best = INFINITY;
        int bk = 1;
#pragma unroll
        for (int k = 1; k < j; ++k) {
            const float v = cl[k - 1] + cr[j - k - 1];
            if (v < best) { best = v; bk = k; }
        }
        dist[j - 1] = best;
        dk[j - 1] = (uint8_t)bk;
    }
    const float A = area_f(b);
    const float cint = A * kCollapseNodeCost + dist[7];
    const float cleaf = b.count <= kLeafMax ? A * kCollapseTriCost * (float)b.count : INFINITY;
    r.leaf = b.count <= kLeafMax && cleaf <= cint ? 1 : 0;   // cint, too, is infinite where an area overflows
    r.split8 = dk[7];
    r.pad0 = r.pad1 = 0;
    r.c[0] = fminf(cleaf, cint);
    r.k[0] = 0;
#pragma unroll
    for (int j = 2; j <= 8; ++j) {
        if (dist[j - 1] < r.c[j - 2]) { r.c[j - 1] = dist[j - 1]; r.k[j - 1] = dk[j - 1]; }
        else { r.c[j - 1] = r.c[j - 2]; r.k[j - 1] = 0; }
    }
    return r;
}

// The records of one small task's subtree by one wave: its internal nodes are
// the ids n + begin .. n + begin + count - 2, one per lane; a lane computes its
// node once both children are done (at most 63 rounds: the subtree's height).
// Costs pass through LDS, so the bottom of the tree (98% of its nodes) needs no
// device-scope fence: climbing from every triangle took 1,950 us for 327,686
// triangles, this takes 20 us and the climb above 78 us.
__global__ __launch_bounds__(256) void k_collapse_dp_small(const SmallTask* __restrict__ small, uint32_t nsmall,
                                                           uint32_t n, const BNode* __restrict__ nodes, DpRec* dp) {
    __shared__ float s_c[4][64][9];   // 9: odd stride
    const uint32_t ti = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (ti >= nsmall) return;   // whole waves only; no block barrier below
    const uint32_t lane = __lane_id();
    float (*c)[9] = s_c[threadIdx.x >> 6];
    const uint32_t first = n + small[ti].begin, inner_n = small[ti].count - 1u;
    const bool mine = lane < inner_n;
    BNode b;
    float cl[8], cr[8];
    bool ll = false, rl = false;   // the child is a triangle
    uint32_t li = 0, ri = 0;
    if (mine) {
        b = nodes[first + lane];
        ll = b.left < n;
        rl = b.right < n;
        li = (b.left - first) & 63u;
        ri = (b.right - first) & 63u;
        const float al = ll ? area_f(nodes[b.left]) * kCollapseTriCost : 0.0f;
        const float ar = rl ? area_f(nodes[b.right]) * kCollapseTriCost : 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) { cl[j] = al; cr[j] = ar; }
    }
    uint64_t done = 0ull;
    for (int round = 0; round < 64; ++round) {
        const bool ready = mine && !(done >> lane & 1ull) && (ll || (done >> li & 1ull)) && (rl || (done >> ri & 1ull));
        const uint64_t now = __ballot(ready);
        if (now == 0ull) break;
        if (ready) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (!ll) cl[j] = c[li][j];
                if (!rl) cr[j] = c[ri][j];
            }
            const DpRec r = dp_node(b, cl, cr);
            dp[first + lane - n] = r;
#pragma unroll
            for (int j = 0; j < 8; ++j) c[lane][j] = r.c[j];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the costs before the next round's reads
        done |= now;
    }
}

// The nodes above the small tasks: one thread per small task and one per
// triangle walk up from a small task's root or a triangle whose parent is such
// a node; the second thread to reach a node (both children done) computes its
// record and goes on, the first stops. The fences publish a record before its
// arrival is counted and order the sibling's record before it is read (device
// scope: the XCDs' L2s).
__global__ void k_collapse_dp(const BNode* __restrict__ nodes, uint32_t n, const SmallTask* __restrict__ small,
                              uint32_t nsmall, const uint32_t* __restrict__ parent, uint32_t* __restrict__ arrive,
                              DpRec* dp) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n + nsmall) return;
    uint32_t x = t < n ? parent[t] : small[t - n].parent;
    if (t < n && x != kNone && nodes[x].count <= kSmall) return;   // inside a small task
    while (x != kNone) {
        __threadfence();
        if (atomicAdd(&arrive[x - n], 1u) == 0u) return;
        __threadfence();
        const BNode& b = nodes[x];
        float cl[8], cr[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            cl[j] = dp_cost(nodes, dp, n, b.left, j + 1);
            cr[j] = dp_cost(nodes, dp, n, b.right, j + 1);
        }
        dp[x - n] = dp_node(b, cl, cr);
        x = parent[x];
    }
}

// Whether binary node x becomes a BVH8 node (else a leaf slot).
__device__ __forceinline__ bool inner(const DpRec* dp, uint32_t n, uint32_t x) {
    return x >= n && dp[x - n].leaf == 0;
}

// Children of one BVH8 node in slot order (kNone = empty slot): the 8-slot
// distribution of binary node bn, expanded.
__device__ void collapse_children(const BNode* nodes, const DpRec* dp, uint32_t n, uint32_t bn, uint32_t* slot_child) {
    uint32_t ch[8];
    int nc = 0;
    const BNode& b = nodes[bn];
    if (!inner(dp, n, bn)) {
        ch[nc++] = bn;   // a leaf root
    } else {
        uint32_t sx[8];
        int sj[8], sp = 0;
        const int k8 = dp[bn - n].split8;
        sx[sp] = b.right; sj[sp++] = 8 - k8;
        sx[sp] = b.left; sj[sp++] = k8;
        while (sp > 0) {
            const uint32_t m = sx[--sp];
            int j = sj[sp];
            if (m < n) j = 1;
            while (j > 1 && dp[m - n].k[j - 1] == 0) j--;
            if (j == 1) { ch[nc++] = m; continue; }
            const int k = dp[m - n].k[j - 1];
            const BNode& o = nodes[m];
            sx[sp] = o.right; sj[sp++] = j - k;
            sx[sp] = o.left; sj[sp++] = k;
        }
    }
    // octant slots: greedy on the signed centroid offsets from the node centre
    float pc[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) pc[a] = 0.5f * (b.lo[a] + b.hi[a]);
    // cost(c, s) = the child's centroid offset along slot s's signs, recomputed at
    // each step: a table of 64 would be scratch memory
    float d[8][3];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
#pragma unroll
        for (int a = 0; a < 3; ++a) d[c][a] = c < nc ? 0.5f * (nodes[ch[c]].lo[a] + nodes[ch[c]].hi[a]) - pc[a] : 0.0f;
    }
    for (int s = 0; s < 8; ++s) slot_child[s] = kNone;
    uint32_t cused = nc < 8 ? 0xFFu << nc : 0u, sused = 0;   // children that are not there count as placed
    for (int it = 0; it < nc; ++it) {
        int bc = -1, bs = -1;
        float bv = -INFINITY;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            if (cused >> c & 1u) continue;
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const float v = ((s & 1) ? d[c][0] : -d[c][0]) + ((s & 2) ? d[c][1] : -d[c][1]) +
                                ((s & 4) ? d[c][2] : -d[c][2]);
                if (!(sused >> s & 1u) && (bc < 0 || v > bv)) { bv = v; bc = c; bs = s; }
            }
        }
        cused |= 1u << bc;
        sused |= 1u << bs;
        slot_child[bs] = ch[bc];
    }
}

__global__ void k_collapse_count(const BNode* __restrict__ nodes, const DpRec* __restrict__ dp, uint32_t n,
                                 const Item* __restrict__ items, uint32_t nitems,
                                 uint32_t* __restrict__ kids, uint32_t* __restrict__ n_int, uint32_t* __restrict__ n_tri) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nitems) return;
    uint32_t sc[8];
    collapse_children(nodes, dp, n, items[i].bnode, sc);
    uint32_t ni = 0, nt = 0;
    for (int s = 0; s < 8; ++s) {
        kids[8 * i + s] = sc[s];
        if (sc[s] == kNone) continue;
        if (inner(dp, n, sc[s])) ni++;
        else nt += nodes[sc[s]].count;
    }
    n_int[i] = ni;
    n_tri[i] = nt;
}

__global__ void k_collapse_write(const BNode* __restrict__ nodes, const DpRec* __restrict__ dp, uint32_t n,
                                 const Item* __restrict__ items, uint32_t nitems,
                                 const uint32_t* __restrict__ kids, const uint32_t* __restrict__ scan_int,
                                 const uint32_t* __restrict__ scan_tri, uint32_t node_base, uint32_t tri_base0,
                                 const float* __restrict__ wtri,
                                 Bvh8Node* __restrict__ out, float4* __restrict__ out_tris, Item* __restrict__ next) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nitems) return;
    Bvh8Node nd;
    const uint32_t child_base = node_base + scan_int[i];
    const uint32_t tri_base = tri_base0 + scan_tri[i];
    uint32_t rank = 0, toff = 0, imask = 0, lmask = 0;
    uint8_t meta[8];
    for (int s = 0; s < 8; ++s) {
        const uint32_t c = kids[8 * i + s];
        if (c == kNone) {
            nd.lo_x[s] = nd.lo_y[s] = nd.lo_z[s] = 0.0f;
            nd.hi_x[s] = nd.hi_y[s] = nd.hi_z[s] = 0.0f;
            meta[s] = 0;
            continue;
        }
        const BNode& x = nodes[c];
        nd.lo_x[s] = nextafterf(x.lo[0], -INFINITY);
        nd.lo_y[s] = nextafterf(x.lo[1], -INFINITY);
        nd.lo_z[s] = nextafterf(x.lo[2], -INFINITY);
        nd.hi_x[s] = nextafterf(x.hi[0], INFINITY);
        nd.hi_y[s] = nextafterf(x.hi[1], INFINITY);
        nd.hi_z[s] = nextafterf(x.hi[2], INFINITY);
        if (inner(dp, n, c)) {
            meta[s] = (uint8_t)(0x80u | rank);
            next[scan_int[i] + rank] = Item{c, child_base + rank};
            imask |= 1u << s;
            rank++;
        } else {
            meta[s] = (uint8_t)((x.count << 5) | toff);
            // the subtree's triangles, left first (at most kLeafMax leaves, depth <= kLeafMax - 1)
            uint32_t stk[kLeafMax + 1];
            int sp = 0;
            stk[sp++] = c;
            uint32_t j = 0;
            while (sp > 0) {
                const BNode& y = nodes[stk[--sp]];
                if (y.left != kNone) {
                    stk[sp++] = y.right;
                    stk[sp++] = y.left;
                    continue;
                }
                const uint32_t t = y.tri;
                const float* w = wtri + 9ull * t;
                float4* o = out_tris + 3ull * (tri_base + toff + j);
                o[0] = make_float4(w[0], w[1], w[2], __uint_as_float(t));
                o[1] = make_float4(w[3], w[4], w[5], 0.0f);
                o[2] = make_float4(w[6], w[7], w[8], 0.0f);
                j++;
            }
            lmask |= 1u << s;
            toff += x.count;
        }
    }
    nd.child_base = (rank ? child_base : 0u) | (imask << 24);
    nd.tri_base = tri_base | (lmask << 24);
    for (int s = 0; s < 8; ++s) nd.meta[s] = meta[s];
    for (int k = 0; k < 12; ++k) nd.pad[k] = 0u;
    out[items[i].out] = nd;
}

// One device allocation for every buffer of a build: a hipMalloc and a hipFree
// for each of the ~30 of them took 2.2 of a 327,686-triangle build's 14 ms.
// take() is called in the same order twice, first with no base to add up the
// bytes.
struct Carver {
    char* base = nullptr;
    size_t bytes = 0;
    template <typename T>
    void take(T*& p, size_t n) {
        p = reinterpret_cast<T*>(base + bytes);
        bytes += ((n ? n : 1) * sizeof(T) + 255) & ~(size_t)255;
    }
};

inline uint32_t blocks(uint64_t n, uint32_t b = 256) { return (uint32_t)((n + b - 1) / b); }

// ---- exclusive scan of uint32 (node and triangle offsets of the collapse) ------
constexpr uint32_t kScanBlock = 1024;   // 256 threads x 4 elements

__global__ __launch_bounds__(256) void k_scan_blocks(const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
                                                     uint32_t n, uint32_t* __restrict__ sums) {
    __shared__ uint32_t s_w[4];
    const uint32_t lane = __lane_id(), w = threadIdx.x >> 6;
    const uint64_t base = (uint64_t)blockIdx.x * kScanBlock + 4ull * threadIdx.x;
    uint32_t v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = base + q < n ? in[base + q] : 0u;
    const uint32_t t0 = v[0], t1 = t0 + v[1], t2 = t1 + v[2], t3 = t2 + v[3];
    uint32_t x = t3;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(x, d);
        if (lane >= (uint32_t)d) x += y;
    }
    if (lane == 63u) s_w[w] = x;
    __syncthreads();
    uint32_t woff = 0, total = 0;
    for (uint32_t q = 0; q < 4u; ++q) {
        if (q < w) woff += s_w[q];
        total += s_w[q];
    }
    const uint32_t ex = woff + x - t3;
    const uint32_t r[4] = {ex, ex + t0, ex + t1, ex + t2};
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (base + q < n) out[base + q] = r[q];
    if (threadIdx.x == 0 && sums) sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(256) void k_scan_add(uint32_t* __restrict__ out, uint32_t n,
                                                  const uint32_t* __restrict__ offs) {
    const uint64_t base = (uint64_t)blockIdx.x * kScanBlock + 4ull * threadIdx.x;
    const uint32_t o = offs[blockIdx.x];
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (base + q < n) out[base + q] += o;
}

// Exclusive scans of two arrays of n by one block.
constexpr uint32_t kScanSmall = 16384;   // one block: 16 steps; more items take the multi-block scans
__global__ __launch_bounds__(1024) void k_scan_pair(const uint32_t* __restrict__ in0, const uint32_t* __restrict__ in1,
                                                    uint32_t* __restrict__ out0, uint32_t* __restrict__ out1, uint32_t n,
                                                    uint32_t* __restrict__ totals) {
    __shared__ uint32_t s_w[2][16];
    const uint32_t lane = __lane_id(), w = threadIdx.x >> 6;
    uint32_t carry0 = 0, carry1 = 0;
    for (uint32_t base = 0; base < n; base += 1024u) {
        const uint32_t i = base + threadIdx.x;
        const uint32_t v0 = i < n ? in0[i] : 0u, v1 = i < n ? in1[i] : 0u;
        uint32_t x0 = v0, x1 = v1;
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y0 = __shfl_up(x0, d), y1 = __shfl_up(x1, d);
            if (lane >= (uint32_t)d) { x0 += y0; x1 += y1; }
        }
        if (lane == 63u) { s_w[0][w] = x0; s_w[1][w] = x1; }
        __syncthreads();
        uint32_t o0 = carry0, o1 = carry1;
        for (uint32_t q = 0; q < 16u; ++q) {
            if (q < w) { o0 += s_w[0][q]; o1 += s_w[1][q]; }
            carry0 += s_w[0][q];
            carry1 += s_w[1][q];
        }
        if (i < n) { out0[i] = o0 + x0 - v0; out1[i] = o1 + x1 - v1; }
        __syncthreads();
    }
    if (threadIdx.x == 0) { totals[0] = carry0; totals[1] = carry1; }
}

// Scratch for the per-block sums of every recursion level (2^32 elements
// need at most 4 levels of 1024-element blocks).
struct ScanTmp {
    static constexpr int kLevels = 4;
    uint32_t* lv[2 * kLevels] = {};
    void carve(Carver& a, uint32_t n) {
        size_t k = 0;
        for (uint32_t m = n; m > kScanBlock; m = (m + kScanBlock - 1) / kScanBlock, ++k) {
            const uint32_t nb = (m + kScanBlock - 1) / kScanBlock;
            a.take(lv[2 * k], nb);
            a.take(lv[2 * k + 1], nb);
        }
    }
};

// out[i] = in[0] + ... + in[i - 1]; tmp must have been carved for n or more.
hipError_t scan_u32(const uint32_t* in, uint32_t* out, uint32_t n, ScanTmp& tmp, size_t level, hipStream_t st) {
    if (n == 0) return hipSuccess;
    const uint32_t nb = (n + kScanBlock - 1) / kScanBlock;
    if (nb == 1) {
        hipLaunchKernelGGL(k_scan_blocks, dim3(1), dim3(256), 0, st, in, out, n, nullptr);
        return hipGetLastError();
    }
    uint32_t* sums = tmp.lv[2 * level];
    uint32_t* offs = tmp.lv[2 * level + 1];
    hipLaunchKernelGGL(k_scan_blocks, dim3(nb), dim3(256), 0, st, in, out, n, sums);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    e = scan_u32(sums, offs, nb, tmp, level + 1, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_scan_add, dim3(nb), dim3(256), 0, st, out, n, offs);
    return hipGetLastError();
}

// Terms of bvh8_sah_cost, the sum over the nodes in FP64: each block's part in
// part[block], the root's area in part[gridDim.x]. The blocks' parts are added
// in order on the host, so the result does not depend on the schedule. 13 us
// for 65,000 nodes (16 MB); bringing them to the host for it took 2.5 ms.
__device__ __forceinline__ double area6(double lx, double ly, double lz, double hx, double hy, double hz) {
    const double dx = hx - lx, dy = hy - ly, dz = hz - lz;
    return 2.0 * (dx * dy + dy * dz + dz * dx);
}

constexpr uint32_t kSahBlocks = 256;

__global__ __launch_bounds__(256) void k_sah(const Bvh8Node* __restrict__ nodes, uint32_t n, double* __restrict__ part) {
    __shared__ double s_p[256];
    double rl[3] = {INFINITY, INFINITY, INFINITY}, rh[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int k = 0; k < 8; ++k) {
        if (!nodes[0].meta[k]) continue;
        const double l[3] = {nodes[0].lo_x[k], nodes[0].lo_y[k], nodes[0].lo_z[k]};
        const double h[3] = {nodes[0].hi_x[k], nodes[0].hi_y[k], nodes[0].hi_z[k]};
        for (int a = 0; a < 3; ++a) { rl[a] = l[a] < rl[a] ? l[a] : rl[a]; rh[a] = rh[a] < h[a] ? h[a] : rh[a]; }
    }
    const double ra = area6(rl[0], rl[1], rl[2], rh[0], rh[1], rh[2]);
    double sum = 0.0;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) {
        const Bvh8Node& nd = nodes[i];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const uint8_t m = nd.meta[k];
            if (!m) continue;
            const double a = area6(nd.lo_x[k], nd.lo_y[k], nd.lo_z[k], nd.hi_x[k], nd.hi_y[k], nd.hi_z[k]) / ra;
            sum += (m & 0x80) ? a : a * ((m >> 5) & 3);
        }
    }
    s_p[threadIdx.x] = sum;
    for (uint32_t d = 128; d > 0; d /= 2) {
        __syncthreads();
        if (threadIdx.x < d) s_p[threadIdx.x] += s_p[threadIdx.x + d];
    }
    if (threadIdx.x == 0) {
        part[blockIdx.x] = s_p[0];
        if (blockIdx.x == 0) part[gridDim.x] = ra;
    }
}

struct BuildBufs {
    float* w;
    float4 *plo, *phi;
    uint32_t *ref0, *ref1;
    SceneBounds* sb;
    BuildCtl* ctl;
    BNode* nodes;
    Task *t0, *t1, *b0, *b1;
    BigState *s0, *s1;
    uint32_t *ct0, *ct1, *cl;
    SmallTask* small;
    uint32_t *parent, *arrive;
    DpRec* dp;
    Bvh8Node* out;
    float4* otri;
    Item *it0, *it1;
    uint32_t *ck, *ni, *nt, *si, *stri, *tot;
    double* sah;
    ScanTmp scan;
    // sizes of the task lists and of the tree
    uint32_t cap_large, cap_small, cap_big, cap_chunks, out_cap;

    void carve(Carver& a, uint32_t n) {
        cap_large = n / (kSmall + 1) + 2;
        cap_small = n / 2 + 2;
        cap_big = n / (kBig + 1) + 2;
        cap_chunks = n / kChunk + cap_big + 2;
        out_cap = std::max(1u, n - 1) + 1;
        a.take(w, 9ull * n);
        a.take(plo, n); a.take(phi, n); a.take(ref0, n); a.take(ref1, n);
        a.take(sb, 1); a.take(ctl, 1); a.take(nodes, 2ull * n);
        a.take(t0, cap_large); a.take(t1, cap_large); a.take(small, cap_small);
        a.take(b0, cap_big); a.take(b1, cap_big); a.take(s0, cap_big); a.take(s1, cap_big);
        a.take(ct0, cap_chunks); a.take(ct1, cap_chunks); a.take(cl, cap_chunks);
        a.take(parent, 2ull * n); a.take(arrive, n); a.take(dp, n);
        a.take(out, out_cap); a.take(otri, 3ull * n);
        a.take(it0, out_cap); a.take(it1, out_cap);
        a.take(ck, 8ull * out_cap); a.take(ni, out_cap + 1); a.take(nt, out_cap + 1);
        a.take(si, out_cap + 1); a.take(stri, out_cap + 1); a.take(tot, 2);
        a.take(sah, kSahBlocks + 1);
        scan.carve(a, out_cap + 1);
    }
};

}  // namespace

#define D_TRY(expr)                                                               \
    do {                                                                          \
        hipError_t e_ = (expr);                                                   \
        if (e_ != hipSuccess) {                                                   \
            err = std::string(#expr) + ": " + hipGetErrorString(e_);              \
            return false;                                                         \
        }                                                                         \
    } while (0)

hipError_t launch_triangle_ids(const DeviceMesh& m, hipStream_t st) {
    if (m.num_tris == 0) return hipSuccess;
    hipLaunchKernelGGL(k_flatten, dim3(blocks(m.num_tris)), dim3(256), 0, st, m.inst, m.num_inst, m.vertices, m.indices,
                       m.num_tris, (float*)nullptr, m.tri_inst, m.tri_prim, (SceneBounds*)nullptr);
    return hipGetLastError();
}

DeviceBvh::~DeviceBvh() {
    if (scratch) (void)hipFree(scratch);
}

bool build_bvh8_device(const DeviceMesh& mesh, const std::function<void(std::vector<float>&)>& flatten, DeviceBvh& out,
                       std::string& err) {
    const uint32_t n = mesh.num_tris;
    if (n >= (1u << 24)) {
        err = "more than 2^24 triangles";
        return false;
    }
    hipStream_t st = nullptr;
    D_TRY(hipStreamCreate(&st));
    struct StreamGuard { hipStream_t s; ~StreamGuard() { (void)hipStreamDestroy(s); } } sg{st};
    if (n == 0) {   // one empty root node, as the host builder
        Bvh8Node empty;
        std::memset(&empty, 0, sizeof empty);
        D_TRY(hipMalloc(&out.scratch, sizeof empty));
        D_TRY(hipMemcpy(out.scratch, &empty, sizeof empty, hipMemcpyHostToDevice));
        out.nodes = (const Bvh8Node*)out.scratch;
        out.num_nodes = out.max_depth = 1;
        return true;
    }
    BuildBufs B;
    Carver carver;
    B.carve(carver, n);
    D_TRY(hipMalloc(&out.scratch, carver.bytes));
    carver = Carver{(char*)out.scratch, 0};
    B.carve(carver, n);
    SceneBounds sb;
    for (int pass = 0;; ++pass) {
        for (int a = 0; a < 3; ++a) {
            sb.b.lo[a] = sb.c.lo[a] = 0xFFFFFFFFu;
            sb.b.hi[a] = sb.c.hi[a] = 0u;
        }
        sb.nonfinite = 0;
        D_TRY(hipMemcpyAsync(B.sb, &sb, sizeof sb, hipMemcpyHostToDevice, st));
        if (pass == 0) {
            BuildCtl c{0u, 0u, 0u, 0u, 0u, kNone};
            D_TRY(hipMemcpyAsync(B.ctl, &c, sizeof c, hipMemcpyHostToDevice, st));
            hipLaunchKernelGGL(k_flatten, dim3(blocks(n)), dim3(256), 0, st, mesh.inst, mesh.num_inst, mesh.vertices,
                               mesh.indices, n, B.w, mesh.tri_inst, mesh.tri_prim, B.sb);
            D_TRY(hipGetLastError());
        }
        hipLaunchKernelGGL(k_prep, dim3(std::min(blocks(n), kPrepBlocks)), dim3(256), 0, st, B.w, n, B.plo, B.phi, B.ref0, B.sb);
        D_TRY(hipGetLastError());
        D_TRY(hipMemcpyAsync(&sb, B.sb, sizeof sb, hipMemcpyDeviceToHost, st));
        D_TRY(hipStreamSynchronize(st));
        if (!sb.nonfinite) break;
        // sign and payload of a NaN differ between the device's and the host's
        // arithmetic and take part in the bounds' keys: such a scene keeps the
        // host's coordinates
        std::vector<float> w;
        flatten(w);
        D_TRY(hipMemcpy(B.w, w.data(), 36ull * n, hipMemcpyHostToDevice));
    }
    auto unkey = [](uint32_t k) {
        const uint32_t u = (k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k;
        float f;
        std::memcpy(&f, &u, 4);
        return f;
    };
    // binary build: levels of large tasks, then every small task
    uint32_t root = kNone;
    uint32_t n_small = 0;
    if (n == 1) {
        root = 0;   // a single triangle: the root is its leaf
        float4 lo = make_float4(unkey(sb.b.lo[0]), unkey(sb.b.lo[1]), unkey(sb.b.lo[2]), 0.0f);
        float4 hi = make_float4(unkey(sb.b.hi[0]), unkey(sb.b.hi[1]), unkey(sb.b.hi[2]), 0.0f);
        BNode b;
        b.left = b.right = kNone;
        b.count = 1;
        b.tri = 0;
        b.lo[0] = lo.x; b.lo[1] = lo.y; b.lo[2] = lo.z;
        b.hi[0] = hi.x; b.hi[1] = hi.y; b.hi[2] = hi.z;
        D_TRY(hipMemcpyAsync(B.nodes, &b, sizeof b, hipMemcpyHostToDevice, st));
    } else if (n <= kSmall) {
        SmallTask t{0u, n, kNone, 0u};
        D_TRY(hipMemcpyAsync(B.small, &t, sizeof t, hipMemcpyHostToDevice, st));
        n_small = 1;
    } else {
        Task t;
        t.begin = 0; t.count = n; t.parent = kNone; t.side = 0; t.buf = 0;
        t.chunk0 = t.pad = 0;
        t.nchunks = (n + kChunk - 1) / kChunk;
        for (int a = 0; a < 3; ++a) {
            t.lo[a] = unkey(sb.b.lo[a]); t.hi[a] = unkey(sb.b.hi[a]);
            t.clo[a] = unkey(sb.c.lo[a]); t.chi[a] = unkey(sb.c.hi[a]);
        }
        uint32_t ntasks = n > kBig ? 0 : 1, nbig = n > kBig ? 1 : 0, nchunks = n > kBig ? t.nchunks : 0, levels = 0;
        Task *cur = B.t0, *nxt = B.t1, *bcur = B.b0, *bnxt = B.b1;
        BigState *scur = B.s0, *snxt = B.s1;
        uint32_t *ccur = B.ct0, *cnxt = B.ct1;
        D_TRY(hipMemcpyAsync(nbig ? bcur : cur, &t, sizeof t, hipMemcpyHostToDevice, st));
        if (nbig) {
            hipLaunchKernelGGL(k_big_root, dim3(1), dim3(256), 0, st, bcur, scur, ccur);
            D_TRY(hipGetLastError());
        }
        while (ntasks + nbig > 0) {
            if (++levels > n) {   // every level shrinks the largest task
                err = "device BVH build did not converge";
                return false;
            }
            D_TRY(hipMemsetAsync(&B.ctl->n_next, 0, 12, st));   // n_next, n_big, n_chunks
            if (nbig) {
                hipLaunchKernelGGL(k_big_bin, dim3(nchunks), dim3(256), 0, st, bcur, ccur, B.plo, B.phi, B.ref0,
                                   B.ref1, scur);
                D_TRY(hipGetLastError());
                hipLaunchKernelGGL(k_big_plan, dim3(nbig), dim3(256), 0, st, bcur, scur);
                D_TRY(hipGetLastError());
                hipLaunchKernelGGL(k_big_count, dim3(nchunks), dim3(256), 0, st, bcur, ccur, B.plo, B.phi, B.ref0,
                                   B.ref1, scur, B.cl);
                D_TRY(hipGetLastError());
                hipLaunchKernelGGL(k_big_partition, dim3(nchunks), dim3(256), 0, st, bcur, ccur, B.plo, B.phi,
                                   B.ref0, B.ref1, scur, B.cl, B.nodes);
                D_TRY(hipGetLastError());
                hipLaunchKernelGGL(k_big_emit, dim3(nbig), dim3(256), 0, st, bcur, scur, n, B.nodes, nxt, bnxt, snxt,
                                   cnxt, B.small, B.ctl);
                D_TRY(hipGetLastError());
            }
            if (ntasks) {
                hipLaunchKernelGGL(k_split_tasks, dim3(ntasks), dim3(256), 0, st, cur, n, B.plo, B.phi, B.ref0,
                                   B.ref1, B.nodes, nxt, B.small, B.ctl);
                D_TRY(hipGetLastError());
            }
            BuildCtl c;
            D_TRY(hipMemcpyAsync(&c, B.ctl, sizeof c, hipMemcpyDeviceToHost, st));
            D_TRY(hipStreamSynchronize(st));
            if (c.n_next > B.cap_large || c.n_small > B.cap_small || c.n_big > B.cap_big || c.n_chunks > B.cap_chunks) {
                err = "device BVH build task list overflow";
                return false;
            }
            ntasks = c.n_next;
            nbig = c.n_big;
            nchunks = c.n_chunks;
            n_small = c.n_small;
            std::swap(cur, nxt);
            std::swap(bcur, bnxt);
            std::swap(scur, snxt);
            std::swap(ccur, cnxt);
        }
    }
    if (n_small) {
        hipLaunchKernelGGL(k_small_tasks, dim3((n_small + 3) / 4), dim3(256), 0, st, B.small, n_small, n, B.plo,
                           B.phi, B.ref0, B.ref1, B.nodes, B.ctl);
        D_TRY(hipGetLastError());
    }
    if (n > 1) {
        BuildCtl c;
        D_TRY(hipMemcpyAsync(&c, B.ctl, sizeof c, hipMemcpyDeviceToHost, st));
        D_TRY(hipStreamSynchronize(st));
        root = c.root;
        if (root < n || root >= 2 * n - 1) {
            err = "device BVH build produced no root";
            return false;
        }
    }
    // collapse: the SAH-optimal slot distribution of every binary node, bottom-up
    D_TRY(hipMemsetAsync(B.parent, 0xFF, sizeof(uint32_t) * (2ull * n), st));
    if (n > 1) {
        hipLaunchKernelGGL(k_parents, dim3(blocks(n - 1)), dim3(256), 0, st, B.nodes, n, B.parent, B.arrive);
        D_TRY(hipGetLastError());
        if (n_small) {
            hipLaunchKernelGGL(k_collapse_dp_small, dim3((n_small + 3) / 4), dim3(256), 0, st, B.small, n_small, n,
                               B.nodes, B.dp);
            D_TRY(hipGetLastError());
        }
        hipLaunchKernelGGL(k_collapse_dp, dim3(blocks((uint64_t)n + n_small)), dim3(256), 0, st, B.nodes, n, B.small,
                           n_small, B.parent, B.arrive, B.dp);
        D_TRY(hipGetLastError());
    }
    {
        Item r0{root, 0};
        D_TRY(hipMemcpyAsync(B.it0, &r0, sizeof r0, hipMemcpyHostToDevice, st));
    }
    uint32_t nitems = 1, out_nodes = 1, out_tris = 0, depth = 0;
    Item* items = B.it0;
    Item* nitems_buf = B.it1;
    while (nitems > 0) {
        depth++;
        hipLaunchKernelGGL(k_collapse_count, dim3(blocks(nitems, 64)), dim3(64), 0, st, B.nodes, B.dp, n, items,
                           nitems, B.ck, B.ni, B.nt);
        D_TRY(hipGetLastError());
        uint32_t tot[2] = {0, 0};
        if (nitems <= kScanSmall) {
            hipLaunchKernelGGL(k_scan_pair, dim3(1), dim3(1024), 0, st, B.ni, B.nt, B.si, B.stri, nitems, B.tot);
            D_TRY(hipGetLastError());
            D_TRY(hipMemcpyAsync(tot, B.tot, sizeof tot, hipMemcpyDeviceToHost, st));
        } else {
            D_TRY(hipMemsetAsync(B.ni + nitems, 0, 4, st));
            D_TRY(hipMemsetAsync(B.nt + nitems, 0, 4, st));
            D_TRY(scan_u32(B.ni, B.si, nitems + 1, B.scan, 0, st));
            D_TRY(scan_u32(B.nt, B.stri, nitems + 1, B.scan, 0, st));
            D_TRY(hipMemcpyAsync(&tot[0], B.si + nitems, 4, hipMemcpyDeviceToHost, st));
            D_TRY(hipMemcpyAsync(&tot[1], B.stri + nitems, 4, hipMemcpyDeviceToHost, st));
        }
        D_TRY(hipStreamSynchronize(st));
        if (out_nodes + tot[0] > B.out_cap || out_tris + tot[1] > n) {
            err = "device BVH collapse overflow";
            return false;
        }
        hipLaunchKernelGGL(k_collapse_write, dim3(blocks(nitems, 64)), dim3(64), 0, st, B.nodes, B.dp, n, items,
                           nitems, B.ck, B.si, B.stri, out_nodes, out_tris, B.w, B.out, B.otri, nitems_buf);
        D_TRY(hipGetLastError());
        out_nodes += tot[0];
        out_tris += tot[1];
        nitems = tot[0];
        std::swap(items, nitems_buf);
    }
    if (out_tris != n) {
        err = "device BVH lost triangles";
        return false;
    }
    if (out_nodes >= (1u << 24)) {
        err = "too many BVH8 nodes for the index encoding (max 2^24)";
        return false;
    }
    const uint32_t sah_blocks = std::min(blocks(out_nodes), kSahBlocks);
    hipLaunchKernelGGL(k_sah, dim3(sah_blocks), dim3(256), 0, st, B.out, out_nodes, B.sah);
    D_TRY(hipGetLastError());
    double part[kSahBlocks + 1];
    D_TRY(hipMemcpyAsync(part, B.sah, sizeof(double) * (sah_blocks + 1), hipMemcpyDeviceToHost, st));
    D_TRY(hipStreamSynchronize(st));
    if (part[sah_blocks] > 0.0) {
        double sah = 1.0;   // the root node itself
        for (uint32_t i = 0; i < sah_blocks; ++i) sah += part[i];
        out.sah_cost = (float)sah;
    }
    out.nodes = B.out;
    out.tris = B.otri;
    out.num_nodes = out_nodes;
    out.max_depth = depth;
    return true;
}

}  // namespace rt
