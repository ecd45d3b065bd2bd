// lbvh.hip -- LBVH build and refit on MI355X.
//
// Tree semantics follow lbvh/lbvh.cu:108-385 (Morton quantization, Karras
// split with the index tie-break) and the swept leaf boxes of
// lbvh/lbvh.cu:623-731; the inner boxes are unions of the children. The
// per-level launches and host round trips of the reference are replaced by
// treelets: a node whose leaves lie in one block of 1,024 is refit in that
// block's workgroup, in LDS; the few nodes across block borders follow in one
// launch per 32-fold larger block.
#include "lbvh.hpp"
#include <algorithm>
#include "ppf_mi355x.h"
#include "sort.hpp"

namespace ppf {

namespace {

constexpr int kNT = 256;

// Treelet classes: a node of class c has its leaves in one aligned block of
// 2^class_shift(c) leaves and not in a smaller class's block. A node across a
// border of class c - 1 blocks lies on the nested chain of that border, whose
// members have distinct common-prefix lengths: at most 30 code bits, 32 scene
// bits and class_shift(c) tie bits, so the 31 borders inside a class c block
// (c >= 1) hold at most 31 x 94 = 2,914 nodes (about 320 in meshes).
constexpr uint32_t kTreelet = 1024; // leaves of a class 0 block
constexpr uint32_t kTopCap = 3072;  // nodes of one larger block
constexpr uint32_t kClassBits = 28; // rank word: class << kClassBits | place
__host__ __device__ inline uint32_t class_shift(uint32_t c) { return 10u + 5u * c; }
__host__ __device__ inline uint32_t class_blocks(uint32_t n, uint32_t c) {
    const uint32_t sh = class_shift(c);
    return sh >= 32 ? 1u : (uint32_t)(((uint64_t)n + (1ull << sh) - 1) >> sh);
}
__host__ __device__ inline uint32_t node_class(uint32_t l, uint32_t r) {
    uint32_t c = 0;
    while (class_shift(c) < 32 && (l >> class_shift(c)) != (r >> class_shift(c))) {
        ++c;
    }
    return c;
}
// Classes beyond 0 a tree of n leaves needs, and the first block of class c
// in the lists.
uint32_t top_classes(uint32_t n) {
    uint32_t c = 0;
    while (class_blocks(n, c) > 1) {
        ++c;
    }
    return c;
}
__host__ __device__ inline uint32_t class_base(uint32_t n, uint32_t c) {
    uint32_t b = 0;
    for (uint32_t k = 1; k < c; ++k) {
        b += class_blocks(n, k);
    }
    return b;
}

__device__ inline uint32_t prim_vertex(const PrimSet &p, uint32_t i, int k) {
    return p.elem ? p.elem[(size_t)i * p.arity + k] : i;
}

__device__ inline uint32_t expand_bits(uint32_t v) {
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// Centroids (lbvh.cu:120-167 term order) and per-block min/max partials (part
// null: none, a tree of many scenes has bounds of its own per scene).
__global__ __launch_bounds__(kNT) void k_centroid(PrimSet p, const float *__restrict__ x,
                                                  float *__restrict__ cent,
                                                  float *__restrict__ part) {
    __shared__ float s[6][kNT];
    const uint32_t i = blockIdx.x * kNT + threadIdx.x;
    float c[3] = {3.4e38f, 3.4e38f, 3.4e38f}, mx[3] = {-3.4e38f, -3.4e38f, -3.4e38f};
    if (i < p.n) {
        const f3 a = load3(x + 3 * (size_t)prim_vertex(p, i, 0));
        f3 m;
        if (p.arity == 3) {
            const f3 b = load3(x + 3 * (size_t)prim_vertex(p, i, 1));
            const f3 d = load3(x + 3 * (size_t)prim_vertex(p, i, 2));
            m = mk3((a.x + b.x + d.x) / 3.0f, (a.y + b.y + d.y) / 3.0f,
                    (a.z + b.z + d.z) / 3.0f);
        } else if (p.arity == 2) {
            const f3 b = load3(x + 3 * (size_t)prim_vertex(p, i, 1));
            m = mk3((a.x + b.x) / 2.0f, (a.y + b.y) / 2.0f, (a.z + b.z) / 2.0f);
        } else {
            m = a;
        }
        store3(cent + 3 * (size_t)i, m);
        c[0] = mx[0] = m.x;
        c[1] = mx[1] = m.y;
        c[2] = mx[2] = m.z;
    }
    if (!part) {
        return;
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        s[d][threadIdx.x] = c[d];
        s[3 + d][threadIdx.x] = mx[d];
    }
    __syncthreads();
    for (int w = kNT / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                s[d][threadIdx.x] = fminf(s[d][threadIdx.x], s[d][threadIdx.x + w]);
                s[3 + d][threadIdx.x] =
                    fmaxf(s[3 + d][threadIdx.x], s[3 + d][threadIdx.x + w]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) {
        part[6 * (size_t)blockIdx.x + threadIdx.x] = s[threadIdx.x][0];
    }
}

__global__ __launch_bounds__(kNT) void k_bounds(uint32_t nb, float *__restrict__ part,
                                                float *__restrict__ bounds) {
    __shared__ float s[6][kNT];
    float v[6] = {3.4e38f, 3.4e38f, 3.4e38f, -3.4e38f, -3.4e38f, -3.4e38f};
    for (uint32_t b = threadIdx.x; b < nb; b += kNT) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            v[d] = fminf(v[d], part[6 * (size_t)b + d]);
            v[3 + d] = fmaxf(v[3 + d], part[6 * (size_t)b + 3 + d]);
        }
    }
#pragma unroll
    for (int d = 0; d < 6; ++d) {
        s[d][threadIdx.x] = v[d];
    }
    __syncthreads();
    for (int w = kNT / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                s[d][threadIdx.x] = fminf(s[d][threadIdx.x], s[d][threadIdx.x + w]);
                s[3 + d][threadIdx.x] =
                    fmaxf(s[3 + d][threadIdx.x], s[3 + d][threadIdx.x + w]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) {
        bounds[threadIdx.x] = s[threadIdx.x][0];
    }
}

// 30-bit Morton codes (lbvh.cu:253-279).
__global__ __launch_bounds__(kNT) void k_morton(uint32_t n, const float *__restrict__ cent,
                                                const float *__restrict__ bounds,
                                                uint32_t *__restrict__ code,
                                                uint32_t *__restrict__ idx) {
    const uint32_t i = blockIdx.x * kNT + threadIdx.x;
    if (i >= n) {
        return;
    }
    uint32_t q[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float lo = bounds[d], hi = bounds[3 + d];
        const float sc = (hi - lo) > 1e-10f ? 1023.0f / (hi - lo) : 0.0f;
        q[d] = (uint32_t)fminf(1023.0f, fmaxf(0.0f, (cent[3 * (size_t)i + d] - lo) * sc));
    }
    code[i] = expand_bits(q[0]) | (expand_bits(q[1]) << 1) | (expand_bits(q[2]) << 2);
    idx[i] = i;
}

__device__ inline uint32_t prim_scene(const PrimSet &p, uint32_t prim) {
    return (p.vscene && p.nscene > 1) ? p.vscene[prim_vertex(p, prim, 0)] : 0u;
}

// Float <-> unsigned with the same order (negative floats reversed), so that
// integer atomics take exact float minima and maxima.
__device__ inline uint32_t ord_bits(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ inline float ord_float(uint32_t u) {
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// Per-scene centroid bounds (6 ordered words per scene: min xyz, max xyz).
// Bound by the atomics on a few words: a wave takes kSceneRun x 64 primitives
// and passes its bounds on when the scene changes (16 scenes of 64 x 64 and
// larger sheets: 83 -> 11 us a tree).
constexpr int kSceneRun = 8;
__global__ __launch_bounds__(kNT) void k_scene_bounds(PrimSet p, const float *__restrict__ cent,
                                                      uint32_t *__restrict__ sb) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t base = (blockIdx.x * (kNT / kWave) + threadIdx.x / kWave) * kSceneRun * kWave;
    uint32_t cs = 0; // the scene of lo and hi
    constexpr float kInf = __builtin_inff();
    float lo[3] = {kInf, kInf, kInf}, hi[3] = {-kInf, -kInf, -kInf};
    auto flush = [&] {
        uint32_t w = 0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            for (int o = kWave / 2; o > 0; o >>= 1) {
                lo[d] = fminf(lo[d], __shfl_xor(lo[d], o));
                hi[d] = fmaxf(hi[d], __shfl_xor(hi[d], o));
            }
            w = lane == (uint32_t)d ? ord_bits(lo[d]) : w;
            w = lane == (uint32_t)d + 3 ? ord_bits(hi[d]) : w;
            lo[d] = kInf, hi[d] = -kInf;
        }
        if (lane < 3) {
            atomicMin(sb + 6 * cs + lane, w);
        } else if (lane < 6) {
            atomicMax(sb + 6 * cs + lane, w);
        }
    };
    bool held = false; // lo and hi hold primitives
    for (int r = 0; r < kSceneRun; ++r) {
        const uint32_t i = base + r * kWave + lane;
        const bool ok = i < p.n;
        uint64_t todo = __ballot(ok);
        const uint32_t c = ok ? prim_scene(p, i) : 0u;
        float x[3] = {0.0f, 0.0f, 0.0f};
        if (ok) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                x[d] = cent[3 * (size_t)i + d];
            }
        }
        while (todo) { // one turn per scene among the wave's primitives
            const uint32_t next = __shfl(c, __ffsll((unsigned long long)todo) - 1);
            if (held && next != cs) {
                flush();
            }
            cs = next;
            held = true;
            const bool mine = ok && c == cs;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                lo[d] = mine ? fminf(lo[d], x[d]) : lo[d];
                hi[d] = mine ? fmaxf(hi[d], x[d]) : hi[d];
            }
            todo &= ~__ballot(mine);
        }
    }
    if (held) {
        flush();
    }
}

// Morton codes quantized in each primitive's own scene box.
__global__ __launch_bounds__(kNT) void k_morton_scenes(PrimSet p, const float *__restrict__ cent,
                                                       const uint32_t *__restrict__ sb,
                                                       uint32_t *__restrict__ code,
                                                       uint32_t *__restrict__ idx) {
    const uint32_t i = blockIdx.x * kNT + threadIdx.x;
    if (i >= p.n) {
        return;
    }
    const uint32_t c = prim_scene(p, i);
    uint32_t q[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float lo = ord_float(sb[6 * c + d]), hi = ord_float(sb[6 * c + 3 + d]);
        const float sc = (hi - lo) > 1e-10f ? 1023.0f / (hi - lo) : 0.0f;
        q[d] = (uint32_t)fminf(1023.0f, fmaxf(0.0f, (cent[3 * (size_t)i + d] - lo) * sc));
    }
    code[i] = expand_bits(q[0]) | (expand_bits(q[1]) << 1) | (expand_bits(q[2]) << 2);
    idx[i] = i;
}

// Empty scene boxes (min at the top of the order, max at the bottom).
__global__ void k_scene_bounds_init(uint32_t ns, uint32_t *__restrict__ sb) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < 6 * ns) {
        sb[k] = (k % 6) < 3 ? 0xffffffffu : 0u;
    }
}

// Scene of each sorted leaf (the key of the second, stable sort pass).
__global__ __launch_bounds__(kNT) void k_scene_keys(PrimSet p, const uint32_t *__restrict__ idx,
                                                    uint32_t *__restrict__ key) {
    const uint32_t i = blockIdx.x * kNT + threadIdx.x;
    if (i < p.n) {
        key[i] = prim_scene(p, idx[i]);
    }
}

// Morton codes in the final leaf order (from the per-primitive copy).
__global__ __launch_bounds__(kNT) void k_regather(uint32_t n, const uint32_t *__restrict__ idx,
                                                  const uint32_t *__restrict__ byprim,
                                                  uint32_t *__restrict__ code) {
    const uint32_t i = blockIdx.x * kNT + threadIdx.x;
    if (i < n) {
        code[i] = byprim[idx[i]];
    }
}

// Common-prefix length of the keys of sorted leaves i and j: the Morton code
// with the index as tie-break (lbvh.cu:289-303), preceded by the scene id
// when the tree holds many scenes (sk: scene per sorted leaf, or null).
__device__ inline int lcp(const uint32_t *__restrict__ k, const uint32_t *__restrict__ sk, int n,
                          int i, int j) {
    if (j < 0 || j >= n) {
        return -1;
    }
    int base = 0;
    if (sk) {
        const uint32_t sa = sk[i], sb = sk[j];
        if (sa != sb) {
            return __clz(sa ^ sb);
        }
        base = 32;
    }
    const uint32_t a = k[i], b = k[j];
    if (a == b) {
        return base + 32 + __clz((uint32_t)(i ^ j));
    }
    return base + __clz(a ^ b);
}

// Karras radix tree over the sorted codes (lbvh.cu:305-385), and the treelet
// class of every internal node. Clears the counts of the lists that follow
// (segs of them, fewer than leaves): a build may be captured into a graph.
__global__ __launch_bounds__(kNT) void k_karras(uint32_t n, const uint32_t *__restrict__ k,
                                                const uint32_t *__restrict__ sk,
                                                const uint32_t *__restrict__ idx,
                                                uint32_t *__restrict__ node,
                                                uint32_t *__restrict__ rank, uint32_t segs,
                                                uint32_t *__restrict__ count) {
    const int i = blockIdx.x * kNT + threadIdx.x;
    const int nn = (int)n;
    if ((uint32_t)i < segs) {
        count[i] = 0;
    }
    if (i < nn) {
        node[2 * (size_t)i] = idx[i] + 1;
        node[2 * (size_t)i + 1] = 0;
    }
    if (i >= nn - 1) {
        return;
    }
    const int d = lcp(k, sk, nn, i, i + 1) > lcp(k, sk, nn, i, i - 1) ? 1 : -1;
    const int lmin = lcp(k, sk, nn, i, i - d);
    int lmax = 2;
    while (lcp(k, sk, nn, i, i + lmax * d) > lmin) {
        lmax *= 2;
    }
    int len = 0;
    for (int t = lmax / 2; t >= 1; t /= 2) {
        if (lcp(k, sk, nn, i, i + (len + t) * d) > lmin) {
            len += t;
        }
    }
    const int j = i + len * d;
    const int l = min(i, j), r = max(i, j);
    const int nodelcp = lcp(k, sk, nn, l, r);
    int s = 0, t = r - l;
    do {
        t = (t + 1) / 2;
        if (lcp(k, sk, nn, l, l + s + t) > nodelcp) {
            s += t;
        }
    } while (t > 1);
    const int split = l + s;
    const uint32_t lc = (l == split) ? (uint32_t)l : n + (uint32_t)split;
    const uint32_t rc = (split + 1 == r) ? (uint32_t)r : n + (uint32_t)split + 1;
    node[2 * ((size_t)n + i)] = lc + 1;
    node[2 * ((size_t)n + i) + 1] = rc + 1;
    rank[i] = node_class((uint32_t)l, (uint32_t)r) << kClassBits;
}

// The lists of the nodes across class 0 borders, one workgroup per class 1
// block (32,768 nodes): its class 1 nodes take their places by an LDS counter,
// the nodes of larger classes (at most the chains of the block's two borders)
// by one atomic per workgroup and class on their block's count. The order in
// a list is irrelevant: a node's box depends only on its children's. An
// atomic per listed node in k_karras made that kernel 140 us longer at 3M
// leaves (device-scope atomics on a hundred words).
constexpr uint32_t kListThreads = 1024, kMaxClass = 6, kEdgeCap = 2 * 94;

__global__ __launch_bounds__(1024) void k_top_lists(uint32_t n, uint32_t *__restrict__ rank,
                                                    uint32_t *__restrict__ count,
                                                    uint32_t *__restrict__ list) {
    __shared__ uint32_t cnt[kMaxClass], base[kMaxClass], edge[kEdgeCap], nedge;
    if (threadIdx.x < kMaxClass) {
        cnt[threadIdx.x] = 0;
    }
    if (threadIdx.x == 0) {
        nedge = 0;
    }
    __syncthreads();
    const uint32_t lo = blockIdx.x << class_shift(1);
    const uint32_t hi = min(n - 1, lo + (1u << class_shift(1)));
    const uint32_t seg1 = class_base(n, 1) + blockIdx.x;
    for (uint32_t i = lo + threadIdx.x; i < hi; i += kListThreads) {
        const uint32_t c = rank[i] >> kClassBits;
        if (c == 1) {
            const uint32_t place = atomicAdd(cnt + 1, 1u);
            rank[i] = (1u << kClassBits) | place;
            if (place < kTopCap) {
                list[(size_t)seg1 * kTopCap + place] = i;
            }
        } else if (c > 1) {
            rank[i] = (c << kClassBits) | atomicAdd(cnt + c, 1u);
            const uint32_t e = atomicAdd(&nedge, 1u);
            if (e < kEdgeCap) {
                edge[e] = i;
            }
        }
    }
    __syncthreads();
    auto seg_of = [&](uint32_t c) {
        return class_base(n, c) + (class_shift(c) < 32 ? lo >> class_shift(c) : 0u);
    };
    if (threadIdx.x == 1) {
        count[seg1] = cnt[1];
    } else if (threadIdx.x > 1 && threadIdx.x < kMaxClass && cnt[threadIdx.x]) {
        base[threadIdx.x] = atomicAdd(count + seg_of(threadIdx.x), cnt[threadIdx.x]);
    }
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < min(nedge, kEdgeCap); e += kListThreads) {
        const uint32_t i = edge[e], c = rank[i] >> kClassBits;
        const uint32_t place = base[c] + (rank[i] & ((1u << kClassBits) - 1u));
        rank[i] = (c << kClassBits) | place;
        if (place < kTopCap) {
            list[(size_t)seg_of(c) * kTopCap + place] = i;
        }
    }
}

// Swept leaf box (lbvh.cu:623-731).
__device__ inline Aabb leaf_box(const PrimSet &p, const float *__restrict__ x0,
                                const float *__restrict__ x1, float t, uint32_t prim) {
    const float margin = 0.5f * p.ghat[prim] + p.offset[prim];
    float lo0[3], hi0[3], lo1[3], hi1[3];
    for (int k = 0; k < p.arity; ++k) {
        const uint32_t v = prim_vertex(p, prim, k);
        const f3 y0 = load3(x0 + 3 * (size_t)v);
        f3 z = y0;
        if (x1) {
            const f3 y1 = load3(x1 + 3 * (size_t)v);
            z = mk3(t * (y1.x - y0.x) + y0.x, t * (y1.y - y0.y) + y0.y,
                    t * (y1.z - y0.z) + y0.z);
        }
        const float a[3] = {y0.x, y0.y, y0.z}, b[3] = {z.x, z.y, z.z};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            lo0[d] = k ? fminf(lo0[d], a[d]) : a[d];
            hi0[d] = k ? fmaxf(hi0[d], a[d]) : a[d];
            lo1[d] = k ? fminf(lo1[d], b[d]) : b[d];
            hi1[d] = k ? fmaxf(hi1[d], b[d]) : b[d];
        }
    }
    Aabb bx;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        bx.mn[d] = fminf(lo0[d], lo1[d]) - margin;
        bx.mx[d] = fmaxf(hi0[d], hi1[d]) + margin;
    }
    bx.active = 1.0f;
    bx.pad = __uint_as_float(prim_scene(p, prim));
    return bx;
}

// Tag of a node from its children's: the scene tag in a tree of many scenes,
// else the primitive bound.
__device__ inline uint32_t join_tag(uint32_t a, uint32_t b, bool scenes, int bound) {
    return scenes ? (a == b ? a : kMixedScene) : bound > 0 ? max(a, b) : min(a, b);
}

// One block of 1,024 leaves: their boxes, then the boxes and walk records of
// the class 0 nodes above them, one leaf and one node per thread. Rounds of
// nodes whose children were done in an earlier round, one barrier each (as
// many rounds as the treelet is deep, 11 to 20 in meshes). The boxes stay in
// LDS until the block is done. A refit of 3M independent triangle edges took
// 139 (leaf boxes) + 222 (27 launches of inner levels) + 245 us (records)
// through memory, after 817 us of level tables per build; it takes 276 us here
// and 3 x 34 us in k_refit_top now, with no tables.
constexpr uint32_t kRoundsPerVote = 4; // a vote on the end costs several plain barriers

struct TreeletScratch {
    float lmn[3][kTreelet], lmx[3][kTreelet], nmn[3][kTreelet], nmx[3][kTreelet];
    uint32_t ltag[kTreelet], ntag[kTreelet], prim[kTreelet], done[kTreelet];
    uint16_t c0[kTreelet], c1[kTreelet]; // child of a node: leaf place, or kTreelet + node place
};

__global__ __launch_bounds__(1024) void k_refit_treelet(PrimSet p, const float *__restrict__ x0,
                                                        const float *__restrict__ x1, float t,
                                                        const uint32_t *__restrict__ node,
                                                        const uint32_t *__restrict__ rank,
                                                        bool scenes, Aabb *__restrict__ box,
                                                        uint32_t *__restrict__ ext,
                                                        WalkRec *__restrict__ rec) {
    __shared__ TreeletScratch s;
    const uint32_t n = p.n, tid = threadIdx.x;
    const uint32_t base = blockIdx.x * kTreelet, i = base + tid;
    if (i < n) {
        const uint32_t prim = node[2 * (size_t)i] - 1;
        const Aabb b = leaf_box(p, x0, x1, t, prim);
        box[i] = b;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            s.lmn[d][tid] = b.mn[d];
            s.lmx[d][tid] = b.mx[d];
        }
        s.prim[tid] = prim;
        s.ltag[tid] = scenes ? __float_as_uint(b.pad) : prim;
    }
    const bool mine = i + 1 < n && (rank[i] >> kClassBits) == 0;
    uint32_t c[2] = {0u, 0u};
    if (mine) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint32_t v = node[2 * ((size_t)n + i) + k] - 1;
            c[k] = v < n ? v - base : v - n - base + kTreelet;
        }
        s.c0[tid] = (uint16_t)c[0];
        s.c1[tid] = (uint16_t)c[1];
    }
    s.done[tid] = 0;
    auto mn = [&](uint32_t q, int d) {
        return q < kTreelet ? s.lmn[d][q] : s.nmn[d][q - kTreelet];
    };
    auto mx = [&](uint32_t q, int d) {
        return q < kTreelet ? s.lmx[d][q] : s.nmx[d][q - kTreelet];
    };
    auto tag = [&](uint32_t q) { return q < kTreelet ? s.ltag[q] : s.ntag[q - kTreelet]; };
    bool todo = mine;
    __syncthreads();
    for (uint32_t round = 1; round <= kTreelet; ++round) {
        // done before this round: a mark of this very round may be seen or not
        auto ready = [&](uint32_t q) {
            return q < kTreelet || s.done[q - kTreelet] - 1u < round - 1u;
        };
        if (todo && ready(c[0]) && ready(c[1])) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                s.nmn[d][tid] = fminf(mn(c[0], d), mn(c[1], d));
                s.nmx[d][tid] = fmaxf(mx(c[0], d), mx(c[1], d));
            }
            s.ntag[tid] = join_tag(tag(c[0]), tag(c[1]), scenes, p.bound);
            s.done[tid] = round;
            todo = false;
        }
        if (round % kRoundsPerVote != 0) {
            __syncthreads();
        } else if (!__syncthreads_or(todo)) {
            break;
        }
    }
    if (!mine) {
        return;
    }
    Aabb u;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        u.mn[d] = s.nmn[d][tid];
        u.mx[d] = s.nmx[d][tid];
    }
    u.active = 1.0f;
    u.pad = __uint_as_float(scenes ? s.ntag[tid] : 0u);
    box[(size_t)n + i] = u;
    ext[i] = s.ntag[tid];
    WalkRec w;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const bool leaf = c[k] < kTreelet;
        const uint32_t g[2] = {leaf ? c[k] : s.c0[c[k] - kTreelet],
                               leaf ? 0u : s.c1[c[k] - kTreelet]};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (leaf && h) {
                put_none(w, 2 * k + h);
                continue;
            }
            const uint32_t q = g[h];
            const float a[3] = {mn(q, 0), mn(q, 1), mn(q, 2)};
            const float b[3] = {mx(q, 0), mx(q, 1), mx(q, 2)};
            put_child(w, 2 * k + h,
                      q < kTreelet ? s.prim[q] | kLeafCode : n + base + q - kTreelet, tag(q), a, b);
        }
    }
    rec[i] = w;
}

// The listed nodes of one class c block (c >= 1), after the smaller classes:
// the same rounds over the list, boxes of children of the same class in LDS,
// the others from memory; then the walk records. One workgroup works through
// few hundred nodes, so its time is its chains of dependent loads: everything
// that does not need a box (the grandchildren and their codes) is loaded
// before the rounds, and nothing is stored inside them (a barrier waits for
// stores). 39 us a launch without either, 34 us now (3M leaves; 20 us at 8,000).
struct TopScratch {
    float mn[3][kTopCap], mx[3][kTopCap];
    uint32_t tag[kTopCap], done[kTopCap];
};
constexpr uint32_t kTopThreads = 1024, kTopPer = kTopCap / kTopThreads;

__global__ __launch_bounds__(1024) void k_refit_top(uint32_t n, uint32_t cls, uint32_t seg0,
                                                    const uint32_t *__restrict__ count,
                                                    const uint32_t *__restrict__ list,
                                                    const uint32_t *__restrict__ node,
                                                    const uint32_t *__restrict__ rank,
                                                    bool scenes, int bound, Aabb *box,
                                                    uint32_t *ext, WalkRec *__restrict__ rec) {
    __shared__ TopScratch s;
    const uint32_t seg = seg0 + blockIdx.x;
    const uint32_t cnt = min(count[seg], kTopCap);
    const uint32_t *my = list + (size_t)seg * kTopCap;
    const uint2 *pair = reinterpret_cast<const uint2 *>(node);
    uint32_t self[kTopPer], gc[kTopPer][4], code[kTopPer][4];
    uint32_t pend[kTopPer][2]; // places of children of this class, or kTopCap
    uint32_t todo = 0;
#pragma unroll
    for (uint32_t k = 0; k < kTopPer; ++k) {
        const uint32_t e = k * kTopThreads + threadIdx.x;
        pend[k][0] = pend[k][1] = kTopCap;
        if (e >= cnt) {
            continue;
        }
        todo |= 1u << k;
        s.done[e] = 0;
        self[k] = my[e];
        const uint2 ch = pair[(size_t)n + self[k]];
        const uint32_t c[2] = {ch.x - 1, ch.y - 1};
        const uint2 g[2] = {pair[c[0]], pair[c[1]]};
        float mn[3], mx[3];
        uint32_t tag = 0;
        bool any = false;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bool leaf = c[h] < n;
            const uint32_t r = leaf ? 0u : rank[c[h] - n];
            gc[k][2 * h] = leaf ? c[h] : g[h].x - 1;
            gc[k][2 * h + 1] = leaf ? kNoCode : g[h].y - 1;
            if ((r >> kClassBits) == cls) {
                pend[k][h] = r & ((1u << kClassBits) - 1u);
                continue;
            }
            const Aabb b = box[c[h]];
            const uint32_t bt = scenes ? __float_as_uint(b.pad)
                                       : leaf ? g[h].x - 1 : ext[c[h] - n];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                mn[d] = any ? fminf(mn[d], b.mn[d]) : b.mn[d];
                mx[d] = any ? fmaxf(mx[d], b.mx[d]) : b.mx[d];
            }
            tag = any ? join_tag(tag, bt, scenes, bound) : bt;
            any = true;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t v = gc[k][q];
            code[k][q] = v == kNoCode ? kNoCode
                         : v < n      ? (node[2 * (size_t)v] - 1) | kLeafCode
                                      : v;
        }
        if (any) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                s.mn[d][e] = mn[d];
                s.mx[d][e] = mx[d];
            }
            s.tag[e] = tag;
        }
    }
    __syncthreads();
    for (uint32_t round = 1; round <= kTopCap; ++round) {
        auto ready = [&](uint32_t q) {
            return q == kTopCap || s.done[q] - 1u < round - 1u;
        };
#pragma unroll
        for (uint32_t k = 0; k < kTopPer; ++k) {
            if (!(todo & (1u << k)) || !ready(pend[k][0]) || !ready(pend[k][1])) {
                continue;
            }
            const uint32_t e = k * kTopThreads + threadIdx.x;
            bool any = pend[k][0] == kTopCap || pend[k][1] == kTopCap;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t q = pend[k][h];
                if (q == kTopCap) {
                    continue;
                }
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    s.mn[d][e] = any ? fminf(s.mn[d][e], s.mn[d][q]) : s.mn[d][q];
                    s.mx[d][e] = any ? fmaxf(s.mx[d][e], s.mx[d][q]) : s.mx[d][q];
                }
                s.tag[e] = any ? join_tag(s.tag[e], s.tag[q], scenes, bound) : s.tag[q];
                any = true;
            }
            s.done[e] = round;
            todo &= ~(1u << k);
        }
        if (round % kRoundsPerVote != 0) {
            __syncthreads();
        } else if (!__syncthreads_or(todo != 0)) {
            break;
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < kTopPer; ++k) {
        const uint32_t e = k * kTopThreads + threadIdx.x;
        if (e >= cnt) {
            continue;
        }
        Aabb u;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            u.mn[d] = s.mn[d][e];
            u.mx[d] = s.mx[d][e];
        }
        u.active = 1.0f;
        u.pad = __uint_as_float(scenes ? s.tag[e] : 0u);
        box[(size_t)n + self[k]] = u;
        ext[self[k]] = s.tag[e];
    }
    __syncthreads(); // the boxes written above are read below
#pragma unroll
    for (uint32_t k = 0; k < kTopPer; ++k) {
        if (k * kTopThreads + threadIdx.x >= cnt) {
            continue;
        }
        WalkRec w;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t v = gc[k][q];
            if (v == kNoCode) {
                put_none(w, q);
                continue;
            }
            const Aabb b = box[v];
            const uint32_t t = scenes  ? __float_as_uint(b.pad)
                               : v < n ? code[k][q] & ~kLeafCode
                                       : ext[v - n];
            put_child(w, q, code[k][q], t, b.mn, b.mx);
        }
        rec[self[k]] = w;
    }
}

uint32_t cdiv(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

} // namespace

Lbvh::~Lbvh() { release(); }

void Lbvh::release() {
    for (void *p : {(void *)node_, (void *)depth_, (void *)rank_, (void *)list_, (void *)code_,
                    (void *)idx_, (void *)scratch_, (void *)cent_, (void *)part_,
                    (void *)box_, (void *)rec_, (void *)ext_, (void *)sb_}) {
        if (p) {
            (void)dev_free(p);
        }
    }
    node_ = depth_ = rank_ = list_ = code_ = idx_ = scratch_ = nullptr;
    cent_ = part_ = nullptr;
    box_ = nullptr;
    rec_ = nullptr;
    ext_ = nullptr;
    sb_ = nullptr;
    sb_cap_ = 0;
    cap_ = 0;
}

int Lbvh::reserve(uint32_t n) {
    if (n <= cap_) {
        return PPF_OK;
    }
    release();
    const size_t nodes = 2 * (size_t)n;
    const size_t nb = cdiv(n, kNT);
    PPF_HIP(dev_alloc(&node_, 2 * nodes * sizeof(uint32_t)));
    PPF_HIP(dev_alloc(&depth_, n * sizeof(uint32_t)));
    PPF_HIP(dev_alloc(&rank_, n * sizeof(uint32_t)));
    const size_t segs = class_base(n, top_classes(n) + 1);
    PPF_HIP(dev_alloc(&list_, std::max<size_t>(segs * (kTopCap + 1), 1) * sizeof(uint32_t)));
    PPF_HIP(dev_alloc(&code_, n * sizeof(uint32_t)));
    PPF_HIP(dev_alloc(&idx_, n * sizeof(uint32_t)));
    PPF_HIP(dev_alloc(&scratch_, radix_sort_scratch_words(n) * sizeof(uint32_t)));
    PPF_HIP(dev_alloc(&cent_, 3 * (size_t)n * sizeof(float)));
    PPF_HIP(dev_alloc(&part_, (6 * nb + 6) * sizeof(float)));
    PPF_HIP(dev_alloc(&box_, nodes * sizeof(Aabb)));
    PPF_HIP(dev_alloc(&rec_, std::max<size_t>(n, 1) * sizeof(WalkRec)));
    PPF_HIP(dev_alloc(&ext_, std::max<size_t>(n, 1) * sizeof(uint32_t)));
    cap_ = n;
    return PPF_OK;
}

int Lbvh::build(const PrimSet &p, const float *x0, const float *x1, float t,
                hipStream_t s) {
    int rc = reserve(p.n);
    if (rc != PPF_OK) {
        return rc;
    }
    if (p.n >= kLeafCode) {
        set_error("Lbvh: %u primitives exceed the walk records' index range", p.n);
        return PPF_ERR_ARG;
    }
    n_ = p.n;
    bound_ = p.bound;
    scenes_ = p.vscene && p.nscene > 1;
    root_ = n_ == 1 ? 0 : n_;
    if (n_ == 0) {
        return PPF_OK;
    }
    const uint32_t nb = cdiv(n_, kNT);
    const bool scenes = scenes_;
    k_centroid<<<nb, kNT, 0, s>>>(p, x0, cent_, scenes ? nullptr : part_);
    PPF_HIP(hipGetLastError());
    if (scenes) {
        // each scene quantized in its own box: a scene's tree does not depend
        // on the other scenes of the mesh
        if (6 * (size_t)p.nscene > sb_cap_) {
            if (sb_) {
                PPF_HIP(dev_free(sb_));
                sb_ = nullptr;
            }
            PPF_HIP(dev_alloc(&sb_, 6 * (size_t)p.nscene * sizeof(uint32_t)));
            sb_cap_ = 6 * (size_t)p.nscene;
        }
        k_scene_bounds_init<<<cdiv(6 * p.nscene, kNT), kNT, 0, s>>>(p.nscene, sb_);
        k_scene_bounds<<<cdiv(p.n, kNT * kSceneRun), kNT, 0, s>>>(p, cent_, sb_);
        k_morton_scenes<<<nb, kNT, 0, s>>>(p, cent_, sb_, code_, idx_);
    } else {
        float *bounds = part_ + 6 * (size_t)nb;
        k_bounds<<<1, kNT, 0, s>>>(nb, part_, bounds);
        k_morton<<<nb, kNT, 0, s>>>(n_, cent_, bounds, code_, idx_);
    }
    PPF_HIP(hipGetLastError());
    if (scenes) { // per-primitive codes, kept for the regather after the scene pass
        PPF_HIP(hipMemcpyAsync(rank_, code_, n_ * sizeof(uint32_t), hipMemcpyDeviceToDevice,
                               s));
    }
    PPF_HIP(radix_sort_pairs(code_, idx_, n_, 30, scratch_, s));
    const uint32_t *sk = nullptr;
    if (scenes) {
        // stable second pass by scene: leaves ordered by (scene, code, index)
        uint32_t bits = 1;
        while (bits < 32 && ((p.nscene - 1) >> bits) != 0) {
            ++bits;
        }
        k_scene_keys<<<nb, kNT, 0, s>>>(p, idx_, depth_);
        PPF_HIP(hipGetLastError());
        PPF_HIP(radix_sort_pairs(depth_, idx_, n_, bits, scratch_, s));
        k_regather<<<nb, kNT, 0, s>>>(n_, idx_, rank_, code_);
        PPF_HIP(hipGetLastError());
        sk = depth_;
    }
    // lists of the nodes across treelet borders: counts, then places
    const uint32_t segs = class_base(n_, top_classes(n_) + 1);
    k_karras<<<nb, kNT, 0, s>>>(n_, code_, sk, idx_, node_, rank_, segs, list_);
    PPF_HIP(hipGetLastError());
    if (segs) {
        k_top_lists<<<class_blocks(n_, 1), kListThreads, 0, s>>>(n_, rank_, list_, list_ + segs);
        PPF_HIP(hipGetLastError());
    }
    return refit(p, x0, x1, t, s);
}

int Lbvh::refit(const PrimSet &p, const float *x0, const float *x1, float t,
                hipStream_t s) {
    if (p.n != n_) {
        set_error("Lbvh::refit: primitive count %u differs from the build (%u)",
                  p.n, n_);
        return PPF_ERR_ARG;
    }
    if (n_ == 0) {
        return PPF_OK;
    }
    k_refit_treelet<<<cdiv(n_, kTreelet), kTreelet, 0, s>>>(p, x0, x1, t, node_, rank_, scenes_,
                                                            box_, ext_, rec_);
    PPF_HIP(hipGetLastError());
    const uint32_t top = top_classes(n_), segs = class_base(n_, top + 1);
    for (uint32_t c = 1; c <= top; ++c) {
        k_refit_top<<<class_blocks(n_, c), kTopThreads, 0, s>>>(
            n_, c, class_base(n_, c), list_, list_ + segs, node_, rank_, scenes_, bound_, box_,
            ext_, rec_);
        PPF_HIP(hipGetLastError());
    }
    return PPF_OK;
}

int Lbvh::follow(const PrimSet &p, const float *x, hipStream_t s, bool fresh) {
    if (!fresh && followed_x_ == x && followed_elem_ == p.elem && n_ == p.n && bound_ == p.bound &&
        scenes_ == (p.vscene && p.nscene > 1)) {
        return refit(p, x, nullptr, 0.0f, s);
    }
    followed_x_ = nullptr;
    const int rc = build(p, x, nullptr, 0.0f, s);
    if (rc == PPF_OK) {
        followed_x_ = x;
        followed_elem_ = p.elem;
    }
    return rc;
}

BvhView Lbvh::view() const {
    BvhView v;
    v.n = n_;
    v.root = root_;
    v.node = node_;
    v.box = box_;
    v.rec = rec_;
    v.scenes = scenes_;
    v.bound = scenes_ ? 0 : bound_;
    return v;
}

} // namespace ppf
