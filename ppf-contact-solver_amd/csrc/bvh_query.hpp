// bvh_query.hpp -- box queries over an LBVH (device).
//
// aabb::overlap / aabb::query of contact/aabb.hpp:70-107: depth-first from the
// root, inactive boxes never overlap. One thread per query; the per-thread
// stack lives in LDS, strided by the workgroup size so a wave's stack slots
// fall in distinct banks. Children are tested before they are pushed, so the
// stack only ever holds overlapping nodes. A query that would push past the
// stack flags `overflow` and stops (the caller runs the pass again with deep
// stacks, and reports a capacity error if those overflow too).
#pragma once
#include "lbvh.hpp"

namespace ppf {

constexpr int kQueryThreads = 128; // threads per query workgroup
// Stack entries per thread. A walk enters one record (two levels of the tree)
// at a time and keeps at most three of its children for later, and on its way
// to the k-th record of a path it holds 3 (k - 1) of them. The walks first run
// with kQueryStack entries (16 KB of LDS per workgroup, ten per CU); a walk that
// needs more raises the overflow flag and never writes past the stack, and the
// caller runs the pass again with kDeepStack entries. traverse() goes on with the
// rightmost child: 3 k <= kDeepStack, 32 records or trees of 64 levels.
// traverse_wave() pushes all four: 3 (k - 1) + 4 <= kDeepStack, 31 records or 62
// levels. A Karras tree is at most as deep as its keys have bits: log2 of the
// scene count, 30 of the Morton code, and log2 of the largest run of equal codes
// (ties split by index).
constexpr int kQueryStack = 32;
constexpr int kDeepStack = 96;

// A query box and the scene of its query element (0 in a one-scene mesh).
struct QBox {
    float mn[3], mx[3];
    uint32_t scene = 0;
};

// Box overlap (aabb::overlap), restricted to nodes holding the query's scene:
// a node whose leaves all belong to another scene is never entered.
__device__ inline bool overlaps(const Aabb &a, const QBox &q) {
    const uint32_t tag = __float_as_uint(a.pad);
    return a.active != 0.0f && (tag == q.scene || tag == kMixedScene) &&
           (a.mn[0] <= q.mx[0] && a.mx[0] >= q.mn[0]) &&
           (a.mn[1] <= q.mx[1] && a.mx[1] >= q.mn[1]) &&
           (a.mn[2] <= q.mx[2] && a.mx[2] >= q.mn[2]);
}

// Scene id of a vertex (0 when the mesh holds one scene).
__device__ inline uint32_t vertex_scene(const uint32_t *vscene, uint32_t nscene, uint32_t v) {
    return (vscene && nscene > 1) ? vscene[v] : 0u;
}

__device__ inline Aabb load_box(const Aabb *b, uint32_t i) {
    const float4 *p = reinterpret_cast<const float4 *>(b + i);
    const float4 lo = p[0];
    const float4 hi = p[1];
    Aabb r;
    r.mn[0] = lo.x, r.mn[1] = lo.y, r.mn[2] = lo.z, r.active = lo.w;
    r.mx[0] = hi.x, r.mx[1] = hi.y, r.mx[2] = hi.z, r.pad = hi.w;
    return r;
}

// Box of the points a, b (min / max), then -/+ margin when it is non-zero
// (aabb::make, contact/aabb.hpp:45-60).
__device__ inline QBox seg_box(f3 a, f3 b, float margin) {
    QBox q{{fminf(a.x, b.x), fminf(a.y, b.y), fminf(a.z, b.z)},
           {fmaxf(a.x, b.x), fmaxf(a.y, b.y), fmaxf(a.z, b.z)},
           0u};
    if (margin != 0.0f) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            q.mn[d] -= margin;
            q.mx[d] += margin;
        }
    }
    return q;
}

// A box that overlaps nothing: the query of an element outside its
// collision window (an inactive query box, contact.cu:1637, 1728, 2563).
__device__ inline QBox empty_box() {
    const float inf = __builtin_inff();
    return QBox{{inf, inf, inf}, {-inf, -inf, -inf}, 0u};
}

// Point +/- margin (aabb::make, contact/aabb.hpp:62-69).
__device__ inline QBox point_box(f3 p, float margin) {
    return QBox{{p.x - margin, p.y - margin, p.z - margin},
                {p.x + margin, p.y + margin, p.z + margin},
                0u};
}

// The stack code of the root: its node id, or for a one-leaf tree its
// primitive | kLeafCode.
__device__ inline uint32_t root_code(const BvhView &bvh) {
    return bvh.n == 1 ? (bvh.node[2 * (size_t)bvh.root] - 1) | kLeafCode : bvh.root;
}

// Which leaves a query pairs with: all, or only primitives above (below) its
// own. The bound prunes subtrees (tags of a tree built with the same bound)
// and leaves.
enum Pairing { kPairAll = 0, kPairAbove = 1, kPairBelow = -1 };

// Tests the children of a walk record against q: a bit per overlapping child
// (aabb::overlap on the stored boxes and scene tags; bound: BvhView's). The
// comparisons keep out unused places, whose boxes are NaN. own: the query's
// primitive for kPairAbove / kPairBelow. With `inner` (statistics) adds the
// number of the node's own internal children that overlap q: their boxes are
// the unions of the stored pairs.
template <int PAIR>
PPF_HD uint32_t record_hits(const uint32_t code[4], const uint32_t tag[4], const float b[24],
                            const QBox &q, uint32_t own, bool scenes, int bound,
                            uint32_t *inner = nullptr) {
    uint32_t hit = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float *bx = b + 6 * k;
        bool ok = (bx[0] <= q.mx[0]) & (bx[3] >= q.mn[0]) & (bx[1] <= q.mx[1]) &
                  (bx[4] >= q.mn[1]) & (bx[2] <= q.mx[2]) & (bx[5] >= q.mn[2]);
        if (scenes) {
            ok &= tag[k] == q.scene || tag[k] == kMixedScene;
        }
        if (PAIR != kPairAll) {
            const uint32_t key = (code[k] & kLeafCode) ? code[k] & ~kLeafCode : tag[k];
            const bool bounded = (code[k] & kLeafCode) != 0 || bound == PAIR;
            ok &= !bounded || (PAIR == kPairAbove ? key > own : key < own);
        }
        hit |= ok ? 1u << k : 0u;
    }
    if (inner) {
#pragma unroll
        for (int k = 0; k < 4; k += 2) {
            const float *u = b + 6 * k, *w = u + 6;
            bool ok = code[k + 1] != kNoCode;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                ok &= fminf(u[d], w[d]) <= q.mx[d] && fmaxf(u[3 + d], w[3 + d]) >= q.mn[d];
            }
            if (scenes) {
                ok &= tag[k] != tag[k + 1] || tag[k] == q.scene || tag[k] == kMixedScene;
            }
            *inner += ok ? 1u : 0u;
        }
    }
    return hit;
}

// Reads internal node v's walk record and tests its children (record_hits).
template <int PAIR>
__device__ inline uint32_t enter(const BvhView &bvh, uint32_t v, const QBox &q, uint32_t own,
                                 uint32_t code[4], uint32_t *inner = nullptr) {
    const uint4 *r = reinterpret_cast<const uint4 *>(bvh.rec + (v - bvh.n));
    const uint4 a = r[0], t = r[1];
    float b[24];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const uint4 w = r[2 + k];
        b[4 * k] = __uint_as_float(w.x), b[4 * k + 1] = __uint_as_float(w.y);
        b[4 * k + 2] = __uint_as_float(w.z), b[4 * k + 3] = __uint_as_float(w.w);
    }
    code[0] = a.x, code[1] = a.y, code[2] = a.z, code[3] = a.w;
    const uint32_t tag[4] = {t.x, t.y, t.z, t.w};
    return record_hits<PAIR>(code, tag, b, q, own, bvh.scenes, bvh.bound, inner);
}

// Work of one lane's tree walks, for the walk statistics: tree nodes whose
// box overlaps the query's (what a walk of the binary tree takes off its
// stack, the root included: the measure of a scene, whatever the records'
// width), leaves among them, and candidates swept (queued CCD work). The
// statistics variants of the kernels (STATS) walk without the pairing bounds.
struct WalkCount {
    uint32_t nodes = 0, leaves = 0, work = 0;
};

// Walk statistics of one kind of query, accumulated on the device (u64):
// launches, queries, nodes, leaves, work. Kinds: line-search vertex sweeps,
// line-search edge sweeps, proximity vertex queries, proximity edge queries.
enum WalkKind { kWalkLsVertex = 0, kWalkLsEdge = 1, kWalkProxVertex = 2, kWalkProxEdge = 3 };
constexpr int kWalkKinds = 4, kWalkFields = 5;

// Adds a workgroup's counts to stats[kind] (null: statistics off). Every
// thread calls it; `query` marks a lane that had a query.
__device__ inline void walk_flush(unsigned long long *stats, int kind, const WalkCount &wc,
                                  bool query) {
    if (!stats) {
        return;
    }
    unsigned long long *s = stats + kWalkFields * kind;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    uint32_t v[4] = {query ? 1u : 0u, wc.nodes, wc.leaves, wc.work};
#pragma unroll
    for (int f = 0; f < 4; ++f) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            v[f] += __shfl_xor(v[f], off, kWave);
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            atomicAdd(s + 1 + f, (unsigned long long)v[f]);
        }
    }
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        atomicAdd(s, 1ull);
    }
}

// Visits every leaf whose box overlaps q (and that PAIR keeps), from the last
// leaf to the first; `leaf(prim)` returns whether the candidate was accepted.
// Returns the accepted count. `stk` is this thread's first LDS slot (stride
// kQueryThreads). Bound by the dependent record loads and by divergence: two
// tree levels per load, and lanes walk until every lane holds a leaf or is
// done, then all run `leaf`, so the candidates' work is not paid for lane by
// lane. Against one level per 64 B record, leaves taken off one at a time and
// no pairing bound: vertex queries of 1M independent triangles 3,792 -> 2,378
// us, their edge queries 2,878 -> 1,885 us; on 8 x 201 x 201 sheets 1,715 ->
// 1,030 us and 2,401 -> 1,448 us.
template <int STACK, int PAIR = kPairAll, bool STATS = false, class F>
__device__ uint32_t traverse(const BvhView &bvh, const QBox &q, uint32_t *stk,
                             uint32_t *overflow, F &&leaf, uint32_t own = 0,
                             WalkCount *wc = nullptr) {
    if (bvh.n == 0 || !overlaps(load_box(bvh.box, bvh.root), q)) {
        return 0;
    }
    uint32_t count = 0;
    uint32_t sp = 0;
    uint32_t v = root_code(bvh);
    bool more = true;
    while (true) {
        while (more && !(v & kLeafCode)) {
            uint32_t code[4];
            const uint32_t hit =
                enter<STATS ? kPairAll : PAIR>(bvh, v, q, own, code, STATS ? &wc->nodes : nullptr);
            if (STATS) {
                ++wc->nodes;
            }
            if (sp + 3 > (uint32_t)STACK) {
                atomicOr(overflow, 1u);
                return count;
            }
            bool next = false;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (hit & (1u << k)) {
                    if (next) {
                        stk[(sp++) * kQueryThreads] = v;
                    }
                    v = code[k];
                    next = true;
                }
            }
            if (!next) {
                more = sp != 0;
                if (more) {
                    v = stk[(--sp) * kQueryThreads];
                }
            }
        }
        if (!more) {
            return count;
        }
        if (STATS) {
            ++wc->nodes;
            ++wc->leaves;
        }
        if (leaf(v & ~kLeafCode)) {
            ++count;
        }
        more = sp != 0;
        if (more) {
            v = stk[(--sp) * kQueryThreads];
        }
    }
}

// ---- wave-cooperative traversal --------------------------------------------
//
// For queries whose per-candidate work is long and data dependent (the CCD
// sweeps): a workgroup is one wave of kWaveQueries queries. Every lane walks
// its own query one node per round; a leaf that `accept(prim)` keeps enters a
// queue in LDS as (query id, prim). Whenever the queue holds a wave's worth of
// entries, and when the walks are over, every lane takes one entry and runs
// `work(qid, prim)`, so the long work runs with (nearly) all lanes active
// instead of with the few lanes that happen to sit on a leaf.

constexpr int kWaveQueries = 64;        // one wave per workgroup
constexpr int kWaveQueue = 2 * kWaveQueries;

template <int STACK> struct WaveScratchT {
    uint32_t stk[STACK * kWaveQueries];
    uint32_t qid[kWaveQueue], prim[kWaveQueue];
};

__device__ inline uint32_t lanes_below(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Line search of 8 x 129 x 129 falling sheets, one-level against two-level
// records: edge sweeps 1,950 -> 1,692 us, vertex sweeps 810 -> 640 us.
// `active`: this lane has a query (lanes past the end pass false). All lanes
// of the workgroup must call it (the rounds are wave uniform).
template <int PAIR, bool STATS, int STACK, class A, class W>
__device__ void traverse_wave(const BvhView &bvh, const QBox &q, bool active, uint32_t qid,
                              WaveScratchT<STACK> &ws, uint32_t *overflow, A &&accept, W &&work,
                              WalkCount *wc = nullptr) {
    const uint32_t lane = threadIdx.x;
    uint32_t *stk = ws.stk + lane;
    uint32_t sp = 0;
    if (active && bvh.n != 0 && overlaps(load_box(bvh.box, bvh.root), q)) {
        stk[0] = root_code(bvh);
        sp = 1;
    }
    uint32_t queued = 0; // wave uniform
    while (true) {
        uint32_t cand = 0xffffffffu;
        if (sp) {
            const uint32_t v = stk[(--sp) * kWaveQueries];
            if (STATS) {
                ++wc->nodes;
            }
            if (v & kLeafCode) {
                const uint32_t prim = v & ~kLeafCode;
                if (STATS) {
                    ++wc->leaves;
                }
                if (accept(prim)) {
                    cand = prim;
                }
            } else {
                uint32_t code[4];
                const uint32_t hit = enter<STATS ? kPairAll : PAIR>(bvh, v, q, qid, code,
                                                                    STATS ? &wc->nodes : nullptr);
                if (sp + 4 > (uint32_t)STACK) {
                    atomicOr(overflow, 1u);
                    sp = 0;
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        if (hit & (1u << k)) {
                            stk[(sp++) * kWaveQueries] = code[k];
                        }
                    }
                }
            }
        }
        const uint64_t m = __ballot(cand != 0xffffffffu);
        if (cand != 0xffffffffu) {
            const uint32_t at = queued + lanes_below(m);
            ws.qid[at] = qid;
            ws.prim[at] = cand;
        }
        queued += (uint32_t)__popcll(m);
        const bool walking = __ballot(sp != 0) != 0;
        if (queued >= (uint32_t)kWaveQueries || (!walking && queued)) {
            __syncthreads();
            const uint32_t take = min(queued, (uint32_t)kWaveQueries);
            if (lane < take) {
                const uint32_t at = queued - 1 - lane;
                work(ws.qid[at], ws.prim[at]);
                if (STATS) {
                    ++wc->work;
                }
            }
            queued -= take;
            __syncthreads();
        }
        if (!walking && !queued) {
            break;
        }
    }
}

} // namespace ppf
