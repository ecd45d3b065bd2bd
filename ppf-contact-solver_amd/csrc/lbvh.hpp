// lbvh.hpp -- linear BVH over faces, edges or vertices (device).
//
// Same tree as the reference's LBVH (lbvh/lbvh.cu:108-385): centroids, scene
// bounds of the centroids, 10-bit-per-axis Morton codes, a stable sort of
// (code, index), and the Karras radix tree with the index tie-break on equal
// codes. Node i < n is leaf i (prim + 1, 0); node n + i is internal node i
// (left + 1, right + 1); the root is node n (leaf 0 when n == 1).
#pragma once
#include "common.hpp"

namespace ppf {

// Box of one node: min xyz, active flag, max xyz, scene tag (32 B, two 16 B
// loads). The tag holds the bits of the scene id every leaf below the node
// belongs to, or kMixedScene when they belong to several (0 throughout for a
// one-scene tree).
struct alignas(32) Aabb {
    float mn[3];
    float active;
    float mx[3];
    float pad;
};
constexpr uint32_t kMixedScene = 0xffffffffu;

// Walk record of internal node n + i (128 B, one L2 line, eight 16 B loads):
// the node's grandchildren in leaf order, two places per child (a leaf child
// stands for itself in the first; an unused place holds kNoCode and NaN), so a
// walk takes two levels of the tree per record. A code is the child's node id,
// or for a leaf its primitive | kLeafCode. The tag is the scene tag of the
// child's box in a tree of many scenes; in a one-scene tree it is the child's
// primitive bound (PrimSet::bound), which lets a query skip subtrees without
// partners.
// The records are the largest part of a tree: 128 B per leaf beside 80 B of
// nodes and boxes (two trees of 6M leaves: 1.5 GB of records).
struct alignas(128) WalkRec {
    uint32_t code[4];
    uint32_t tag[4];
    float box[24]; // child 0 min xyz, max xyz, then children 1 to 3
};
constexpr uint32_t kLeafCode = 0x80000000u;
constexpr uint32_t kNoCode = 0xffffffffu;
constexpr uint32_t kInactiveTag = 0xfffffffeu;

PPF_HD void put_child(WalkRec &w, int k, uint32_t code, uint32_t tag, const float mn[3],
                      const float mx[3]) {
    w.code[k] = code;
    w.tag[k] = tag;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        w.box[6 * k + d] = mn[d];
        w.box[6 * k + 3 + d] = mx[d];
    }
}
// A NaN box compares false with every query box. An empty one (+inf, -inf)
// would overlap the box of a query with an infinite gap, offset or position.
// (A test of the code in the walk instead: 3.05 -> 3.16 ms of line search.)
PPF_HD void put_none(WalkRec &w, int k) {
    const float nan = __builtin_nanf("");
    const float box[3] = {nan, nan, nan};
    put_child(w, k, kNoCode, kInactiveTag, box, box);
}

struct BvhView {
    uint32_t n = 0;            // leaves
    uint32_t root = 0;
    const uint32_t *node = nullptr; // 2 words per node
    const Aabb *box = nullptr;
    const WalkRec *rec = nullptr;   // n - 1 records (internal nodes)
    bool scenes = false;       // tags are scene tags
    int bound = 0;             // tags are primitive bounds: +1 largest, -1 smallest
};

// The trees of a collision mesh.
struct StaticTrees {
    BvhView face, edge;
};

// Primitive set a tree is built over: `arity` vertex indices per primitive
// (3 faces, 2 edges, 1 vertices; index = element for vertices), margin
// 0.5*ghat + offset per primitive.
struct PrimSet {
    uint32_t n = 0;
    int arity = 1;
    const uint32_t *elem = nullptr;  // n * arity vertex indices (null: identity)
    const float *ghat = nullptr;     // per primitive
    const float *offset = nullptr;   // per primitive
    // Many scenes: scene id per vertex (a primitive's scene is its first
    // vertex's) and the scene count. The tree then orders its leaves by
    // (scene, Morton code), so each scene is one subtree, and tags every node
    // with its scene. Null / nscene <= 1: one scene.
    const uint32_t *vscene = nullptr;
    uint32_t nscene = 0;
    // Primitive bound the walk records of a one-scene tree carry per child: the
    // largest (+1) or smallest (-1) primitive below it, or none (0). Queries
    // that pair with higher (lower) primitives only skip the other subtrees.
    int bound = 0;
};

class Lbvh {
  public:
    ~Lbvh();
    // Allocates for up to n primitives (grows when needed).
    int reserve(uint32_t n);
    // Full build from positions x0 (swept to x0 + t (x1 - x0) when x1 is set).
    int build(const PrimSet &p, const float *x0, const float *x1, float t,
              hipStream_t s);
    // Refit the leaf boxes and the inner boxes, same topology.
    int refit(const PrimSet &p, const float *x0, const float *x1, float t,
              hipStream_t s);
    // The tree of arrays that their owner may rewrite between calls: refit to
    // what they hold now, or built where they are others than at the last
    // call. A refit takes any contents (every primitive keeps a leaf); the
    // addresses only decide whether the tree is a fresh one, as `fresh` asks for.
    int follow(const PrimSet &p, const float *x, hipStream_t s, bool fresh = false);
    BvhView view() const;
    uint32_t *nodes() { return node_; }
    Aabb *boxes() { return box_; }

  private:
    uint32_t cap_ = 0, n_ = 0, root_ = 0;
    uint32_t *node_ = nullptr, *depth_ = nullptr;
    uint32_t *rank_ = nullptr; // treelet class and place of every internal node
    uint32_t *list_ = nullptr; // nodes across treelet borders, per block: counts, places
    uint32_t *code_ = nullptr, *idx_ = nullptr, *scratch_ = nullptr;
    float *cent_ = nullptr, *part_ = nullptr;
    Aabb *box_ = nullptr;
    WalkRec *rec_ = nullptr;
    uint32_t *ext_ = nullptr; // tag of every internal node (scene or primitive bound)
    int bound_ = 0;
    bool scenes_ = false;
    const float *followed_x_ = nullptr; // arrays of the last follow() that built
    const uint32_t *followed_elem_ = nullptr;
    uint32_t *sb_ = nullptr; // per-scene centroid bounds (many scenes)
    size_t sb_cap_ = 0;
    void release();
};

} // namespace ppf
