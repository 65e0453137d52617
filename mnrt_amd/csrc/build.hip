// build.hip — kd-tree construction on gfx950 for triangles (SAH) and photons (VVH).
//
// Follows the two-stage build of KDTreeGPU::BuildTree (KDTreeGPU.cpp:175-209):
//
//   large-node stage (LargeNodeStage / ProcessLargeNodes, KDTreeGPU.cpp:247-782):
//     per level, for all active nodes at once:
//       classification counts       k_count     (kdtree.cu:467-682, 752-824, 1986-2033)
//       compaction offsets, children, small/large partition
//                                   k_children  (CompactElementData / UpdateSmallList, KDTreeGPU.cpp:664-941)
//       scatter + tight bounds      k_scatter   (kdtree_chunklist.cu:73-184, kdtree.cu:310-445)
//       split clipping              k_clip      (kdtree_tri.cu:190-489)
//     All counts stay on the device; the host waits for a run of levels at a time (the
//     reference synchronises about ten times per level).
//
//   small-node stage (PreProcessSmallNodes / ProcessSmallNodes, KDTreeGPU.cpp:945-1154):
//     one wave64 per small root builds the whole subtree in LDS: split candidates and
//     their 64-bit element masks (kdtree.cu:1035-1251), exact SAH / VVH per node with a
//     wave argmin over (cost, candidate index) (kdtree.cu:1288-1471), preorder emission.
//
//   layout: subtree sizes climb from the leaves, addresses are sums over the ancestors
//   (KDTreeGPU::PreorderTraversal, KDTreeGPU.cpp:1156-1209): two launches.
//
// Deterministic rules replace the reference's random and racy choices (elements in a
// split plane go left for even index, right for odd; equal SAH costs resolve to the
// lowest candidate index), so the tree is identical, word for word, to the one the host
// oracle builds.
#include <algorithm>
#include <type_traits>
#include <vector>

#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "batch_dev.h"
#include "scan.h"

namespace mnrt {

constexpr uint32_t kNone = 0xFFFFFFFFu;

enum : uint32_t { BN_LEAF = 3, BN_SMALL = 4, BN_PENDING = 5 };
// Build nodes: one 64-byte record (a cache line) per node of the large-stage tree (inner nodes,
// empty and capped leaves, small roots), written and read as quads.  Build nodes 0..S-1 are the
// roots of the S scenes built together.
struct alignas(64) BnRec {
    uint32_t type;   // 0..2 inner split axis, BN_LEAF, BN_SMALL, BN_PENDING
    uint32_t split;  // split position bits (inner)
    uint32_t left, right;
    uint32_t level;
    uint32_t aux;  // small-root index (BN_SMALL) or first copied element (BN_LEAF)
    uint32_t cnt;  // element count (BN_LEAF)
    uint32_t scene;
    uint32_t parent;  // kNone for a root; kCutParent | node below an empty-space cut
    uint32_t pad;
    uint32_t size, rsize;  // nodes and references in the subtree
    unsigned long long acc;  // what the children that have arrived brought (k_layout_sizes)
    uint32_t addr, rbase;  // small roots: subtree start in the scene's tree
};
static_assert(sizeof(BnRec) == 64, "one line");
constexpr uint32_t kCutParent = 0x80000000u;

struct alignas(16) SmallRec {  // small roots
    uint32_t first, cnt, level, bn;
    float lo[3];
    uint32_t scene;
    float hi[3];
    uint32_t pad;
};
static_assert(sizeof(SmallRec) == 48, "three quads");

// Writes quad q of a record.
__device__ __forceinline__ void put4(void* rec, uint32_t q, uint32_t x, uint32_t y, uint32_t z, uint32_t w) {
    ((uint4*)rec)[q] = make_uint4(x, y, z, w);
}

// Concatenated input of S scenes: element e of scene s is entry base[s] + e; element
// indices inside a build are scene-local, as a single-scene build would number them.
struct Geometry {
    int kind;
    const float4* v0;
    const float4* v1;
    const float4* v2;
    const uint32_t* base;  // S + 1 offsets
    uint32_t num_scenes;
};

__device__ __forceinline__ uint32_t scene_of(const uint32_t* base, uint32_t nscenes, uint32_t g) {
    uint32_t lo = 0, hi = nscenes;  // last s with base[s] <= g
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (base[mid] <= g) lo = mid;
        else hi = mid;
    }
    return lo;
}

__device__ __forceinline__ uint32_t fenc(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float fdec(uint32_t u) {
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u);
}
__device__ __forceinline__ float f4c(const float4& v, uint32_t a) { return a == 0 ? v.x : (a == 1 ? v.y : v.z); }
__device__ __forceinline__ void f4set(float4& v, uint32_t a, float x) {
    if (a == 0) v.x = x;
    else if (a == 1) v.y = x;
    else v.z = x;
}
// -0 -> +0 so min/max and stored split words never depend on the sign of zero
__device__ __forceinline__ float canon(float x) { return x + 0.0f; }

__device__ __forceinline__ bool plane_goes_left(uint32_t idx) { return (idx & 1u) == 0u; }

// Large-node classification (kernel_MarkLeftRightElements, kdtree.cu:752-824) with the
// even/odd rule for elements in the split plane.
__device__ __forceinline__ void classify(int kind, uint32_t idx, const float4& lo, const float4& hi,
                                         uint32_t axis, float s, bool& L, bool& R) {
    if (kind == MNRT_KIND_TRI) {
        float mn = f4c(lo, axis), mx = f4c(hi, axis);
        bool planar_on = (mn == s && mn == mx);
        L = mn < s || (planar_on && plane_goes_left(idx));
        R = s < mx || (planar_on && !plane_goes_left(idx));
    } else {
        float p = f4c(lo, axis);
        if (plane_goes_left(idx)) {
            L = p <= s;
            R = s < p;
        } else {
            L = p < s;
            R = s <= p;
        }
    }
}

// Triangles that go to both children (and are clipped there).
__device__ __forceinline__ bool straddles(int kind, const float4& lo, const float4& hi, uint32_t axis, float s) {
    return kind == MNRT_KIND_TRI && f4c(lo, axis) < s && s < f4c(hi, axis);
}

// ---- split clipping (dev_ClipSegment / dev_ClipTriToBounds, kdtree_tri.cu:190-316) ----

// Vertex lists of the clipping in LDS (a per-lane array indexed by the running vertex
// count would live in scratch memory): per lane two lists of up to kClipVerts vertices,
// coordinate-major with the lane innermost, so the lanes of a wave touch consecutive banks.
// k_clip runs kClipBlock lanes per workgroup.
constexpr int kClipBlock = 64;
constexpr int kClipVerts = 12;  // a triangle clipped by six planes has at most 9

struct ClipLists {
    __attribute__((address_space(3))) float* col;  // this lane's column
    int list, n;                                   // current list, its vertices
    __device__ __forceinline__ int at(int l, int v, int c) const { return ((l * kClipVerts + v) * 3 + c) * kClipBlock; }
    __device__ __forceinline__ float get(int v, int c) const { return col[at(list, v, c)]; }
    __device__ __forceinline__ f3 vert(int v) const { return mk3(get(v, 0), get(v, 1), get(v, 2)); }
    __device__ __forceinline__ void put(int l, int v, f3 p) {
        if (v >= kClipVerts) return;  // (cannot happen: at most 9 vertices)
        col[at(l, v, 0)] = p.x;
        col[at(l, v, 1)] = p.y;
        col[at(l, v, 2)] = p.z;
    }
};

__device__ __forceinline__ float f3c(const f3& v, int a) { return a == 0 ? v.x : (a == 1 ? v.y : v.z); }
__device__ __forceinline__ void f3set(f3& v, int a, float x) {
    if (a == 0) v.x = x;
    else if (a == 1) v.y = x;
    else v.z = x;
}

// Sutherland-Hodgman step: the list clipped by the plane x[axis] = val, keeping the side
// where (x[axis] - val) * sense >= 0, into the lane's other list.  A list that lies on that side
// stays as it is: most planes cut few of a wave's triangles, and a step without a cut costs its
// test only (k_clip in the 1.03M-triangle build, 26 levels: 527 -> 412 us, with the vertex loads a
// step ahead and the node's words in the job).
template <int axis>
__device__ __forceinline__ void clip_segments(ClipLists& L, float val, float sense) {
    const int n = min(L.n, kClipVerts);
    bool out = false;
    for (int i = 0; i < n; ++i) out |= !((L.get(i, axis) - val) * sense >= 0.0f);
    if (!out) return;
    const f3 first = L.vert(0);
    f3 a = first, next = L.vert(min(1, n - 1));
    bool ins = (f3c(a, axis) - val) * sense >= 0.0f;
    const int to = L.list ^ 1;
    int m = 0;
    for (int i = 0; i < n; ++i) {
        const f3 b = (i + 1 == n) ? first : next;
        next = L.vert(min(i + 2, n - 1));
        const bool ine = (f3c(b, axis) - val) * sense >= 0.0f;
        if (ins != ine) {
            float t = (val - f3c(a, axis)) / (f3c(b, axis) - f3c(a, axis));
            f3 h = mk3(a.x + t * (b.x - a.x), a.y + t * (b.y - a.y), a.z + t * (b.z - a.z));
            f3set(h, axis, val);
            L.put(to, m++, h);
        }
        if (ine) L.put(to, m++, b);
        a = b;
        ins = ine;
    }
    L.list = to;
    L.n = m;
}

// Clipped bounds of a straddling triangle inside a child box, padded outward by 2^-20 of
// the largest magnitude involved, clamped to the child box and to the previous bounds.
// col: this lane's LDS column (2 * kClipVerts * 3 words at stride kClipBlock).
__device__ void clip_bounds(const Geometry& G, uint32_t idx, float4& lo, float4& hi, const float4& bmin,
                            const float4& bmax, __attribute__((address_space(3))) float* col) {
    ClipLists L;
    L.col = col;
    L.list = 0;
    L.n = 3;
    const float4 v0 = G.v0[idx], v1 = G.v1[idx], v2 = G.v2[idx];
    L.put(0, 0, xyz(v0));
    L.put(0, 1, xyz(v1));
    L.put(0, 2, xyz(v2));
    if (lo.x != hi.x) {
        clip_segments<0>(L, bmin.x, 1.0f);
        clip_segments<0>(L, bmax.x, -1.0f);
    }
    if (lo.y != hi.y) {
        clip_segments<1>(L, bmin.y, 1.0f);
        clip_segments<1>(L, bmax.y, -1.0f);
    }
    if (lo.z != hi.z) {
        clip_segments<2>(L, bmin.z, 1.0f);
        clip_segments<2>(L, bmax.z, -1.0f);
    }
    const int na = min(L.n, kClipVerts);
    for (int ax = 0; ax < 3; ++ax) {
        float l, h;
        float bl = f4c(bmin, ax), bh = f4c(bmax, ax);
        if (na == 0) {
            l = f4c(lo, ax);
            h = f4c(hi, ax);
        } else {
            l = kInf;
            h = -kInf;
            for (int i = 0; i < na; ++i) {
                l = fminf(L.get(i, ax), l);
                h = fmaxf(L.get(i, ax), h);
            }
            float m = fmaxf(fmaxf(fabsf(l), fabsf(h)), fmaxf(fabsf(bl), fabsf(bh)));
            float pad = m * (1.0f / 1048576.0f);
            l = l - pad;
            h = h + pad;
        }
        l = fmaxf(l, bl);
        h = fminf(h, bh);
        l = fmaxf(l, f4c(lo, ax));
        h = fminf(h, f4c(hi, ax));
        f4set(lo, ax, canon(l));
        f4set(hi, ax, canon(h));
    }
}
// ---------------------------------------------------------------------------------------
// large-node stage
// ---------------------------------------------------------------------------------------
// Elements of an active node fill consecutive slots from a multiple of 64 on, so every wave of
// 64 slots belongs to one node: its values are wave-uniform, and a stable partition needs a
// prefix sum over waves (one packed word each), not over elements.  The element record is its
// lower bound with the index in .w and, for triangles, the upper bound.  A level is four launches
// (three for points):
//   k_count     classifies every element, one packed count per wave, summed per chunk of 64 waves;
//   k_children  per node: prefix of its chunks' sums, the children's places and build nodes;
//   k_scatter   classifies again, writes every element into its children (a wave sums the counts
//               of its chunk before it) and accumulates the next level's tight bounds;
//   k_clip      bounds of straddling triangles, from a queue.
// Places are handed out by atomics, aggregated per workgroup, so nodes and small roots lie in an
// arbitrary order (the tree does not depend on it: a node's elements keep theirs, and the final
// addresses come from the layout).  All counts stay on the device: a launch reads the level's
// (nodes, waves) from the level table, an empty level returns at once, and whatever would
// outgrow a buffer sets kErrRoom instead, after which every later kernel returns.
// Measured against one launch per step over chunk lists, element flags and three-pass scans (16
// launches a level and a host synchronisation): 1.03M triangles 5.6 -> 2.6 ms, 1M photons 3.5 ->
// 1.3 ms, 3001 triangles 1.34 -> 0.53 ms, 32 scenes' triangle and photon trees recorded 4.0 -> 1.75
// ms.

// Device words of a build: totals, then the level table.
enum : uint32_t {
    W_ERR = 0,
    W_MAXLEVEL,    // deepest build node
    W_SMALL_OVF,   // small roots whose subtree outgrew its staging area
    W_ERRLEVEL,    // with kErrRoom: the level that outgrew a buffer
    W_NBN = 4,     // build nodes, elements of large-stage leaves: one 64-bit word
    W_LL = 5,
    W_NSE = 6,     // small-root elements, small roots: one 64-bit word
    W_NSMALL = 7,
    // per level: waves, nodes (one 64-bit word), clip jobs, 0 (another), W_NBN .. W_NSMALL before it
    W_LEVELS = 8,
};
constexpr uint32_t kLevelWords = 8;
constexpr uint32_t kLevels = MNRT_MAX_LEVEL + 2;  // every level's nodes are deeper than the last's
constexpr uint32_t kWords = W_LEVELS + kLevelWords * (kLevels + 1);

constexpr uint32_t kErrRoom = 64u;          // a buffer was outgrown
constexpr uint32_t kErrLevels = 128u;       // active nodes left after the last recorded level
constexpr uint32_t kErrOutputRoom = 256u;   // the trees outgrew the output arrays
constexpr uint32_t kErrLayoutDepth = 512u;  // a leaf deeper than a recording promises (kLayoutSpareLevels)

struct BuildCaps {
    uint32_t na;     // active nodes of a level
    uint32_t nw;     // waves of a level (64 slots each)
    uint32_t bn;     // build nodes
    uint32_t small;  // small roots
    uint32_t se;     // small-root elements
    uint32_t ll;     // elements of large-stage leaves
};

// An active node: 18 of 32 words, which a wave loads at once, a word per lane.  tb: tight bounds,
// the minima of fenc(lo) and of ~fenc(hi).
struct alignas(128) NodeRec {
    float lo[3], hi[3];
    uint32_t first, cnt, level, bn, scene;
    uint32_t base;  // of the scene's elements in the input
    uint32_t tb[6];
    uint32_t pad[14];
};
static_assert(sizeof(NodeRec) == 128, "one line");
enum : uint32_t { ND_LO = 0, ND_HI = 3, ND_FIRST = 6, ND_CNT, ND_LEVEL, ND_BN, ND_SCENE, ND_BASE, ND_TB = 12, ND_WORDS = 18 };

// Element arrays: lower bound and original index (.w), upper bound; wnode: active node of every
// wave.
struct ElemView {
    float4* lo;
    float4* hi;
    uint32_t* wnode;
};

// What k_children decided about a node: child 0 and 1 as CH_*, first destination (CH_LEAF: first
// copied element) and next-level node, and the box after the empty-space cuts.
enum : uint32_t { CH_DEAD = 0, CH_SMALL, CH_LARGE, CH_LEAF };
struct alignas(64) SplitRec {
    uint32_t axis;
    float split;
    uint32_t type[2], at[2], to[2];
    float lo[3];
    uint32_t base;  // of the scene's elements in the input
    float hi[3];
    uint32_t job;  // first clip job
};
static_assert(sizeof(SplitRec) == 64, "one line");

// Everything the level kernels work on.
struct LevelArgs {
    uint32_t* W;
    uint32_t level;
    BuildCaps cap;
    float ratio;
    uint32_t small_max;
    NodeRec *A, *An;
    ElemView E, Nx, Sm;
    uint32_t* wc;  // per wave: left, right and straddling counts, a byte each
    unsigned long long *cs, *csn;  // sums per chunk (chunk_of) of this level and the next
    uint4* coff;   // per chunk: elements of its node before it, left and right; its first clip job
    SplitRec* P;
    SmallRec* S;
    BnRec* B;
    uint32_t* ll_idx;
    uint4* q;      // clip jobs, one per straddling element: slot, destinations left and right, node
};

// Chunks: 64 consecutive waves of a node, counted from its first.  Nodes and their waves are handed
// out together, so a later node's waves come later, and chunk w0 / 64 + p on belong to node p alone.
__host__ __device__ inline uint64_t chunks_for(uint64_t nw, uint64_t na) { return nw / 64u + na + 1u; }
__device__ __forceinline__ uint32_t chunk_of(uint32_t p, uint32_t w0, uint32_t w) { return (w0 >> 6) + p + ((w - w0) >> 6); }
// A chunk's sums: left, right and straddling counts (at most 4096 each).
constexpr uint32_t kSumBits = 21u;
__device__ __forceinline__ uint32_t sum_part(unsigned long long v, uint32_t k) {
    return (uint32_t)(v >> (kSumBits * k)) & ((1u << kSumBits) - 1u);
}

__device__ __forceinline__ uint32_t level_waves(const LevelArgs& L) {
    return L.W[W_ERR] != 0u ? 0u : min(L.W[W_LEVELS + kLevelWords * L.level], L.cap.nw);
}
__device__ __forceinline__ uint32_t level_nodes(const LevelArgs& L) {
    return L.W[W_ERR] != 0u ? 0u : min(L.W[W_LEVELS + kLevelWords * L.level + 1], L.cap.na);
}

// Empty-space cuts then the spatial median split (kernel_CanCutOffEmptySpace,
// kernel_EmptySpaceCutting, kernel_SplitLargeNodes; kdtree.cu:467-682).  Sides are cut in
// the reference's order (min x, y, z, then max x, y, z); each cut turns the node into an
// inner node with an empty leaf and a tighter copy.  The median splits the longest axis
// of the cut box, ties to the lower axis.
struct Plan {
    float lo[3], hi[3];  // the box after the cuts
    float tight[6];
    uint32_t cuts;   // sides that are cut, one bit each
    uint32_t level;  // of the node that is split
    uint32_t axis;
    float split;
    bool leaf;  // level cap reached: the node is a leaf with its elements
};

// w: this lane's word of the node record.  Whole wave; the result is uniform.
__device__ __forceinline__ uint32_t rec_word(uint32_t w, uint32_t i) {
    return (uint32_t)__builtin_amdgcn_readlane((int)w, (int)i);
}
__device__ __forceinline__ uint32_t load_rec(const NodeRec* A, uint32_t p, uint32_t lane) {
    return ((const uint32_t*)(A + p))[min(lane, (uint32_t)ND_WORDS - 1u)];
}

__device__ __forceinline__ Plan plan_node(uint32_t w, float ratio) {
    Plan R;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        R.lo[k] = __uint_as_float(rec_word(w, ND_LO + k));
        R.hi[k] = __uint_as_float(rec_word(w, ND_HI + k));
    }
    R.level = rec_word(w, ND_LEVEL);
    R.cuts = 0;
#pragma unroll
    for (int side = 0; side < 6; ++side) {
        const int ax = side % 3;
        const bool is_max = side >= 3;
        const uint32_t t = rec_word(w, ND_TB + side);
        R.tight[side] = fdec(is_max ? ~t : t);
        if (R.level >= MNRT_MAX_LEVEL) continue;
        const float total = R.hi[ax] - R.lo[ax];
        const float empty = is_max ? R.hi[ax] - R.tight[side] : R.tight[side] - R.lo[ax];
        if (!(empty > total * ratio)) continue;
        R.cuts |= 1u << side;
        ++R.level;
        if (is_max) R.hi[ax] = R.tight[side];
        else R.lo[ax] = R.tight[side];
    }
    R.leaf = R.level >= MNRT_MAX_LEVEL;
    const float ex = R.hi[0] - R.lo[0], ey = R.hi[1] - R.lo[1], ez = R.hi[2] - R.lo[2];
    R.axis = 0;
    float emax = ex, lo = R.lo[0], hi = R.hi[0];
    if (ey > emax) { R.axis = 1; emax = ey; lo = R.lo[1]; hi = R.hi[1]; }
    if (ez > emax) { R.axis = 2; lo = R.lo[2]; hi = R.hi[2]; }
    R.split = lo + 0.5f * (hi - lo);
    R.axis = uniform(R.axis);
    R.cuts = uniform(R.cuts);
    R.level = uniform(R.level);
    return R;
}

// Clears a build's words and sets its first level (na nodes in nw waves), small roots and build
// nodes; the scenes' tight bounds start empty, their deepest levels and the first level's chunk sums
// at 0.
__global__ __launch_bounds__(256) void k_build_init(uint32_t* __restrict__ W, uint32_t na, uint32_t nw, uint32_t nsmall,
                                                    uint32_t nse, uint32_t nscenes, uint32_t* __restrict__ stb,
                                                    uint32_t* __restrict__ maxlvl,
                                                    unsigned long long* __restrict__ cs) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kWords)
        W[i] = i == W_NBN ? nscenes : i == W_NSE ? nse : i == W_NSMALL ? nsmall : i == W_LEVELS ? nw
               : i == W_LEVELS + 1 ? na : 0u;
    for (uint32_t j = i; j < 6 * nscenes; j += gridDim.x * blockDim.x) stb[j] = 0xFFFFFFFFu;
    for (uint32_t j = i; j < nscenes; j += gridDim.x * blockDim.x) maxlvl[j] = 0u;
    for (uint32_t j = i; j < chunks_for(nw, na); j += gridDim.x * blockDim.x) cs[j] = 0ull;
}

// Puts a build back to where it was before `level`, which outgrew a buffer: totals, the level's clip
// jobs, the next level, and the level's chunk sums.
__global__ __launch_bounds__(256) void k_level_again(uint32_t* __restrict__ W, uint32_t level, uint64_t nchunks,
                                                     unsigned long long* __restrict__ cs) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t* const T = W + W_LEVELS + kLevelWords * level;
    if (i < 4u) {
        W[W_NBN + i] = T[4 + i];
        T[kLevelWords + i] = 0u;
    }
    if (i < 2u) T[2 + i] = 0u;
    if (i == 0u) W[W_ERR] = 0u;
    for (uint64_t j = i; j < nchunks; j += (uint64_t)gridDim.x * blockDim.x) cs[j] = 0ull;
}

// Per-scene placement decided on the host: an active (large) root or a small root, its index in
// that list and its first slot there.
struct RootPlan {
    const uint32_t* kind;  // 0 active, 1 small
    const uint32_t* index;
    const uint32_t* off;
};

__device__ __forceinline__ void tight_words(const float4& lo, const float4& hi, uint32_t (&v)[6]) {
    v[0] = fenc(lo.x);
    v[1] = fenc(lo.y);
    v[2] = fenc(lo.z);
    v[3] = ~fenc(hi.x);
    v[4] = ~fenc(hi.y);
    v[5] = ~fenc(hi.z);
}

// Adds the lanes' tight words to their targets tb[stride * to ..] (kNone: none), lanes that share
// a target reduced first: one atomic per component and distinct target.  Whole wave.
__device__ __forceinline__ void tight_by_key(uint32_t to, const uint32_t (&v)[6], uint32_t* __restrict__ tb,
                                             uint32_t stride, uint32_t lane) {
    for (uint64_t m = ballot(to != kNone); m != 0ull;) {
        const uint32_t t = (uint32_t)__builtin_amdgcn_readlane((int)to, (int)__builtin_ctzll(m));
        const bool mine = to == t;
        uint32_t best = ~0u;
#pragma unroll
        for (uint32_t k = 0; k < 6; ++k) {
            const uint32_t r = wave_min_u32(mine ? v[k] : ~0u);
            if (lane == k) best = r;
        }
        if (lane < 6u) atomicMin(&tb[(size_t)stride * t + lane], best);
        m &= ~ballot(mine);
    }
}

// Input elements: bounds, placed with their scene's root (elements of a small scene with the small
// roots), and the scenes' tight bounds.  A workgroup takes kInitPer elements per thread, so a
// scene's bounds cost one atomic per component and workgroup unless the workgroup spans scenes.
constexpr uint32_t kInitBlock = 1024, kInitPer = 4;

__global__ __launch_bounds__(kInitBlock) void k_init_elems(Geometry G, uint32_t n, RootPlan R, ElemView E, ElemView Sm,
                                                           uint32_t* __restrict__ stb) {
    __shared__ uint32_t s_min[kInitBlock / 64][6];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t b0 = blockIdx.x * (kInitBlock * kInitPer), b1 = min(b0 + kInitBlock * kInitPer, n);
    const uint32_t s0 = scene_of(G.base, G.num_scenes, b0);
    const bool one = b1 <= G.base[s0 + 1];  // the workgroup's elements are one scene's
    uint32_t acc[6] = {~0u, ~0u, ~0u, ~0u, ~0u, ~0u};
    for (uint32_t t = 0; t < kInitPer; ++t) {
        const uint32_t i = b0 + t * kInitBlock + threadIdx.x;
        uint32_t s = kNone;
        uint32_t v[6] = {~0u, ~0u, ~0u, ~0u, ~0u, ~0u};
        if (i < b1) {
            s = one ? s0 : scene_of(G.base, G.num_scenes, i);
            const float4 a = G.v0[i];
            float4 lo, hi;
            if (G.kind == MNRT_KIND_TRI) {
                const float4 b = G.v1[i], c = G.v2[i];
                lo = make_float4(canon(fminf(a.x, fminf(b.x, c.x))), canon(fminf(a.y, fminf(b.y, c.y))),
                                 canon(fminf(a.z, fminf(b.z, c.z))), 0.0f);
                hi = make_float4(canon(fmaxf(a.x, fmaxf(b.x, c.x))), canon(fmaxf(a.y, fmaxf(b.y, c.y))),
                                 canon(fmaxf(a.z, fmaxf(b.z, c.z))), 0.0f);
            } else {
                lo = hi = make_float4(canon(a.x), canon(a.y), canon(a.z), 0.0f);
            }
            const uint32_t local = i - G.base[s], d = R.off[s] + local;
            const bool small = R.kind[s] != 0u;
            const ElemView& D = small ? Sm : E;
            D.lo[d] = make_float4(lo.x, lo.y, lo.z, __uint_as_float(local));
            if (G.kind == MNRT_KIND_TRI) D.hi[d] = hi;
            if (!small && (d & 63u) == 0u) E.wnode[d >> 6] = R.index[s];
            tight_words(lo, hi, v);
        }
        if (one) {
#pragma unroll
            for (int k = 0; k < 6; ++k) acc[k] = min(acc[k], v[k]);
        } else {
            tight_by_key(s, v, stb, 6u, lane);
        }
    }
    if (!one) return;  // uniform per workgroup
#pragma unroll
    for (int k = 0; k < 6; ++k) acc[k] = wave_min_u32(acc[k]);
    if (lane == 0)
        for (int k = 0; k < 6; ++k) s_min[wave][k] = acc[k];
    __syncthreads();
    if (threadIdx.x < 6) {
        uint32_t m = ~0u;
        for (uint32_t w = 0; w < kInitBlock / 64; ++w) m = min(m, s_min[w][threadIdx.x]);
        atomicMin(&stb[6 * s0 + threadIdx.x], m);
    }
}

// Root boxes (given, or the tight bounds of the scene's elements; (+max, -max) for an
// empty scene) and the root entries of the active / small lists.
__global__ __launch_bounds__(256) void k_roots_setup(uint32_t nscenes, const uint32_t* __restrict__ base,
                                                     const uint32_t* __restrict__ stb, const float* __restrict__ given,
                                                     RootPlan R, NodeRec* A, SmallRec* S, BnRec* B,
                                                     float* __restrict__ out_box) {
    uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nscenes) return;
    const uint32_t cnt = base[s + 1] - base[s];
    float4 lo, hi;
    if (given) {
        lo = make_float4(canon(given[6 * s + 0]), canon(given[6 * s + 1]), canon(given[6 * s + 2]), 0.0f);
        hi = make_float4(canon(given[6 * s + 3]), canon(given[6 * s + 4]), canon(given[6 * s + 5]), 0.0f);
    } else if (cnt == 0) {
        lo = make_float4(kInf, kInf, kInf, 0.0f);
        hi = make_float4(-kInf, -kInf, -kInf, 0.0f);
    } else {
        lo = make_float4(fdec(stb[6 * s]), fdec(stb[6 * s + 1]), fdec(stb[6 * s + 2]), 0.0f);
        hi = make_float4(fdec(~stb[6 * s + 3]), fdec(~stb[6 * s + 4]), fdec(~stb[6 * s + 5]), 0.0f);
    }
    const uint32_t i = R.index[s];
    const bool small = R.kind[s] != 0u;
    put4(&B[s], 0, small ? BN_SMALL : BN_PENDING, 0u, 0u, 0u);
    put4(&B[s], 1, 0u, i, 0u, s);
    put4(&B[s], 2, kNone, 0u, 0u, 0u);
    put4(&B[s], 3, 0u, 0u, 0u, 0u);
    if (!small) {
        NodeRec& a = A[i];
        a.lo[0] = lo.x; a.lo[1] = lo.y; a.lo[2] = lo.z;
        a.hi[0] = hi.x; a.hi[1] = hi.y; a.hi[2] = hi.z;
        a.first = R.off[s];
        a.cnt = cnt;
        a.level = 0;
        a.bn = s;
        a.scene = s;
        a.base = base[s];
        for (int k = 0; k < 6; ++k) a.tb[k] = stb[6 * s + k];
    } else {
        put4(&S[i], 0, R.off[s], cnt, 0u, s);
        put4(&S[i], 1, __float_as_uint(lo.x), __float_as_uint(lo.y), __float_as_uint(lo.z), s);
        put4(&S[i], 2, __float_as_uint(hi.x), __float_as_uint(hi.y), __float_as_uint(hi.z), 0u);
    }
    out_box[6 * s + 0] = lo.x;
    out_box[6 * s + 1] = lo.y;
    out_box[6 * s + 2] = lo.z;
    out_box[6 * s + 3] = hi.x;
    out_box[6 * s + 4] = hi.y;
    out_box[6 * s + 5] = hi.z;
}

// Left, right and straddling counts of every wave, and their sums per chunk.  Bound by reading the elements (33 MB a
// level at 1.03M triangles: 10-12 us).  The wave makes its node's plan itself: about 100 instructions on
// values it shares, less than another launch and its latency.
constexpr uint32_t kCountBlock = 1024, kCountWaves = kCountBlock / 64;

template <int kKind>
__global__ __launch_bounds__(kCountBlock) __attribute__((amdgpu_waves_per_eu(8))) void k_count(LevelArgs L) {
    // two sets, used in turn: one barrier a step
    __shared__ unsigned long long s_sum[2][kCountWaves];
    __shared__ uint32_t s_chunk[2][kCountWaves];
    const uint32_t nw = level_waves(L), lane = threadIdx.x & 63u, wave = uniform(threadIdx.x >> 6);
    // the totals before the level, for a build that goes on from here in larger buffers
    if (blockIdx.x == 0 && threadIdx.x < 4u && L.W[W_ERR] == 0u)
        L.W[W_LEVELS + kLevelWords * L.level + 4 + threadIdx.x] = L.W[W_NBN + threadIdx.x];
    uint32_t set = 0;
    for (uint32_t w0 = blockIdx.x * kCountWaves; w0 < nw; w0 += gridDim.x * kCountWaves) {  // uniform per workgroup
        const uint32_t w = w0 + wave;
        uint32_t c = 0, chunk = kNone;
        if (w < nw) {
            const uint32_t p = uniform(L.E.wnode[w]), e = 64u * w + lane;
            const float4 lo = L.E.lo[e];  // (slots past the node's last element hold anything)
            const float4 hi = (kKind == MNRT_KIND_TRI) ? L.E.hi[e] : lo;
            const uint32_t nd = load_rec(L.A, p, lane);
            const Plan R = plan_node(nd, L.ratio);
            bool l = false, r = false, both = false;
            if (!R.leaf && e - rec_word(nd, ND_FIRST) < rec_word(nd, ND_CNT)) {
                classify(kKind, __float_as_uint(lo.w), lo, hi, R.axis, R.split, l, r);
                both = straddles(kKind, lo, hi, R.axis, R.split);
            }
            c = (uint32_t)__popcll(ballot(l)) | (uint32_t)__popcll(ballot(r)) << 8 | (uint32_t)__popcll(ballot(both)) << 16;
            chunk = chunk_of(p, rec_word(nd, ND_FIRST) >> 6, w);
            if (lane == 0) L.wc[w] = c;
        }
        if (lane == 0) {
            s_chunk[set][wave] = chunk;
            s_sum[set][wave] = (unsigned long long)(c & 0xFFu) | (unsigned long long)(c >> 8 & 0xFFu) << kSumBits |
                               (unsigned long long)(c >> 16) << (2u * kSumBits);
        }
        __syncthreads();
        if (threadIdx.x < kCountWaves) {  // one atomic per run of waves of one chunk
            const uint32_t i = threadIdx.x, ch = s_chunk[set][i];
            if (ch != kNone && (i == 0u || s_chunk[set][i - 1u] != ch)) {
                unsigned long long v = s_sum[set][i];
                for (uint32_t j = i + 1u; j < kCountWaves && s_chunk[set][j] == ch; ++j) v += s_sum[set][j];
                atomicAdd(&L.cs[ch], v);
            }
        }
        set ^= 1u;
    }
}

// Children of 16 nodes per workgroup step, one wave per node.  Bound by latency: the node's
// record, its chunk sums, one atomic for the places of the 16 nodes' children (a lane per 64-bit
// total) and the records, written by a lane each, every record a line or part of one.  With
// column arrays, a field per store, a serial sum over the 16 nodes and one lane writing, and each
// node's sum over all its waves (16 k for the root), the 26 levels of 1.03M triangles took 493 us
// (35 at the root, 14 between); now 248 (6.5 and 9).
constexpr uint32_t kChildBlock = 1024, kChildNodes = kChildBlock / 64;
__global__ __launch_bounds__(kChildBlock) __attribute__((amdgpu_waves_per_eu(8))) void k_children(LevelArgs L) {
    __shared__ uint32_t s_need[kChildNodes][8], s_base[kChildNodes][8];
    __shared__ uint32_t s_na;  // one read for the workgroup: others may set the error while it runs
    if (threadIdx.x == 0) s_na = level_nodes(L);
    __syncthreads();
    const uint32_t na = uniform(s_na), lane = threadIdx.x & 63u, wave = uniform(threadIdx.x >> 6);
    for (uint32_t p0 = blockIdx.x * kChildNodes; p0 < na; p0 += gridDim.x * kChildNodes) {  // uniform per workgroup
        const uint32_t p = p0 + wave;
        const bool live = p < na;
        Plan R{};
        uint32_t nd = 0, n[2] = {0u, 0u}, nq = 0;
        uint32_t type[2] = {CH_DEAD, CH_DEAD};
        bool leaf = false;
        uint32_t m = 0;
        // what the node asks for, lane by lane: build nodes, leaf elements, small elements and
        // roots, next-level waves and nodes, clip jobs, 0
        uint32_t need = 0;
        if (live) {
            nd = load_rec(L.A, p, lane);
            m = rec_word(nd, ND_CNT);
            // the chunks' offsets
            const uint32_t c0 = chunk_of(p, rec_word(nd, ND_FIRST) >> 6, rec_word(nd, ND_FIRST) >> 6), nc = (m + 4095u) >> 12;
            unsigned long long c = lane < nc ? L.cs[c0 + lane] : 0ull;
            for (uint32_t b = 0; b < nc; b += 64u) {
                const uint32_t i = b + lane;
                const uint32_t v[3] = {sum_part(c, 0), sum_part(c, 1), sum_part(c, 2)};
                if (i + 64u < nc) c = L.cs[c0 + i + 64u];
                else c = 0ull;
                uint32_t incl[3];
#pragma unroll
                for (uint32_t k = 0; k < 3; ++k) incl[k] = wave_scan_u32(v[k]);
                if (i < nc)
                    L.coff[c0 + i] = make_uint4(n[0] + incl[0] - v[0], n[1] + incl[1] - v[1], nq + incl[2] - v[2], 0u);
                n[0] += rec_word(incl[0], 63u);
                n[1] += rec_word(incl[1], 63u);
                nq += rec_word(incl[2], 63u);
            }
            R = plan_node(nd, L.ratio);
            // no progress: every element went to both children
            leaf = R.leaf || (n[0] == m && n[1] == m);
            uint32_t v[7] = {2u * (uint32_t)__popc(R.cuts) + (leaf ? 0u : 2u), 0u, 0u, 0u, 0u, 0u, leaf ? 0u : nq};
            if (leaf) {
                type[0] = CH_LEAF;
                v[1] = m;
            } else {
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    // small iff count <= smallNodeMax (kernel_MarkSmallNodes, kdtree.cu:849-875)
                    type[s] = n[s] <= L.small_max ? CH_SMALL : CH_LARGE;
                    if (type[s] == CH_SMALL) {
                        v[2] += n[s];
                        v[3] += 1u;
                    } else {
                        v[4] += (n[s] + 63u) >> 6;
                        v[5] += 1u;
                    }
                }
            }
#pragma unroll
            for (uint32_t k = 0; k < 7; ++k)
                if (lane == k) need = v[k];
        }
        if (lane < 8u) s_need[wave][lane] = need;
        __syncthreads();
        if (wave == 0) {
            // lane 16 k + i: 64-bit total k (build nodes | leaf elements, small elements | small
            // roots, next waves | next nodes, clip jobs) of node i
            const uint32_t i = lane & 15u, k = lane >> 4;
            const uint32_t a = s_need[i][2u * k], b = s_need[i][2u * k + 1u];
            const uint32_t ia = row_scan_u32(a), ib = row_scan_u32(b);
            unsigned long long at = 0;
            if (i == 15u) {
                const uint32_t word = k == 0u ? W_NBN : k == 1u ? W_NSE
                                      : k == 2u ? W_LEVELS + kLevelWords * (L.level + 1u) : W_LEVELS + kLevelWords * L.level + 2u;
                if ((ia | ib) != 0u) at = atomicAdd((unsigned long long*)&L.W[word], (unsigned long long)ib << 32 | ia);
                const uint32_t ca = k == 0u ? L.cap.bn : k == 1u ? L.cap.se : L.cap.nw;
                const uint32_t cb = k == 0u ? L.cap.ll : k == 1u ? L.cap.small : L.cap.na;
                if (k < 3u && ((at & 0xFFFFFFFFull) + ia > ca || (at >> 32) + ib > cb)) {
                    L.W[W_ERRLEVEL] = L.level;
                    atomicOr(&L.W[W_ERR], kErrRoom);
                    at = ~0ull;
                }
            }
            const uint32_t lo = row_last((uint32_t)at), hi = row_last((uint32_t)(at >> 32));
            const bool none = ballot(lo == kNone && hi == kNone) != 0ull;  // nothing of these nodes is written
            s_base[i][2u * k] = none ? kNone : lo + ia - a;
            s_base[i][2u * k + 1u] = none ? kNone : hi + ib - b;
        }
        __syncthreads();
        const uint32_t base = s_base[wave][min(lane, 7u)];  // (rewritten after the next step's barrier)
        if (!live || rec_word(base, 0u) == kNone) continue;
        const uint32_t scene = rec_word(nd, ND_SCENE), bn0 = rec_word(nd, ND_BN);
        const uint32_t id0 = rec_word(base, 0u), ncuts = (uint32_t)__popc(R.cuts), level0 = rec_word(nd, ND_LEVEL);
        const uint32_t cur = ncuts ? id0 + 2u * ncuts - 1u : bn0, id = id0 + 2u * ncuts;
        const uint32_t tw = __shfl(nd, ND_TB + min(lane, 5u), 64);
        // lanes 0..5: the cuts
        if (lane < 6u && (R.cuts >> lane & 1u)) {
            const uint32_t k = (uint32_t)__popc(R.cuts & ((1u << lane) - 1u)), above = k ? id0 + 2u * k - 1u : bn0;
            const uint32_t empty = id0 + 2u * k, cont = empty + 1u, lv = level0 + k + 1u;
            const bool is_max = lane >= 3u;
            put4(&L.B[above], 0, is_max ? lane - 3u : lane, __float_as_uint(fdec(is_max ? ~tw : tw)),
                 is_max ? cont : empty, is_max ? empty : cont);
            put4(&L.B[empty], 0, BN_LEAF, 0u, 0u, 0u);
            put4(&L.B[empty], 1, lv, 0u, 0u, scene);
            put4(&L.B[empty], 2, above | kCutParent, 0u, 1u, 0u);
            put4(&L.B[cont], 1, lv, 0u, 0u, scene);
            put4(&L.B[cont], 2, above | kCutParent, 0u, 0u, 0u);
            put4(&L.B[cont], 3, 0u, 0u, 0u, 0u);
        }
        const uint32_t bx[3] = {__float_as_uint(R.lo[0]), __float_as_uint(R.lo[1]), __float_as_uint(R.lo[2])};
        const uint32_t bh[3] = {__float_as_uint(R.hi[0]), __float_as_uint(R.hi[1]), __float_as_uint(R.hi[2])};
        if (leaf) {
            if (lane == 0) {
                const uint32_t at = rec_word(base, 1u);
                put4(&L.B[cur], 0, BN_LEAF, 0u, 0u, 0u);
                L.B[cur].aux = at;
                L.B[cur].cnt = m;
                put4(&L.P[p], 0, 0u, 0u, CH_LEAF, CH_DEAD);
                put4(&L.P[p], 1, at, 0u, 0u, 0u);
            }
            continue;
        }
        const uint32_t spl = __float_as_uint(R.split);
        auto clear_sums = [&](uint32_t to, uint32_t at, uint32_t cnt) {
            for (uint32_t i = lane; i < (cnt + 4095u) >> 12; i += 64u) L.csn[(at >> 12) + to + i] = 0ull;
        };
        const uint32_t se = rec_word(base, 2u), sr = rec_word(base, 3u), nw0 = rec_word(base, 4u), nx = rec_word(base, 5u);
        const bool small0 = type[0] == CH_SMALL, small1 = type[1] == CH_SMALL;
        // places of the two children: the left one's first
        const uint32_t at0 = small0 ? se : 64u * nw0, at1 = small1 ? se + (small0 ? n[0] : 0u)
                                                                   : 64u * (nw0 + (small0 ? 0u : (n[0] + 63u) >> 6));
        const uint32_t to0 = small0 ? sr : nx, to1 = small1 ? sr + (small0 ? 1u : 0u) : nx + (small0 ? 0u : 1u);
        if (!small0) clear_sums(to0, at0, n[0]);
        if (!small1) clear_sums(to1, at1, n[1]);
        if (lane == 2u) {
            put4(&L.P[p], 0, R.axis, spl, type[0], type[1]);
            put4(&L.P[p], 1, at0, at1, to0, to1);
            put4(&L.P[p], 2, bx[0], bx[1], bx[2], rec_word(nd, ND_BASE));
            put4(&L.P[p], 3, bh[0], bh[1], bh[2], rec_word(base, 6u));
            put4(&L.B[cur], 0, R.axis, spl, id, id + 1u);
        } else if (lane < 2u) {
            const bool right = lane == 1u, sm = right ? small1 : small0;
            const uint32_t at = right ? at1 : at0, to = right ? to1 : to0, cnt = right ? n[1] : n[0];
            const uint32_t bn = id + lane;
            uint32_t x[3], y[3];
#pragma unroll
            for (uint32_t k = 0; k < 3; ++k) {
                x[k] = right && R.axis == k ? spl : bx[k];
                y[k] = !right && R.axis == k ? spl : bh[k];
            }
            put4(&L.B[bn], 0, sm ? BN_SMALL : BN_PENDING, 0u, 0u, 0u);
            put4(&L.B[bn], 1, R.level + 1u, to, 0u, scene);
            put4(&L.B[bn], 2, cur, 0u, 0u, 0u);
            put4(&L.B[bn], 3, 0u, 0u, 0u, 0u);
            if (sm) {
                put4(&L.S[to], 0, at, cnt, R.level + 1u, bn);
                put4(&L.S[to], 1, x[0], x[1], x[2], scene);
                put4(&L.S[to], 2, y[0], y[1], y[2], 0u);
            } else {
                put4(&L.An[to], 0, x[0], x[1], x[2], y[0]);
                put4(&L.An[to], 1, y[1], y[2], at, cnt);
                put4(&L.An[to], 2, R.level + 1u, bn, scene, rec_word(nd, ND_BASE));
                put4(&L.An[to], 3, ~0u, ~0u, ~0u, ~0u);
                put4(&L.An[to], 4, ~0u, ~0u, 0u, 0u);
            }
        }
    }
}

// Scatter each element into its children: small roots append to the small-element
// buffer, large children to the next level's arrays, whose tight bounds (kernel_GenChunkAABB and
// two segmented reductions, kdtree.cu:310-445) are accumulated on the way: per wave, then per
// run of waves of one node in the workgroup, one atomic per component and run.  A straddling
// triangle's bounds in a child are its clip to the child box (kernel_PerformSplitClipping,
// kdtree_tri.cu:389-489), which k_clip computes from the queue written here, 64 to a wave
// rather than one pass of a whole wave per straddler.  Bound by memory (66 MB a level at 1.03M
// triangles: 20 us, 3.3 TB/s; 28 with one 1024-thread workgroup on a CU instead of two) and, below
// about 10^5 elements, by latency (7 us).
constexpr uint32_t kScatterBlock = 1024, kScatterWaves = kScatterBlock / 64;

template <int kKind>
__global__ __launch_bounds__(kScatterBlock) __attribute__((amdgpu_waves_per_eu(8))) void k_scatter(LevelArgs L) {
    // two sets, used in turn: one barrier a step
    __shared__ uint32_t s_tb[2][kScatterWaves][12];
    __shared__ uint32_t s_node[2][kScatterWaves];
    __shared__ uint32_t s_to[2][kScatterWaves][2];  // next-level nodes of the wave's children, or kNone
    const uint32_t nw = level_waves(L), lane = threadIdx.x & 63u, wave = uniform(threadIdx.x >> 6);
    uint32_t set = 0;
    for (uint32_t w0 = blockIdx.x * kScatterWaves; w0 < nw; w0 += gridDim.x * kScatterWaves) {  // uniform per workgroup
        const uint32_t w = w0 + wave, e = 64u * w + lane;
        uint32_t p = kNone, to[2] = {kNone, kNone}, mine = ~0u;  // mine: lane k < 12, tight word k
        if (w < nw) {
            p = uniform(L.E.wnode[w]);
            const float4 lo = L.E.lo[e];  // (slots past the node's last element hold anything)
            const float4 hi = (kKind == MNRT_KIND_TRI) ? L.E.hi[e] : lo;
            const uint32_t sp = ((const uint32_t*)(L.P + p))[lane & 15u];
            const uint32_t fc = ((const uint32_t*)(L.A + p))[ND_FIRST + (lane & 1u)];
            const uint32_t idx = __float_as_uint(lo.w), local = e - rec_word(fc, 0u);
            const bool in = local < rec_word(fc, 1u);
            const uint32_t type0 = rec_word(sp, 2u), type1 = rec_word(sp, 3u);
            if (type0 == CH_LEAF) {
                if (in) L.ll_idx[rec_word(sp, 4u) + local] = idx;
            } else if (type0 != CH_DEAD) {
                const uint32_t axis = rec_word(sp, 0u);
                const float s = __uint_as_float(rec_word(sp, 1u));
                bool go[2] = {false, false}, both = false;
                if (in) {
                    classify(kKind, idx, lo, hi, axis, s, go[0], go[1]);
                    both = straddles(kKind, lo, hi, axis, s);
                }
                // the waves of the chunk before this one
                const uint32_t wf = rec_word(fc, 0u) >> 6, ch = chunk_of(p, wf, w), wl = wf + ((w - wf) & ~63u) + lane;
                const uint32_t cw = wl < w ? L.wc[wl] : 0u;
                uint4 off = L.coff[ch];
                const uint32_t before = wave_sum_u32((cw & 0xFFu) | (cw & 0xFF00u) << 8);
                off.x += before & 0xFFFFu;
                off.y += before >> 16;
                if (kKind == MNRT_KIND_TRI) off.z += wave_sum_u32(cw >> 16);
                uint32_t v[6], dst[2];
                tight_words(lo, hi, v);
#pragma unroll
                for (int side = 0; side < 2; ++side) {
                    const bool large = (side ? type1 : type0) == CH_LARGE;
                    const uint32_t child = rec_word(sp, 6u + side);
                    dst[side] = rec_word(sp, 4u + side) + (side ? off.y : off.x) + mask_prefix(ballot(go[side]));
                    const ElemView& D = large ? L.Nx : L.Sm;
                    if (go[side] && !both) {  // (a straddler's record comes with its clip)
                        D.lo[dst[side]] = lo;
                        if (kKind == MNRT_KIND_TRI) D.hi[dst[side]] = hi;
                    }
                    if (go[side]) {
                        if (large && (dst[side] & 63u) == 0u) L.Nx.wnode[dst[side] >> 6] = child;
                    }
                    if (large) {
                        to[side] = child;
#pragma unroll
                        for (uint32_t k = 0; k < 6; ++k) {
                            const uint32_t t = wave_min_u32(go[side] && !both ? v[k] : ~0u);
                            if (lane == 6u * side + k) mine = t;
                        }
                    }
                }
                if (kKind == MNRT_KIND_TRI) {
                    const uint64_t mq = ballot(both);
                    if (both) L.q[rec_word(sp, 15u) + off.z + mask_prefix(mq)] = make_uint4(e, dst[0], dst[1], p);
                }
            }
        }
        if (lane == 0) {
            s_node[set][wave] = p;
            s_to[set][wave][0] = to[0];
            s_to[set][wave][1] = to[1];
        }
        if (lane < 12u) s_tb[set][wave][lane] = mine;
        __syncthreads();
        if (threadIdx.x < 12u * kScatterWaves) {
            const uint32_t i = threadIdx.x / 12u, k = threadIdx.x % 12u, node = s_node[set][i], t = s_to[set][i][k / 6u];
            if (t != kNone && (i == 0u || s_node[set][i - 1u] != node)) {
                uint32_t v = s_tb[set][i][k];
                for (uint32_t j = i + 1u; j < kScatterWaves && s_node[set][j] == node; ++j) v = min(v, s_tb[set][j][k]);
                if (v != ~0u) atomicMin(&L.An[t].tb[k % 6u], v);
            }
        }
        set ^= 1u;
    }
}

// The clip queue of a triangle level: two lanes per job clip its triangle to the child boxes, write
// the record at the place k_scatter found and add them to a large child's tight bounds (lanes
// that share a child reduce first).
__global__ __launch_bounds__(kClipBlock) void k_clip(LevelArgs L, Geometry G) {
    __shared__ float s_lists[2 * kClipVerts * 3 * kClipBlock];
    __attribute__((address_space(3))) float* col = (__attribute__((address_space(3))) float*)(s_lists + threadIdx.x);
    if (L.W[W_ERR] != 0u) return;
    const uint32_t nq = 2u * L.W[W_LEVELS + kLevelWords * L.level + 2], lane = threadIdx.x;
    for (uint32_t j0 = blockIdx.x * kClipBlock; j0 < nq; j0 += gridDim.x * kClipBlock) {
        const uint32_t j = j0 + lane;
        uint32_t to = kNone;
        uint32_t v[6] = {~0u, ~0u, ~0u, ~0u, ~0u, ~0u};
        if (j < nq) {
            const uint4 job = L.q[j >> 1];
            const uint32_t e = job.x, side = j & 1u;
            const uint4* P = (const uint4*)&L.P[job.w];
            const uint4 p0 = P[0], p1 = P[1], p2 = P[2], p3 = P[3];
            const uint32_t axis = p0.x, type = side ? p0.w : p0.z;
            float4 lo = L.E.lo[e], hi = L.E.hi[e];
            float4 bmin = make_float4(__uint_as_float(p2.x), __uint_as_float(p2.y), __uint_as_float(p2.z), 0.0f);
            float4 bmax = make_float4(__uint_as_float(p3.x), __uint_as_float(p3.y), __uint_as_float(p3.z), 0.0f);
            if (side == 0) f4set(bmax, axis, __uint_as_float(p0.y));
            else f4set(bmin, axis, __uint_as_float(p0.y));
            clip_bounds(G, p2.w + __float_as_uint(lo.w), lo, hi, bmin, bmax, col);
            const ElemView& D = type == CH_LARGE ? L.Nx : L.Sm;
            const uint32_t d = side ? job.z : job.y;
            D.lo[d] = lo;
            D.hi[d] = hi;
            if (type == CH_LARGE) {
                to = side ? p1.w : p1.z;
                tight_words(lo, hi, v);
            }
        }
        tight_by_key(to, v, (uint32_t*)L.An + ND_TB, sizeof(NodeRec) / 4u, lane);
    }
}

// ---- small-node stage: one wave64 per small root ----------------------------------------

// one small root per wave and one wave per workgroup: a workgroup's LDS (the candidate
// masks, about 10 KB for triangles) is released when its own root is done, not when the
// slowest of several roots is (measured: the recorded 1.03M-triangle build 4.97 -> 4.78 ms)
constexpr int kSmallWaves = 1;
constexpr int kSmallStack = MNRT_MAX_LEVEL + 4;

struct SmallStackEnt {
    uint64_t mask;
    float lo[3], hi[3];
    uint32_t lvl_ax;  // level | axis << 30 (axis: of the split whose right child this is)
    uint32_t patch;   // node whose right-child word gets this entry's address, or kNone
    __device__ uint32_t level() const { return lvl_ax & 0x3FFFFFFFu; }
    __device__ uint32_t axis() const { return lvl_ax >> 30; }
};

// Staging area of a small root with n elements: stage_mul * n + stage_add node words and
// as many references (4n + 64 by default; the environment variable MNRT_SMALL_STAGE_CAP
// = "mul,add" overrides it, so tests can force the fallback).  The subtree is written
// there with subtree-local addresses while its size is counted, then moved into place
// once the layout is known.  A subtree that does not fit (rare) is counted on without
// being written and emitted by a second pass at its final address.
struct StageCap {
    uint32_t mul, add;
    __host__ __device__ uint32_t of(uint32_t n) const { return mul * n + add; }
    // first slot of root r, whose elements start at `first` (both grow together over the roots)
    __device__ uint32_t begin(uint32_t r, uint32_t first) const { return mul * first + add * r; }
};

enum : int { kSmallStage = 0, kSmallEmit = 1 };

struct SmallOut {
    uint32_t* nsize;  // stage: nodes per small subtree
    uint32_t* rsize;  // stage: references per small subtree
    uint32_t* mlvl;   // stage: deepest level in the small subtree
    uint2* st_nodes;         // stage: node words, subtree-local addresses
    uint32_t* st_refs;       // stage: references, subtree-local
    uint32_t* st_ovf;        // stage: 1 where the subtree did not fit; emit: only these
    StageCap st_cap;
    const BnRec* bn;  // emit: subtree start address / reference base
    uint32_t* nodes;
    uint32_t* refs;
    uint32_t* W;
    uint32_t max_nodes;
    uint32_t max_refs;
    const uint32_t* node_base;  // per scene: first node / reference of its tree
    const uint32_t* ref_base;
};

// m = 2 m + (u < v) and 2 m + (u > v), u wave-uniform: the comparison's result is the carry.
__device__ __forceinline__ void shift_in_less(uint32_t& m, float u, float v) {
    asm("v_cmp_lt_f32 vcc, %1, %2\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc" : "+v"(m) : "s"(u), "v"(v) : "vcc");
}
__device__ __forceinline__ void shift_in_greater(uint32_t& m, float u, float v) {
    asm("v_cmp_gt_f32 vcc, %1, %2\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc" : "+v"(m) : "s"(u), "v"(v) : "vcc");
}
// The floats next to a finite one (+0 for either zero).
__device__ __forceinline__ float next_down(float f) {
    const uint32_t u = __float_as_uint(f);
    return __uint_as_float(f > 0.0f ? u - 1u : (f < 0.0f ? u + 1u : 0x80000001u));
}
__device__ __forceinline__ float next_up(float f) {
    const uint32_t u = __float_as_uint(f);
    return __uint_as_float(f > 0.0f ? u + 1u : (f < 0.0f ? u - 1u : 1u));
}

// Bound by instruction issue: 7.0 k vector instructions per root of the 1.03M-triangle build (42 k
// roots, 439 us; 586 us with the masks built candidate by candidate, both children through the stack and
// every node's candidates evaluated).
// kMode kSmallStage: subtree sizes, and the subtree written to its staging area while it
// fits; kSmallEmit: written at its final address (only roots with st_ovf set
// when st_ovf is given).
// The element kind is a template argument so that LDS holds what the kind needs: point
// elements have no upper bounds and 3n candidates (triangles: 6n), which halves the mask
// arrays and lets more waves share a CU.
template <int kMode, int kKind>
__global__ __launch_bounds__(64 * kSmallWaves) void k_small(DN dnsmall, const SmallRec* __restrict__ S,
                                                            ElemView Sm,
                                                            const float* __restrict__ scene_qr, SmallOut O) {
    constexpr int kind = kKind;
    // candidate slots of an element: (isMax, axis), slot = isMax * 3 + axis
    constexpr int kSlots = (kKind == MNRT_KIND_TRI) ? 6 : 3;
    __shared__ SmallStackEnt s_stack[kSmallWaves][kSmallStack];

    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const uint32_t r = blockIdx.x * kSmallWaves + wave;
    if (r >= dnsmall.get() || O.W[W_ERR] != 0u) return;  // uniform per wave
    if (kMode == kSmallEmit && O.st_ovf && O.st_ovf[r] == 0u) return;
    SmallStackEnt* stack = s_stack[wave];

    const SmallRec root = S[r];
    const uint32_t first = root.first, n = root.cnt;
    // lane j holds element j (n <= 64)
    const bool valid = lane < n;
    float4 mlo = make_float4(0.0f, 0.0f, 0.0f, 0.0f), mhi = mlo;
    uint32_t midx = 0;
    if (valid) {
        mlo = Sm.lo[first + lane];
        mhi = (kKind == MNRT_KIND_TRI) ? Sm.hi[first + lane] : mlo;
        midx = __float_as_uint(mlo.w);
    }
    const bool mleft = plane_goes_left(midx);
    // Candidates axis-major, minimums then maximums (kernel_CreateSplitCandidates,
    // kdtree.cu:1035-1082), c = isMax * 3n + axis * n + i; masks as kernel_InitSplitMasks
    // (kdtree.cu:1110-1251).  Lane i holds its element's candidates and compares them with one element
    // per step, whose bounds are broadcast; a comparison's result is shifted into the lane's mask
    // by an add with carry, so a step is 10 instructions for four masks (one lane mask per
    // candidate, combined and written to its lane, took about 50).  Lane i keeps the masks of its
    // element's candidates in registers (slot isMax * 3 + axis: candidate c = slot * n + i).
    //   triangles: L = min < s, R = s < max; the candidate's own element goes right of
    //              its minimum and left of its maximum; a flat element in the plane goes
    //              left if plane_goes_left, else right;
    //   points:    L = p < s, R = s < p; a point in the plane goes left if
    //              plane_goes_left, else right.
    // "In the plane as well" is a comparison with the next float below or above (no candidate of
    // use is infinite).
    uint64_t cmL[kSlots], cmR[kSlots];
    const uint64_t self = 1ull << lane;
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        const float mn = f4c(mlo, ax), mx = f4c(mhi, ax);
        const bool in_plane = (kind == MNRT_KIND_POINT || mn == mx) && fabsf(mn) < kInf;
        const float below = in_plane && mleft ? next_down(mn) : mn, above = in_plane && !mleft ? next_up(mx) : mx;
        uint32_t w[2][4];  // halves of the masks: left and right of the minimum, of the maximum
#pragma unroll
        for (int half = 1; half >= 0; --half) {
            uint32_t l0 = 0, r0 = 0, l1 = 0, r1 = 0;
            for (int j = (int)min(n, half ? 64u : 32u) - 1; j >= 32 * half; --j) {
                const float lo_j = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(below), j));
                const float hi_j = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(above), j));
                shift_in_less(l0, lo_j, mn);
                shift_in_greater(r0, hi_j, mn);
                if (kind == MNRT_KIND_TRI) {
                    shift_in_less(l1, lo_j, mx);
                    shift_in_greater(r1, hi_j, mx);
                }
            }
            w[half][0] = l0;
            w[half][1] = r0;
            w[half][2] = l1;
            w[half][3] = r1;
        }
        cmL[ax] = (uint64_t)w[1][0] << 32 | w[0][0];
        cmR[ax] = (uint64_t)w[1][1] << 32 | w[0][1];
        if (kind == MNRT_KIND_TRI) {
            cmL[ax] &= ~self;
            cmR[ax] |= self;
            cmL[3 + ax] = ((uint64_t)w[1][2] << 32 | w[0][2]) | self;
            cmR[3 + ax] = ((uint64_t)w[1][3] << 32 | w[0][3]) & ~self;
        }
    }

    uint32_t addr = 0, rbase = 0, maxlvl = 0;
    const uint32_t scene = root.scene;
    // emit: scene-local addresses into the scene's tree; stage: subtree-local addresses
    // into the staging area
    uint32_t* nodes = nullptr;
    uint32_t* refs = nullptr;
    uint32_t lim_nodes = 0u, lim_refs = 0u;
    bool writing = true;
    if (kMode == kSmallEmit) {
        nodes = O.nodes + 2ull * O.node_base[scene];
        refs = O.refs + O.ref_base[scene];
        lim_nodes = O.max_nodes - O.node_base[scene];
        lim_refs = O.max_refs - O.ref_base[scene];
        addr = O.bn[root.bn].addr;
        rbase = O.bn[root.bn].rbase;
    } else if (kMode == kSmallStage) {
        const uint32_t off = O.st_cap.begin(r, first);
        nodes = (uint32_t*)(O.st_nodes + off);
        refs = O.st_refs + off;
        lim_nodes = lim_refs = O.st_cap.of(n);
    }
    // the node at hand; left children follow at once, right ones wait on the stack
    int sp = 0;
    SmallStackEnt e;
    e.mask = (n == 64) ? ~0ull : ((1ull << n) - 1ull);
    for (int k = 0; k < 3; ++k) {
        e.lo[k] = root.lo[k];
        e.hi[k] = root.hi[k];
    }
    e.lvl_ax = root.level;
    e.patch = kNone;
    const float qr2 = 2.0f * scene_qr[scene];
    for (;;) {
        if (writing && (addr >= lim_nodes || rbase > lim_refs)) {
            if (kMode == kSmallEmit) {
                if (lane == 0) atomicOr(&O.W[W_ERR], 4u);
                break;
            }
            writing = false;  // staging area full: counted on, emitted later
        }
        if (writing && e.patch != kNone && lane == 0) nodes[2 * e.patch + 1] = (e.axis() << 30) | addr;
        maxlvl = max(maxlvl, e.level());
        const uint32_t cnt = (uint32_t)__popcll(e.mask);
        float best_cost = kInf;
        uint32_t best = kNone;
        const float ext[3] = {e.hi[0] - e.lo[0], e.hi[1] - e.lo[1], e.hi[2] - e.lo[2]};
        // A split leaves elements on both sides, so it costs kCostTraverse and at least the node's own
        // area or volume once: 4 and more, up to rounding, which three elements never exceed.  (In a box
        // turned inside out, as a caller may give it, areas do not add up.)
        const bool plain = ext[0] >= 0.0f && ext[1] >= 0.0f && ext[2] >= 0.0f && (kind == MNRT_KIND_TRI || qr2 >= 0.0f);
        const bool never = plain && cnt <= 3u;
        if (cnt > 0 && !never && e.level() < MNRT_MAX_LEVEL) {
            float denom;
            if (kind == MNRT_KIND_POINT) {
                float vol = 1.0f;
                for (int i = 0; i < 3; ++i) vol *= ext[i] + qr2;
                denom = 1.0f / vol;
            } else {
                float area = 2.0f * (ext[0] * ext[1] + ext[0] * ext[2] + ext[1] * ext[2]);
                denom = 1.0f / area;
            }
            // lane i evaluates its element's candidates, slot by slot (the axis a constant:
            // the node's bounds and extents on it need no selects); key = slot * 64 + i
            // orders the candidates as c = slot * n + i does
#pragma unroll
            for (int slot = 0; slot < kSlots; ++slot) {
                if (!valid) break;
                const int a = slot % 3;
                const float s = slot < 3 ? f4c(mlo, a) : f4c(mhi, a);
                const float lo_a = e.lo[a], hi_a = e.hi[a];
                if (!(lo_a < s && s < hi_a)) continue;
                const uint64_t bl = cmL[slot] & e.mask, br = cmR[slot] & e.mask;
                const uint32_t nl = (uint32_t)__popc((uint32_t)bl) + (uint32_t)__popc((uint32_t)(bl >> 32));
                const uint32_t nr = (uint32_t)__popc((uint32_t)br) + (uint32_t)__popc((uint32_t)(br >> 32));
                if (nl == 0 || nr == 0) continue;
                // the other two axes' extents, (a + 1) % 3 and (a + 2) % 3
                const float x1 = ext[(a + 1) % 3];
                const float x2 = ext[(a + 2) % 3];
                float cost;
                if (kind == MNRT_KIND_POINT) {
                    float vl = (x1 + qr2) * (s - lo_a + qr2) * (x2 + qr2);
                    float vr = (x1 + qr2) * (hi_a - s + qr2) * (x2 + qr2);
                    cost = ((float)nl * vl + (float)nr * vr) * denom + kCostTraverse;
                } else {
                    float al = 2.0f * (x1 * x2 + (s - lo_a) * (x1 + x2));
                    float ar = 2.0f * (x1 * x2 + (hi_a - s) * (x1 + x2));
                    cost = ((float)nl * al + (float)nr * ar) * denom + kCostTraverse;
                }
                if (cost < best_cost) {
                    best_cost = cost;
                    best = (uint32_t)slot * 64u + lane;
                }
            }
            // lowest cost, ties to the lower candidate (an order-independent minimum)
            auto take = [&](float oc, uint32_t ob) {
                if (oc < best_cost || (oc == best_cost && ob < best)) {
                    best_cost = oc;
                    best = ob;
                }
            };
#define MNRT_ARGMIN_DPP(ctrl) take(__uint_as_float(dpp_mov<ctrl>(__float_as_uint(best_cost))), dpp_mov<ctrl>(best))
            MNRT_ARGMIN_DPP(kDppPairSwap);
            MNRT_ARGMIN_DPP(kDppQuadSwap);
            MNRT_ARGMIN_DPP(kDppHalfMirror);
            MNRT_ARGMIN_DPP(kDppRowMirror);
#undef MNRT_ARGMIN_DPP
            {
                const uint32_t cb = __float_as_uint(best_cost), bb = best;
                best_cost = __uint_as_float(row_lane(cb, 0));
                best = row_lane(bb, 0);
                for (int row = 1; row < 4; ++row) take(__uint_as_float(row_lane(cb, row)), row_lane(bb, row));
            }
        }
        if (best == kNone || !(best_cost < (float)cnt)) {
            if (writing && rbase + cnt > lim_refs) {
                if (kMode == kSmallEmit) {
                    if (lane == 0) atomicOr(&O.W[W_ERR], 8u);
                    break;
                }
                writing = false;
            }
            if (writing) {
                if (lane == 0) {
                    nodes[2 * addr] = cnt;
                    nodes[2 * addr + 1] = (MNRT_LEAF_TAG << 30) | rbase;
                }
                if (lane < n && ((e.mask >> lane) & 1ull)) {
                    uint64_t below = (lane == 0) ? 0ull : (e.mask & ((1ull << lane) - 1ull));
                    refs[rbase + (uint32_t)__popcll(below)] = midx;
                }
            }
            ++addr;
            rbase += cnt;
            if (sp == 0) break;
            --sp;
            wave_sync();
            e = stack[sp];
            continue;
        }
        // the chosen candidate: slot and element lane from the key, its plane and masks
        // read from that lane
        const uint32_t bslot = __builtin_amdgcn_readfirstlane(best) >> 6, blane = __builtin_amdgcn_readfirstlane(best) & 63u;
        const uint32_t a = bslot % 3u;
        float sv = 0.0f;
        uint64_t bmL = 0, bmR = 0;
#pragma unroll
        for (int k = 0; k < kSlots; ++k) {
            if (bslot == (uint32_t)k) {
                sv = k < 3 ? f4c(mlo, k % 3) : f4c(mhi, k % 3);
                bmL = cmL[k];
                bmR = cmR[k];
            }
        }
        // (readlane returns int: each half goes through uint32_t, or the low half would be
        // sign-extended into the high one)
        auto lane_u32 = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane(v, (int)blane); };
        const float s = __uint_as_float(lane_u32(__float_as_uint(sv)));
        const uint64_t selL = ((uint64_t)lane_u32((uint32_t)(bmL >> 32)) << 32) | (uint64_t)lane_u32((uint32_t)bmL);
        const uint64_t selR = ((uint64_t)lane_u32((uint32_t)(bmR >> 32)) << 32) | (uint64_t)lane_u32((uint32_t)bmR);
        if (writing && lane == 0) {
            nodes[2 * addr] = __float_as_uint(s);
            nodes[2 * addr + 1] = a << 30;
        }
        if (lane == 0) {
            SmallStackEnt R = e;
            R.mask = selR & e.mask;
            for (uint32_t k = 0; k < 3; ++k) R.lo[k] = (a == k) ? s : e.lo[k];  // (selects, not indexing)
            R.lvl_ax = (e.level() + 1) | (a << 30);
            R.patch = addr;
            stack[sp] = R;
        }
        ++sp;
        ++addr;
        e.mask &= selL;
        for (uint32_t k = 0; k < 3; ++k) e.hi[k] = (a == k) ? s : e.hi[k];
        e.lvl_ax = e.level() + 1;
        e.patch = kNone;
    }
    if (kMode == kSmallStage && lane == 0) {
        O.nsize[r] = addr;
        O.rsize[r] = rbase;
        O.mlvl[r] = maxlvl;
        O.st_ovf[r] = writing ? 0u : 1u;
        if (!writing) atomicAdd(&O.W[W_SMALL_OVF], 1u);
    }
}

StageCap stage_cap_setting() {
    StageCap c{4u, 64u};
    if (const char* e = std::getenv("MNRT_SMALL_STAGE_CAP")) {
        unsigned m = 0, a = 0;
        if (std::sscanf(e, "%u,%u", &m, &a) == 2 && m <= 64 && a <= 4096) c = StageCap{m, a};
    }
    return c;
}

// Moves staged small subtrees to their final addresses (one wave per small root):
// inner words get the subtree's first address added to the right-child index, leaf words
// its first reference added to the reference offset.
__global__ __launch_bounds__(64 * kSmallWaves) void k_small_place(DN dnsmall, const SmallRec* __restrict__ S, SmallOut O) {
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const uint32_t r = blockIdx.x * kSmallWaves + wave;
    if (r >= dnsmall.get() || O.st_ovf[r] != 0u || O.W[W_ERR] != 0u) return;
    const uint32_t scene = S[r].scene;
    const BnRec& bn = O.bn[S[r].bn];
    const uint32_t a0 = bn.addr, r0 = bn.rbase;
    const uint32_t nn = O.nsize[r], nr = O.rsize[r];
    const uint32_t lim_nodes = O.max_nodes - O.node_base[scene], lim_refs = O.max_refs - O.ref_base[scene];
    if (a0 + nn > lim_nodes || r0 + nr > lim_refs) {
        if (lane == 0) atomicOr(&O.W[W_ERR], 4u);
        return;
    }
    uint2* nodes = (uint2*)(O.nodes + 2ull * O.node_base[scene]) + a0;
    uint32_t* refs = O.refs + O.ref_base[scene] + r0;
    const uint32_t off = O.st_cap.begin(r, S[r].first);
    for (uint32_t j = lane; j < nn; j += 64) {
        uint2 w = O.st_nodes[off + j];
        const uint32_t tag = w.y >> 30;
        w.y = (tag << 30) | ((w.y & MNRT_INDEX_MASK) + (tag == MNRT_LEAF_TAG ? r0 : a0));
        nodes[j] = w;
    }
    for (uint32_t j = lane; j < nr; j += 64) refs[j] = O.st_refs[off + j];
}

// ---- layout ---------------------------------------------------------------------------
// (KDTreeGPU::PreorderTraversal launches two kernels per level over all nodes,
// KDTreeGPU.cpp:1156-1209.)  Subtree sizes climb from the leaves in one launch: a child brings
// its sizes to its parent by one atomic, whose old value tells the second child to arrive what the
// first brought, and that one goes on.  Below an empty-space cut the sibling is an empty leaf, so
// the climb passes without an exchange.  A node's address is the sum over its ancestors, so one
// more launch places and emits every node at once.  58 launches, one per level and direction, took
// 234 us of the 1.03M-triangle build, these two 73 us.
constexpr uint32_t kAccBits = 31u;  // acc: references, nodes, arrivals (31 + 31 + 2 bits)

// top: the deepest level the build may reach; a leaf below it sets kErrLayoutDepth.
__global__ __launch_bounds__(256) void k_layout_sizes(DN dnbn, BnRec* __restrict__ B,
                                                      const uint32_t* __restrict__ s_nsize,
                                                      const uint32_t* __restrict__ s_rsize,
                                                      const uint32_t* __restrict__ s_mlvl, uint32_t top,
                                                      uint32_t* __restrict__ maxlvl, uint32_t* __restrict__ W) {
    if (W[W_ERR] != 0u) return;  // (per wave: another's error only ends the climb early)
    const uint32_t nbn = dnbn.get(), lane = threadIdx.x & 63u;
    for (uint32_t j0 = blockIdx.x * blockDim.x; j0 < nbn; j0 += gridDim.x * blockDim.x) {  // uniform per wave
        const uint32_t j = j0 + threadIdx.x;
        uint32_t scene = kNone, depth = 0, deepest = 0;
        if (j < nbn) {
            const uint4 q0 = ((const uint4*)&B[j])[0], q1 = ((const uint4*)&B[j])[1];
            uint32_t parent = B[j].parent;
            const uint32_t t = q0.x, x = q1.y;
            // (an empty leaf of a cut has its size already and is no deeper than its sibling)
            const bool cut_leaf = t == BN_LEAF && q1.z == 0u && parent != kNone && (parent & kCutParent);
            if ((t == BN_LEAF || t == BN_SMALL) && !cut_leaf) {
                uint32_t i = j, size = 1u, rsize = q1.z;
                scene = q1.w;
                deepest = depth = q1.x;
                if (t == BN_SMALL) {
                    size = s_nsize[x];
                    rsize = s_rsize[x];
                    depth = s_mlvl[x];
                }
                for (;;) {
                    if (size > MNRT_INDEX_MASK || rsize > MNRT_INDEX_MASK) {
                        atomicOr(&W[W_ERR], kErrOutputRoom);
                        break;
                    }
                    *(uint2*)&B[i].size = make_uint2(size, rsize);
                    if (parent == kNone) break;
                    const uint32_t p = parent & ~kCutParent;
                    const bool cut = (parent & kCutParent) != 0u;
                    parent = B[p].parent;
                    i = p;
                    if (cut) {
                        size += 2u;
                        continue;
                    }
                    const unsigned long long old =
                        atomicAdd(&B[p].acc, 1ull << 62 | (unsigned long long)size << kAccBits | rsize);
                    if ((old >> 62) == 0ull) break;
                    size += 1u + ((uint32_t)(old >> kAccBits) & 0x7FFFFFFFu);
                    rsize += (uint32_t)old & 0x7FFFFFFFu;
                }
            }
        }
        deepest = wave_max_u32(deepest);
        if (lane == 0u && deepest != 0u) {
            atomicMax(&W[W_MAXLEVEL], deepest);
            if (deepest > top) atomicOr(&W[W_ERR], kErrLayoutDepth);
        }
        for (uint64_t m = ballot(scene != kNone); m != 0ull;) {
            const uint32_t s = (uint32_t)__builtin_amdgcn_readlane((int)scene, (int)__builtin_ctzll(m));
            const uint32_t d = wave_max_u32(scene == s ? depth : 0u);
            if (lane == 0u) atomicMax(&maxlvl[s], d);
            m &= ~ballot(scene == s);
        }
    }
}

// Per scene (root = build node s): nodes, references and leaves, and the trees' places
// in the shared arrays.  Every inner node has two children, so leaves = (nodes + 1) / 2.
// max_nodes / max_refs: room of the output arrays.
__global__ __launch_bounds__(1024) void k_scene_totals(uint32_t nscenes, const BnRec* __restrict__ B,
                                                       uint32_t* __restrict__ nodes, uint32_t* __restrict__ refs,
                                                       uint32_t* __restrict__ nbase, uint32_t* __restrict__ rbase,
                                                       uint32_t* __restrict__ leaves, uint32_t max_nodes,
                                                       uint32_t max_refs, uint32_t* __restrict__ W) {
    __shared__ uint64_t s_wave[16], s_rwave[16];
    if (W[W_ERR] != 0u) return;  // (uniform: this launch sets it after its last barrier only)
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    uint64_t n0 = 0, r0 = 0;
    for (uint32_t b = 0; b < nscenes; b += 1024u) {
        const uint32_t s = b + tid;
        const uint32_t n = s < nscenes ? B[s].size : 0u, r = s < nscenes ? B[s].rsize : 0u;
        uint64_t incl = n, rincl = r;  // (64 sizes of at most 2^30 - 1 pass 32 bits)
#pragma unroll
        for (uint32_t o = 1; o < 64; o <<= 1) {
            const uint64_t a = __shfl_up((unsigned long long)incl, o, 64), c = __shfl_up((unsigned long long)rincl, o, 64);
            if (lane >= o) {
                incl += a;
                rincl += c;
            }
        }
        if (lane == 63u) {
            s_wave[wave] = incl;
            s_rwave[wave] = rincl;
        }
        __syncthreads();
        uint64_t nb = n0, rb = r0;
        for (uint32_t i = 0; i < 16u; ++i) {
            if (i < wave) {
                nb += s_wave[i];
                rb += s_rwave[i];
            }
            n0 += s_wave[i];
            r0 += s_rwave[i];
        }
        if (s < nscenes) {
            nodes[s] = n;
            refs[s] = r;
            nbase[s] = (uint32_t)(nb + incl - n);
            rbase[s] = (uint32_t)(rb + rincl - r);
            leaves[s] = (n + 1u) / 2u;
        }
        __syncthreads();  // the LDS words are rewritten by the next step
    }
    if (tid == 0) {
        nbase[nscenes] = (uint32_t)n0;
        rbase[nscenes] = (uint32_t)r0;
        if (n0 == 0u || n0 > max_nodes || r0 > max_refs) atomicOr(&W[W_ERR], kErrOutputRoom);
    }
}

// Places every build node and writes the large stage's inner nodes and leaves.
__global__ __launch_bounds__(256) void k_emit_large(DN dnbn, BnRec* __restrict__ B,
                                                    const uint32_t* __restrict__ ll_idx,
                                                    uint32_t* __restrict__ nodes_all, uint32_t* __restrict__ refs_all,
                                                    const uint32_t* __restrict__ W,
                                                    const uint32_t* __restrict__ node_base,
                                                    const uint32_t* __restrict__ ref_base) {
    if (W[W_ERR] != 0u) return;  // failed build: nothing is emitted
    const uint32_t nbn = dnbn.get();
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nbn; i += gridDim.x * blockDim.x) {
        const uint4 q0 = ((const uint4*)&B[i])[0], q1 = ((const uint4*)&B[i])[1];
        const uint32_t t = q0.x, sc = q1.w;
        uint32_t a = 0, rb = 0;
        for (uint32_t c = i, up = B[i].parent; up != kNone;) {
            const uint32_t p = up & ~kCutParent, l = B[p].left;
            const uint32_t above = B[p].parent;
            a += 1u;
            if (l != c) {
                const uint2 z = *(const uint2*)&B[l].size;
                a += z.x;
                rb += z.y;
            }
            c = p;
            up = above;
        }
        if (t == BN_SMALL) {
            *(uint2*)&B[i].addr = make_uint2(a, rb);
            continue;
        }
        uint2* nodes = (uint2*)nodes_all + node_base[sc];
        if (t == BN_LEAF) {
            const uint32_t m = q1.z, from = q1.y;
            uint32_t* refs = refs_all + ref_base[sc];
            nodes[a] = make_uint2(m, (MNRT_LEAF_TAG << 30) | rb);
            for (uint32_t k = 0; k < m; ++k) refs[rb + k] = ll_idx[from + k];
        } else {
            nodes[a] = make_uint2(q0.y, (t << 30) | (a + 1u + B[q0.z].size));
        }
    }
}

}  // namespace mnrt

// =========================================================================================
// host driver
// =========================================================================================
namespace {

using namespace mnrt;

// Build workspace: one device block per host thread and device, kept across builds and
// grown to the largest build seen, so a build in steady state allocates nothing but its
// output arrays (allocation calls that must grow device memory cost milliseconds each; buffers that a
// build replaces by larger ones, taken from the stream-ordered pool and given back at once, made
// 205001 triangles with small roots of one take 250 ms, 25 from the block).
// Buffers are carved bump-wise and not reused within a build; a build that outgrows the
// block takes the rest from the stream-ordered pool, and the block grows to fit when that
// build ends.  The blocks live until the process ends.
constexpr int kArenaDevices = 64;
struct Arena {
    char* base = nullptr;
    size_t cap = 0;
};
thread_local Arena t_arena[kArenaDevices];

class Pool {
   public:
    explicit Pool(hipStream_t st) : st_(st) {
        int dev = -1;
        if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < kArenaDevices) arena_ = &t_arena[dev];
    }
    ~Pool() {
        // nothing may still use the workspace when the next build on this thread reuses it
        (void)hipStreamSynchronize(st_);
        for (void* p : ptrs_) (void)pool_free(p, st_);
        if (arena_ && peak_ > arena_->cap) {
            (void)hipStreamSynchronize(st_);
            if (arena_->base) (void)hipFree(arena_->base);
            *arena_ = Arena{};
            void* nb = nullptr;
            const size_t ncap = peak_ + std::min(peak_ / 4, size_t(1) << 30) + (size_t(64) << 20);
            // (what this build had from the pool lies there unused: it goes back to the device if need be)
            if (device_alloc(&nb, ncap) == hipSuccess || (pool_trim(), device_alloc(&nb, ncap) == hipSuccess))
                *arena_ = Arena{(char*)nb, ncap};
        }
    }
    template <typename T>
    T* get(uint64_t count) {
        const size_t bytes = (std::max<size_t>(count * sizeof(T), 16) + 255) & ~size_t(255);
        total_ += bytes;
        peak_ = std::max(peak_, total_);
        if (arena_ && top_ + bytes <= arena_->cap) {
            void* p = arena_->base + top_;
            top_ += bytes;
            return (T*)p;
        }
        void* p = nullptr;
        if (pool_alloc(&p, bytes, st_) != hipSuccess) {
            ok = false;
            return nullptr;
        }
        ptrs_.push_back(p);
        return (T*)p;
    }
    bool ok = true;

   private:
    hipStream_t st_;
    Arena* arena_ = nullptr;
    size_t top_ = 0;
    size_t total_ = 0, peak_ = 0;
    std::vector<void*> ptrs_;
};

// Bump carving of one device block: a first pass (base null) measures, the second carves.
class Carver {
   public:
    explicit Carver(char* base) : base_(base) {}
    template <typename T>
    T* get(uint64_t count) {
        const uint64_t bytes = (std::max<uint64_t>(count * sizeof(T), 16) + 255) & ~uint64_t(255);
        T* p = base_ ? (T*)(base_ + top_) : nullptr;
        top_ += bytes;
        return p;
    }
    uint64_t size() const { return top_; }

   private:
    char* base_;
    uint64_t top_ = 0;
};

inline dim3 blocks_for(uint64_t n, uint32_t bs = 256) { return dim3((uint32_t)std::max<uint64_t>(1, (n + bs - 1) / bs)); }
// Grid of a launch that strides: at most `most` workgroups.
inline dim3 blocks_to(uint64_t n, uint32_t bs, uint32_t most) {
    return dim3(std::min<uint32_t>(blocks_for(std::min<uint64_t>(n, 1ull << 40), bs).x, most));
}

// Placement of the scenes' roots: large scenes become active nodes, whose elements start at a
// multiple of 64 slots, small ones small roots.
struct RootCounts {
    uint32_t na = 0, nw = 0, nsmall = 0, nse = 0, largest = 0;
};
RootCounts plan_roots(const uint32_t* h_base, uint32_t S_, uint32_t small_max, uint32_t* kind, uint32_t* index,
                      uint32_t* off) {
    RootCounts c;
    for (uint32_t s = 0; s < S_; ++s) {
        const uint32_t cnt = h_base[s + 1] - h_base[s];
        c.largest = std::max(c.largest, cnt);
        if (cnt > small_max) {
            kind[s] = 0;
            index[s] = c.na++;
            off[s] = 64u * c.nw;
            c.nw += (cnt + 63u) / 64u;
        } else {
            kind[s] = 1;
            index[s] = c.nsmall++;
            off[s] = c.nse;
            c.nse += cnt;
        }
    }
    return c;
}

// Buffers of the large-node stage.
struct LevelBufs {
    uint32_t* W;
    uint32_t* stb;  // tight bounds per scene
    NodeRec* N[2];
    ElemView X[2], Sm;
    SmallRec* S;
    BnRec* B;
    uint32_t* wc;
    unsigned long long* cs[2];
    uint4* coff;
    SplitRec* P;
    uint32_t* ll_idx;
    uint4* q;
};

template <typename A>
ElemView take_elems(A& a, int kind, uint64_t slots, bool waves) {
    ElemView V{};
    V.lo = a.template get<float4>(slots);
    V.hi = kind == MNRT_KIND_TRI ? a.template get<float4>(slots) : V.lo;
    V.wnode = waves ? a.template get<uint32_t>(slots / 64u) : nullptr;
    return V;
}

template <typename A>
LevelBufs take_levels(A& a, int kind, uint32_t S_, const BuildCaps& C) {
    LevelBufs b{};
    b.W = a.template get<uint32_t>(kWords);
    b.stb = a.template get<uint32_t>(6ull * S_);
    for (NodeRec*& n : b.N) n = a.template get<NodeRec>(C.na);
    const uint64_t slots = 64ull * C.nw;
    for (ElemView& V : b.X) V = take_elems(a, kind, slots, true);
    b.Sm = take_elems(a, kind, C.se, false);
    b.S = a.template get<SmallRec>(C.small);
    b.B = a.template get<BnRec>(C.bn);
    b.wc = a.template get<uint32_t>(C.nw);
    for (unsigned long long*& v : b.cs) v = a.template get<unsigned long long>(chunks_for(C.nw, C.na));
    b.coff = a.template get<uint4>(chunks_for(C.nw, C.na));
    b.P = a.template get<SplitRec>(C.na);
    b.ll_idx = a.template get<uint32_t>(C.ll);
    b.q = kind == MNRT_KIND_TRI ? a.template get<uint4>(slots) : nullptr;
    return b;
}

// Input elements, their tight bounds per scene and the root entries.
void launch_roots(const LevelBufs& b, const Geometry& G, uint32_t ntot, const RootPlan& R, const RootCounts& c,
                  const float* given, float* rootbox, uint32_t* maxlvl, hipStream_t st) {
    const uint32_t S_ = G.num_scenes;
    hipLaunchKernelGGL(k_build_init, blocks_to(std::max<uint64_t>({kWords, 6ull * S_, chunks_for(c.nw, c.na)}), 256, 256), dim3(256), 0, st, b.W, c.na, c.nw,
                       c.nsmall, c.nse, S_, b.stb, maxlvl, b.cs[0]);
    if (ntot > 0)
        hipLaunchKernelGGL(k_init_elems, blocks_for(ntot, kInitBlock * kInitPer), dim3(kInitBlock), 0, st, G, ntot, R,
                           b.X[0], b.Sm, b.stb);
    hipLaunchKernelGGL(k_roots_setup, blocks_for(S_), dim3(256), 0, st, S_, G.base, b.stb, given, R, b.N[0], b.S, b.B,
                       rootbox);
}

// One level of the large-node stage, for about na nodes in nw waves (the grids' sizes only).
void launch_level(const LevelBufs& b, const Geometry& G, const mnrt_build_params& prm, const BuildCaps& C,
                  uint32_t level, uint64_t na, uint64_t nw, hipStream_t st) {
    LevelArgs L{};
    L.W = b.W;
    L.level = level;
    L.cap = C;
    L.ratio = prm.empty_space_ratio;
    L.small_max = prm.small_node_max;
    L.A = b.N[level & 1u];
    L.An = b.N[(level + 1u) & 1u];
    L.E = b.X[level & 1u];
    L.Nx = b.X[(level + 1u) & 1u];
    L.Sm = b.Sm;
    L.wc = b.wc;
    L.cs = b.cs[level & 1u];
    L.csn = b.cs[(level + 1u) & 1u];
    L.coff = b.coff;
    L.P = b.P;
    L.S = b.S;
    L.B = b.B;
    L.ll_idx = b.ll_idx;
    L.q = b.q;
    const dim3 gc = blocks_to(nw, kCountWaves, 512), gn = blocks_to(na, kChildNodes, 512), gs = blocks_to(nw, kScatterWaves, 512);
    if (G.kind == MNRT_KIND_TRI) {
        hipLaunchKernelGGL((k_count<MNRT_KIND_TRI>), gc, dim3(kCountBlock), 0, st, L);
        hipLaunchKernelGGL(k_children, gn, dim3(kChildBlock), 0, st, L);
        hipLaunchKernelGGL((k_scatter<MNRT_KIND_TRI>), gs, dim3(kScatterBlock), 0, st, L);
        hipLaunchKernelGGL(k_clip, blocks_to(nw, 1, 2048), dim3(kClipBlock), 0, st, L, G);
    } else {
        hipLaunchKernelGGL((k_count<MNRT_KIND_POINT>), gc, dim3(kCountBlock), 0, st, L);
        hipLaunchKernelGGL(k_children, gn, dim3(kChildBlock), 0, st, L);
        hipLaunchKernelGGL((k_scatter<MNRT_KIND_POINT>), gs, dim3(kScatterBlock), 0, st, L);
    }
}

// Buffers of the small-node stage.
template <typename A>
SmallOut take_small(A& a, uint32_t* W, const StageCap& cap, uint64_t nsmall, uint64_t nse) {
    const uint64_t total = (uint64_t)cap.mul * nse + (uint64_t)cap.add * nsmall;  // sum over the roots
    SmallOut O{};
    O.nsize = a.template get<uint32_t>(nsmall);
    O.rsize = a.template get<uint32_t>(nsmall);
    O.mlvl = a.template get<uint32_t>(nsmall);
    O.st_ovf = a.template get<uint32_t>(nsmall);
    O.st_nodes = a.template get<uint2>(total);
    O.st_refs = a.template get<uint32_t>(total);
    O.st_cap = cap;
    O.W = W;
    return O;
}

template <int kMode>
void launch_small(int kind, DN nsmall, const SmallRec* S, const ElemView& Sm, const float* qr, const SmallOut& O,
                  hipStream_t st) {
    const dim3 grid((nsmall.v + kSmallWaves - 1) / kSmallWaves), block(64 * kSmallWaves);
    if (kind == MNRT_KIND_TRI)
        hipLaunchKernelGGL((k_small<kMode, MNRT_KIND_TRI>), grid, block, 0, st, nsmall, S, Sm, qr, O);
    else
        hipLaunchKernelGGL((k_small<kMode, MNRT_KIND_POINT>), grid, block, 0, st, nsmall, S, Sm, qr, O);
}

// Per-scene device table: everything from rootbox to smaxlvl is one consecutive result block.
struct SceneTab {
    uint32_t *base, *pkind, *pindex, *poff;  // S + 1 element offsets, the roots' placement
    float *qr, *given, *rootbox;
    uint32_t *snodes, *srefs, *nbase, *rbase, *sleaves, *smaxlvl;  // nbase, rbase: S + 1
    uint32_t *slot_begin, *box_begin;  // photon_tables (recorded builds)
};
constexpr uint64_t scene_tab_words(uint64_t S_) { return 32ull * S_ + 64; }
constexpr uint64_t scene_input_words(uint64_t S_) { return 11ull * S_ + 1; }    // base .. given
constexpr uint64_t scene_result_words(uint64_t S_) { return 12ull * S_ + 2; }   // rootbox .. smaxlvl

SceneTab scene_tab(uint32_t* t, uint32_t S_) {
    SceneTab T;
    T.base = t;
    T.pkind = T.base + S_ + 1;
    T.pindex = T.pkind + S_;
    T.poff = T.pindex + S_;
    T.qr = (float*)(T.poff + S_);
    T.given = T.qr + S_;
    T.rootbox = T.given + 6 * S_;
    T.snodes = (uint32_t*)(T.rootbox + 6 * S_);
    T.srefs = T.snodes + S_;
    T.nbase = T.srefs + S_;
    T.rbase = T.nbase + S_ + 1;
    T.sleaves = T.rbase + S_ + 1;
    T.smaxlvl = T.sleaves + S_;
    T.slot_begin = T.smaxlvl + S_;
    T.box_begin = T.slot_begin + S_ + 1;
    return T;
}

// Tree s of a batch from the result block r; its arrays start at nodes / refs.
void set_tree(mnrt_tree& t, int kind, uint32_t s, uint32_t S_, const uint32_t* r, const uint32_t* h_base,
              uint32_t* nodes, uint32_t* refs) {
    const float* box = (const float*)r + 6ull * s;
    const uint32_t* n = r + 6ull * S_;
    const uint32_t *nb = n + 2ull * S_, *rb = nb + S_ + 1, *lv = rb + S_ + 1;
    std::memset(&t, 0, sizeof(t));
    t.kind = (uint32_t)kind;
    t.num_nodes = n[s];
    t.num_refs = n[S_ + s];
    t.num_elems = h_base[s + 1] - h_base[s];
    t.num_leaves = lv[s];
    t.max_level = lv[S_ + s];
    for (int k = 0; k < 3; ++k) {
        t.root_min[k] = box[k];
        t.root_max[k] = box[3 + k];
    }
    t.d_nodes = nodes + 2ull * nb[s];
    t.d_refs = refs + rb[s];
}

// Sizes a host-driven build met, from which a recorded device-driven build sizes its
// fixed buffers.
struct BuildStats {
    RootCounts roots;
    std::vector<uint32_t> level_na, level_nw;
    uint32_t max_na = 0, max_nw = 0;
    uint32_t nbn = 0, nsmall = 0, nse = 0, ll = 0, maxlvl = 0, total_nodes = 0, total_refs = 0;
};

// Buffer sizes a host-driven build starts with.  Points never straddle, so a level holds at
// most the input and small_max + 1 elements per node; triangles are duplicated, and the rest is
// what ordinary trees stay below.  A build that outgrows one of them moves to larger ones and goes on
// from the level that did (grow_caps, grow_levels).
BuildCaps first_caps(int kind, uint32_t S_, uint32_t ntot, uint32_t small_max, const RootCounts& c) {
    const uint64_t ne = (kind == MNRT_KIND_TRI ? 2ull : 1ull) * ntot, lim = MNRT_INDEX_MASK;
    const uint64_t per = ntot / small_max;
    BuildCaps C{};
    C.na = (uint32_t)std::min<uint64_t>(lim, ne / (small_max + 1) + c.na + 1);
    C.nw = (uint32_t)std::min<uint64_t>(lim / 64, ne / 64 + C.na + c.nw);
    C.bn = (uint32_t)std::min<uint64_t>(lim, S_ + 8 * per + 1024);
    C.small = (uint32_t)std::min<uint64_t>(lim, c.nsmall + 4 * per + 256);
    C.se = (uint32_t)std::min<uint64_t>(lim, ne + 1024);
    C.ll = (uint32_t)std::min<uint64_t>(lim, ntot + 1024ull);
    return C;
}

// The sizes that level `level` of an outgrown build exceeds, at least doubled, and with them those
// of the totals that are more than half full: deeper levels add to them, and each time a build goes on
// costs a synchronisation and copies.  An element of a level or a small root ends in a leaf, a
// build node in the tree: beyond MNRT_INDEX_MASK of them the tree itself has no room (false).
bool grow_caps(BuildCaps& C, const uint32_t* W, uint32_t level) {
    bool room = true, grown = false;
    auto grow = [&](uint32_t& cap, uint64_t need, uint64_t lim, bool total) {
        if (need <= cap && !(total && 2 * need > cap)) return;
        if (need > cap) {
            grown = true;
            if (cap >= lim) room = false;
        }
        cap = (uint32_t)std::min<uint64_t>(lim, std::max<uint64_t>(2ull * cap, need + need / 4));
    };
    const uint64_t lim = MNRT_INDEX_MASK;
    const uint32_t* next = W + W_LEVELS + kLevelWords * (level + 1);
    grow(C.nw, next[0], lim / 64, false);
    grow(C.na, next[1], lim, false);
    grow(C.bn, W[W_NBN], lim, true);
    grow(C.small, W[W_NSMALL], lim, true);
    grow(C.se, W[W_NSE], lim, true);
    grow(C.ll, W[W_LL], lim, true);
    return room && grown;
}

// Moves a build that outgrew the sizes C at level `level` (device words W) to buffers of the sizes D:
// what the levels before it left, which the level reads or adds to; the rest is written before
// it is read.  A build that started over each time it outgrew a size (up to 13 times): 3001 triangles, small
// roots of at most 4: 8.6 ms, now 2.4; 205001, at most 4: 15.7, now 5.7, at most one: 57, now 25;
// 1.03M, at most 16: 7.0, now 3.7; 500000 points in 4913 places 6.6, now 2.5.
int grow_levels(Pool& pool, int kind, LevelBufs& b, const BuildCaps& C, const BuildCaps& D, const uint32_t* W,
                uint32_t level, hipStream_t st) {
    const uint32_t* T = W + W_LEVELS + kLevelWords * level;
    const uint64_t nw = T[0], na = T[1], nbn = T[4], ll = T[5], nse = T[6], nsmall = T[7];
    hipError_t err = hipSuccess;
    auto move = [&](auto*& p, uint64_t from, uint64_t to, uint64_t used) {
        using E = std::remove_reference_t<decltype(*p)>;
        if (to == from || !pool.ok || err != hipSuccess) return;
        E* n = pool.get<E>(to);
        if (!pool.ok) return;
        if (used != 0) err = hipMemcpyAsync(n, p, used * sizeof(E), hipMemcpyDeviceToDevice, st);
        p = n;
    };
    auto move_elems = [&](ElemView& V, uint64_t from, uint64_t to, uint64_t used) {
        move(V.lo, from, to, used);
        if (kind == MNRT_KIND_TRI) move(V.hi, from, to, used);
        else V.hi = V.lo;
    };
    const uint64_t chunks = chunks_for(C.nw, C.na), more_chunks = chunks_for(D.nw, D.na);
    for (uint32_t i = 0; i < 2; ++i) {
        const bool cur = i == (level & 1u);
        move(b.N[i], C.na, D.na, cur ? na : 0u);
        move_elems(b.X[i], 64ull * C.nw, 64ull * D.nw, cur ? 64u * nw : 0u);
        move(b.X[i].wnode, C.nw, D.nw, cur ? nw : 0u);
        move(b.cs[i], chunks, more_chunks, 0u);
    }
    move_elems(b.Sm, C.se, D.se, nse);
    move(b.S, C.small, D.small, nsmall);
    move(b.B, C.bn, D.bn, nbn);
    move(b.wc, C.nw, D.nw, 0u);
    move(b.coff, chunks, more_chunks, 0u);
    move(b.P, C.na, D.na, 0u);
    move(b.ll_idx, C.ll, D.ll, ll);
    if (kind == MNRT_KIND_TRI) move(b.q, 64ull * C.nw, 64ull * D.nw, 0u);
    if (!pool.ok) return MNRT_ERR_NOMEM;
    const uint64_t n = chunks_for(nw, na);
    hipLaunchKernelGGL(k_level_again, blocks_to(n, 256, 256), dim3(256), 0, st, b.W, level, n, b.cs[level & 1u]);
    return err == hipSuccess && hipGetLastError() == hipSuccess ? MNRT_OK : MNRT_ERR_HIP;
}

// Builds the trees of S scenes together: one level loop over the active nodes of all
// scenes, one small-node launch for all small roots, one layout / emission pass.  Each
// scene's tree equals the tree a single-scene build of it gives (indices are
// scene-local, all decisions are per node).
//   h_base: S + 1 element offsets into the concatenated input.
//   h_roots: 6 floats per scene (or null: tight bounds).  h_qr: VVH radius per scene
//   (or null: params->max_query_radius).
//   out[s] views into shared arrays; out[0] owns them (mnrt_tree_release(&out[0])
//   frees every tree of the batch).
// The host waits for the device after the levels (to see whether there are more, and to size the
// small stage), after the layout (to allocate the trees) and at the end.
int build_batch_impl(int kind, const float* d_v0, const float* d_v1, const float* d_v2, const uint32_t* h_base,
                     uint32_t nscenes, const mnrt_build_params* prm, const float* h_roots, const float* h_qr,
                     mnrt_tree* out, hipStream_t st, BuildStats* stats = nullptr) {
    if (!out || !prm || !h_base || nscenes == 0) return MNRT_ERR_ARG;
    const uint32_t ntot = h_base[nscenes];
    for (uint32_t s = 0; s < nscenes; ++s)
        if (h_base[s + 1] < h_base[s]) return MNRT_ERR_ARG;
    if (ntot > 0 && !d_v0) return MNRT_ERR_ARG;
    if (kind == MNRT_KIND_TRI && ntot > 0 && (!d_v1 || !d_v2)) return MNRT_ERR_ARG;
    if (prm->small_node_max < 1 || prm->small_node_max > 64) return MNRT_ERR_ARG;
    if (ntot > (MNRT_INDEX_MASK >> 2)) return MNRT_ERR_CAPACITY;
    const uint32_t S_ = nscenes;
    Pool pool(st);
    uint32_t* d_tab = pool.get<uint32_t>(scene_tab_words(S_));
    if (!pool.ok) return MNRT_ERR_NOMEM;
    const SceneTab T = scene_tab(d_tab, S_);

    // host staging in pinned memory: device words, the per-scene tables
    const uint32_t hw = (kWords + 15u) & ~15u;
    uint32_t* h_pin = (uint32_t*)host_staging(0, (hw + scene_tab_words(S_)) * 4);
    if (!h_pin) return MNRT_ERR_NOMEM;
    uint32_t* h_W = h_pin;
    uint32_t* h_tab = h_pin + hw;
    RootCounts c;
    {
        const SceneTab H = scene_tab(h_tab, S_);
        for (uint32_t s = 0; s <= S_; ++s) H.base[s] = h_base[s];
        c = plan_roots(h_base, S_, prm->small_node_max, H.pkind, H.pindex, H.poff);
        for (uint32_t s = 0; s < S_; ++s) {
            H.qr[s] = h_qr ? h_qr[s] : prm->max_query_radius;
            for (int k = 0; k < 6; ++k) H.given[6 * s + k] = h_roots ? h_roots[6 * s + k] : 0.0f;
        }
        MNRT_HIP_CHECK(hipMemcpyAsync(d_tab, h_tab, scene_input_words(S_) * 4, hipMemcpyHostToDevice, st));
    }
    Geometry G{kind, (const float4*)d_v0, d_v1 ? (const float4*)d_v1 : (const float4*)d_v0,
               d_v2 ? (const float4*)d_v2 : (const float4*)d_v0, T.base, S_};
    const RootPlan RP{T.pkind, T.pindex, T.poff};

    // ---- large-node stage ----
    // Levels are enqueued ahead of the counts (a middle split halves a node's box, so about log2
    // of the elements per small root, half as many again where they lie unevenly), then a few at
    // a time until a level has no nodes.
    uint32_t first_levels = 0;
    if (c.na > 0) {
        uint32_t lg = 1;
        while ((c.largest >> lg) >= prm->small_node_max) ++lg;
        first_levels = std::min<uint32_t>(lg + lg / 2 + 1, kLevels);
    }
    BuildCaps C = first_caps(kind, S_, ntot, prm->small_node_max, c);
    LevelBufs b = take_levels(pool, kind, S_, C);
    if (!pool.ok) return MNRT_ERR_NOMEM;
    launch_roots(b, G, ntot, RP, c, h_roots ? (const float*)T.given : (const float*)nullptr, T.rootbox, T.smaxlvl, st);
    uint32_t levels = 0;
    for (uint32_t until = first_levels;;) {
        for (; levels < until; ++levels)
            launch_level(b, G, *prm, C, levels, std::min<uint64_t>(C.na, (uint64_t)c.na << levels), C.nw, st);
        MNRT_HIP_CHECK(hipGetLastError());
        MNRT_HIP_CHECK(hipMemcpyAsync(h_W, b.W, kWords * 4, hipMemcpyDeviceToHost, st));
        MNRT_HIP_CHECK(hipStreamSynchronize(st));
        if (h_W[W_ERR] == 0u) {
            if (h_W[W_LEVELS + kLevelWords * levels + 1] == 0u) break;
            if (levels == kLevels) return MNRT_ERR_STATE;
            until = std::min(levels + 4u, kLevels);
            continue;
        }
        if (h_W[W_ERR] != kErrRoom || h_W[W_ERRLEVEL] >= levels) return MNRT_ERR_STATE;
        levels = h_W[W_ERRLEVEL];
        BuildCaps D = C;
        if (!grow_caps(D, h_W, levels)) return MNRT_ERR_CAPACITY;
        const int rc = grow_levels(pool, kind, b, C, D, h_W, levels, st);
        if (rc != MNRT_OK) return rc;
        C = D;
    }
    const uint32_t nbn = h_W[W_NBN], nsmall = h_W[W_NSMALL], nse = h_W[W_NSE];
    if (stats) {
        *stats = BuildStats{};
        stats->roots = c;
        for (uint32_t l = 0; l < levels && h_W[W_LEVELS + kLevelWords * l + 1] != 0u; ++l) {
            stats->level_nw.push_back(h_W[W_LEVELS + kLevelWords * l]);
            stats->level_na.push_back(h_W[W_LEVELS + kLevelWords * l + 1]);
            stats->max_nw = std::max(stats->max_nw, stats->level_nw.back());
            stats->max_na = std::max(stats->max_na, stats->level_na.back());
        }
        stats->nbn = nbn;
        stats->nsmall = nsmall;
        stats->nse = nse;
        stats->ll = h_W[W_LL];
    }

    // ---- small-node stage: subtree sizes, each subtree written to its staging area ----
    const StageCap st_cap = stage_cap_setting();
    if ((uint64_t)st_cap.mul * nse + (uint64_t)st_cap.add * nsmall > 0xFFFFFFFFull) return MNRT_ERR_CAPACITY;
    SmallOut O = take_small(pool, b.W, st_cap, nsmall, nse);
    if (!pool.ok) return MNRT_ERR_NOMEM;
    if (nsmall > 0) launch_small<kSmallStage>(kind, hn(nsmall), b.S, b.Sm, T.qr, O, st);
    // ---- layout ----
    const dim3 lgrid = blocks_for(nbn);
    hipLaunchKernelGGL(k_layout_sizes, lgrid, dim3(256), 0, st, hn(nbn), b.B, (const uint32_t*)O.nsize,
                       (const uint32_t*)O.rsize, (const uint32_t*)O.mlvl, (uint32_t)MNRT_MAX_LEVEL, T.smaxlvl, b.W);
    hipLaunchKernelGGL(k_scene_totals, dim3(1), dim3(1024), 0, st, S_, (const BnRec*)b.B, T.snodes, T.srefs, T.nbase,
                       T.rbase, T.sleaves, (uint32_t)MNRT_INDEX_MASK, (uint32_t)MNRT_INDEX_MASK, b.W);
    MNRT_HIP_CHECK(hipGetLastError());
    uint32_t* h_res = h_tab;
    MNRT_HIP_CHECK(hipMemcpyAsync(h_res, T.rootbox, scene_result_words(S_) * 4, hipMemcpyDeviceToHost, st));
    MNRT_HIP_CHECK(hipMemcpyAsync(h_W, b.W, W_LEVELS * 4, hipMemcpyDeviceToHost, st));
    MNRT_HIP_CHECK(hipStreamSynchronize(st));
    if (h_W[W_ERR] != 0u) return h_W[W_ERR] == kErrOutputRoom ? MNRT_ERR_CAPACITY : MNRT_ERR_STATE;
    const uint32_t total_nodes = h_res[9ull * S_], total_refs = h_res[10ull * S_ + 1];
    if (stats) {
        stats->maxlvl = h_W[W_MAXLEVEL];
        stats->total_nodes = total_nodes;
        stats->total_refs = total_refs;
    }

    // ---- emission into the caller-visible trees ----
    uint32_t* d_nodes = nullptr;
    uint32_t* d_refs = nullptr;
    if (pool_alloc((void**)&d_nodes, (size_t)total_nodes * 8, st) != hipSuccess) return MNRT_ERR_NOMEM;
    if (pool_alloc((void**)&d_refs, (size_t)total_refs * 4, st) != hipSuccess) {
        (void)pool_free(d_nodes, st);
        return MNRT_ERR_NOMEM;
    }
    hipLaunchKernelGGL(k_emit_large, lgrid, dim3(256), 0, st, hn(nbn), b.B, (const uint32_t*)b.ll_idx, d_nodes,
                       d_refs, (const uint32_t*)b.W, (const uint32_t*)T.nbase, (const uint32_t*)T.rbase);
    O.bn = b.B;
    O.nodes = d_nodes;
    O.refs = d_refs;
    O.max_nodes = total_nodes;
    O.max_refs = total_refs;
    O.node_base = T.nbase;
    O.ref_base = T.rbase;
    if (nsmall > 0) {
        hipLaunchKernelGGL(k_small_place, dim3((nsmall + kSmallWaves - 1) / kSmallWaves), dim3(64 * kSmallWaves), 0, st,
                           hn(nsmall), b.S, O);
        // subtrees that outgrew their staging area are built again at their final address
        if (h_W[W_SMALL_OVF] > 0) launch_small<kSmallEmit>(kind, hn(nsmall), b.S, b.Sm, T.qr, O, st);
    }
    int rc = MNRT_OK;
    if (hipMemcpyAsync(h_W, b.W, W_LEVELS * 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess || hipGetLastError() != hipSuccess)
        rc = MNRT_ERR_HIP;
    else if (h_W[W_ERR] != 0u)
        rc = MNRT_ERR_STATE;
    if (rc != MNRT_OK) {
        (void)pool_free(d_nodes, st);
        (void)pool_free(d_refs, st);
        return rc;
    }
    for (uint32_t s = 0; s < S_; ++s) {
        set_tree(out[s], kind, s, S_, h_res, h_base, d_nodes, d_refs);
        out[s].owns_nodes = (s == 0) ? 1u : 0u;
    }
    return MNRT_OK;
}

// =========================================================================================
// device-driven build, recorded once into a hipGraph
// =========================================================================================
// The same kernels as build_batch_impl, with every buffer fixed and the level loop unrolled to
// a recorded number of levels.  Capacities come from a host-driven build of the same scenes (its
// BuildStats) with a margin; whatever would outgrow them sets an error bit instead.

// Levels a recorded build covers beyond the first build's deepest large-stage node.  The layout climbs
// parent links and could place deeper trees too: the limit is what mnrt_build_graph_status states.
constexpr uint32_t kLayoutSpareLevels = 6u;

// Active nodes left after the last recorded level.
__global__ __launch_bounds__(64) void k_levels_done(uint32_t* __restrict__ W, uint32_t level) {
    if (threadIdx.x == 0 && blockIdx.x == 0 && W[W_ERR] == 0u && W[W_LEVELS + kLevelWords * level + 1] != 0u) W[W_ERR] = kErrLevels;
}

}  // namespace

struct mnrt_build_graph {
    int kind = 0;
    uint32_t ns = 0, ntot = 0;
    std::vector<uint32_t> h_base;      // ns + 1
    std::vector<uint32_t> h_plan;      // kind / index / offset per scene
    std::vector<uint32_t> h_photon;    // slot_begin, box_begin (ns + 1 each, photon_tables)
    std::vector<float> h_qr, h_roots;  // per scene (roots: empty when not given)
    mnrt_build_params prm{};
    const float *v0 = nullptr, *v1 = nullptr, *v2 = nullptr, *pow4 = nullptr, *dir4 = nullptr;
    BuildStats stats;
    BuildCaps cap{};
    uint32_t cap_nodes = 0, cap_refs = 0;  // output arrays (all trees)
    uint32_t levels = 0;
    float margin = 0.25f;
    char* dbuf = nullptr;
    uint64_t dbytes = 0;
    uint32_t* W = nullptr;
    uint32_t* d_tab = nullptr;
    uint32_t* nodes = nullptr;
    uint32_t* refs = nullptr;
    float* recs = nullptr;
    uint32_t* qnodes = nullptr;
    hipStream_t cap_stream = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};

namespace {

// Carves g's device block (base null: measures it) and, when st is given, enqueues the
// whole build on st (which is capturing).  Every launch is a kernel: the sequence has no
// memset, copy or allocation nodes.
int graph_record(mnrt_build_graph& g, char* base, hipStream_t st) {
    const uint32_t S_ = g.ns, ntot = g.ntot;
    const int kind = g.kind;
    const BuildCaps C = g.cap;
    Carver cv(base);
    uint32_t* tab = cv.get<uint32_t>(scene_tab_words(S_));
    const SceneTab T = scene_tab(tab, S_);
    const LevelBufs b = take_levels(cv, kind, S_, C);
    const StageCap st_cap = stage_cap_setting();
    if ((uint64_t)st_cap.mul * C.se + (uint64_t)st_cap.add * C.small > 0xFFFFFFFFull) return MNRT_ERR_CAPACITY;
    SmallOut O = take_small(cv, b.W, st_cap, C.small, C.se);
    // outputs
    uint32_t* nodes = cv.get<uint32_t>(2ull * g.cap_nodes);
    uint32_t* refs = cv.get<uint32_t>(g.cap_refs);
    float* recs = cv.get<float>((uint64_t)g.cap_refs * (kind == MNRT_KIND_TRI ? 12u : 8u));
    // box hierarchies and query-time node words (box_block)
    uint32_t* qnodes = kind == MNRT_KIND_POINT
                           ? cv.get<uint32_t>(box_block(g.h_photon[2 * S_ + 1], S_, g.cap_nodes) + 8u)
                           : nullptr;
    if (!base) {
        g.dbytes = cv.size();
        return MNRT_OK;
    }
    g.W = b.W;
    g.d_tab = tab;
    g.nodes = nodes;
    g.refs = refs;
    g.recs = recs;
    g.qnodes = qnodes;
    if (!st) return MNRT_OK;

    // ---- the recorded sequence ----
    const BuildStats& bs = g.stats;
    const double grow = 1.0 + (double)g.margin;
    auto planned = [&](uint64_t x, uint64_t slack, uint64_t cap) {
        return std::min<uint64_t>(cap, (uint64_t)((double)x * grow) + slack);
    };
    Geometry G{kind, (const float4*)g.v0, g.v1 ? (const float4*)g.v1 : (const float4*)g.v0,
               g.v2 ? (const float4*)g.v2 : (const float4*)g.v0, T.base, S_};
    launch_roots(b, G, ntot, RootPlan{T.pkind, T.pindex, T.poff}, bs.roots,
                 g.h_roots.empty() ? (const float*)nullptr : (const float*)T.given, T.rootbox, T.smaxlvl, st);
    MNRT_HIP_CHECK(hipGetLastError());
    for (uint32_t l = 0; l < g.levels; ++l) {
        const size_t pl = std::min<size_t>(l, bs.level_na.size() - 1);
        launch_level(b, G, g.prm, C, l, planned(bs.level_na[pl], 256, C.na), planned(bs.level_nw[pl], 64, C.nw), st);
        MNRT_HIP_CHECK(hipGetLastError());
    }
    hipLaunchKernelGGL(k_levels_done, dim3(1), dim3(64), 0, st, b.W, g.levels);

    // small-node stage
    const DN nbn = dn(b.W + W_NBN, C.bn), nsm = dn(b.W + W_NSMALL, C.small);
    launch_small<kSmallStage>(kind, nsm, b.S, b.Sm, T.qr, O, st);
    // layout
    // a replay deeper than the first build's depth and a few levels more sets kErrLayoutDepth
    const uint32_t top = std::min<uint32_t>(bs.maxlvl + kLayoutSpareLevels, MNRT_MAX_LEVEL);
    const dim3 lgrid = blocks_for(planned(bs.nbn, 256, C.bn));
    hipLaunchKernelGGL(k_layout_sizes, lgrid, dim3(256), 0, st, nbn, b.B, (const uint32_t*)O.nsize,
                       (const uint32_t*)O.rsize, (const uint32_t*)O.mlvl, top, T.smaxlvl, b.W);
    hipLaunchKernelGGL(k_scene_totals, dim3(1), dim3(1024), 0, st, S_, (const BnRec*)b.B, T.snodes, T.srefs, T.nbase,
                       T.rbase, T.sleaves, g.cap_nodes, g.cap_refs, b.W);
    // emission (each kernel returns at once when W[W_ERR] is set)
    hipLaunchKernelGGL(k_emit_large, lgrid, dim3(256), 0, st, nbn, b.B, (const uint32_t*)b.ll_idx, nodes, refs,
                       (const uint32_t*)b.W, (const uint32_t*)T.nbase, (const uint32_t*)T.rbase);
    O.bn = b.B;
    O.nodes = nodes;
    O.refs = refs;
    O.max_nodes = g.cap_nodes;
    O.max_refs = g.cap_refs;
    O.node_base = T.nbase;
    O.ref_base = T.rbase;
    hipLaunchKernelGGL(k_small_place, dim3((C.small + kSmallWaves - 1) / kSmallWaves), dim3(64 * kSmallWaves), 0, st,
                       nsm, b.S, O);
    // subtrees that outgrew their staging area, built again at their final address
    launch_small<kSmallEmit>(kind, nsm, b.S, b.Sm, T.qr, O, st);
    // records and query-time node words
    const DN nrefs = dn(T.rbase + S_, g.cap_refs), nnodes = dn(T.nbase + S_, g.cap_nodes);
    if (kind == MNRT_KIND_TRI) {
        int rc = launch_tri_records_batch(refs, nrefs, T.rbase, T.base, S_, (const float4*)g.v0, (const float4*)g.v1,
                                          (const float4*)g.v2, (float4*)recs, b.W + W_ERR, st);
        if (rc != MNRT_OK) return rc;
    } else if (g.pow4 && g.dir4) {
        uint32_t max_elems = 0;
        for (uint32_t s = 0; s < S_; ++s) max_elems = std::max(max_elems, g.h_base[s + 1] - g.h_base[s]);
        const PhotonTables tab{S_, T.nbase, T.rbase, T.base, T.slot_begin, T.box_begin};
        int rc = launch_photon_records_batch(refs, tab, g.h_photon[S_], max_elems, (const float4*)g.v0,
                                             (const float4*)g.pow4, (const float4*)g.dir4, (float4*)recs,
                                             (float4*)qnodes, b.W + W_ERR, st);
        if (rc == MNRT_OK)
            rc = launch_collapse_batch((const uint2*)nodes, nnodes, T.nbase, S_, T.box_begin, kQueryLeafRefs,
                                       (uint2*)qnodes, b.W + W_ERR, st);
        if (rc != MNRT_OK) return rc;
    }
    MNRT_HIP_CHECK(hipGetLastError());
    return MNRT_OK;
}

}  // namespace

extern "C" int mnrt_build_tri(const float* d_v0, const float* d_v1, const float* d_v2, uint32_t n,
                              const mnrt_build_params* params, mnrt_tree* out, void* stream) {
    if (!params || !out) return MNRT_ERR_ARG;
    uint32_t base[2] = {0, n};
    const float* root = params->has_root_box ? params->root_min : nullptr;
    float r6[6];
    if (root) {
        for (int k = 0; k < 3; ++k) {
            r6[k] = params->root_min[k];
            r6[3 + k] = params->root_max[k];
        }
    }
    int rc = build_batch_impl(MNRT_KIND_TRI, d_v0, d_v1, d_v2, base, 1, params, root ? r6 : nullptr, nullptr, out,
                              (hipStream_t)stream);
    if (rc != MNRT_OK) return rc;
    rc = mnrt_tree_attach_tri_records(out, d_v0, d_v1, d_v2, stream);
    if (rc != MNRT_OK) mnrt_tree_release(out);
    return rc;
}

extern "C" int mnrt_build_points(const float* d_pos4, uint32_t n, const mnrt_build_params* params, mnrt_tree* out,
                                 void* stream) {
    if (!params || !out) return MNRT_ERR_ARG;
    uint32_t base[2] = {0, n};
    float r6[6];
    for (int k = 0; k < 3; ++k) {
        r6[k] = params->root_min[k];
        r6[3 + k] = params->root_max[k];
    }
    return build_batch_impl(MNRT_KIND_POINT, d_pos4, nullptr, nullptr, base, 1, params,
                            params->has_root_box ? r6 : nullptr, nullptr, out, (hipStream_t)stream);
}

extern "C" int mnrt_build_tri_batch(const float* d_v0, const float* d_v1, const float* d_v2,
                                    const uint32_t* h_offsets, uint32_t num_scenes, const mnrt_build_params* params,
                                    const float* h_root_boxes, mnrt_tree* out, void* stream) {
    int rc = build_batch_impl(MNRT_KIND_TRI, d_v0, d_v1, d_v2, h_offsets, num_scenes, params, h_root_boxes, nullptr,
                              out, (hipStream_t)stream);
    if (rc != MNRT_OK) return rc;
    rc = mnrt_tree_attach_tri_records_batch(out, num_scenes, d_v0, d_v1, d_v2, h_offsets, stream);
    if (rc != MNRT_OK) mnrt_tree_release(out);
    return rc;
}

extern "C" int mnrt_build_points_batch(const float* d_pos4, const uint32_t* h_offsets, uint32_t num_scenes,
                                       const mnrt_build_params* params, const float* h_root_boxes,
                                       const float* h_max_query_radius, mnrt_tree* out, void* stream) {
    return build_batch_impl(MNRT_KIND_POINT, d_pos4, nullptr, nullptr, h_offsets, num_scenes, params, h_root_boxes,
                            h_max_query_radius, out, (hipStream_t)stream);
}

// ---- device-driven batched build (mnrt_build_graph_*) ------------------------------------

extern "C" int mnrt_build_graph_create(const mnrt_build_graph_desc* d, mnrt_tree* out, mnrt_build_graph** g_out,
                                       void* stream) {
    using namespace mnrt;
    if (!d || !out || !g_out || !d->params || !d->h_offsets || d->num_scenes == 0) return MNRT_ERR_ARG;
    if (d->kind != MNRT_KIND_TRI && d->kind != MNRT_KIND_POINT) return MNRT_ERR_ARG;
    if (!(d->margin >= 0.0f && d->margin <= 16.0f)) return MNRT_ERR_ARG;
    *g_out = nullptr;
    const uint32_t S_ = d->num_scenes;
    const uint32_t ntot = d->h_offsets[S_];
    if (ntot > 0 && (!d->d_v0 || (d->kind == MNRT_KIND_TRI && (!d->d_v1 || !d->d_v2)))) return MNRT_ERR_ARG;
    if (d->kind == MNRT_KIND_POINT && (!d->d_power4) != (!d->d_dir4)) return MNRT_ERR_ARG;
    hipStream_t st = (hipStream_t)stream;
    auto* g = new (std::nothrow) mnrt_build_graph;
    if (!g) return MNRT_ERR_NOMEM;
    auto fail = [&](int rc) {
        (void)mnrt_build_graph_destroy(g);
        return rc;
    };
    g->kind = d->kind;
    g->ns = S_;
    g->ntot = ntot;
    g->prm = *d->params;
    g->v0 = d->d_v0;
    g->v1 = d->d_v1;
    g->v2 = d->d_v2;
    g->pow4 = d->d_power4;
    g->dir4 = d->d_dir4;
    g->margin = d->margin;
    g->h_base.assign(d->h_offsets, d->h_offsets + S_ + 1);
    if (d->h_root_boxes) g->h_roots.assign(d->h_root_boxes, d->h_root_boxes + 6ull * S_);
    g->h_qr.assign(S_, d->params->max_query_radius);
    if (d->h_max_query_radius)
        for (uint32_t s = 0; s < S_; ++s) g->h_qr[s] = d->h_max_query_radius[s];

    // 1. a host-driven build of the same scenes: sizes for the fixed buffers
    {
        std::vector<mnrt_tree> tmp(S_);
        int rc = build_batch_impl(d->kind, d->d_v0, d->d_v1, d->d_v2, d->h_offsets, S_, d->params, d->h_root_boxes,
                                  d->h_max_query_radius, tmp.data(), st, &g->stats);
        if (rc != MNRT_OK) return fail(rc);
        (void)hipStreamSynchronize(st);
        (void)mnrt_tree_release(&tmp[0]);
    }
    const BuildStats& bs = g->stats;
    const double grow = 1.0 + (double)d->margin;
    auto cap = [&](uint64_t x, uint64_t slack) -> uint32_t {
        return (uint32_t)std::min<uint64_t>(MNRT_INDEX_MASK, (uint64_t)((double)x * grow) + slack);
    };
    // room for a replay that needs, at any level, the children of the widest level on top of the
    // first build's totals
    BuildCaps& C = g->cap;
    C.na = cap(bs.max_na, 64);
    C.nw = cap(bs.max_nw, 16ull + C.na);
    C.bn = cap(bs.nbn + 14ull * bs.max_na, 1024);
    C.small = cap(bs.nsmall + 2ull * bs.max_na, 256);
    C.se = cap(bs.nse + 128ull * bs.max_nw, 1024);
    C.ll = cap(bs.ll + 64ull * bs.max_nw, 1024);
    C.nw = std::min<uint32_t>(C.nw, MNRT_INDEX_MASK / 64u);
    g->cap_nodes = cap(bs.total_nodes, 1024);
    g->cap_refs = cap(bs.total_refs, 1024);
    g->levels = bs.level_na.empty() ? 0u
                                    : std::min<uint32_t>((uint32_t)bs.level_na.size() + 2u, MNRT_MAX_LEVEL + 1u);
    g->h_plan.assign(3ull * S_, 0u);
    (void)plan_roots(g->h_base.data(), S_, g->prm.small_node_max, g->h_plan.data(), g->h_plan.data() + S_,
                     g->h_plan.data() + 2ull * S_);

    g->h_photon.assign(2ull * (S_ + 1), 0u);
    if (g->kind == MNRT_KIND_POINT) {
        std::vector<uint32_t> elems(S_);
        for (uint32_t s = 0; s < S_; ++s) elems[s] = g->h_base[s + 1] - g->h_base[s];
        photon_tables(elems.data(), S_, g->h_photon.data(), g->h_photon.data() + S_ + 1);
    }

    // 2. the fixed device block, and the per-scene tables in it
    int rc = graph_record(*g, nullptr, nullptr);
    if (rc != MNRT_OK) return fail(rc);
    if (device_alloc((void**)&g->dbuf, g->dbytes) != hipSuccess) {
        g->dbuf = nullptr;
        return fail(MNRT_ERR_NOMEM);
    }
    rc = graph_record(*g, g->dbuf, nullptr);
    if (rc != MNRT_OK) return fail(rc);
    {
        const SceneTab T = scene_tab(g->d_tab, S_);
        std::vector<float> fq(S_ + 6ull * S_, 0.0f);
        for (uint32_t s = 0; s < S_; ++s) fq[s] = g->h_qr[s];
        for (size_t i = 0; i < g->h_roots.size(); ++i) fq[S_ + i] = g->h_roots[i];
        if (hipMemcpy(T.base, g->h_base.data(), 4ull * (S_ + 1), hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(T.pkind, g->h_plan.data(), 12ull * S_, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(T.qr, fq.data(), 4ull * fq.size(), hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(T.slot_begin, g->h_photon.data(), 8ull * (S_ + 1), hipMemcpyHostToDevice) != hipSuccess)
            return fail(MNRT_ERR_HIP);
    }

    // 3. record the device-driven build
    if (hipStreamCreateWithFlags(&g->cap_stream, hipStreamNonBlocking) != hipSuccess) {
        g->cap_stream = nullptr;
        return fail(MNRT_ERR_HIP);
    }
    if (hipStreamBeginCapture(g->cap_stream, hipStreamCaptureModeThreadLocal) != hipSuccess) return fail(MNRT_ERR_HIP);
    rc = graph_record(*g, g->dbuf, g->cap_stream);
    hipGraph_t graph = nullptr;
    const hipError_t ce = hipStreamEndCapture(g->cap_stream, &graph);
    g->graph = graph;
    if (rc != MNRT_OK) return fail(rc);
    if (ce != hipSuccess || !graph) return fail(MNRT_ERR_HIP);
    if (hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0) != hipSuccess) {
        g->exec = nullptr;
        return fail(MNRT_ERR_HIP);
    }

    // 4. one replay: the trees in out[], which must equal the host-driven build's
    rc = mnrt_build_graph_replay(g, stream);
    uint32_t flags = 0;
    if (rc == MNRT_OK) rc = mnrt_build_graph_status(g, out, &flags, stream);
    if (rc == MNRT_OK && flags != 0u) rc = MNRT_ERR_STATE;
    if (rc != MNRT_OK) return fail(rc);
    *g_out = g;
    return MNRT_OK;
}

extern "C" int mnrt_build_graph_replay(mnrt_build_graph* g, void* stream) {
    if (!g || !g->exec) return MNRT_ERR_ARG;
    MNRT_HIP_CHECK(hipGraphLaunch(g->exec, (hipStream_t)stream));
    return MNRT_OK;
}

extern "C" int mnrt_build_graph_status(mnrt_build_graph* g, mnrt_tree* out, uint32_t* h_flags, void* stream) {
    using namespace mnrt;
    if (!g || !g->dbuf || !h_flags) return MNRT_ERR_ARG;
    hipStream_t st = (hipStream_t)stream;
    const uint32_t S_ = g->ns;
    const SceneTab T = scene_tab(g->d_tab, S_);
    uint32_t err = 0;
    std::vector<uint32_t> res(scene_result_words(S_));
    MNRT_HIP_CHECK(hipStreamSynchronize(st));
    MNRT_HIP_CHECK(hipMemcpy(&err, g->W + W_ERR, 4, hipMemcpyDeviceToHost));
    MNRT_HIP_CHECK(hipMemcpy(res.data(), T.rootbox, 4ull * res.size(), hipMemcpyDeviceToHost));
    *h_flags = err;
    if (err != 0u || !out) return MNRT_OK;
    const uint32_t* hnb = res.data() + 8ull * S_;
    const uint32_t* hrb = hnb + S_ + 1;
    const uint32_t per = g->kind == MNRT_KIND_TRI ? 12u : 8u;
    const bool recs = g->kind == MNRT_KIND_TRI || (g->pow4 && g->dir4);
    for (uint32_t s = 0; s < S_; ++s) {
        mnrt_tree& t = out[s];
        // the arrays belong to the graph (mnrt_build_graph_destroy frees them)
        set_tree(t, g->kind, s, S_, res.data(), g->h_base.data(), g->nodes, g->refs);
        t.d_recs = recs ? g->recs + (uint64_t)per * hrb[s] : nullptr;
        if (g->kind == MNRT_KIND_POINT && recs) {
            const uint32_t* bb = g->h_photon.data() + S_ + 1;
            t.d_qnodes = g->qnodes + box_block(bb[s], s, hnb[s]) + (bb[s + 1] - bb[s]);
            t.qleaf_max = kQueryLeafRefs;
            t.owns_qnodes = MNRT_QNODES_BOXES;
        }
    }
    return MNRT_OK;
}

extern "C" int mnrt_build_graph_destroy(mnrt_build_graph* g) {
    if (!g) return MNRT_OK;
    (void)hipDeviceSynchronize();
    if (g->exec) (void)hipGraphExecDestroy(g->exec);
    if (g->graph) (void)hipGraphDestroy(g->graph);
    if (g->cap_stream) (void)hipStreamDestroy(g->cap_stream);
    if (g->dbuf) (void)hipFree(g->dbuf);
    delete g;
    return MNRT_OK;
}
