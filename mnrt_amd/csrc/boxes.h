// boxes.h — box hierarchy over a photon tree's leaf-ordered records, which the kNN kernels
// walk instead of the binary node words.
//
// The records lie in the kd-tree's leaf order, so 64 consecutive ones (a group: one wave's
// batch) are close in space whatever leaves they come from.  Level 0 holds the exact bounds
// of every group, level 1 those of 64 consecutive groups, level 2 those of 64 level-1
// boxes: three wave-wide box tests lead to the groups that can hold a neighbour.  Against
// query-time leaves of up to 512 photons reached through binary nodes a query (1M photons,
// k = 100) tests 13 groups instead of 27 batches of 64 and makes 8 box tests instead of
// visiting 28 inner nodes one dependent scalar load after the other.
//
// A box is two float4 (lo, hi).  Levels are padded to whole waves with empty boxes (+inf,
// -inf), whose distance is +inf, so box tests need no lane masks.  The hierarchy lies right
// before the tree's query-time node words (d_qnodes) and its size depends on num_elems only;
// MNRT_QNODES_BOXES in owns_qnodes says that it is there.
#pragma once

#include <type_traits>

#include "mnrt_common.h"

namespace mnrt {

__host__ __device__ constexpr uint32_t pad64(uint32_t n) { return (n + 63u) & ~63u; }

struct BoxGeom {
    uint32_t g0, s0;  // groups; slots of level 0 (padded to 64)
    uint32_t g1, s1;
    uint32_t g2, s2;
};
// Hierarchy of a tree of at most `elems` references.
__host__ __device__ constexpr BoxGeom box_geom(uint32_t elems) {
    BoxGeom g{};
    g.g0 = (elems + 63u) / 64u;
    g.s0 = pad64(g.g0);
    g.g1 = g.s0 / 64u;
    g.s1 = pad64(g.g1);
    g.g2 = g.s1 / 64u;
    g.s2 = pad64(g.g2);
    return g;
}
// 4-byte words of the hierarchy (a multiple of 8; 0 for an empty tree).
__host__ __device__ constexpr uint64_t box_words(uint32_t elems) {
    const BoxGeom g = box_geom(elems);
    return 8ull * ((uint64_t)g.s0 + g.s1 + g.s2);
}

// Batches: one array holds, scene by scene, the hierarchy and then the query-time node words.
// First word of scene s's hierarchy: box_begin[s] is the sum of box_words over the scenes
// before it, nbase[s] the nodes of the trees before it; 8 words of slack a scene let every
// hierarchy start 32-byte aligned.
__host__ __device__ constexpr uint64_t box_block(uint64_t box_begin_s, uint32_t s, uint64_t nbase_s) {
    return box_begin_s + 8ull * s + ((2ull * nbase_s + 7ull) & ~7ull);
}

// What a query needs of a tree's hierarchy (p null: the tree has none).
struct BoxTree {
    const float4* p;
    uint32_t nrefs;   // references (the last group may be partial)
    uint32_t o1, o2;  // first box of levels 1 and 2
    uint32_t g1, g2;  // boxes of levels 1 and 2
    uint32_t end;     // boxes of all levels, padding included
};

inline BoxTree box_tree(const mnrt_tree& t) {
    BoxTree b{};
    if (!(t.owns_qnodes & MNRT_QNODES_BOXES) || !t.d_qnodes) return b;
    const BoxGeom g = box_geom(t.num_elems);
    b.p = (const float4*)(t.d_qnodes - box_words(t.num_elems));
    b.nrefs = t.num_refs;
    b.o1 = g.s0;
    b.o2 = g.s0 + g.s1;
    b.end = g.s0 + g.s1 + g.s2;
    b.g1 = g.g1;
    b.g2 = g.g2;
    return b;
}

__device__ __forceinline__ float wave_min_f32(float v) {
    auto dpp = [](float x, auto ctrl) { return __uint_as_float(dpp_mov<decltype(ctrl)::value>(__float_as_uint(x))); };
    v = fminf(v, dpp(v, std::integral_constant<int, kDppPairSwap>{}));
    v = fminf(v, dpp(v, std::integral_constant<int, kDppQuadSwap>{}));
    v = fminf(v, dpp(v, std::integral_constant<int, kDppHalfMirror>{}));
    v = fminf(v, dpp(v, std::integral_constant<int, kDppRowMirror>{}));
    const uint32_t u = __float_as_uint(v);
    return fminf(fminf(__uint_as_float(row_lane(u, 0)), __uint_as_float(row_lane(u, 1))),
                 fminf(__uint_as_float(row_lane(u, 2)), __uint_as_float(row_lane(u, 3))));
}

struct Box {
    float4 lo, hi;
};

__device__ __forceinline__ Box empty_box() {
    const float inf = __uint_as_float(0x7F800000u);
    return Box{make_float4(inf, inf, inf, 0.0f), make_float4(-inf, -inf, -inf, 0.0f)};
}

// Bounds of the boxes held one per lane, in every lane (NaN coordinates are ignored:
// fminf returns the other operand).
__device__ __forceinline__ Box wave_box(const Box& b) {
    return Box{make_float4(wave_min_f32(b.lo.x), wave_min_f32(b.lo.y), wave_min_f32(b.lo.z), 0.0f),
               make_float4(-wave_min_f32(-b.hi.x), -wave_min_f32(-b.hi.y), -wave_min_f32(-b.hi.z), 0.0f)};
}

}  // namespace mnrt
