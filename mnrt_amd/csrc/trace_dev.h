// trace_dev.h — closest-hit and any-hit traversal of the packed preorder kd-tree (device
// functions), shared by the ray kernels (trace.hip, shadow.hip) and the photon tracer
// (photon.hip).
//
// dev_FindNextIntersectionKDWhileWhile (raytracing.cu:503-645) restated for the SoA node
// words and leaf-ordered triangle records:
//   * interval decisions are widened by a relative 2^-16 (split parameter NaN for a ray
//     lying in the plane: both children; tsplit < 0 or beyond tmax: near child; before
//     tmin: far child; else both), and equal lambdas resolve to the lower triangle
//     index, so the hit equals the brute-force closest hit whatever the tree;
//   * a popped node is skipped when the best hit lies before its tmin (the reference
//     ends the search at the first leaf whose tmax exceeds the best hit, which misses
//     hits in a sibling pushed for a ray lying in the split plane);
//   * the stack is bounded by the build's level cap; its top kLds entries per lane live
//     in LDS, deeper ones in the lane's private array (the reference keeps the whole
//     stack in local memory).
//
// A wave traces windows of rays (trace_stream), not one ray per lane to its end.  With a lane per
// ray the wave steps until its longest ray is done and tests as many triangles per leaf as the
// fullest leaf among its lanes holds: for bounce rays 10 % of the lanes worked (47 k wave
// instructions per 64 rays, 68 triangle tests a ray).  So, unless the rays go together (kTogether),
//   * a lane whose ray is done takes the next ray, kRefill lanes at a time;
//   * lanes walk to their next leaf until fewer than kWalkMin still walk, and wait there;
//   * the waiting leaves' (ray, triangle) pairs are dealt to all lanes, 64 at a time, unless
//     the lanes' own leaves are about as full as each other, when each lane tests its own.
// Bound by instruction issue: about 25 k vector instructions per 64 bounce rays of the 1.03M-triangle
// scene (206 walk steps with 29 lanes, 85 dealt tests with 49 pairs, 37 own tests), 83 tests and 93
// steps a ray.  A lane per ray and now, us: 2.07M bounce rays of 1.03M triangles 2698 and 1738, 785 k
// area-light shadow rays of 205001 triangles 981 and 781, 6144 camera rays of 1294 triangles 63 and 46;
// 2.07M camera rays of 1.03M triangles 1043 and 977, of 205001 1172 and 1264, of 1294 213 and 221.
#pragma once

#include "mnrt_common.h"

namespace mnrt {

struct RootBox {
    float lo[3], hi[3];
};

struct Hit {
    int32_t tri;
    float t;
    uint32_t rec;  // the triangle's record
};

constexpr int kTraceStack = MNRT_MAX_LEVEL + 2;

// LDS entries per lane of the traversal stack: as many as leave room for 24 waves on a CU.  On
// the 1M-triangle workload 5 % of pushes land deeper than 6 entries, so some lane of a wave often
// goes to scratch memory there; 6 entries instead of 7: 1670 -> 1721 us.
constexpr int kTraceLds = 7;

// Waves that run at once: 24 per CU (80 registers, 6.4 KB of LDS).
constexpr uint32_t kTraceWaves = 6144, kWindowWaves = kTraceWaves + kTraceWaves / 2u;

// Rays a wave traces at once: 64, or fewer while all the waves run at once: a wave's longest ray
// and fullest leaves are then shorter, and the spare lanes test triangles.  6144 camera rays: 16 a
// wave 44 us, 64 a wave 69 us; 131044 bounce rays (205001 triangles): 32 a wave 421 us, 64 466 us.
inline uint32_t trace_width(uint64_t n) { return n > 32u * kTraceWaves ? 64u : n > 16u * kTraceWaves ? 32u : 16u; }
inline uint32_t trace_windows(uint64_t n, uint32_t width) { return (uint32_t)((n + width - 1u) / width); }

// Of 64 rays, the lanes that take new rays together and the least number that goes on walking while
// others wait at leaves.  16..32 and 6..16 are within 4 % of each other on bounce rays, shadow rays
// and photon paths; fewer walkers suit small launches.
constexpr uint32_t kRefill = 24, kWalkMin = 10;
// A set of 64 rays of which on average at least kTogether lanes walk, while at least kEarly are
// still traced, is traced to its end as it is: for camera rays every refill, wait and dealt test is
// overhead.  Between 24 and 36, bounce rays gain 2 % and camera rays lose 10 %; at 18 bounce rays
// lose 10 %.  So is a set of which fewer than kEarly have anything to trace (the others miss the root box, or
// a light's back): dealt and refilled instead, camera rays past an object take 77 -> 95 us (784 k, 205001
// triangles), bounce rays of an open scene and shadow rays the same within 2 %.  A source whose kTogether is
// above 64 has no such sets.
constexpr uint32_t kEarly = 48, kRaysTogether = 24;

// LDS words of a wave: pair owners and best records (64 each), best keys (64 x 2), stack.
constexpr uint32_t kTraceWords = 256u + 3u * 64u * (uint32_t)kTraceLds;

// Rays of a wave: a window of `width` consecutive ones, a wave per window, which the hardware starts as
// others end.  In launches of more than kWindowWaves windows a wave whose rays do not go together takes
// further ones, from the launch's end, whose own waves then find them taken: lanes that refill gain more
// than new waves do (1.69M bounce rays 1483 us with windows from a counter, a wave per window 2093).  Rays
// that go together, or miss the root box, leave the rest to the hardware.  2.07M rays with a window from
// a counter for every 64, whose atomics come 12 ns apart, and now: camera rays of 1294 triangles 420 and
// 221 us, of which most miss the box 398 and 50, of 1.03M triangles 1002 and 977; bounce rays of 1.03M 1713 and
// 1738 (two atomics a window, and waves that find theirs taken).  (From the end by a fixed stride
// instead of a count: bounce rays 5 to 10 % slower, camera rays up to 9 % faster; 128 rays a window: bounce
// rays 4 to 7 % slower; a fixed share of the rays for every wave that fits at once: waves of slow rays end
// late, camera rays up to 40 % slower.)  Shadow rays always have a wave per window: 1.76M from a point
// light (20000 triangles) 427 us, with windows from a counter 592.
struct RayWindow {
    uint32_t next, end;  // rays of the window not handed out yet
    uint32_t n, width;
    uint32_t* shared;    // kShared*; null: the wave's own window is all
    bool open;           // there may be more windows

    // span: the first window's rays, if more than width.
    __device__ __forceinline__ RayWindow(uint32_t first, uint32_t n_, uint32_t width_, uint32_t* shared_, uint32_t span = 0u)
        : next(min(first, n_)), end(next + min(max(width_, span), n_ - next)), n(n_), width(width_), shared(shared_), open(shared_ != nullptr) {}
    // Words that the waves of a launch share: windows taken from the end, then, from kSharedTaken on, a
    // word for every window but the first kTraceWaves, whose waves start at once: 1 when it is taken.
    static constexpr uint32_t kSharedTaken = 32;
    static constexpr uint64_t shared_words(uint32_t windows) { return kSharedTaken + (windows - kTraceWaves); }
    // Takes window w for this wave; false if another has it (uniform, whole wave).
    static __device__ __forceinline__ bool claim(uint32_t* shared, uint32_t w, uint32_t lane) {
        if (w < kTraceWaves) return true;
        uint32_t old = 0;
        if (lane == 0u) old = atomicExch(shared + kSharedTaken + (w - kTraceWaves), 1u);
        return uniform(old) == 0u;
    }
    // Another window, if there is one (uniform, whole wave).  A window that is taken already has been
    // started by the hardware, and so have those before it.
    __device__ __forceinline__ void take(uint32_t lane) {
        uint32_t c = 0;
        if (lane == 0u) c = atomicAdd(shared, 1u);
        c = uniform(c);
        const uint32_t w = gridDim.x - 1u - c;
        open = c < gridDim.x - kTraceWaves && claim(shared, w, lane);
        next = open ? w * width : n;
        end = next + min(width, n - next);
    }
};

// The shared words of a launch of `windows` on a stream, or null where none are needed or to be had (then
// every wave has its own window).  They live until the launch is done.
class RayShared {
   public:
    RayShared(uint32_t windows, hipStream_t st);
    ~RayShared();
    uint32_t* p = nullptr;

   private:
    hipStream_t st_;
};

// Per-lane traversal stack of kStack entries (node, tmin, tmax).  Entry e < kTraceLds is in
// LDS, (node, tmin) at pair e * 64 + lane and tmax at word e * 64 + lane of an array of its own
// (lanes of a wave touch consecutive banks); deeper entries in a private array.  kStack entries
// suffice for a tree of max level <= kStack: the entries are far children of distinct levels of the
// current path.
// (Only the array is a struct in memory: a pointer beside it would be loaded from scratch too.)
template <int kStack>
struct DeepStack {
    static constexpr int kPriv = kStack > kTraceLds ? kStack - kTraceLds : 1;
    unsigned long long lo[kPriv];
    float hi[kPriv];
};
struct LdsStack {
    __attribute__((address_space(3))) unsigned long long* lo;
    __attribute__((address_space(3))) float* hi;
};
template <int kStack>
__device__ __forceinline__ void stack_put(const LdsStack& l, DeepStack<kStack>& m, int e, uint32_t node, float a, float b) {
    const unsigned long long v = (unsigned long long)__float_as_uint(a) << 32 | node;
    if (e < kTraceLds) {
        l.lo[e * 64] = v;
        l.hi[e * 64] = b;
    } else {
        m.lo[e - kTraceLds] = v;
        m.hi[e - kTraceLds] = b;
    }
}
template <int kStack>
__device__ __forceinline__ void stack_get(const LdsStack& l, const DeepStack<kStack>& m, int e, uint32_t& node, float& a,
                                          float& b) {
    unsigned long long v;
    if (e < kTraceLds) {
        v = l.lo[e * 64];
        b = l.hi[e * 64];
    } else {
        v = m.lo[e - kTraceLds];
        b = m.hi[e - kTraceLds];
    }
    node = (uint32_t)v;
    a = __uint_as_float((uint32_t)(v >> 32));
}

// Calls test(a, e1, e2, r) on the count triangle records from rec (3 float4 each) until it
// returns true; returns whether it did.  Two record buffers alternate, so the next record
// loads while the current one is tested and no registers are copied between tests; the
// loads are unconditional (past the leaf's end they re-read its last record, which is
// not tested again), so the wait before a test leaves the next record's loads in flight.
template <typename F>
__device__ __forceinline__ bool for_leaf_tris(const float4* rec, uint32_t count, F&& test) {
    if (count == 0) return false;
    float4 a0 = rec[0], b0 = rec[1], c0 = rec[2];
    const uint32_t last = count - 1u;
    for (uint32_t r = 0;; r += 2) {
        const float4* p1 = rec + 3u * min(r + 1u, last);
        const float4 a1 = p1[0], b1 = p1[1], c1 = p1[2];
        if (test(a0, b0, c0, r)) return true;
        if (r + 1 >= count) return false;
        const float4* p2 = rec + 3u * min(r + 2u, last);
        a0 = p2[0];
        b0 = p2[1];
        c0 = p2[2];
        if (test(a1, b1, c1, r + 1u)) return true;
        if (r + 2 >= count) return false;
    }
}

// Order of floats as unsigned words (any sign).
__device__ __forceinline__ uint32_t order_bits(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float order_float(uint32_t u) {
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u);
}

__device__ __forceinline__ uint32_t from_lane(uint32_t v, uint32_t lane) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(lane * 4u), (int)v);
}
__device__ __forceinline__ float from_lane(float v, uint32_t lane) {
    return __uint_as_float(from_lane(__float_as_uint(v), lane));
}

// Traces the rays a source hands out to the wave's lanes, until it has no more.
//   src.rays: ray numbers to hand out (RayWindow);
//   src.start(i, o, d, dist): ray i; false when there is nothing to trace;
//   src.finish(o, d, dist, hit): result of the lane's ray; true when the lane goes on with
//     another ray that it put in o, d.
// Closest hit (kAny false): the brute-force closest hit, lambda > eps, up to where the ray leaves
// the root box, + eps.
// Any hit (dev_FindNextIntersectionKDWhileWhile<false>, raytracing.cu:503-645, as the
// shadow-ray kernels use it, raytracing.cu:1019-1114): hit.tri >= 0 iff some triangle is hit at
// lambda with
//     lambda > eps,  lambda < min(t_exit, dist) + eps,  lambda + slack < dist
// (t_exit: where the ray leaves the root box).  The reference tests only the first
// hit it meets against the light distance (`lambda >= distance`, `lambda + eps >=
// distance`), so which triangle decides depends on the order of a leaf's list; here
// any occluding triangle decides, so the result equals the brute-force predicate
// whatever the tree.  The search ends at the first occluder.
// lds: the wave's kTraceWords.  Whole wave, every lane active.
template <bool kAny, int kStack, typename Src>
__device__ __forceinline__ void trace_stream(const uint2* __restrict__ nodes, const float4* __restrict__ recs,
                                             const RootBox& root, float eps, float slack, uint32_t* lds, Src& src) {
    typedef __attribute__((address_space(3))) uint32_t lds_u32;
    typedef __attribute__((address_space(3))) unsigned long long lds_u64;
    enum : uint32_t { kIdle, kDone, kWalk, kLeaf };
    const uint32_t lane = threadIdx.x & 63u;
    lds_u32* own = (lds_u32*)lds;
    lds_u32* brec = own + 64;
    lds_u64* key = (lds_u64*)(own + 128);
    DeepStack<kStack> deep;
    const LdsStack top{(lds_u64*)(own + 256) + lane, (__attribute__((address_space(3))) float*)(own + 256 + 128 * kTraceLds) + lane};
    const uint32_t width = src.rays.width;
    uint32_t steps = 0, lanes = 0;
    const uint32_t refill = width * kRefill / 64u, walk_min = width * kWalkMin / 64u;
    uint32_t state = kIdle, node = 0, best_rec = 0;
    int32_t best_tri = -1;
    f3 o = mk3(0.0f, 0.0f, 0.0f), d = o, inv = o;
    float dist = 0.0f, best_t = 0.0f, tmin = 0.0f, tmax = 0.0f;  // best_t: any hit: the limit on lambda
    int sp = 0;
    uint2 nd = make_uint2(0u, 0u);

    auto pop = [&]() {
        state = kDone;
        while (sp > 0) {
            stack_get(top, deep, --sp, node, tmin, tmax);
            if (!kAny && best_tri >= 0 && best_t < tmin) continue;
            nd = nodes[node];
            state = kWalk;
            break;
        }
    };
    // One step of a walking lane.
    auto step = [&]() {
        if (is_leaf(nd.y)) {
            if (nd.x != 0u) state = kLeaf;
            else pop();
        } else {
            const uint32_t a = nd.y >> 30;
            const float s = __uint_as_float(nd.x);
            const uint32_t left = node + 1, right = nd.y & MNRT_INDEX_MASK;
            const float oa = comp(o, a), da = comp(d, a), ia = comp(inv, a);
            const float tsplit = (s - oa) * ia;
            const bool below = (oa < s) | ((oa == s) & (da > 0.0f));
            const uint32_t first = below ? left : right, second = below ? right : left;
            // (a NaN tsplit compares false throughout: both children over the whole interval)
            const bool near = (tsplit < 0.0f) | (tsplit > tmax * kTravTolHi);
            const bool far = !near & (tsplit < tmin * kTravTolLo);
            node = far ? second : first;
            nd = nodes[node];
            if (!(near | far)) {
                if (sp < kStack) stack_put(top, deep, sp++, second, fmaxf(tmin, tsplit * kTravTolLo), tmax);
                tmax = fminf(tmax, tsplit * kTravTolHi);
            }
        }
    };
    // The lane's own leaf.
    auto own_tests = [&]() {
        const uint32_t begin = nd.y & MNRT_INDEX_MASK;
        for_leaf_tris(recs + 3ull * begin, nd.x, [&](const float4& a4, const float4& e14, const float4& e24, uint32_t r) {
            float lam, u, v;
            if (!(ray_tri(xyz(a4), xyz(e14), xyz(e24), o, d, lam, u, v) && lam > eps)) return false;
            if (kAny) {
                if (!(lam < best_t && lam + slack < dist)) return false;
                best_tri = 0;
                return true;
            }
            const int32_t tri = (int32_t)__float_as_uint(a4.w);
            if (lam < best_t || (lam == best_t && best_tri >= 0 && tri < best_tri)) {
                best_t = lam;
                best_tri = tri;
                best_rec = begin + r;
            }
            return false;
        });
    };
    for (;;) {
        const bool together = Src::kTogether <= 64u && width == 64u && lanes >= steps * Src::kTogether;
        const uint32_t busy = (uint32_t)__popcll(ballot(state >= kWalk));
        const uint32_t done = (uint32_t)__popcll(ballot(state == kDone));
        // rays that walk together (steps, lanes: of the set so far) end together: the wave waits for them
        if (busy == 0u || ((src.rays.open || src.rays.next < src.rays.end ? width - busy : done) >= refill && !together)) {
            if (busy == 0u) {
                if (src.rays.next == src.rays.end && lanes >= steps * Src::kTogether) src.rays.open = false;
                steps = lanes = 0u;
            }
            bool ray = false;
            if (state == kDone) {
                ray = src.finish(o, d, dist, Hit{best_tri, best_t, best_rec});
                state = kIdle;
            }
            const bool want = state == kIdle && !ray && lane < width;
            if (src.rays.next == src.rays.end && src.rays.open) src.rays.take(lane);
            const uint64_t m = ballot(want);
            const uint32_t rank = mask_prefix(m), left = src.rays.end - src.rays.next;
            if (want && rank < left) ray = src.start(src.rays.next + rank, o, d, dist);
            src.rays.next += min((uint32_t)__popcll(m), left);
            if (ray) {
                inv = mk3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
                best_tri = -1;
                sp = 0;
                node = 0;
                float t0, t1;
                state = kDone;
                if (ray_box(root.lo, root.hi, o, inv, eps, kInf, t0, t1)) {
                    best_t = (kAny ? fminf(t1, dist) : t1) + eps;
                    tmin = t0;
                    tmax = best_t;
                    nd = nodes[0];
                    state = kWalk;
                }
            }
            if (ballot(state != kIdle) == 0ull && left == 0u && !src.rays.open) break;
        }
        if (together) {
            // every lane to its leaf, and through it
            for (;;) {
                const uint32_t walking = (uint32_t)__popcll(ballot(state == kWalk));
                if (walking == 0u) break;
                if (busy >= kEarly) {
                    ++steps;
                    lanes += walking;
                }
                if (state == kWalk) step();
            }
            if (state == kLeaf) {
                own_tests();
                if (kAny && best_tri >= 0) state = kDone;
                else pop();
            }
            continue;
        }
        // to the next leaf
        for (;;) {
            const uint64_t m = ballot(state == kWalk);
            const uint32_t walking = (uint32_t)__popcll(m);
            if (walking == 0u || (walking < walk_min && ballot(state == kLeaf) != 0ull)) break;
            if (state == kWalk) step();
        }
        const bool at_leaf = state == kLeaf;
        if (ballot(at_leaf) == 0ull) continue;
        const uint32_t cnt = at_leaf ? nd.x : 0u, begin = nd.y & MNRT_INDEX_MASK;
        const uint32_t incl = wave_scan_u32(cnt), total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        const uint32_t most = wave_max_u32(cnt);
        if (3u * ((total + 63u) >> 6) >= 2u * most) {
            // about equally full leaves (a lane's own test costs two thirds of a dealt one)
            if (at_leaf)
                own_tests();
        } else {
            const uint32_t first = incl - cnt, shift = begin - first;
            // a key is (lambda, triangle); before any hit (limit, 0), which no hit equals or
            // exceeds and counts
            const unsigned long long key0 =
                (unsigned long long)order_bits(best_t) << 32 | (uint32_t)(best_tri < 0 ? 0 : best_tri);
            key[lane] = kAny ? 1ull : key0;
            uint32_t carry = 0;
            for (uint32_t base = 0; base < total; base += 64u) {
                // the lane whose leaf holds pair base + lane
                own[lane] = 0u;
                wave_sync();
                if (cnt != 0u && first - base < 64u) own[first - base] = lane + 1u;
                wave_sync();
                uint32_t w = own[lane];
                if (lane == 0u) w = max(w, carry);
                w = wave_max_scan_u32(w);
                carry = (uint32_t)__builtin_amdgcn_readlane((int)w, 63);
                const uint32_t r = w - 1u, pair = base + lane;
                const bool valid = pair < total;
                const uint32_t rec = from_lane(shift, r) + pair;
                const f3 ro = mk3(from_lane(o.x, r), from_lane(o.y, r), from_lane(o.z, r));
                const f3 rd = mk3(from_lane(d.x, r), from_lane(d.y, r), from_lane(d.z, r));
                const float rt = from_lane(best_t, r), rdist = kAny ? from_lane(dist, r) : 0.0f;
                const float4* t = recs + 3ull * (valid ? rec : begin);
                bool hit = false;
                float lam = 0.0f;
                uint32_t tri = 0;
                if (valid) {
                    const float4 a4 = t[0], e14 = t[1], e24 = t[2];
                    float u, v;
                    hit = ray_tri(xyz(a4), xyz(e14), xyz(e24), ro, rd, lam, u, v) && lam > eps;
                    hit = hit && (kAny ? lam < rt && lam + slack < rdist : lam <= rt);
                    tri = __float_as_uint(a4.w);
                }
                if (ballot(hit) != 0ull) {
                    if (kAny) {
                        if (hit) key[r] = 0ull;
                    } else {
                        const unsigned long long mine = (unsigned long long)order_bits(lam) << 32 | tri;
                        if (hit) __hip_atomic_fetch_min(&key[r], mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        wave_sync();
                        if (hit && key[r] == mine) brec[r] = rec;
                    }
                }
                wave_sync();
            }
            if (at_leaf) {
                const unsigned long long k = key[lane];
                if (kAny) {
                    if (k == 0ull) best_tri = 0;
                } else if (k != key0) {
                    best_t = order_float((uint32_t)(k >> 32));
                    best_tri = (int32_t)(uint32_t)k;
                    best_rec = brec[lane];
                }
            }
            wave_sync();
        }
        if (at_leaf) {
            if (kAny && best_tri >= 0) state = kDone;
            else pop();
        }
    }
}

}  // namespace mnrt
