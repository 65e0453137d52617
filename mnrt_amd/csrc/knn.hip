// knn.hip — exact k-nearest-photon radiance estimate on gfx950.
//
// Replaces the reference's query-radius estimate + range search + gather:
//   KDTreePoint::ComputeQueryRadii (KDTreePoint.cpp:229-248, kdtree_point.cu:229-546),
//   dev_RangeSearch (photon_knn.cu:113-235) and kernel_PhotonGather
//   (photon_knn.cu:487-552, wrapper KernelPMPhotonGather :833-844).
//
// Design (one wave64 per query):
//   * the photons come in groups of 64 consecutive leaf-ordered records, which the whole wave
//     finds with wave-uniform control flow through the box hierarchy over them (boxes.h): one
//     box per lane and test, three levels, boxes beyond the limit skipped.  (dev_RangeSearch
//     walks the binary tree per thread, photon_knn.cu:146-171.)  A tree without a hierarchy
//     (node words supplied by the caller) is walked node by node over its query-time node
//     words with far children on a per-wave LDS stack;
//   * a group's photon records are tested one per lane with one coalesced buffer load each
//     (bounded at the last record);
//   * candidates (d2 bits << 32 | record position) are appended to a per-wave LDS buffer
//     with ballot + mbcnt compaction; when k are known or the buffer would overflow, the
//     candidates above a threshold are dropped (at least k stay) and the pruning limit
//     tightens; the exact k best, ties by photon index, are selected once at the end;
//   * each lane fetches the records of its slots of the set and the front-facing powers are
//     summed per channel as exact 64-bit fixed-point integers (the reference adds floats in
//     its range-search order, photon_knn.cu:506-516, so its sums depend on that order); the
//     set is sorted only when the caller asks for the neighbour lists;
//   * a wave answers a chain of neighbouring queries: one load brings all their inputs, one
//     query after the other is searched with the whole wave, and one pass at the end computes
//     the outputs of all of them, one per lane.
//
// Bound: instruction issue, on the vector and the scalar unit alike (4 cycles each per wave64
// instruction and SIMD); HBM traffic is a tenth of the bytes the searches touch.  Per query of
// 2.07M bounce hits (k = 100, 1M photons): 1297 vector and 980 scalar instructions with binary
// nodes, query-time leaves of 512 photons and outputs per query (5.12 ms), 773 and 651 with the
// hierarchy (3.62 ms), then 3.14 ms with radii for the searches that have no previous query and
// chains of 16.
#include <algorithm>
#include <type_traits>
#include <cmath>
#include <cstring>
#include <mutex>

#include "batch_dev.h"
#include "order.h"

// Device scratch of mnrt_knn_gather_noalloc (the query processing order and, with slot
// indices, the per-query values before their runs are summed): 64 MiB per device, held
// for the process's lifetime.  Host code never passes this name to a kernel or a copy: it
// is a host-side stand-in; the device address comes from hipGetSymbolAddress, once per
// device (g_scratch_addr).
static __device__ __align__(256) uint32_t scratch[(64u << 20) / 4];

namespace mnrt {

constexpr int kWavesPerBlock = 4;
constexpr int kKnnStack = 64;
// relative margin of the node pruning limit over the photon limit (see knn_query)
constexpr float kPruneMargin = 1.0f + 0x1p-20f;
// word 3 of a raw (untyped, stride 0) buffer descriptor on gfx9-family parts: 32-bit data
// format; reads at or past num_records bytes return zero
constexpr int kBufferWord3 = 0x00020000;

enum : int { kModeRadii = 0, kModeRadiance = 1, kModeBackward = 2 };

// Sorts keys[0..size) ascending, size a power of two.
__device__ __forceinline__ void wave_bitonic(uint64_t* keys, uint32_t size, uint32_t lane) {
    for (uint32_t k2 = 2; k2 <= size; k2 <<= 1) {
        for (uint32_t j = k2 >> 1; j > 0; j >>= 1) {
            for (uint32_t t = lane; t < (size >> 1); t += 64) {
                uint32_t i = 2 * j * (t / j) + (t % j);
                uint32_t l = i + j;
                uint64_t a = keys[i], b = keys[l];
                bool asc = (i & k2) == 0;
                if ((a > b) == asc) {
                    keys[i] = b;
                    keys[l] = a;
                }
            }
            wave_sync();
        }
    }
}

// Exact channel sums of the front-facing powers, RK <= 4 slots per lane (unused slots 0), as
// 64-bit fixed-point integers: with m a channel's largest |v| (m = f 2^e, f in [0.5, 1)), every
// term is rounded to a multiple of 2^(e-40) (exact for terms down to 2^-17 m), ties to even, the
// integers are added in any order (|sum| < 2^48) and the total is rounded to float once
// (power_sum).  A term v = q 2^(e-40) is split as q = hi 2^23 + lo: hi the nearest integer to
// v 2^(17-e) (|hi| <= 2^17), lo the nearest to the exactly representable rest times 2^23
// (|lo| <= 2^22; hi 2^23 is even, so ties of lo fall as ties of q), in five fp32 instructions.
// A lane's up to 4 parts are exact in fp32 and the wave's 256 fit 32 bits.  The nine wave
// reductions share their steps: permlane swaps fold two registers into one, so three channels
// cost 13 instructions for the largest |v| and 24 for the six sums (one by one: 27 and 54).
// Finite inputs; wave-uniform results.
struct LaneSwap {
    uint32_t a, b;
};
// lanes 0..31 of a and of b, and lanes 32..63 of a and of b, each pair joined in one register
__device__ __forceinline__ LaneSwap swap32(uint32_t a, uint32_t b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    return LaneSwap{(uint32_t)r[0], (uint32_t)r[1]};
}
// rows of 16 lanes: (a0, b0, a2, b2) and (a1, b1, a3, b3)
__device__ __forceinline__ LaneSwap swap16(uint32_t a, uint32_t b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    return LaneSwap{(uint32_t)r[0], (uint32_t)r[1]};
}

template <int RK>
__device__ __forceinline__ void wave_power_sums(const float (&vx)[RK], const float (&vy)[RK], const float (&vz)[RK],
                                                uint32_t (&m)[3], int32_t (&hi)[3], int32_t (&lo)[3]) {
    static_assert(RK <= 4, "32-bit part sums hold at most 256 terms");
    uint32_t mx = 0, my = 0, mz = 0;  // max |v| as bits: non-negative floats order as their bits
#pragma unroll
    for (int t = 0; t < RK; ++t) {
        mx = max(mx, __float_as_uint(vx[t]) & 0x7FFFFFFFu);
        my = max(my, __float_as_uint(vy[t]) & 0x7FFFFFFFu);
        mz = max(mz, __float_as_uint(vz[t]) & 0x7FFFFFFFu);
    }
    {
        const LaneSwap s = swap32(mx, my), z = swap32(mz, mz);
        const LaneSwap r = swap16(max(s.a, s.b), max(z.a, z.b));  // rows x z y z
        uint32_t v = max(r.a, r.b);
        v = max(v, dpp_mov<kDppPairSwap>(v));
        v = max(v, dpp_mov<kDppQuadSwap>(v));
        v = max(v, dpp_mov<kDppHalfMirror>(v));
        v = max(v, dpp_mov<kDppRowMirror>(v));
        m[0] = row_lane(v, 0);
        m[1] = row_lane(v, 2);
        m[2] = row_lane(v, 1);
    }
    uint32_t h[3], l[3];
    auto parts = [&](const float (&v)[RK], int c) {
        const int sh = 17 - __builtin_amdgcn_frexp_expf(__uint_as_float(m[c]));
        float fh = 0.0f, fl = 0.0f;
#pragma unroll
        for (int t = 0; t < RK; ++t) {
            const float s = ldexpf(v[t], sh), r = rintf(s);
            fh += r;
            fl += rintf((s - r) * 0x1p23f);
        }
        h[c] = (uint32_t)(int32_t)fh;
        l[c] = (uint32_t)(int32_t)fl;
    };
    parts(vx, 0);
    parts(vy, 1);
    parts(vz, 2);
    const LaneSwap sx = swap32(h[0], l[0]), sy = swap32(h[1], l[1]), sz = swap32(h[2], l[2]);
    const uint32_t z = sz.a + sz.b;  // halves hi, lo
    const LaneSwap r = swap16(sx.a + sx.b, sy.a + sy.b), rz = swap16(z, z);
    auto row_sum = [](uint32_t v) {
        v += dpp_mov<kDppPairSwap>(v);
        v += dpp_mov<kDppQuadSwap>(v);
        v += dpp_mov<kDppHalfMirror>(v);
        v += dpp_mov<kDppRowMirror>(v);
        return v;
    };
    const uint32_t xy = row_sum(r.a + r.b), zz = row_sum(rz.a + rz.b);  // rows x.hi y.hi x.lo y.lo
    hi[0] = (int32_t)row_lane(xy, 0);
    hi[1] = (int32_t)row_lane(xy, 1);
    hi[2] = (int32_t)row_lane(zz, 0);
    lo[0] = (int32_t)row_lane(xy, 2);
    lo[1] = (int32_t)row_lane(xy, 3);
    lo[2] = (int32_t)row_lane(zz, 2);
}

// The channel sum of wave_power_sums' parts, rounded to float once.
__device__ __forceinline__ float power_sum(uint32_t m_bits, int32_t hi, int32_t lo) {
    const float m = __uint_as_float(m_bits);
    if (!(m > 0.0f)) return 0.0f;
    int ex;
    (void)frexpf(m, &ex);
    const double acc = (double)hi * 0x1p23 + (double)lo;  // exact: |acc| < 2^49
    return (float)ldexp(acc, ex - 40);
}

__device__ __forceinline__ uint32_t pow2_at_least(uint32_t v) {
    uint32_t p = 1;
    while (p < v) p <<= 1;
    return p;
}

constexpr uint32_t kInterpolations = 6;

// Candidates are d2 bits << 32 | record position.  The photon index, which breaks ties of
// d2, is in the record and read only when a tie straddles the k-th place, so a candidate
// costs one 8-byte LDS write.

// Masks of the k smallest (d2, photon index) among the cnt > k candidates held R per lane (d2
// bits h below those of lim, ~0 in empty slots; record positions pos).  Search over the d2
// bits, one ballot per slot and probe, that ends at the first probe with exactly k candidates
// below it: distances are mostly distinct, so it needs no walk down to the k-th distance's last
// bit (20 to 25 probes).  On surfaces the photons within d2 grow linearly with d2, so the first
// probes interpolate in the counts (about 4 instead of the 9 of a bisection); then it bisects.
// Returns the k-th d2's bits.
template <int R>
__device__ __forceinline__ uint32_t wave_select_k(const uint32_t (&h)[R], const uint32_t (&pos)[R], uint32_t cnt,
                                                  uint32_t k, float lim, const float4* __restrict__ recs,
                                                  uint64_t (&keep)[R]) {
    // count(h < lo) = c_lo < k < c_hi = count(h < hi)
    uint32_t lo = 0u, hi = uniform(__float_as_uint(lim)), c_lo = 0u, c_hi = cnt;
    for (uint32_t it = 0; hi - lo > 1u; ++it) {
        uint32_t probe = lo + ((hi - lo) >> 1);
        if (it < kInterpolations) {
            const float f = ((float)(k - c_lo) + 0.5f) * __builtin_amdgcn_rcpf((float)(c_hi - c_lo) + 1.0f);
            const float x = __uint_as_float(lo) + (__uint_as_float(hi) - __uint_as_float(lo)) * f;
            probe = uniform(min(max(__float_as_uint(x), lo + 1u), hi - 1u));
        }
        uint32_t c = 0;
#pragma unroll
        for (int t = 0; t < R; ++t) {
            keep[t] = ballot(h[t] < probe);
            c += (uint32_t)__popcll(keep[t]);
        }
        if (c == k) {
            uint32_t m = 0;
#pragma unroll
            for (int t = 0; t < R; ++t) m = max(m, h[t] < probe ? h[t] : 0u);
            return wave_max_u32(m);
        }
        if (c < k) {
            lo = probe;
            c_lo = c;
        } else {
            hi = probe;
            c_hi = c;
        }
    }
    hi = lo;
    // hi is the k-th d2 and more than one candidate has it
    uint32_t below = 0, tie = 0;
    uint64_t eq[R];
#pragma unroll
    for (int t = 0; t < R; ++t) {
        keep[t] = ballot(h[t] < hi);
        eq[t] = ballot(h[t] == hi);
        below += (uint32_t)__popcll(keep[t]);
        tie += (uint32_t)__popcll(eq[t]);
    }
    const uint32_t need = k - below;  // 1 <= need <= tie
    if (need < tie) {
        uint32_t idx[R];  // photon indices of the ties; the `need` lowest are kept
#pragma unroll
        for (int t = 0; t < R; ++t) {
            idx[t] = 0xFFFFFFFFu;
            if (__builtin_amdgcn_inverse_ballot_w64(eq[t])) idx[t] = __float_as_uint(recs[2ull * pos[t]].w);
        }
        lo = 0u;  // the need-th lowest index
        for (int b = 31; b >= 0; --b) {
            const uint32_t probe = lo | (1u << b);
            uint32_t c = 0;
#pragma unroll
            for (int t = 0; t < R; ++t) c += (uint32_t)__popcll(eq[t] & ballot(idx[t] < probe));
            if (c < need) lo = probe;
        }
#pragma unroll
        for (int t = 0; t < R; ++t) eq[t] &= ballot(idx[t] <= lo);
    }
#pragma unroll
    for (int t = 0; t < R; ++t) keep[t] |= eq[t];
    return hi;
}

// A pruning threshold on the high word (d2 bits) that keeps between k and hi_k of the cnt
// candidates' d2 bits h held R per lane (~0 for empty slots): *upper = count(h <= T).  Binary search over
// the high word that stops as soon as the keys at or below the range top number at most
// hi_k (far fewer steps than the exact k-th); *upper > hi_k means ties made it impossible.
template <int R>
__device__ __forceinline__ uint32_t wave_window_hi(const uint32_t (&h)[R], uint32_t k, uint32_t hi_k, uint32_t cnt,
                                                   uint32_t* upper_out) {
    if (cnt <= hi_k) {
        uint32_t m = 0;
#pragma unroll
        for (int t = 0; t < R; ++t) m = max(m, h[t] != 0xFFFFFFFFu ? h[t] : 0u);
        *upper_out = cnt;
        return wave_max_u32(m);
    }
    // [prefix, prefix + width) holds the k-th high word; upper = count(h < prefix + width)
    uint32_t prefix = 0, upper = cnt;
    uint64_t width = 1ull << 32;
    while (width > 1 && upper > hi_k) {
        width >>= 1;
        const uint32_t probe = prefix + (uint32_t)width;
        uint32_t c = 0;
#pragma unroll
        for (int t = 0; t < R; ++t) c += (uint32_t)__popcll(ballot(h[t] < probe));
        if (c >= k) upper = c;
        else prefix = probe;
    }
    *upper_out = upper;
    return prefix + (uint32_t)(width - 1);
}

// The tree a query walks: from the launch arguments (one tree) or the query's scene.
struct KnnTree {
    const uint2* nodes;
    const float4* recs;
    BoxTree boxes;
    float r2max;
    float r_max;
};

// Backward mode: the front-facing neighbours of a chunk of queries as (photon << 8 | slot) in a
// per-wave LDS list, which the caller merges before touching memory.
struct PairSink {
    uint64_t* pairs;
    uint32_t n;      // wave-uniform
    uint32_t slot;   // the query's
    uint32_t pbase;  // added to the photon index (offset of the scene's photons in a batch)
};

// A wave's block of up to 64 consecutive queries, lane j holding query j: what the searches
// read (one coalesced load each instead of a dependent uniform load per query) ...
struct QueryLanes {
    uint32_t q;
    float x, y, z;
    float step;        // distance to the query before it
    float nx, ny, nz;  // normal turned toward the source ray (photon_knn.cu:500-505)
    float sure;        // see front_facing
};
// ... and what they found, in lane j, for the outputs (knn_finish), which are then computed for
// all queries of the block at once rather than by a whole wave for each.
struct FoundLanes {
    float r2;
    uint32_t found;
    uint32_t m[3];   // channel sums of the front-facing powers as wave_power_sums gives them
    int32_t hi[3], lo[3];
};

__device__ __forceinline__ float lane_f32(float v, uint32_t j) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), (int)j));
}

template <int kMode>
__device__ __forceinline__ QueryLanes load_queries(const KnnArgs& A, uint32_t q, bool in, uint32_t lane) {
    QueryLanes Q{};
    Q.q = q;
    if (in) {
        const float4 p = A.pos[q];
        Q.x = p.x;
        Q.y = p.y;
        Q.z = p.z;
        if (kMode != kModeRadii) {
            f3 n = xyz(A.nrm[q]);
            const f3 rd = xyz(A.dir[q]);
            if (dot3(mk3(-rd.x, -rd.y, -rd.z), n) < 0.0f) n = mk3(n.x * -1.0f, n.y * -1.0f, n.z * -1.0f);
            Q.nx = n.x;
            Q.ny = n.y;
            Q.nz = n.z;
            const float n1 = fabsf(n.x) + fabsf(n.y) + fabsf(n.z);
            Q.sure = n1 > 1e-30f ? n1 * 0.0625f : __uint_as_float(0x7F800000u);
        }
    }
    const float dx = Q.x - __shfl_up(Q.x, 1, 64), dy = Q.y - __shfl_up(Q.y, 1, 64), dz = Q.z - __shfl_up(Q.z, 1, 64);
    Q.step = __builtin_amdgcn_sqrtf(dx * dx + dy * dy + dz * dz);
    return Q;
}

// dot3(n, oct_decode(c)) < 0, from the direction scaled by 32767, whose coordinates are integers
// and need no division: the scaled product differs from 32767 times the fp32 one by at most
// about 0.02 (|nx| + |ny| + |nz|) (a few roundings of terms up to 32767), so its sign is the
// fp32 one's outside `sure` = 1/16 of that sum, and *unsure asks for the exact expression inside.
__device__ __forceinline__ bool front_facing(float nx, float ny, float nz, uint32_t c, float sure, bool* unsure) {
    const float u = (float)(int32_t)(int16_t)(uint16_t)c, v = (float)((int32_t)c >> 16);
    const float z = (32767.0f - fabsf(u)) - fabsf(v);
    const float fu = z < 0.0f ? copysignf(32767.0f - fabsf(v), u) : u;
    const float fv = z < 0.0f ? copysignf(32767.0f - fabsf(u), v) : v;
    const float d = __builtin_fmaf(nz, z, __builtin_fmaf(ny, fv, nx * fu));
    *unsure = !(fabsf(d) > sure);
    return d < 0.0f;
}

// Warm start for consecutive queries of one wave on one tree: every one of the previous
// query's k neighbours lies within d_k(prev) + |prev - q| of q, so that radius (rounded
// up) bounds this query's k-th distance and the search starts with it instead of r_max.
constexpr float kNoHint = -1.0f, kFew = -2.0f;
struct WarmHint {
    float r2;  // previous query's k-th d2; kNoHint: first query; kFew: it found fewer than k
    // Queries in spatial-cell order (incoherent hits) lie farther apart than the previous
    // query's k-th distance more often, so that the bound above is loose: they search first
    // within d_k(prev) + 0.3 |prev - q|, a guess, and within the bound only when it holds
    // fewer than k (0.5: 2 % slower).  Camera hits in tile order lie close together and use the
    // bound.
    bool guess;
};

// Margin on the squared radius estimated from a group's density (1: 5 % of the searches need a
// second pass; 0.7 and 1.4 were slower by 8 and 2 %), and the squared radius, in squared k-th
// distances of the previous query, up to which a warm start is near enough to take the boxes in
// any order (1.5, 2.5 and 4: 61,440 queries 164 / 128 / 121 us).
constexpr float kColdMargin = 1.0f;
constexpr float kWarmMost = 4.0f;

// One query by one wave: query j of the block.  cand: CAP LDS entries, snode / soff: kKnnStack
// (kBoxes: unused).  kBoxes: the tree has a box hierarchy, which is walked instead of the
// node words.  Returns what was found in lane j of F.
template <int CAP, int kMode, bool kBoxes>
__device__ __forceinline__ void knn_query(const KnnArgs& A, const KnnTree& Tr, const QueryLanes& Q, uint32_t j,
                                          uint32_t lane, uint64_t* cand, uint32_t* snode, float4* soff, WarmHint& hint,
                                          FoundLanes& F, PairSink* sink = nullptr) {
    const float qx = lane_f32(Q.x, j), qy = lane_f32(Q.y, j), qz = lane_f32(Q.z, j);
    const uint32_t lane32 = lane * 32u;  // this lane's byte offset in a 64-record batch
    const uint32_t k = A.k;
    float r2max = Tr.r2max;
    if (A.r_query) {
        const float rq = ld_uniform(A.r_query, (uint32_t)__builtin_amdgcn_readlane((int)Q.q, (int)j));
        r2max = rq * rq;
    }
    // search radius: r_max, or the warm-start bound when smaller, and for queries in
    // spatial-cell order first the guess of WarmHint::guess.  The bound is computed in fp32 with
    // the hardware square root; margins of 2^-16 per step are far above its and the fp32
    // distances' roundings (a few units of 2^-24), and the bound is exclusive, hence the next
    // float up.  The search stays exact whatever it is: a bound holding fewer than k photons is
    // searched again with r2max, and one holding k or more holds the k nearest.
    float r2lim = r2max;
    float r2next = r2max;  // the next pass's limit when this one holds fewer than k
    bool tight = false;    // the radius comes from a near previous query
    const float step = lane_f32(Q.step, j);
    // a near previous query found fewer than k: so will this one, most likely, and then no smaller radius
    // and no order of the boxes saves anything (784,641 queries of radius 0.02 in a room, k = 50, 20,001 photons,
    // camera hits 628 -> 458 us, bounce hits 686 -> 518; 500 photons, radius 0.35, radii alone: 379 -> 269)
    const bool few = kBoxes && hint.r2 == kFew && step * step < 4.0f * r2max;
    if (hint.r2 >= 0.0f) {
        constexpr float kMargin = 1.0f + 0x1p-16f;
        const float dk = __builtin_amdgcn_sqrtf(hint.r2);
        const float b = (dk + step) * kMargin;
        const float b2 = (b * b) * kMargin;
        r2lim = r2next = b2 < r2max ? __uint_as_float(__float_as_uint(b2) + 1u) : r2max;
        if (hint.guess) {
            const float g = dk + 0.3f * step;
            r2lim = fminf(r2next, g * g);
        }
        tight = r2lim < r2max && r2lim <= kWarmMost * hint.r2;
    }

    uint32_t cnt = 0;        // candidates in the buffer
    bool full = false;       // the buffer holds the k best so far (after a window: more)
    float thr_d2 = kInf;     // with full: the k best so far lie at d2 <= thr_d2
    // a photon is taken when d2 < tlim (r2lim, and with full also d2 bits <= thr_d2 bits:
    // a superset of the keys below the k-th; the exact selection at the end trims it)
    float tlim = r2lim, plim = r2lim * kPruneMargin;
    auto set_limits = [&]() {
        tlim = r2lim;
        if (full) {
            const uint32_t tb = __float_as_uint(thr_d2);
            tlim = fminf(r2lim, __uint_as_float(tb < 0x7F800000u ? tb + 1u : tb));
        }
        plim = (full ? fminf(r2lim, thr_d2) : r2lim) * kPruneMargin;
    };

    // loads the candidates of R slots per lane
    auto load_cands = [&](auto& h, auto& pos) {
        constexpr int R = sizeof(h) / sizeof(h[0]);
#pragma unroll
        for (int t = 0; t < R; ++t) {
            const uint32_t i = lane + 64u * t;
            const uint64_t c = cand[i];
            h[t] = i < cnt ? (uint32_t)(c >> 32) : 0xFFFFFFFFu;
            pos[t] = (uint32_t)c;
        }
    };
    // writes the candidates of the masks back, in order, from slot 0
    auto store_cands = [&](const auto& h, const auto& pos, const auto& keep) {
        constexpr int R = sizeof(h) / sizeof(h[0]);
        wave_sync();
        uint32_t base = 0;
#pragma unroll
        for (int t = 0; t < R; ++t) {
            if (__builtin_amdgcn_inverse_ballot_w64(keep[t]))
                cand[mask_prefix_from(keep[t], base)] = ((uint64_t)h[t] << 32) | pos[t];
            base += (uint32_t)__popcll(keep[t]);
        }
        wave_sync();
    };
    // keeps the k best, unsorted (cnt > k)
    auto exact_keep_slots = [&](auto slots) {
        constexpr int R = decltype(slots)::value;
        uint32_t h[R], pos[R];
        uint64_t keep[R];
        load_cands(h, pos);
        thr_d2 = __uint_as_float(wave_select_k<R>(h, pos, cnt, k, tlim, Tr.recs, keep));
        store_cands(h, pos, keep);
        cnt = k;
        full = true;
        set_limits();
    };
    // keeps the k best, unsorted (cnt > k); looks only at the ceil(cnt / 64) slots per lane that
    // hold candidates
    auto exact_keep = [&]() {
        constexpr int R = CAP / 64;
        if (R > 2 && cnt <= 128u) exact_keep_slots(std::integral_constant<int, (R > 2 ? 2 : R)>{});
        else if (R > 3 && cnt <= 192u) exact_keep_slots(std::integral_constant<int, (R > 3 ? 3 : R)>{});
        else if (R > 4 && cnt <= 256u) exact_keep_slots(std::integral_constant<int, (R > 4 ? 4 : R)>{});
        else exact_keep_slots(std::integral_constant<int, R>{});
    };
    // when the buffer fills up: keeps at least k and at most CAP - 64 candidates under a
    // threshold on d2 (the exact k best are selected once, at the end); false when equal
    // distances leave only the exact selection
    auto window_keep = [&]() {
        constexpr int R = CAP / 64;
        wave_sync();  // the lanes' candidates of the batches before
        uint32_t h[R], pos[R];
        uint64_t keep[R];
        load_cands(h, pos);
        uint32_t upper = 0;
        uint32_t T = wave_window_hi<R>(h, k, (uint32_t)CAP - 64u, cnt, &upper);
        if (upper > (uint32_t)CAP - 64u) {
            T = wave_select_k<R>(h, pos, cnt, k, tlim, Tr.recs, keep);
            upper = k;
        } else {
#pragma unroll
            for (int t = 0; t < R; ++t) keep[t] = ballot(h[t] <= T);
        }
        store_cands(h, pos, keep);
        cnt = upper;
        full = true;
        thr_d2 = __uint_as_float(T);
        set_limits();
    };
    // tests one record per lane at byte offset lane32 + soffset of rsrc (part: only the first n < 64
    // lanes), record position first + lane, and appends the ones closer than the limit; returns
    // whether the limit tightened
    auto test_batch = [&](__amdgpu_buffer_rsrc_t rsrc, uint32_t soffset, bool part, uint32_t n, uint32_t first) {
        const auto w = __builtin_amdgcn_raw_buffer_load_b96(rsrc, (int)lane32, (int)soffset, 0);
        const float dx = __uint_as_float(w[0]) - qx, dy = __uint_as_float(w[1]) - qy, dz = __uint_as_float(w[2]) - qz;
        const float d2 = dx * dx + dy * dy + dz * dz;
        uint64_t m = ballot(d2 < tlim);
        if (__builtin_expect(part, 0)) {  // past the buffer's end lanes read zeros
            m &= (1ull << n) - 1ull;
            asm volatile("");  // a branch, not selects: it is rarely taken and scalar issue is what bounds this loop
        }
        if (m == 0ull) return false;
        uint32_t after = cnt + (uint32_t)__popcll(m);
        bool tighter = false;
        if (__builtin_expect(after > (uint32_t)CAP, 0)) {
            window_keep();
            m &= ballot(d2 < tlim);
            after = cnt + (uint32_t)__popcll(m);
            tighter = true;
        }
        if (__builtin_amdgcn_inverse_ballot_w64(m))
            cand[mask_prefix_from(m, cnt)] = ((uint64_t)__float_as_uint(d2) << 32) | (first + lane);
        cnt = after;
        return tighter;
    };
    // squared distance from the query to box `lane` of the 64 from box `at` on (0 inside): each
    // term and the sum round like a photon's d2 in the box, whose terms are no smaller, so a photon
    // closer than the limit lies in a box closer than the limit: no margin is needed
    auto box_dist = [&](__amdgpu_buffer_rsrc_t rsrc, uint32_t at) {
        const auto lo = __builtin_amdgcn_raw_buffer_load_b96(rsrc, (int)lane32, (int)(at * 32u), 0);
        const auto hi = __builtin_amdgcn_raw_buffer_load_b96(rsrc, (int)lane32 + 16, (int)(at * 32u), 0);
        const float dx = fmaxf(fmaxf(__uint_as_float(lo[0]) - qx, qx - __uint_as_float(hi[0])), 0.0f);
        const float dy = fmaxf(fmaxf(__uint_as_float(lo[1]) - qy, qy - __uint_as_float(hi[1])), 0.0f);
        const float dz = fmaxf(fmaxf(__uint_as_float(lo[2]) - qz, qz - __uint_as_float(hi[2])), 0.0f);
        return dx * dx + dy * dy + dz * dz;
    };
    // takes a box from the mask (not empty): any of them under a warm-start radius, the nearest
    // when the search starts from r_max (its limit then tightens with the first groups)
    auto take_box = [&](auto nearest, uint64_t& m, float d) {
        uint64_t c = m;
        if (decltype(nearest)::value) {
            const uint32_t v = __builtin_amdgcn_inverse_ballot_w64(m) ? __float_as_uint(d) : 0xFFFFFFFFu;
            c &= ballot(v == wave_min_u32(v));
        }
        const uint32_t i = (uint32_t)__builtin_ctzll(c);
        m = bit_clear(m, i);
        return i;
    };
    auto walk_boxes = [&](auto nearest) {
        const BoxTree& B = Tr.boxes;
        const __amdgpu_buffer_rsrc_t boxes =
            __builtin_amdgcn_make_buffer_rsrc((void*)B.p, (short)0, (int)(B.end * 32u), kBufferWord3);
        for (uint32_t b2 = 0; b2 < B.g2; b2 += 64u) {
            float e2 = 0.0f, e1 = 0.0f;
            uint64_t m2 = 1ull, m1 = 1ull;
            if (B.g2 > 1u) {
                e2 = box_dist(boxes, B.o2 + b2);
                m2 = ballot(e2 < tlim);
            }
            while (m2) {
                const uint32_t i2 = b2 + take_box(nearest, m2, e2);
                if (B.g1 > 1u) {
                    e1 = box_dist(boxes, B.o1 + 64u * i2);
                    m1 = ballot(e1 < tlim);
                }
                bool tight1 = false;
                while (m1) {
                    const uint32_t i1 = 64u * i2 + take_box(nearest, m1, e1);
                    const float e0 = box_dist(boxes, 64u * i1);
                    uint64_t m0 = ballot(e0 < tlim);
                    // the 4096 records below the box, up to the last one, and the group that the
                    // last one leaves partial
                    const uint32_t left = min(B.nrefs - 4096u * i1, 4096u);
                    const uint32_t last = (left & 63u) ? left >> 6 : 64u;
                    const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
                        (void*)(Tr.recs + (uint64_t)8192u * i1), (short)0, (int)(left * 32u), kBufferWord3);
                    while (m0) {
                        const uint32_t g = take_box(nearest, m0, e0);
                        bool tight = test_batch(rr, g * 2048u, g == last, left & 63u, 4096u * i1 + 64u * g);
                        if (decltype(nearest)::value && !full && cnt >= k) {
                            window_keep();
                            tight = true;
                        }
                        if (tight) {
                            m0 &= ballot(e0 < tlim);
                            tight1 = true;
                        }
                    }
                    if (tight1) m1 &= ballot(e1 < tlim);
                }
                if (tight1) m2 &= ballot(e2 < tlim);
            }
        }
    };

    if (kBoxes && !tight && !few && Tr.boxes.g2 <= 64u) {
        // no warm start: a radius from the density around the query instead of r_max.  64 photons
        // on a surface (or in a volume: about the same number) in a box whose largest face has
        // area a have their k nearest within sqrt(k a / (64 pi)); of the boxes that hold the query
        // (or are nearest) the smallest is taken, as boxes can straddle distant photons.
        const BoxTree& B = Tr.boxes;
        const __amdgpu_buffer_rsrc_t boxes =
            __builtin_amdgcn_make_buffer_rsrc((void*)B.p, (short)0, (int)(B.end * 32u), kBufferWord3);
        float d2 = 0.0f, a = 0.0f;
        auto nearest_of = [&](uint32_t at) {
            const auto lo = __builtin_amdgcn_raw_buffer_load_b96(boxes, (int)lane32, (int)(at * 32u), 0);
            const auto hi = __builtin_amdgcn_raw_buffer_load_b96(boxes, (int)lane32 + 16, (int)(at * 32u), 0);
            const float lx = __uint_as_float(lo[0]), ly = __uint_as_float(lo[1]), lz = __uint_as_float(lo[2]);
            const float hx = __uint_as_float(hi[0]), hy = __uint_as_float(hi[1]), hz = __uint_as_float(hi[2]);
            const float dx = fmaxf(fmaxf(lx - qx, qx - hx), 0.0f), dy = fmaxf(fmaxf(ly - qy, qy - hy), 0.0f),
                        dz = fmaxf(fmaxf(lz - qz, qz - hz), 0.0f);
            const uint32_t e = __float_as_uint(dx * dx + dy * dy + dz * dz), m = wave_min_u32(e);
            const float ex = hx - lx, ey = hy - ly, ez = hz - lz;
            const uint32_t f = e == m ? __float_as_uint(fmaxf(ex * ey, fmaxf(ey * ez, ex * ez))) : 0xFFFFFFFFu;
            const uint32_t fm = wave_min_u32(f);
            d2 = __uint_as_float(m);
            a = __uint_as_float(fm);
            return (uint32_t)__builtin_ctzll(ballot(f == fm));
        };
        uint32_t i = B.g2 > 1u ? nearest_of(B.o2) : 0u;
        i = B.g1 > 1u ? 64u * i + nearest_of(B.o1 + 64u * i) : 0u;
        (void)nearest_of(64u * i);
        const float g = __builtin_amdgcn_sqrtf(a * ((float)k * (kColdMargin / 64.0f * kInvPi))) + __builtin_amdgcn_sqrtf(d2);
        if (g * g < r2lim) {
            r2next = fminf(r2lim, 4.0f * (g * g));
            r2lim = g * g;
            set_limits();
        }
    }
    for (;;) {  // another pass when the radius held fewer than k
        // (a NaN coordinate has no neighbours, and no box to skip)
        if (kBoxes && qx == qx && qy == qy && qz == qz) {
            if (tight || few) walk_boxes(std::false_type{});
            else walk_boxes(std::true_type{});
        }
        if (!kBoxes) {
            int sp = 0;
            uint32_t node = 0;
            // Squared per-axis distances from the query to the current node's box (0 inside) and,
            // per split axis, the sum of the other two: a far child's box distance is
            // diff^2 + rest[a].  A photon's d2 sums its terms in x, y, z order; the box distance's
            // other order can round a few units in the last place differently, so the pruning
            // limit plim carries a relative margin of 2^-20 (far above those roundings): a node is
            // dropped only when every photon in it lies beyond the limit.
            float ox2 = 0.0f, oy2 = 0.0f, oz2 = 0.0f;
            // lanes 0-2 hold the query's x, y, z and the three rest sums: a split axis picks its
            // value with one lane read
            const float qlane = lane == 0 ? qx : (lane == 1 ? qy : qz);
            float rlane = 0.0f;
            for (;;) {
                node = uniform(node);
                uint2 nd = ld_uniform8(Tr.nodes, node);
                nd.x = uniform(nd.x);
                nd.y = uniform(nd.y);
                while (!is_leaf(nd.y)) {
                    const uint32_t a = nd.y >> 30;
                    const float s = __uint_as_float(nd.x);
                    const float qa = lane_f32(qlane, a), rest = lane_f32(rlane, a);
                    const float diff = qa - s;  // > 0 exactly when qa > s
                    const float d2a = diff * diff;
                    // far child's box distance: the split plane replaces this axis' offset
                    const float bd2 = d2a + rest;
                    const uint32_t left = node + 1, right = nd.y & MNRT_INDEX_MASK;
                    const bool gr = diff > 0.0f;
                    // entries are far children of distinct levels of the current path, so a
                    // tree of max_level <= MNRT_MAX_LEVEL < kKnnStack never fills the stack; the
                    // slot clamp only keeps a malformed tree's writes inside it
                    if (bd2 <= plim) {
                        if (lane == 0) {
                            const int e = min(sp, kKnnStack - 1);
                            snode[e] = gr ? left : right;
                            soff[e] = make_float4(a == 0 ? d2a : ox2, a == 1 ? d2a : oy2, a == 2 ? d2a : oz2, bd2);
                        }
                        ++sp;
                    }
                    node = uniform(gr ? right : left);
                    nd = ld_uniform8(Tr.nodes, node);
                    nd.x = uniform(nd.x);
                    nd.y = uniform(nd.y);
                }
                wave_sync();
                const uint32_t count = nd.x, begin = nd.y & MNRT_INDEX_MASK;
                // the leaf's records (32 B each, position and photon index first) through a buffer
                // descriptor that ends with the leaf
                const __amdgpu_buffer_rsrc_t lr = __builtin_amdgcn_make_buffer_rsrc(
                    (void*)(Tr.recs + 2ull * begin), (short)0, (int)(count * 32u), kBufferWord3);
                for (uint32_t base = 0; base < count; base += 64) {
                    (void)test_batch(lr, base * 32u, count - base < 64u, (count - base) & 63u, begin + base);
                    wave_sync();
                }
                if (!full && cnt >= k) window_keep();
                bool found = false;
                while (sp > 0) {
                    --sp;
                    const int e = min(sp, kKnnStack - 1);
                    const float4 f = soff[e];
                    if (uniformf(f.w) > plim) continue;
                    node = uniform(snode[e]);
                    ox2 = uniformf(f.x);
                    oy2 = uniformf(f.y);
                    oz2 = uniformf(f.z);
                    rlane = lane == 0 ? oy2 + oz2 : (lane == 1 ? ox2 + oz2 : ox2 + oy2);
                    found = true;
                    break;
                }
                wave_sync();
                if (!found) break;
            }
        }
        if (cnt >= k || !(r2lim < r2max)) break;
        // a guess that held fewer than k: the bound next; the bound holds k (the r_max pass
        // after it keeps the search exact whatever the roundings)
        r2lim = r2lim < r2next ? r2next : r2max;
        tight = false;
        cnt = 0;
        full = false;
        thr_d2 = kInf;
        set_limits();
    }
    wave_sync();
    // the buffer holds exactly the set after this, in no particular order
    const uint32_t found = min(cnt, k);  // min(#photons closer than r_max, k)
    float r2 = r2max;
    if (cnt > k) {
        exact_keep();
        r2 = thr_d2;
    } else if (cnt == k) {
        // the k-th distance: the largest d2 of the set
        uint32_t hi = 0;
        for (uint32_t i = lane; i < found; i += 64) hi = max(hi, (uint32_t)(cand[i] >> 32));
        r2 = __uint_as_float(wave_max_u32(hi));
    }
    hint.r2 = found >= k ? r2 : kFew;
    if (lane == j) {
        F.r2 = r2;
        F.found = found;
    }

    if (kMode != kModeRadii) {
        // Front-facing powers: each lane fetches the records of its slots of the set.  The set
        // has at most k <= CAP - 64 entries (the launch picks CAP >= k + 64), so ceil(k / 64)
        // slots per lane hold it; slots beyond would only add zeros.
        const float nx = lane_f32(Q.nx, j), ny = lane_f32(Q.ny, j), nz = lane_f32(Q.nz, j);
        const float sure = lane_f32(Q.sure, j);
        auto front_sums = [&](auto slots) {
            constexpr int R = decltype(slots)::value;
            float vx[R], vy[R], vz[R];
#pragma unroll
            for (int t = 0; t < R; ++t) {
                const uint32_t i = lane + 64u * (uint32_t)t;
                vx[t] = vy[t] = vz[t] = 0.0f;
                bool front = false;
                uint64_t key = 0;
                if (i < found) {
                    const float4* rec = Tr.recs + 2ull * (uint32_t)cand[i];
                    const float4 pw = rec[1];
                    const uint32_t c = __float_as_uint(pw.w);
                    bool unsure;
                    front = front_facing(nx, ny, nz, c, sure, &unsure);
                    if (unsure) front = dot3(mk3(nx, ny, nz), oct_decode(c)) < 0.0f;
                    if (front) {
                        vx[t] = pw.x;
                        vy[t] = pw.y;
                        vz[t] = pw.z;
                        if (kMode == kModeBackward)
                            key = (((uint64_t)__float_as_uint(rec[0].w) + sink->pbase) << 8) | sink->slot;
                    }
                }
                if (kMode == kModeBackward) {
                    const uint64_t m = ballot(front);
                    if (front) sink->pairs[mask_prefix_from(m, sink->n)] = key;
                    sink->n += (uint32_t)__popcll(m);
                }
            }
            uint32_t m[3];
            int32_t hi[3], lo[3];
            wave_power_sums<R>(vx, vy, vz, m, hi, lo);
            if (lane == j) {
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    F.m[c] = m[c];
                    F.hi[c] = hi[c];
                    F.lo[c] = lo[c];
                }
            }
        };
        constexpr int RK = std::min<int>((CAP - 64) / 64, (int)((MNRT_KNN_MAX_K + 63u) / 64u));
        if (RK >= 2 && k <= 64u) front_sums(std::integral_constant<int, 1>{});
        else if (RK >= 3 && k <= 128u) front_sums(std::integral_constant<int, (RK >= 3 ? 2 : RK)>{});
        else if (RK >= 4 && k <= 192u) front_sums(std::integral_constant<int, (RK >= 4 ? 3 : RK)>{});
        else front_sums(std::integral_constant<int, RK>{});
    }
    // neighbour lists, for callers that ask for them: (d2, photon index) order
    if (A.out_nbr) {
        const uint32_t q = (uint32_t)__builtin_amdgcn_readlane((int)Q.q, (int)j);
        const uint32_t size = pow2_at_least(found);
        wave_sync();
        for (uint32_t i = lane; i < size; i += 64) {
            const uint64_t c = cand[i];
            cand[i] = i < found ? ((c >> 32) << 32) | __float_as_uint(Tr.recs[2ull * (uint32_t)c].w) : ~0ull;
        }
        wave_sync();
        wave_bitonic(cand, size, lane);
        for (uint32_t i = lane; i < k; i += 64)
            A.out_nbr[(size_t)q * k + i] = (i < found) ? (uint32_t)cand[i] : 0xFFFFFFFFu;
    }
    wave_sync();
}

// The launch's KnnArgs (its kernel's first argument) read anew: what only the outputs need is
// then not held in scalar registers, of which 8 waves per SIMD leave 80 each, through the search.
__device__ __forceinline__ KnnArgs late_args() {
#if defined(__HIP_DEVICE_COMPILE__)
    uint64_t p = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return ld_uniform((const KnnArgs*)p, 0u);
#else
    return KnnArgs{};
#endif
}

// Outputs of the block's queries, one lane each (in: the lane's query was answered).
// Backward: also the query's fixed-point weights w[3 lane ..], fix_scale units per unit
// gradient.
template <int kMode>
__device__ __forceinline__ void knn_finish(const KnnArgs& A, const QueryLanes& Q, const FoundLanes& F, bool in,
                                           float r_max, uint32_t lane, double fix_scale = 0.0, long long* w = nullptr) {
    if (!in) return;
    const uint32_t q = Q.q, found = F.found;
    const float r2 = F.r2;
    if (A.out_count) A.out_count[q] = found;
    if (kMode == kModeRadii) {
        if (A.out_radius) A.out_radius[q] = found >= A.k ? sqrtf(r2) : (A.r_query ? A.r_query[q] : r_max);
        if (A.out_r2) A.out_r2[q] = r2;
        return;
    }
    float ix = 0.0f, iy = 0.0f, iz = 0.0f;
    if (r2 > 0.0f) {
        const float den = r2 * kPi;
        ix = power_sum(F.m[0], F.hi[0], F.lo[0]) / den;
        iy = power_sum(F.m[1], F.hi[1], F.lo[1]) / den;
        iz = power_sum(F.m[2], F.hi[2], F.lo[2]) / den;
    }
    float4 c4 = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
    if (A.clr) {
        c4 = A.clr[q];
        if (found < 8) ix = iy = iz = 0.0f;
    }
    const float4 in4 = A.infl[q];
    if (kMode == kModeBackward) {
        // Adjoint with the neighbour set fixed: L_c = ((alpha rho_c / pi) S_c / (pi r2)) infl_c,
        // so dLoss/dS_c = G_c (alpha rho_c / pi) infl_c / (pi r2) for every front-facing
        // neighbour's power, and dLoss/drho_c = G_c (alpha / pi) E_c infl_c.
        const float4 g = A.grad[q];
        const bool gated = (A.clr && found < 8) || !(r2 > 0.0f);
        const float den = r2 * kPi;
        const float wx = gated ? 0.0f : (g.x * (((c4.w * c4.x) * kInvPi) * in4.x)) / den;
        const float wy = gated ? 0.0f : (g.y * (((c4.w * c4.y) * kInvPi) * in4.y)) / den;
        const float wz = gated ? 0.0f : (g.z * (((c4.w * c4.z) * kInvPi) * in4.z)) / den;
        if (A.out_grad_clr)
            A.out_grad_clr[q] = make_float4(g.x * (((c4.w * kInvPi) * ix) * in4.x),
                                            g.y * (((c4.w * kInvPi) * iy) * in4.y),
                                            g.z * (((c4.w * kInvPi) * iz) * in4.z), 0.0f);
        // fixed-point adds are associative, so the per-photon sums do not depend on the
        // order in which queries arrive
        const bool sum = fix_scale > 0.0;
        w[3 * lane + 0] = sum ? __double2ll_rn((double)wx * fix_scale) : 0ll;
        w[3 * lane + 1] = sum ? __double2ll_rn((double)wy * fix_scale) : 0ll;
        w[3 * lane + 2] = sum ? __double2ll_rn((double)wz * fix_scale) : 0ll;
        return;
    }
    const float rx = (((c4.w * c4.x) * kInvPi) * ix) * in4.x;
    const float ry = (((c4.w * c4.y) * kInvPi) * iy) * in4.y;
    const float rz = (((c4.w * c4.z) * kInvPi) * iz) * in4.z;
    if (A.inv_dist) {
        // reciprocal distance from the source ray's origin (photon_knn.cu:529-535)
        const f3 od = sub3(mk3(Q.x, Q.y, Q.z), xyz(A.orig[q]));
        const float v = 1.0f / sqrtf(dot3(od, od));
        A.inv_dist[q] = A.inv_accumulate ? A.inv_dist[q] + v : v;
    }
    if (A.out_r2) A.out_r2[q] = r2;
    if (A.out_irr) A.out_irr[q] = make_float4(ix, iy, iz, 0.0f);
    if (A.accumulate) {
        const float4 o = A.rad_out[q];
        A.rad_out[q] = make_float4(o.x + rx, o.y + ry, o.z + rz, o.w + 0.0f);
    } else {
        A.rad_out[q] = make_float4(rx, ry, rz, 0.0f);
    }
}

// Consecutive queries per wave: each after the first starts from the previous one's k-th
// distance (WarmHint), which neighbouring queries nearly share, and the block's loads and
// outputs are shared too.  Long chains take fewer searches from scratch, but leave too few waves
// for the chip (8192 at a time) when there are few queries, and then their steps add up to the
// launch's time: k = 100, 1M photons, camera hits, chains of 1 / 8 / 16: 4096 queries 46 / 126 /
// 239 us, 61,440: 235 / 189 / 287 us, 524,288: 1747 / 812 / 810 us, 2.07M: 6.60 / 2.87 / 2.73 ms.
// Neighbouring queries are slow together where the map is uneven, so the slowest chain, not the mean, ends the
// launch: chains of 16 wait until it has a dozen rounds of waves (k = 50, 1M photons, chains of 8 / 16, 784,641
// queries: bounce hits 1091 / 1199 us, points anywhere in the room 3164 / 4188; 2.07M: 2591 / 2506 and
// 6701 / 7254), and node words, over which slow searches are slower still, keep to 8 (points anywhere in the
// room: 784,641 queries 4914 / 7049 us, 2.07M 9129 / 11054; bounce hits 1281 / 1382 and 3070 / 3006).
inline uint32_t knn_chain(uint32_t n, bool boxes) {
    return std::min(boxes && n >= 12u * 8192u * 16u ? 16u : 8u, std::max(1u, n / 24576u));
}

template <int CAP, int kMode, bool kBoxes>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_knn(KnnArgs A) {
    __shared__ uint64_t s_cand[kWavesPerBlock][CAP];
    __shared__ uint32_t s_snode[kBoxes ? 1 : kWavesPerBlock][kBoxes ? 1 : kKnnStack];
    __shared__ float4 s_soff[kBoxes ? 1 : kWavesPerBlock][kBoxes ? 1 : kKnnStack];
    const uint32_t wave = uniform(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t j0 = ((uint64_t)blockIdx.x * kWavesPerBlock + wave) * A.chain;
    if (j0 >= A.n) return;  // uniform per wave
    const uint32_t n = (uint32_t)min<uint64_t>(A.chain, A.n - j0);
    const KnnTree Tr{A.nodes, A.recs, A.boxes, A.r2max, A.r_max};
    WarmHint hint{kNoHint, A.order_far && !order_coherent(A.n, A.order_far)};
    const bool in = lane < n;
    const uint32_t jl = (uint32_t)j0 + (in ? lane : 0u);
    const QueryLanes Q = load_queries<kMode>(A, A.order ? A.order[jl] : jl, in, lane);
    FoundLanes F{};
    for (uint32_t j = 0; j < n; ++j)
        knn_query<CAP, kMode, kBoxes>(A, Tr, Q, j, lane, s_cand[wave], s_snode[kBoxes ? 0 : wave],
                                      s_soff[kBoxes ? 0 : wave], hint, F);
    const KnnArgs L = late_args();
    knn_finish<kMode>(L, Q, F, in, L.r_max, lane);
}

// Batched radiance: waves take chunks of `chunk` consecutive query slots from a work
// counter (one counter per XCD share, as k_trace_batch), slot g belonging to the scene
// whose slot range holds it.  Slots at or past a scene's count (count[s], device side:
// the number of shading points the batched compaction wrote) are left untouched.
template <int CAP, int kWaves, bool kBoxes>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_knn_batch(
    KnnArgs G, const KnnScene* __restrict__ scenes, const uint32_t* __restrict__ slot_begin, uint32_t ns,
    const uint32_t* __restrict__ count, uint32_t chunk, uint32_t num_parts, const uint32_t* __restrict__ part_begin,
    const uint32_t* __restrict__ part_end, uint32_t* __restrict__ work) {
    __shared__ uint64_t s_cand[kWaves][CAP];
    __shared__ uint32_t s_snode[kBoxes ? 1 : kWaves][kBoxes ? 1 : kKnnStack];
    __shared__ float4 s_soff[kBoxes ? 1 : kWaves][kBoxes ? 1 : kKnnStack];
    const uint32_t wave = uniform(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t xcd = blockIdx.x % num_parts;
    for (uint32_t part = 0; part < num_parts; ++part) {
        const uint32_t p = (xcd + part) % num_parts;
        const uint32_t pb = part_begin[p], pe = part_end[p];
        const uint32_t units = (uint32_t)(((uint64_t)(pe - pb) + chunk - 1u) / chunk);
        for (;;) {
            const uint32_t c = take_unit(work, p, units, part > 0u, lane);
            if (c >= units) break;
            const uint64_t c0 = (uint64_t)pb + (uint64_t)c * chunk;
            const uint32_t c1 = (uint32_t)min<uint64_t>(c0 + chunk, pe);
            // the scene of the chunk's slots, refreshed only when a slot crosses into the next
            uint32_t s = uniform(seg_of(slot_begin, ns, (uint32_t)c0));
            uint32_t b = 0, e = 0, m = 0;
            KnnTree Tr{};
            WarmHint hint{kNoHint, false};
            auto enter = [&]() {
                b = ld_uniform(slot_begin, s);
                e = ld_uniform(slot_begin, s + 1);
                m = count ? ld_uniform(count, s) : e - b;
                const KnnScene sc = ld_uniform(scenes, s);
                Tr = KnnTree{sc.nodes, sc.recs, sc.boxes, sc.r2max, sc.r_max};
                hint.r2 = kNoHint;  // another scene's photons
            };
            enter();
            for (uint32_t g0 = (uint32_t)c0; g0 < c1; g0 += 64u) {
                const uint32_t n = min(c1 - g0, 64u);
                const QueryLanes Q = load_queries<kModeRadiance>(G, g0 + min(lane, n - 1u), lane < n, lane);
                FoundLanes F{};
                uint64_t done = 0;
                hint.r2 = kNoHint;  // (the step to the first query of the block is not known)
                for (uint32_t j = 0; j < n; ++j) {
                    const uint32_t g = g0 + j;
                    if (g >= e) {
                        do {
                            ++s;
                        } while (g >= ld_uniform(slot_begin, s + 1));
                        enter();
                    }
                    if (g - b >= m) continue;
                    done |= 1ull << j;
                    knn_query<CAP, kModeRadiance, kBoxes>(G, Tr, Q, j, lane, s_cand[wave], s_snode[kBoxes ? 0 : wave],
                                                          s_soff[kBoxes ? 0 : wave], hint, F);
                }
                knn_finish<kModeRadiance>(late_args(), Q, F, (done >> lane) & 1ull, 0.0f, lane);
            }
        }
    }
}

// Backward pass over chunks of `chunk` consecutive queries per wave (chunk x k <= kPairs):
// the chunk's (photon, query) pairs are sorted by photon in LDS and each photon's
// fixed-point contributions summed before one atomic per channel.  Consecutive queries
// (neighbouring pixels) share most of their neighbours, so this issues a fraction of the
// per-pair atomics; the integer sums are the same in any order.
constexpr int kPairCap = 256;
constexpr uint32_t kBwdChunk = 8;  // queries per chunk, at most

// Sorts a wave's (photon << 8 | slot) pairs by photon in LDS and adds each photon's summed
// fixed-point weights with one atomic per channel.  heads: room for kPairCap words.
__device__ __forceinline__ void merge_pairs(uint64_t* pairs, uint32_t np, const long long* w, uint32_t* heads,
                                            unsigned long long* acc, uint32_t lane) {
    if (np == 0) return;
    // sort the pairs by (photon, slot); pad to a power of two with keys above every pair
    uint32_t size = 64;
    while (size < np) size <<= 1;
    for (uint32_t t = np + lane; t < size; t += 64) pairs[t] = ~0ull;
    wave_sync();
    for (uint32_t k2 = 2; k2 <= size; k2 <<= 1) {
        for (uint32_t j = k2 >> 1; j > 0; j >>= 1) {
            for (uint32_t t = lane; t < (size >> 1); t += 64) {
                const uint32_t i = 2 * j * (t / j) + (t % j), l = i + j;
                const uint64_t a = pairs[i], b = pairs[l];
                if ((a > b) == ((i & k2) == 0)) {
                    pairs[i] = b;
                    pairs[l] = a;
                }
            }
            wave_sync();
        }
    }
    // the first pair of every photon's run
    uint32_t runs = 0;
    for (uint32_t t = 0; t < np; t += 64) {
        const uint32_t i = t + lane;
        const bool head = i < np && (i == 0u || (pairs[i - 1] >> 8) != (pairs[i] >> 8));
        const uint64_t m = ballot(head);
        if (head) heads[mask_prefix_from(m, runs)] = i;
        runs += (uint32_t)__popcll(m);
    }
    wave_sync();
    // A lane per (run, channel): sum the run's weights, one atomic.  The three channels of a photon lie
    // together, so an instruction's 64 atomics touch a third of the lines that a lane per run makes:
    // forward and backward of 77361 queries (k = 50, 131072 photons) 565 -> 468 us, the inverse step of
    // 8 scenes 1564 -> 1425 us.
    for (uint32_t t = lane; t < 3u * runs; t += 64) {
        const uint32_t r = t / 3u, ch = t - 3u * r;
        uint32_t i = heads[r];
        const uint64_t p = pairs[i] >> 8;
        const uint32_t e = r + 1u < runs ? heads[r + 1u] : np;
        long long sum = 0;
        for (; i < e; ++i) sum += w[3u * ((uint32_t)pairs[i] & 0xFFu) + ch];
        if (sum) atomicAdd(&acc[3 * p + ch], (unsigned long long)sum);
    }
}

template <int CAP, bool kBoxes>
__global__ __launch_bounds__(256) void k_knn_bwd_chunks(KnnArgs A, uint32_t chunk) {
    __shared__ uint64_t s_cand[kWavesPerBlock][CAP];
    __shared__ uint32_t s_snode[kBoxes ? 1 : kWavesPerBlock][kBoxes ? 1 : kKnnStack];
    __shared__ float4 s_soff[kBoxes ? 1 : kWavesPerBlock][kBoxes ? 1 : kKnnStack];
    __shared__ uint64_t s_pairs[kWavesPerBlock][kPairCap];
    __shared__ long long s_w[kWavesPerBlock][3 * kBwdChunk];
    static_assert(2 * CAP >= kPairCap, "merge_pairs keeps its runs in the candidate buffer");
    const uint32_t wave = uniform(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t j0 = ((uint64_t)blockIdx.x * kWavesPerBlock + wave) * A.chain;
    if (j0 >= A.n) return;  // uniform per wave
    const double fix_scale = ld_uniform(A.fix_scale, 0u);
    if (!(fix_scale > 0.0) && !A.out_grad_clr) return;  // no weight: no gradient of the powers
    const uint32_t n = (uint32_t)min<uint64_t>(A.chain, A.n - j0);
    const KnnTree Tr{A.nodes, A.recs, A.boxes, A.r2max, A.r_max};
    WarmHint hint{kNoHint, A.order_far && !order_coherent(A.n, A.order_far)};
    const bool in = lane < n;
    const uint32_t jl = (uint32_t)j0 + (in ? lane : 0u);
    const QueryLanes Q = load_queries<kModeBackward>(A, A.order ? A.order[jl] : jl, in, lane);
    for (uint32_t c0 = 0; c0 < n; c0 += chunk) {
        const uint32_t c1 = min(c0 + chunk, n);
        FoundLanes F{};
        PairSink sink{s_pairs[wave], 0u, 0u, 0u};
        for (uint32_t j = c0; j < c1; ++j) {
            sink.slot = j - c0;
            knn_query<CAP, kModeBackward, kBoxes>(A, Tr, Q, j, lane, s_cand[wave], s_snode[kBoxes ? 0 : wave],
                                                  s_soff[kBoxes ? 0 : wave], hint, F, &sink);
        }
        const KnnArgs L = late_args();
        knn_finish<kModeBackward>(L, Q, F, lane >= c0 && lane < c1, L.r_max, lane - c0, fix_scale, s_w[wave]);
        wave_sync();
        merge_pairs(s_pairs[wave], sink.n, s_w[wave], (uint32_t*)s_cand[wave], L.acc, lane);
        wave_sync();
    }
}

// Adds per-query radiance into slots given by a slot index per query (final gathering,
// PhotonMap::GatherFor, PhotonMap.cpp:234-270).  A run of equal consecutive slots is
// summed in query order by the run's first query, so sorted slot indices (as final
// gathering produces them) give a deterministic result.
__global__ __launch_bounds__(256) void k_scatter_runs(const float4* __restrict__ per_query,
                                                      const float* __restrict__ per_query_inv,
                                                      const uint32_t* __restrict__ idx_sp, uint32_t n,
                                                      float4* __restrict__ io_rad, float* __restrict__ io_inv) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t slot = idx_sp[i];
    if (i > 0 && idx_sp[i - 1] == slot) return;
    float x = 0.0f, y = 0.0f, z = 0.0f, w = 0.0f;
    for (uint32_t j = i; j < n && idx_sp[j] == slot; ++j) {
        float4 r = per_query[j];
        x = x + r.x;
        y = y + r.y;
        z = z + r.z;
        if (per_query_inv) w = w + per_query_inv[j];
    }
    atomicAdd(&io_rad[slot].x, x);
    atomicAdd(&io_rad[slot].y, y);
    atomicAdd(&io_rad[slot].z, z);
    if (per_query_inv) atomicAdd(&io_inv[slot], w);
}

// Bound on |weight| per query for the fixed-point scale of the backward pass, from the
// forward's r2 and neighbour counts (same expressions as the backward kernel).
// Workgroups of the passes that bound the weights: one atomic each (per scene), or the atomics of all
// waves on one address would take longer than the pass (6.6 ns each).
constexpr uint32_t kWmaxBlock = 1024;

__global__ __launch_bounds__(kWmaxBlock) void k_bwd_wmax(uint32_t n, const float4* __restrict__ grad,
                                                  const float4* __restrict__ clr, const float4* __restrict__ infl,
                                                  const float* __restrict__ r2, const uint32_t* __restrict__ count,
                                                  uint32_t* __restrict__ wmax_bits) {
    uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
    float m = 0.0f;
    if (q < n) {
        float4 g = grad[q], in4 = infl[q];
        float4 c4 = clr ? clr[q] : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
        float rr = r2[q];
        bool gated = (clr && count[q] < 8) || !(rr > 0.0f);
        if (!gated) {
            float den = rr * kPi;
            const float w[3] = {(g.x * (((c4.w * c4.x) * kInvPi) * in4.x)) / den,
                                (g.y * (((c4.w * c4.y) * kInvPi) * in4.y)) / den,
                                (g.z * (((c4.w * c4.z) * kInvPi) * in4.z)) / den};
            m = abs_max3(w);  // (+infinity when a weight is not finite)
        }
    }
    __shared__ uint32_t s_max[kWmaxBlock / 64];
    const uint32_t b = wave_max_u32(__float_as_uint(m));  // (m >= 0: order of the bits)
    if ((threadIdx.x & 63u) == 0) s_max[threadIdx.x >> 6] = b;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (uint32_t w = 0; w < kWmaxBlock / 64; ++w) t = max(t, s_max[w]);
        if (t) atomicMax(wmax_bits, t);
    }
}

// A photon's gradient from its fixed-point sums (scale: bwd_scale).
__device__ __forceinline__ float4 photon_grad(const unsigned long long* __restrict__ acc, double scale) {
    const double inv = scale > 0.0 ? 1.0 / scale : 0.0;
    if (scale < 0.0) {
        const float nan = __uint_as_float(0x7FC00000u);
        return make_float4(nan, nan, nan, 0.0f);
    }
    return make_float4((float)((double)(long long)acc[0] * inv), (float)((double)(long long)acc[1] * inv),
                       (float)((double)(long long)acc[2] * inv), 0.0f);
}

__global__ __launch_bounds__(256) void k_fix_to_float(uint32_t np, const unsigned long long* __restrict__ acc,
                                                      const double* __restrict__ scale, float4* __restrict__ out) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < np) out[p] = photon_grad(acc + 3ull * p, *scale);
}

// --- batched backward (one launch sequence for every scene of a batch) ---------------

// Per-scene weight bounds: slot g of scene s (g - slot_begin[s] < count[s]) adds its
// bound to wmax[s]; a wave whose slots lie in one scene reduces first.
__global__ __launch_bounds__(kWmaxBlock) void k_bwd_wmax_batch(uint32_t n, const uint32_t* __restrict__ slot_begin,
                                                        uint32_t ns, const uint32_t* __restrict__ count,
                                                        const float4* __restrict__ grad,
                                                        const float4* __restrict__ clr,
                                                        const float4* __restrict__ infl,
                                                        const float* __restrict__ r2,
                                                        const uint32_t* __restrict__ nbr_count,
                                                        uint32_t* __restrict__ wmax_bits) {
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    float m = 0.0f;
    uint32_t s = 0;
    if (g < n) {
        s = seg_of(slot_begin, ns, g);
        const uint32_t cnt = count ? count[s] : slot_begin[s + 1] - slot_begin[s];
        if (g - slot_begin[s] < cnt) {
            float4 gr = grad[g], in4 = infl[g];
            float4 c4 = clr ? clr[g] : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
            float rr = r2[g];
            bool gated = (clr && nbr_count[g] < 8) || !(rr > 0.0f);
            if (!gated) {
                float den = rr * kPi;
                const float w[3] = {(gr.x * (((c4.w * c4.x) * kInvPi) * in4.x)) / den,
                                    (gr.y * (((c4.w * c4.y) * kInvPi) * in4.y)) / den,
                                    (gr.z * (((c4.w * c4.z) * kInvPi) * in4.z)) / den};
                m = abs_max3(w);
            }
        }
    }
    __shared__ uint32_t s_max[kWmaxBlock / 64], s_scene[kWmaxBlock / 64];
    const uint32_t s0 = uniform(s), wave = threadIdx.x >> 6;
    const bool one = ballot(s != s0) == 0ull;  // the wave's slots are one scene's
    const uint32_t b = wave_max_u32(one ? __float_as_uint(m) : 0u);  // (m >= 0: order of the bits)
    if ((threadIdx.x & 63u) == 0) {
        s_max[wave] = b;
        s_scene[wave] = s0;
    }
    if (!one && m > 0.0f) atomicMax(&wmax_bits[s], __float_as_uint(m));
    __syncthreads();
    if (threadIdx.x < kWmaxBlock / 64) {  // one atomic per run of waves of one scene
        const uint32_t i = threadIdx.x, sc = s_scene[i];
        if (i == 0u || s_scene[i - 1u] != sc) {
            uint32_t t = 0;
            for (uint32_t w = i; w < kWmaxBlock / 64 && s_scene[w] == sc; ++w) t = max(t, s_max[w]);
            if (t) atomicMax(&wmax_bits[sc], t);
        }
    }
}

// Fixed-point unit per scene from its bound and query count: the largest power of two
// with count * wmax * unit < 2^62 (the same expression as the single-scene entry point); 0 when no
// query has weight, negative when a weight is not finite: no sum is taken then and the photon
// gradients become NaN.
__device__ __forceinline__ double bwd_scale(uint32_t n, uint32_t wmax_bits) {
    const float wm = __uint_as_float(wmax_bits);
    if (!(wm <= kInf)) return -1.0;
    if (!(n > 0 && wm > 0.0f)) return 0.0;
    int e = 0;
    (void)frexp(4.611686018427387904e18 / ((double)n * (double)wm), &e);
    return ldexp(1.0, e - 1);
}

__global__ __launch_bounds__(64) void k_bwd_scale(uint32_t n, const uint32_t* __restrict__ wmax_bits,
                                                  double* __restrict__ scale) {
    if (threadIdx.x == 0) *scale = bwd_scale(n, *wmax_bits);
}

__global__ __launch_bounds__(64) void k_bwd_scale_batch(uint32_t ns, const uint32_t* __restrict__ slot_begin,
                                                        const uint32_t* __restrict__ count,
                                                        const uint32_t* __restrict__ wmax_bits,
                                                        double* __restrict__ scale) {
    for (uint32_t s = threadIdx.x; s < ns; s += blockDim.x) {
        const uint32_t n = count ? count[s] : slot_begin[s + 1] - slot_begin[s];
        scale[s] = bwd_scale(n, wmax_bits[s]);
    }
}

// Batched backward: waves take work items of `chunk` consecutive query slots (chunk x k <=
// kPairCap) from the work counters, as k_knn_batch does.  A pair carries the photon's index
// in the concatenation of the scenes' photon arrays (scene offset + original index) and its
// weight in the scene's own fixed-point unit, so one work item may span scenes.
template <int CAP, bool kBoxes>
__global__ __launch_bounds__(256) void k_knn_bwd_batch(KnnArgs G, const KnnScene* __restrict__ scenes,
                                                       const uint32_t* __restrict__ slot_begin, uint32_t ns,
                                                       const uint32_t* __restrict__ count,
                                                       const uint32_t* __restrict__ photon_begin,
                                                       const double* __restrict__ scale, uint32_t chunk,
                                                       uint32_t num_parts, const uint32_t* __restrict__ part_begin,
                                                       const uint32_t* __restrict__ part_end,
                                                       uint32_t* __restrict__ work) {
    __shared__ uint64_t s_cand[kWavesPerBlock][CAP];
    __shared__ uint32_t s_snode[kBoxes ? 1 : kWavesPerBlock][kBoxes ? 1 : kKnnStack];
    __shared__ float4 s_soff[kBoxes ? 1 : kWavesPerBlock][kBoxes ? 1 : kKnnStack];
    __shared__ uint64_t s_pairs[kWavesPerBlock][kPairCap];
    __shared__ long long s_w[kWavesPerBlock][3 * kBwdChunk];
    static_assert(2 * CAP >= kPairCap, "merge_pairs keeps its runs in the candidate buffer");
    const uint32_t wave = uniform(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t xcd = blockIdx.x % num_parts;
    for (uint32_t part = 0; part < num_parts; ++part) {
        const uint32_t p = (xcd + part) % num_parts;
        const uint32_t pb = part_begin[p], pe = part_end[p];
        const uint32_t units = (uint32_t)(((uint64_t)(pe - pb) + chunk - 1u) / chunk);
        for (;;) {
            const uint32_t c = take_unit(work, p, units, part > 0u, lane);
            if (c >= units) break;
            const uint64_t g0 = (uint64_t)pb + (uint64_t)c * chunk;
            const uint32_t n = (uint32_t)min<uint64_t>(chunk, pe - g0);
            uint32_t s = uniform(seg_of(slot_begin, ns, (uint32_t)g0));
            uint32_t b = 0, e = 0, m = 0;
            double fs = 0.0, fs_lane = 0.0;
            KnnTree Tr{};
            WarmHint hint{kNoHint, false};
            PairSink sink{s_pairs[wave], 0u, 0u, 0u};
            auto enter = [&]() {
                b = ld_uniform(slot_begin, s);
                e = ld_uniform(slot_begin, s + 1);
                m = count ? ld_uniform(count, s) : e - b;
                sink.pbase = ld_uniform(photon_begin, s);
                fs = ld_uniform(scale, s);
                const KnnScene sc = ld_uniform(scenes, s);
                Tr = KnnTree{sc.nodes, sc.recs, sc.boxes, sc.r2max, sc.r_max};
                hint.r2 = kNoHint;
            };
            enter();
            const QueryLanes Q =
                load_queries<kModeBackward>(G, (uint32_t)g0 + min(lane, n - 1u), lane < n, lane);
            FoundLanes F{};
            uint64_t done = 0;
            for (uint32_t j = 0; j < n; ++j) {
                const uint32_t g = (uint32_t)g0 + j;
                if (g >= e) {
                    do {
                        ++s;
                    } while (g >= ld_uniform(slot_begin, s + 1));
                    enter();
                }
                if (g - b >= m) continue;
                done |= 1ull << j;
                sink.slot = j;
                if (lane == j) fs_lane = fs;
                knn_query<CAP, kModeBackward, kBoxes>(G, Tr, Q, j, lane, s_cand[wave], s_snode[kBoxes ? 0 : wave],
                                                      s_soff[kBoxes ? 0 : wave], hint, F, &sink);
            }
            const KnnArgs L = late_args();
            knn_finish<kModeBackward>(L, Q, F, (done >> lane) & 1ull, 0.0f, lane, fs_lane, s_w[wave]);
            wave_sync();
            merge_pairs(s_pairs[wave], sink.n, s_w[wave], (uint32_t*)s_cand[wave], L.acc, lane);
            wave_sync();
        }
    }
}

// Photon gradients of every scene from the fixed-point sums (photon p of the
// concatenation belongs to the scene whose photon range holds it).
__global__ __launch_bounds__(256) void k_fix_to_float_batch(uint32_t np, const uint32_t* __restrict__ photon_begin,
                                                            uint32_t ns, const unsigned long long* __restrict__ acc,
                                                            const double* __restrict__ scale,
                                                            float4* __restrict__ out) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < np) out[p] = photon_grad(acc + 3ull * p, scale[seg_of(photon_begin, ns, p)]);
}

__global__ __launch_bounds__(256) void k_zero_u64(unsigned long long* __restrict__ p, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = 0ull;
}

// Backward launches: a wave's chain of queries in chunks of floor(kPairCap / k).
int launch_knn_bwd(const KnnArgs& A0, hipStream_t st) {
    KnnArgs A = A0;
    const uint32_t chunk = std::max<uint32_t>(1u, std::min<uint32_t>(kBwdChunk, (uint32_t)kPairCap / A.k));
    A.chain = chunk * std::max(1u, std::min(16u, A.n / 24576u) / chunk);  // whole chunks, at most 16 queries
    const uint64_t per_block = (uint64_t)kWavesPerBlock * A.chain;
    dim3 block(64 * kWavesPerBlock), grid((uint32_t)((A.n + per_block - 1) / per_block));
    const uint32_t need = A.k + 64;
#define MNRT_KC(C)                                                                                            \
    do {                                                                                                      \
        if (A.boxes.p) hipLaunchKernelGGL((k_knn_bwd_chunks<C, true>), grid, block, 0, st, A, chunk);         \
        else hipLaunchKernelGGL((k_knn_bwd_chunks<C, false>), grid, block, 0, st, A, chunk);                  \
    } while (0)
    if (need <= 128) MNRT_KC(128);
    else if (need <= 256) MNRT_KC(256);
    else MNRT_KC(512);
#undef MNRT_KC
    MNRT_HIP_CHECK(hipGetLastError());
    return MNRT_OK;
}

template <int kMode>
int launch_knn(const KnnArgs& A0, hipStream_t st) {
    KnnArgs A = A0;
    A.chain = knn_chain(A.n, A.boxes.p != nullptr);
    const uint64_t per_block = (uint64_t)kWavesPerBlock * A.chain;
    dim3 block(64 * kWavesPerBlock), grid((uint32_t)((A.n + per_block - 1) / per_block));
    uint32_t need = A.k + 64;
#define MNRT_KK(C)                                                                                 \
    do {                                                                                           \
        if (A.boxes.p) hipLaunchKernelGGL((k_knn<C, kMode, true>), grid, block, 0, st, A);         \
        else hipLaunchKernelGGL((k_knn<C, kMode, false>), grid, block, 0, st, A);                  \
    } while (0)
    if (need <= 128) MNRT_KK(128);
    else if (need <= 256) MNRT_KK(256);
    else MNRT_KK(512);
#undef MNRT_KK
    MNRT_HIP_CHECK(hipGetLastError());
    return MNRT_OK;
}

int launch_knn_batch(const KnnArgs& G, const KnnScene* scenes, const uint32_t* slot_begin, uint32_t ns,
                     const uint32_t* count, uint32_t chunk, uint32_t num_parts, const uint32_t* part_begin,
                     const uint32_t* part_end, uint32_t* work, uint32_t cap, uint32_t waves,
                     uint32_t grid, bool boxes, hipStream_t st) {
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, st, work, num_parts * kWorkStride, 0u);
#define MNRT_KB(C, W, X)                                                                                   \
    hipLaunchKernelGGL((k_knn_batch<C, W, X>), dim3(grid), dim3(64 * W), 0, st, G, scenes, slot_begin, ns, \
                       count, chunk, num_parts, part_begin, part_end, work)
#define MNRT_KB_W(C)                              \
    do {                                          \
        if (!boxes) MNRT_KB(C, 4, false);         \
        else if (waves == 1) MNRT_KB(C, 1, true); \
        else if (waves == 2) MNRT_KB(C, 2, true); \
        else MNRT_KB(C, 4, true);                 \
    } while (0)
    if (waves != 1 && waves != 2 && waves != 4) return MNRT_ERR_ARG;
    if (cap == 128) MNRT_KB_W(128);
    else if (cap == 256) MNRT_KB_W(256);
    else if (cap == 512) MNRT_KB_W(512);
    else return MNRT_ERR_ARG;
#undef MNRT_KB_W
#undef MNRT_KB
    MNRT_HIP_CHECK(hipGetLastError());
    return MNRT_OK;
}

// Backward of a batch: clears the accumulators, bounds and scales the weights per scene
// (from the forward's r2 and neighbour counts), runs the pair-merging walk and converts
// the sums.  G.out_r2 / G.out_count / G.out_nbr must be null (the walk would rewrite them).
int launch_knn_bwd_batch(const KnnArgs& G, const KnnScene* scenes, const uint32_t* slot_begin, uint32_t ns,
                         const uint32_t* count, const uint32_t* photon_begin, uint32_t total_photons,
                         const float* fwd_r2, const uint32_t* fwd_count, uint32_t* wmax, double* scale, uint32_t num_parts, const uint32_t* part_begin,
                         const uint32_t* part_end, uint32_t* work, uint32_t grid, bool boxes, float* grad_pow4, hipStream_t st) {
    const uint32_t n = G.n;
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, st, work, num_parts * kWorkStride, 0u);
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, st, wmax, ns, 0u);
    const uint64_t words = 3ull * total_photons;
    if (words) {
        const uint32_t zb = (uint32_t)std::min<uint64_t>((words + 255) / 256, 8192);
        hipLaunchKernelGGL(k_zero_u64, dim3(zb), dim3(256), 0, st, G.acc, words);
    }
    if (n)
        hipLaunchKernelGGL(k_bwd_wmax_batch, dim3((n + kWmaxBlock - 1) / kWmaxBlock), dim3(kWmaxBlock), 0, st, n, slot_begin, ns, count,
                           G.grad, G.clr, G.infl, fwd_r2, fwd_count, wmax);
    hipLaunchKernelGGL(k_bwd_scale_batch, dim3(1), dim3(64), 0, st, ns, slot_begin, count, wmax, scale);
    const uint32_t chunk = std::max<uint32_t>(1u, std::min<uint32_t>(kBwdChunk, (uint32_t)kPairCap / G.k));
    const uint32_t need = G.k + 64;
#define MNRT_KBX(C, X)                                                                                              \
    hipLaunchKernelGGL((k_knn_bwd_batch<C, X>), dim3(grid), dim3(64 * kWavesPerBlock), 0, st, G, scenes, slot_begin, \
                       ns, count, photon_begin, scale, chunk, num_parts, part_begin, part_end, work)
#define MNRT_KBB(C)                  \
    do {                             \
        if (boxes) MNRT_KBX(C, true); \
        else MNRT_KBX(C, false);     \
    } while (0)
    if (need <= 128) MNRT_KBB(128);
    else if (need <= 256) MNRT_KBB(256);
    else MNRT_KBB(512);
#undef MNRT_KBB
#undef MNRT_KBX
    if (total_photons)
        hipLaunchKernelGGL(k_fix_to_float_batch, dim3((total_photons + 255) / 256), dim3(256), 0, st, total_photons,
                           photon_begin, ns, G.acc, scale, (float4*)grad_pow4);
    MNRT_HIP_CHECK(hipGetLastError());
    return MNRT_OK;
}
}  // namespace mnrt

namespace {

constexpr size_t kScratchWords = sizeof(scratch) / sizeof(uint32_t);
constexpr int kScratchMaxDevices = 64;
std::mutex g_scratch_mu;
uint32_t* g_scratch_addr[kScratchMaxDevices] = {};

// Words of scratch mnrt_knn_gather_noalloc needs for n queries: the processing order, and
// 5 words per query (radiance + inverse distance) when slot indices are given.
size_t noalloc_words(uint32_t n, bool slots) {
    if (n >= mnrt::kOrderMaxItems) return SIZE_MAX;  // far beyond the array either way
    return mnrt::spatial_order_words(n) + (slots ? 5ull * n : 0ull);
}

}  // namespace

namespace mnrt {

// Looks up this device's address of `scratch` (the device must be current); kept per
// device, so later calls on it reuse the address.
int knn_scratch_init(int device) {
    if (device < 0 || device >= kScratchMaxDevices) return MNRT_ERR_NODEV;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_addr[device]) return MNRT_OK;
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return MNRT_ERR_HIP;
    g_scratch_addr[device] = (uint32_t*)p;
    return MNRT_OK;
}

}  // namespace mnrt

static int knn_check(const mnrt_tree* pmap, uint32_t k) {
    if (!pmap) return MNRT_ERR_ARG;
    if (k == 0 || k > MNRT_KNN_MAX_K) return MNRT_ERR_ARG;
    if (pmap->kind != MNRT_KIND_POINT || !pmap->d_nodes || !pmap->d_recs || pmap->num_nodes == 0)
        return MNRT_ERR_STATE;
    if (pmap->max_level > MNRT_MAX_LEVEL || pmap->num_nodes >= mnrt::kUniform8MaxIndex) return MNRT_ERR_CAPACITY;
    return MNRT_OK;
}

extern "C" int mnrt_knn_gather(const mnrt_tree* pmap, uint32_t k, float r_max, uint32_t n,
                               const float* d_pos4, const float* d_nrm4, const float* d_dir4,
                               const float* d_infl4, const float* d_clr4, const uint32_t* d_idx_sp,
                               const float* d_query_radius, const float* d_orig4, float* d_io_rad4,
                               float* d_io_inv_dist, float* d_out_r2, float* d_out_irr4, uint32_t* d_out_nbr,
                               uint32_t* d_out_count, void* stream) {
    int rc = knn_check(pmap, k);
    if (rc != MNRT_OK) return rc;
    if (n == 0) return MNRT_OK;
    if (!d_pos4 || !d_nrm4 || !d_dir4 || !d_infl4 || !d_io_rad4 || !(r_max > 0.0f)) return MNRT_ERR_ARG;
    if (d_io_inv_dist && !d_orig4) return MNRT_ERR_ARG;
    hipStream_t st = (hipStream_t)stream;
    mnrt::KnnArgs A{};
    A.nodes = (const uint2*)(pmap->d_qnodes ? pmap->d_qnodes : pmap->d_nodes);
    A.recs = (const float4*)pmap->d_recs;
    A.boxes = mnrt::box_tree(*pmap);
    A.k = k;
    A.r2max = r_max * r_max;
    A.r_max = r_max;
    A.n = n;
    A.pos = (const float4*)d_pos4;
    A.nrm = (const float4*)d_nrm4;
    A.dir = (const float4*)d_dir4;
    A.infl = (const float4*)d_infl4;
    A.clr = (const float4*)d_clr4;
    A.r_query = d_query_radius;
    A.orig = (const float4*)d_orig4;
    A.out_r2 = d_out_r2;
    A.out_irr = (float4*)d_out_irr4;
    A.out_nbr = d_out_nbr;
    A.out_count = d_out_count;
    void* obuf = nullptr;
    rc = mnrt::spatial_order(pmap->root_min, pmap->root_max, n, d_pos4, st, &A.order, &obuf, &A.order_far);
    if (rc != MNRT_OK) return rc;
    float4* tmp = nullptr;
    if (d_idx_sp) {
        // per-query values first, then summed into their slots run by run
        MNRT_HIP_CHECK(mnrt::pool_alloc((void**)&tmp, (size_t)n * (sizeof(float4) + sizeof(float)), st));
        A.rad_out = tmp;
        A.accumulate = 0;
        A.inv_dist = d_io_inv_dist ? (float*)(tmp + n) : nullptr;
        A.inv_accumulate = 0;
    } else {
        A.rad_out = (float4*)d_io_rad4;
        A.accumulate = 1;
        A.inv_dist = d_io_inv_dist;
        A.inv_accumulate = 1;
    }
    rc = mnrt::launch_knn<mnrt::kModeRadiance>(A, st);
    if (rc == MNRT_OK && d_idx_sp) {
        hipLaunchKernelGGL(mnrt::k_scatter_runs, dim3((n + 255) / 256), dim3(256), 0, st, tmp,
                           d_io_inv_dist ? (const float*)(tmp + n) : (const float*)nullptr, d_idx_sp, n,
                           (float4*)d_io_rad4, d_io_inv_dist);
        if (hipGetLastError() != hipSuccess) rc = MNRT_ERR_HIP;
    }
    if (tmp && mnrt::pool_free(tmp, st) != hipSuccess && rc == MNRT_OK) rc = MNRT_ERR_HIP;
    if (obuf && mnrt::pool_free(obuf, st) != hipSuccess && rc == MNRT_OK) rc = MNRT_ERR_HIP;
    return rc;
}

extern "C" int mnrt_knn_gather_noalloc(const mnrt_tree* pmap, uint32_t k, float r_max, uint32_t n,
                                       const float* d_pos4, const float* d_nrm4, const float* d_dir4,
                                       const float* d_infl4, const float* d_clr4, const uint32_t* d_idx_sp,
                                       const float* d_query_radius, const float* d_orig4, float* d_io_rad4,
                                       float* d_io_inv_dist, float* d_out_r2, float* d_out_irr4,
                                       uint32_t* d_out_nbr, uint32_t* d_out_count, void* stream) {
    int rc = knn_check(pmap, k);
    if (rc != MNRT_OK) return rc;
    if (n == 0) return MNRT_OK;
    if (!d_pos4 || !d_nrm4 || !d_dir4 || !d_infl4 || !d_io_rad4 || !(r_max > 0.0f)) return MNRT_ERR_ARG;
    if (d_io_inv_dist && !d_orig4) return MNRT_ERR_ARG;
    if (noalloc_words(n, d_idx_sp != nullptr) > kScratchWords) return MNRT_ERR_CAPACITY;
    int dev = 0;
    MNRT_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kScratchMaxDevices) return MNRT_ERR_NODEV;
    uint32_t* scr = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        scr = g_scratch_addr[dev];
    }
    if (!scr) {  // mnrt_device_init was not called for this device
        rc = mnrt::knn_scratch_init(dev);
        if (rc != MNRT_OK) return rc;
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        scr = g_scratch_addr[dev];
    }
    hipStream_t st = (hipStream_t)stream;
    mnrt::KnnArgs A{};
    A.nodes = (const uint2*)(pmap->d_qnodes ? pmap->d_qnodes : pmap->d_nodes);
    A.recs = (const float4*)pmap->d_recs;
    A.boxes = mnrt::box_tree(*pmap);
    A.k = k;
    A.r2max = r_max * r_max;
    A.r_max = r_max;
    A.n = n;
    A.pos = (const float4*)d_pos4;
    A.nrm = (const float4*)d_nrm4;
    A.dir = (const float4*)d_dir4;
    A.infl = (const float4*)d_infl4;
    A.clr = (const float4*)d_clr4;
    A.r_query = d_query_radius;
    A.orig = (const float4*)d_orig4;
    A.out_r2 = d_out_r2;
    A.out_irr = (float4*)d_out_irr4;
    A.out_nbr = d_out_nbr;
    A.out_count = d_out_count;
    // scratch layout: [processing order][per-query radiance (4 n)][per-query inverse distance (n)]
    rc = mnrt::spatial_order_into(pmap->root_min, pmap->root_max, n, d_pos4, st, scr, &A.order, &A.order_far);
    if (rc != MNRT_OK) return rc;
    float4* tmp = nullptr;
    if (d_idx_sp) {
        // every query's value is written before the run sums read it: nothing to clear
        tmp = (float4*)(scr + mnrt::spatial_order_words(n));
        A.rad_out = tmp;
        A.accumulate = 0;
        A.inv_dist = d_io_inv_dist ? (float*)(tmp + n) : nullptr;
        A.inv_accumulate = 0;
    } else {
        A.rad_out = (float4*)d_io_rad4;
        A.accumulate = 1;
        A.inv_dist = d_io_inv_dist;
        A.inv_accumulate = 1;
    }
    rc = mnrt::launch_knn<mnrt::kModeRadiance>(A, st);
    if (rc == MNRT_OK && d_idx_sp) {
        hipLaunchKernelGGL(mnrt::k_scatter_runs, dim3((n + 255) / 256), dim3(256), 0, st, tmp,
                           d_io_inv_dist ? (const float*)(tmp + n) : (const float*)nullptr, d_idx_sp, n,
                           (float4*)d_io_rad4, d_io_inv_dist);
        if (hipGetLastError() != hipSuccess) rc = MNRT_ERR_HIP;
    }
    return rc;
}

extern "C" int mnrt_knn_radii(const mnrt_tree* pmap, uint32_t k, float r_max, uint32_t n,
                              const float* d_pos4, float* d_out_radius, void* stream) {
    int rc = knn_check(pmap, k);
    if (rc != MNRT_OK) return rc;
    if (n == 0) return MNRT_OK;
    if (!d_pos4 || !d_out_radius || !(r_max > 0.0f)) return MNRT_ERR_ARG;
    mnrt::KnnArgs A{};
    A.nodes = (const uint2*)(pmap->d_qnodes ? pmap->d_qnodes : pmap->d_nodes);
    A.recs = (const float4*)pmap->d_recs;
    A.boxes = mnrt::box_tree(*pmap);
    A.k = k;
    A.r2max = r_max * r_max;
    A.r_max = r_max;
    A.n = n;
    A.pos = (const float4*)d_pos4;
    A.out_radius = d_out_radius;
    hipStream_t st = (hipStream_t)stream;
    void* obuf = nullptr;
    rc = mnrt::spatial_order(pmap->root_min, pmap->root_max, n, d_pos4, st, &A.order, &obuf, &A.order_far);
    if (rc != MNRT_OK) return rc;
    rc = mnrt::launch_knn<mnrt::kModeRadii>(A, st);
    if (obuf && mnrt::pool_free(obuf, st) != hipSuccess && rc == MNRT_OK) rc = MNRT_ERR_HIP;
    return rc;
}

extern "C" int mnrt_knn_gather_bwd(const mnrt_tree* pmap, uint32_t k, float r_max, uint32_t n,
                                   const float* d_pos4, const float* d_nrm4, const float* d_dir4,
                                   const float* d_infl4, const float* d_clr4, const float* d_query_radius,
                                   const float* d_grad_rad4,
                                   const float* d_r2, const uint32_t* d_count, float* d_grad_pow4,
                                   float* d_grad_clr4, void* stream) {
    int rc = knn_check(pmap, k);
    if (rc != MNRT_OK) return rc;
    if (!d_grad_pow4) return MNRT_ERR_ARG;
    hipStream_t st = (hipStream_t)stream;
    const uint32_t np = pmap->num_elems;
    if (n == 0 || np == 0) {
        if (np) MNRT_HIP_CHECK(hipMemsetAsync(d_grad_pow4, 0, (size_t)np * 16, st));
        return MNRT_OK;
    }
    if (!d_pos4 || !d_nrm4 || !d_dir4 || !d_infl4 || !d_grad_rad4 || !d_r2 || !d_count || !(r_max > 0.0f))
        return MNRT_ERR_ARG;
    // (not for a stream that is being captured: the workspace is given back on return)
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    MNRT_HIP_CHECK(hipStreamIsCapturing(st, &cs));
    if (cs != hipStreamCaptureStatusNone) return MNRT_ERR_HIP;
    void* buf = nullptr;
    MNRT_HIP_CHECK(mnrt::pool_alloc(&buf, (size_t)np * 24 + 256, st));
    // accumulators, the largest weight, the scale: all on the device, so the call waits for nothing
    // (reading the weight back and scaling on the host left the GPU idle for a fifth of a 131072-photon,
    // 77361-query call)
    unsigned long long* acc = (unsigned long long*)buf;
    uint32_t* wmax = (uint32_t*)(acc + 3ull * np);
    double* scale = (double*)(acc + 3ull * np + 1u);
    const uint64_t words = 3ull * np + 1u;
    hipLaunchKernelGGL(mnrt::k_zero_u64, dim3((uint32_t)std::min<uint64_t>((words + 255) / 256, 8192)), dim3(256), 0, st,
                       acc, words);
    hipLaunchKernelGGL(mnrt::k_bwd_wmax, dim3((n + mnrt::kWmaxBlock - 1) / mnrt::kWmaxBlock), dim3(mnrt::kWmaxBlock), 0,
                       st, n, (const float4*)d_grad_rad4, (const float4*)d_clr4, (const float4*)d_infl4, d_r2, d_count,
                       wmax);
    hipLaunchKernelGGL(mnrt::k_bwd_scale, dim3(1), dim3(64), 0, st, n, (const uint32_t*)wmax, scale);
    rc = hipGetLastError() == hipSuccess ? MNRT_OK : MNRT_ERR_HIP;
    const uint32_t* order = nullptr;
    const uint32_t* order_far = nullptr;
    void* obuf = nullptr;
    if (rc == MNRT_OK)
        rc = mnrt::spatial_order(pmap->root_min, pmap->root_max, n, d_pos4, st, &order, &obuf, &order_far);
    if (rc == MNRT_OK) {
        mnrt::KnnArgs A{};
        A.order = order;
        A.order_far = order_far;
        A.nodes = (const uint2*)(pmap->d_qnodes ? pmap->d_qnodes : pmap->d_nodes);
        A.recs = (const float4*)pmap->d_recs;
        A.boxes = mnrt::box_tree(*pmap);
        A.k = k;
        A.r2max = r_max * r_max;
        A.r_max = r_max;
        A.n = n;
        A.pos = (const float4*)d_pos4;
        A.nrm = (const float4*)d_nrm4;
        A.dir = (const float4*)d_dir4;
        A.infl = (const float4*)d_infl4;
        A.clr = (const float4*)d_clr4;
        A.r_query = d_query_radius;
        A.grad = (const float4*)d_grad_rad4;
        A.acc = acc;
        A.fix_scale = scale;
        A.out_grad_clr = (float4*)d_grad_clr4;
        rc = mnrt::launch_knn_bwd(A, st);
    }
    if (rc == MNRT_OK) {
        hipLaunchKernelGGL(mnrt::k_fix_to_float, dim3((np + 255) / 256), dim3(256), 0, st, np, acc,
                           (const double*)scale, (float4*)d_grad_pow4);
        if (hipGetLastError() != hipSuccess) rc = MNRT_ERR_HIP;
    }
    if (obuf) (void)mnrt::pool_free(obuf, st);
    (void)mnrt::pool_free(buf, st);
    return rc;
}
