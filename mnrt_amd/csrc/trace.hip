// trace.hip — closest-hit ray traversal of the packed preorder kd-tree on gfx950.
//
// Replaces kernel_FindIntersections + dev_FindNextIntersectionKDWhileWhile<true>
// (raytracing.cu:503-645, 854-879) and its wrapper KernelRTTraceRays
// (raytracing.cu:1617-1635).  One wave per run of rays (trace_dev.h).  Differences from
// the reference, all deliberate:
//   * the tree and triangles are kernel arguments (no __constant__ / texture binding),
//     so several trees can be traced at once;
//   * leaves address contiguous leaf-ordered triangle records (v0, e1, e2: 48 B), not
//     texture fetches of three vertices through an index list;
//   * interval decisions are widened by a relative 2^-16 and equal lambdas resolve to
//     the lower triangle index, so the hit equals the brute-force closest hit over all
//     triangles whatever the tree;
//   * the traversal stack is bounded by the build's level cap instead of KD_MAX_HEIGHT
//     local-memory arrays with no overflow check, and its top entries live in LDS.
#include "batch_dev.h"
#include "trace_dev.h"

namespace mnrt {

__global__ __launch_bounds__(256) void k_clear_words(uint32_t* __restrict__ p, uint64_t n) {
    for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < n; i += gridDim.x * 256ull) p[i] = 0u;
}

RayShared::RayShared(uint32_t windows, hipStream_t st) : st_(st) {
    if (windows <= kWindowWaves) return;
    // (a captured launch does without: no allocation is recorded)
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    hipError_t rc = hipStreamIsCapturing(st, &cs);
    if (cs != hipStreamCaptureStatusNone) return;
    const uint64_t words = RayWindow::shared_words(windows);
    void* buf = nullptr;
    if (rc == hipSuccess) rc = pool_alloc(&buf, 4u * words, st);
    if (rc != hipSuccess) {  // the launch does without; its own check is for the launch
        (void)hipGetLastError();
        return;
    }
    p = (uint32_t*)buf;
    hipLaunchKernelGGL(k_clear_words, dim3((uint32_t)std::min<uint64_t>((words + 255u) / 256u, 1024u)), dim3(256), 0, st, p, words);
}
RayShared::~RayShared() {
    if (p) (void)pool_free(p, st_);
}

// Rays first..last of arrays; results as they are asked for.
struct RaySource {
    static constexpr uint32_t kTogether = kRaysTogether;
    RayWindow rays;
    uint32_t first;  // of the scene's rays
    const float4* __restrict__ orig;
    const float4* __restrict__ dir;
    const float4* __restrict__ recs;
    int32_t* __restrict__ out_tri;
    float* __restrict__ out_t;
    float2* __restrict__ out_bary;
    float4* __restrict__ out_pt;
    uint32_t* __restrict__ out_valid;
    uint32_t ray = 0;

    __device__ __forceinline__ bool start(uint32_t i, f3& o, f3& d, float&) {
        i = ray = first + i;
        o = xyz(orig[i]);
        d = xyz(dir[i]);
        return true;
    }
    __device__ __forceinline__ bool finish(f3& o, f3& d, float, const Hit& h) {
        const bool hit = h.tri >= 0;
        const float t = hit ? h.t : 0.0f;
        out_tri[ray] = h.tri;
        if (out_t) out_t[ray] = t;
        if (out_bary) {
            float lam, u = 0.0f, v = 0.0f;
            if (hit) {  // the hit's test again: the same operations, the same bits
                const float4* r = recs + 3ull * h.rec;
                ray_tri(xyz(r[0]), xyz(r[1]), xyz(r[2]), o, d, lam, u, v);
            }
            out_bary[ray] = make_float2(u, v);
        }
        if (out_pt) out_pt[ray] = make_float4(o.x + d.x * t, o.y + d.y * t, o.z + d.z * t, 0.0f);
        if (out_valid) out_valid[ray] = hit ? 1u : 0u;
        return false;
    }
};

// One wave per workgroup: its LDS goes to the next when its own run is done.  kShared: the launch has shared
// words (the same kernel with and without them: 6144 camera rays 50 us, 49 without).
template <bool kShared>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6))) void k_trace_closest(
    const uint2* __restrict__ nodes, const float4* __restrict__ recs, RootBox root, uint32_t n, uint32_t width, uint32_t* shared,
    const float4* __restrict__ orig, const float4* __restrict__ dir, float eps,
    int32_t* __restrict__ out_tri, float* __restrict__ out_t, float2* __restrict__ out_bary,
    float4* __restrict__ out_pt, uint32_t* __restrict__ out_valid) {
    __shared__ __align__(8) uint32_t s_wave[kTraceWords];
    if (kShared && !RayWindow::claim(shared, blockIdx.x, threadIdx.x)) return;
    RaySource src{RayWindow(blockIdx.x * width, n, width, kShared ? shared : nullptr), 0u, orig, dir, recs, out_tri, out_t, out_bary, out_pt, out_valid};
    trace_stream<false, kTraceStack>(nodes, recs, root, eps, 0.0f, s_wave, src);
}

}  // namespace mnrt

extern "C" int mnrt_trace_closest(const mnrt_tree* tree, uint32_t n, const float* d_orig4,
                                  const float* d_dir4, float eps, int32_t* d_out_tri,
                                  float* d_out_t, float* d_out_bary2, float* d_out_pt4,
                                  uint32_t* d_out_valid, void* stream) {
    if (!tree || (n > 0 && (!d_out_tri || !d_orig4 || !d_dir4))) return MNRT_ERR_ARG;
    if (tree->kind != MNRT_KIND_TRI || !tree->d_nodes || !tree->d_recs || tree->num_nodes == 0)
        return MNRT_ERR_STATE;
    if (tree->max_level > MNRT_MAX_LEVEL) return MNRT_ERR_CAPACITY;
    if (n == 0) return MNRT_OK;
    mnrt::RootBox rb;
    for (int a = 0; a < 3; ++a) {
        rb.lo[a] = tree->root_min[a];
        rb.hi[a] = tree->root_max[a];
    }
    const uint32_t width = mnrt::trace_width(n), windows = mnrt::trace_windows(n, width);
    const mnrt::RayShared shared(windows, (hipStream_t)stream);
    hipLaunchKernelGGL(shared.p ? mnrt::k_trace_closest<true> : mnrt::k_trace_closest<false>, dim3(windows), dim3(64), 0,
                       (hipStream_t)stream, (const uint2*)tree->d_nodes, (const float4*)tree->d_recs, rb, n, width, shared.p,
                       (const float4*)d_orig4, (const float4*)d_dir4, eps, d_out_tri, d_out_t,
                       (float2*)d_out_bary2, (float4*)d_out_pt4, d_out_valid);
    MNRT_HIP_CHECK(hipGetLastError());
    return MNRT_OK;
}

// ---- batches: many trees, one persistent launch ----------------------------------------

namespace mnrt {

// Waves take units of consecutive rays, parts of a tile, from a work counter until every tile
// is done; tile t belongs to the scene whose tile range holds it.  Each XCD (workgroup id
// mod 8 on MI355X) has its own counter over a contiguous share of the tiles, so an
// XCD's L2 holds the trees of the scenes it traces; a wave whose share is done
// takes units from the next XCD's share.
template <int kStack>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void k_trace_batch(TraceBatchArgs B) {
    extern __shared__ __align__(8) uint32_t s_waves[];
    const uint32_t xcd = blockIdx.x % B.num_parts, wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const uint32_t per_tile = B.tile_rays / B.unit;
    for (uint32_t part = 0; part < B.num_parts; ++part) {
        const uint32_t p = (xcd + part) % B.num_parts;
        const uint32_t begin = B.part_begin[p], units = (B.part_end[p] - begin) * per_tile;
        for (;;) {
            const uint32_t u = take_unit(B.work, p, units, part > 0u, lane);
            if (u >= units) break;
            const uint32_t t = begin + u / per_tile;
            const uint32_t s = seg_of(B.tile_begin, B.num_scenes, t);
            const TraceScene& d = B.scenes[s];
            const uint32_t first = d.ray_begin + (t - B.tile_begin[s]) * B.tile_rays + (u % per_tile) * B.unit;
            if (first >= d.ray_end) continue;
            RootBox root;
            for (int a = 0; a < 3; ++a) {
                root.lo[a] = d.lo[a];
                root.hi[a] = d.hi[a];
            }
            const float4* recs = global_ptr(d.recs);
            RaySource src{RayWindow(0u, min(B.unit, d.ray_end - first), min(B.unit, 64u), nullptr, B.unit), first, B.orig, B.dir, recs, B.out_tri, B.out_t, B.out_bary, nullptr,
                          nullptr};
            trace_stream<false, kStack>(global_ptr(d.nodes), recs, root, d.eps, 0.0f, s_waves + wave * kTraceWords,
                                        src);
        }
    }
}

// A set of rays while there are at most sixteen a wave, then four sets (61.5M rays of 256 scenes:
// 15.3 ms by single sets, a million atomics on eight counters, 14.5 by four; 1.69M rays of 32 scenes:
// the frame takes 4.2 ms by single sets, 4.5 by four, whose ends are uneven).
uint32_t trace_unit(uint64_t rays, uint32_t tile) {
    return rays > 1024u * (uint64_t)kTraceWaves && tile % 256u == 0u ? 256u : trace_width(rays);
}

int launch_trace_batch(const TraceBatchArgs& B, int stack, uint32_t grid, uint32_t block, hipStream_t st) {
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, st, B.work, B.num_parts * kWorkStride, 0u);
    const uint32_t lds = 4u * kTraceWords * (block / 64u);
    switch (stack) {
        case 16: hipLaunchKernelGGL(k_trace_batch<16>, dim3(grid), dim3(block), lds, st, B); break;
        case 24: hipLaunchKernelGGL(k_trace_batch<24>, dim3(grid), dim3(block), lds, st, B); break;
        case 32: hipLaunchKernelGGL(k_trace_batch<32>, dim3(grid), dim3(block), lds, st, B); break;
        case kTraceStack: hipLaunchKernelGGL(k_trace_batch<kTraceStack>, dim3(grid), dim3(block), lds, st, B); break;
        default: return MNRT_ERR_ARG;
    }
    MNRT_HIP_CHECK(hipGetLastError());
    return MNRT_OK;
}

}  // namespace mnrt
