// trace.hip -- BVH8 closest-hit traversal, alone or fused with the diffuse
// path it serves.
//
// Replaces IntersectorStreamCuda::intersect (core/intersector_stream_cuda.h:27-34),
// which the reference forwards to OptiX Prime's closest query
// (accel/optix/optix_intersector_stream_cuda.cpp:77-82), and, in the fused
// modes, the raygen / shade kernels and the per-bounce host loop of
// DiffuseRendererCuda::render (render/diffuse_renderer_cuda.cu:27-120,159-212).
//
// One ray per lane.  The kernel is persistent: each wave takes work from the
// launch's counters; when at least kRefill of its 64 lanes are idle, the wave
// ballots them, takes that many work items with one atomic and hands them out
// by lane prefix, so lanes stay busy on incoherent bounces.  The traversal
// stack is a per-lane ring of kStackLds entries in LDS; deeper entries spill
// to a per-lane slice of global memory.  Each entry keeps the entry distance
// of its box, so nodes behind the closest hit are dropped when popped.
//
// The loop is bound by VALU issue (every slot taken, with 27 to 34 % of the
// lanes active), so a step costs what it issues.  A push wraps its positions only in
// waves where some stack has passed the ring's end, the node's exponents scale
// by ldexp, the near and far offsets share one fma, a leaf slot's byte comes
// out by one permute, and hit coordinates are computed once per ray: 1.3 M
// triangles of spheres at 1080p 4806 -> 4936 Mrays/s batched and 2930 -> 3005
// in plain frames, 0.4 M triangles at 720p 2760 -> 2830 and 1073 -> 1110.
//
// Modes:
//   kModeTrace    work item = a ray of the input array; writes its hit record.
//   kModeDiffuse  work item = a path (one pixel sample).  The lane generates
//                 the camera ray, and when a ray finishes it shades it in
//                 place: a miss adds the path throughput, a hit at max depth
//                 adds 0, any other hit bounces (cosine hemisphere) and the
//                 lane traces the next ray of the same path.  Paths of every
//                 depth share the launch, so a frame pays the latency of its
//                 slowest path once instead of once per bounce, and no ray or
//                 hit record goes through HBM.
//   kModePrimary  as kModeDiffuse with the primary shading ((N+1)/2, 0.05).
//   kModeDiffuse2 as kModeDiffuse with next-event shadow rays: at each hit the
//                 lane traces an any-hit shadow ray, then the path's next ray.
//   kModeOccluded work item = a ray of the input array; any-hit query, writes
//                 the distance of a blocking triangle or -1.
//
// Result of a query: the hit with the smallest (t, primId) among triangles
// that the watertight test says the ray crosses with tnear <= t <= tfar, t
// being the plane distance computed in double -- the same answer as testing
// every triangle, whatever the visiting order.
#include <algorithm>
#include <type_traits>

#include "launch_shape.h"
#include "prt_internal.h"

namespace prt {
namespace {

constexpr int kStackLds = 16;      // default LDS entries per lane (power of two)
constexpr int kRefill = 32;        // default: refill when this many lanes are idle
// In launches of at least so many waves a wave stops when its own work counter
// has run out: 64 waves serve each of the 16, which hold about the same work
// (work_deal.h), and a look at all counters for items left queues up at their lines when all waves
// take it at the end.  With / without that look, us: closest hits 300 k 206 /
// 186, 600 k 262 / 223, 1 M 432 / 398, any hit 500 k 214 / 177; Mrays/s of plain
// frames 3270 / 3630, 2100 / 2270, 1390 / 1500, 2320 / 2500 (four scenes); 300 k
// rays on each of three streams at once 127 / 105 us.
constexpr uint32_t kOwnCounterWaves = 1024;

enum {
    kModeTrace = 0, kModeDiffuse = 1, kModePrimary = 2, kModeBatch = 3, kModeRgb = 4, kModeAdjoint = 5,
    kModeDiffuse2 = 6, kModeOccluded = 7
};

__device__ __forceinline__ float as_f(uint32_t u) { return __uint_as_float(u); }

// Minimum over the 8 lanes of an aligned group, in every lane of it: three
// DPP steps (lane ^ 1, lane ^ 2, then the mirror of the 8 lanes, whose halves
// hold one value each by then) instead of three trips through the LDS crossbar.
__device__ __forceinline__ uint32_t dpp8(uint32_t v, int step)
{
    const int x = (int)v;
    return (uint32_t)(step == 0 ? __builtin_amdgcn_update_dpp(x, x, 0xB1, 0xF, 0xF, true)
                      : step == 1 ? __builtin_amdgcn_update_dpp(x, x, 0x4E, 0xF, 0xF, true)
                                  : __builtin_amdgcn_update_dpp(x, x, 0x141, 0xF, 0xF, true));
}
__device__ __forceinline__ uint32_t min8(uint32_t v)
{
    v = min(v, dpp8(v, 0));
    v = min(v, dpp8(v, 1));
    return min(v, dpp8(v, 2));
}
__device__ __forceinline__ uint32_t or8(uint32_t v)
{
    v |= dpp8(v, 0);
    v |= dpp8(v, 1);
    return v | dpp8(v, 2);
}

// Position of the r-th (from 0) set bit of m, which has more than r.
__device__ __forceinline__ uint32_t nth_bit(uint32_t m, uint32_t r)
{
    uint32_t pos = 0;
#pragma unroll
    for (int w = 16; w >= 1; w >>= 1) {
        const uint32_t c = (uint32_t)__popc((m >> pos) & ((1u << w) - 1u));
        const bool up = r >= c;
        pos += up ? (uint32_t)w : 0u;
        r -= up ? c : 0u;
    }
    return pos;
}

// kLook: the fused diffuse frame with the frame lookahead compiled in.
template <bool kCount, int kMode, int kBlock = kTraceBlock, int kStack = kStackLds, bool kLook = false>
__global__ __launch_bounds__(kBlock, kMode == kModeBatch || kMode == kModeAdjoint || kMode == kModeDiffuse2 || kLook ? 4 : 1) void k_trace(SceneDevice sc, TraceLaunch tl, PathLaunch pl, BatchLaunch bl,
                                                  uint2* spill, int stack_entries, int refill, uint32_t* err)
{
    static_assert((kStack & (kStack - 1)) == 0, "LDS stack depth must be a power of two");
    constexpr bool kRayQuery = kMode == kModeTrace || kMode == kModeOccluded;
    __shared__ uint32_t st_node[kStack * kBlock];
    __shared__ float st_t[kStack * kBlock];
    // rays per depth: an LDS histogram in the instrumented variant only, so
    // the timed variant keeps 32 KiB of LDS per block (5 blocks per CU)
    uint32_t* depth_hist = nullptr;
    if constexpr (kCount && !kRayQuery && kMode != kModeBatch) {
        __shared__ uint32_t hist[kMaxQueueDepth];
        depth_hist = hist;
    }
    uint32_t n_rays = 0;
    uint4* grad_sums = nullptr;  // add_gradient
    if constexpr (kMode == kModeAdjoint) {
        __shared__ uint4 sums[kBlock];
        grad_sums = sums;
    }

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    // LDS ring entry q of this lane: byte offset ((q mod kStack) * kBlock + tid) * 4
    constexpr int kRingShift = kBlock == 256 ? 10 : (kBlock == 128 ? 9 : 8);
    static_assert(kBlock == 256 || kBlock == 128 || kBlock == 64, "ring layout");
    constexpr uint32_t kRingMask = (uint32_t)(kStack - 1) << kRingShift;
    const uint32_t tid4 = (uint32_t)tid * 4u;
    auto ring_off = [&](int q) -> uint32_t { return (((uint32_t)q << kRingShift) & kRingMask) | tid4; };
    auto ring_node = [&](uint32_t off) -> uint32_t& { return *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(st_node) + off); };
    auto ring_t = [&](uint32_t off) -> float& { return *reinterpret_cast<float*>(reinterpret_cast<char*>(st_t) + off); };
    const uint64_t lane_lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const uint32_t count = kRayQuery ? (tl.count_ptr ? *tl.count_ptr : tl.count)
                         : (kMode == kModeBatch ? bl.total_work
                                                : (kMode == kModeAdjoint || (kMode == kModeRgb && pl.rgb_planes)
                                                       ? pl.entries * (uint32_t)pl.spp
                                                       : pl.entries));
    uint2* my_spill = spill + ((size_t)blockIdx.x * kBlock + tid) * (size_t)stack_entries;
    const int spill_cap = stack_entries;
    if constexpr (kCount && !kRayQuery && kMode != kModeBatch) {
        if (tid < kMaxQueueDepth) depth_hist[tid] = 0;
        __syncthreads();
    }

    // A stack overflow.  A small query's flag is in pinned host memory, where the
    // link may not carry an atomic OR; a query raises nothing else, so it stores.
    auto raise_overflow = [&]() {
        if constexpr (kRayQuery) __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        else atomicOr(err, 1u);
    };

    bool active = false;   // the lane holds a ray or path
    bool tracing = false;  // ... and is traversing (else its ray waits for shading)
    uint32_t ray_idx = 0;
    f3 o{0, 0, 0}, d{0, 0, 0};
    float tmin = 0.0f, tbest = 0.0f;
    float inv_x = 0, inv_y = 0, inv_z = 0;
    bool neg_x = false, neg_y = false, neg_z = false;
    WatertightRay wr{};
    int32_t best_prim = -1;
    uint32_t best_rec = 0;
    int sp = 0, bottom = 0;
    int32_t node = -1;
    float node_t = 0.0f;        // entry distance of `node`
    uint32_t pend = 0, pend_base = 0;  // triangle records still to test: pend_base + bit index
    uint32_t pend2 = 0, pend2_base = 0;  // a second leaf group, found while the first is tested
    // path state (fused modes)
    int32_t pixel = 0;
    uint32_t rng = 0;
    int depth = 0;
    float lw = 1.0f;
    int max_depth = pl.max_depth;
    float albedo = pl.albedo;
    // scene of the lane's current ray (per lane in the batch mode)
    const PRT_GLOBAL Bvh8Node* nodes = global_view(sc.nodes);
    const PRT_GLOBAL float* tris = global_view(sc.tris);
    const PRT_GLOBAL int32_t* prim_ids = global_view(sc.prim_ids);
    int32_t scene_id = 0;  // batch mode: the lane's scene (for its shading attributes)
    float* sample_out = nullptr;
    // RGB throughput (RGB and adjoint modes); adjoint: per-channel product of
    // the path's nonzero albedos and count of zero albedos from the primal
    // pass, and the path's weight dLoss/dI / spp
    float lg = 1.0f, lb = 1.0f;
    float pr = 1.0f, pg = 1.0f, pb = 1.0f;
    uint32_t zeros = 0;  // 8 bits per channel
    float gw_r = 0.0f, gw_g = 0.0f, gw_b = 0.0f;
    bool replay = false;
    uint32_t hit_slot = 0;  // the path's column of PathLaunch::path_hits
    int path_pass = 0;
    // diffuse2: the current ray is a shadow ray; the path's next ray waits in
    // (eo, ed); radiance gathered so far
    bool shadow = false;
    f3 eo{0, 0, 0}, ed{0, 0, 0};
    float lsum = 0.0f;
    unsigned long long n_nodes = 0, n_tris = 0, n_spill = 0;
    unsigned long long n_wsteps = 0, n_lsteps = 0, n_wshade = 0;  // instrumented SIMT occupancy
    unsigned long long n_dwsteps = 0, n_dlsteps = 0;              // ... after the work ran out
    unsigned long long t_exhausted = 0;                           // wall clock when it ran out
    bool exhausted = false;  // wave-uniform: the work is handed out
    // Cooperative traversal of a wave's last paths (see coop_traverse below)
    constexpr bool kCoop = !kLook;
    const bool coop_on = kCoop && pl.coop != 0;
    uint64_t coop_paths = 0;                 // lanes whose paths the wave goes on with in groups
    const int gj = lane & 7;                 // this lane's place in its group
    const int gbase = lane & ~7;             // first lane of the group
    constexpr int kGStack = 8 * kStack;      // a group's stack: its lanes' LDS rings joined
    uint2* const g_spill = spill + ((size_t)blockIdx.x * kBlock + (tid & ~7)) * (size_t)stack_entries;
    auto group_slot = [&](int q) -> int { return ((q >> 3) & (kStack - 1)) * kBlock + (tid & ~7) + (q & 7); };

    // Frame lookahead (diffuse and diffuse2, LookState); a path of frame pass + l is
    // at level l.  This frame's space, from LookState::counter: [0, F) are
    // its items S_0..entries-1 (F = entries - S_0), then the paths the
    // previous call suspended, level by level: queue l holds lk_res[l + 1] -
    // lk_res[l] of them from lk_res[l] on (they are part way through, so
    // they go last).
    //  - A wave whose work counter has none of them left (in small launches:
    //    no counter has) takes items of the
    //    later frames from LookState::spec_counter (level l: path S_l + j
    //    for the j-th item of its share), but only while it holds no path of
    //    this frame: waves that do take nothing more, stay sparse and issue
    //    first (s_setprio).
    //  - Every wave starts registered in LookState::live and leaves it once,
    //    at that same point (none left for it, no level-0 path held); every
    //    counter has waves that stay until it has run out, so all are handed
    //    out when the last leaves, which writes this call's tag into each
    //    block's stop flag.
    //  - After the stop no more items are taken, and paths of later frames
    //    leave for the queue of their level: at a bounce, or in the middle
    //    of a ray, which the next call then traces again from its origin.
    constexpr bool kLookMode = (kMode == kModeDiffuse || kMode == kModeDiffuse2) && kLook;
    constexpr int kLookItem = look_item(kMode == kModeDiffuse2 ? PRT_RENDERER_DIFFUSE2 : PRT_RENDERER_DIFFUSE);
    LookState* const look = kLookMode ? pl.look : nullptr;
    uint32_t lk_F = 0, lk_fresh_end = 0, lk_target = 0;
    uint32_t lk_S[kLookLevels + 1] = {};         // S_l
    uint32_t lk_res[kLookLevels + 1] = {};       // this frame's space: queue l from lk_res[l]
    uint32_t lk_spec[kLookLevels + 2] = {};      // later frames' space: level l from lk_spec[l]
    if (kLookMode && look) {
#pragma unroll
        for (int l = 0; l <= kLookLevels; ++l) lk_S[l] = look->started[l];
        lk_F = count - lk_S[0];
        lk_target = look->target;
        lk_res[0] = lk_F;
#pragma unroll
        for (int l = 0; l < kLookLevels; ++l) lk_res[l + 1] = lk_res[l] + look->resume_in[l];
        lk_fresh_end = lk_res[kLookLevels];
#pragma unroll
        for (int l = 1; l <= kLookLevels + 1; ++l) lk_spec[l] = look->spec_begin[l];
    }
    bool stop = kLookMode && look && lk_target == 0;  // wave-uniform: this frame is finished
    bool fresh_out = false;  // wave-uniform: this wave takes no more of this frame's space
    bool live = kLookMode && look;  // wave-uniform: registered in LookState::live
    int level = 0;           // the lane's path belongs to frame pass + level
    bool suspend = false;    // the lane's later-frame path waits in (o, d) for the queue
    uint32_t poll_steps = 0;
    uint32_t* const stop_flag = kLookMode && look ? pl.look_flags + (size_t)blockIdx.x * kLookFlagStride : nullptr;
    // leaves LookState::live; the last wave to leave raises every stop flag
    auto look_leave = [&]() {
        uint32_t old = 0;
        if (lane == 0) old = atomicSub(&look->live, 1u);
        old = (uint32_t)__builtin_amdgcn_readfirstlane((int)old);
        if (old == 1u)
            for (uint32_t b = (uint32_t)lane; b < gridDim.x; b += 64u)
                __hip_atomic_store(pl.look_flags + (size_t)b * kLookFlagStride, pl.look_gen, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        live = false;
    };
    unsigned long long n_ahead[kLookLevels] = {};  // rays of frame pass + l + 1
    if (stop) exhausted = true;

    auto start_ray = [&](f3 org, f3 dir, float near, float far) {
        o = org;
        d = dir;
        tmin = near;
        tbest = far;
        const float dx = fabsf(d.x) < 1e-20f ? copysignf(1e-20f, d.x) : d.x;
        const float dy = fabsf(d.y) < 1e-20f ? copysignf(1e-20f, d.y) : d.y;
        const float dz = fabsf(d.z) < 1e-20f ? copysignf(1e-20f, d.z) : d.z;
        inv_x = __builtin_amdgcn_rcpf(dx);
        inv_y = __builtin_amdgcn_rcpf(dy);
        inv_z = __builtin_amdgcn_rcpf(dz);
        neg_x = dx < 0.0f;
        neg_y = dy < 0.0f;
        neg_z = dz < 0.0f;
        wr = watertight_setup(d);
        best_prim = -1;
        sp = bottom = 0;
        node = 0;
        node_t = near;
        pend = 0;
        pend2 = 0;
        tracing = true;
    };

    // Shading frame of the current ray's closest hit (triangle p0, p1, p2):
    // the full ShadingContext when the scene has per-vertex attributes (the
    // hit coordinates are recomputed from the winner's edge functions), else
    // the frame of the ray-facing geometric normal.
    auto hit_frame = [&](f3 p0, f3 p1, f3 p2) -> Frame {
        const int32_t* aidx = sc.idx;
        const float* an = pl.fast ? nullptr : sc.normals;
        const float* at = pl.fast ? nullptr : sc.texcoords;
        if (kMode == kModeBatch) {
            const SceneDevice& js = bl.scenes[scene_id];
            aidx = js.idx;
            an = js.normals;
            at = js.texcoords;
        }
        if (an != nullptr || at != nullptr) {
            float hu, hv;
            tri_barycentrics(wr, o, p0, p1, p2, hu, hv);
            return attribute_frame(aidx, an, at, best_prim, p0, p1, p2, d, hu, hv);
        }
        return make_frame(face_normal(p0, p1, p2, d));
    };

    // Starts work item `my` (a ray, or a path's camera ray) in this lane.
    // spec_claim: an item of a later frame (lookahead).
    auto start_item = [&](uint32_t my, bool spec_claim) __attribute__((always_inline)) {
        if (kRayQuery) {
            ray_idx = my;
            const float4 r0 = tl.rays[2 * (size_t)my];
            const float4 r1 = tl.rays[2 * (size_t)my + 1];
            if (r1.w < 0.0f) {
                if (kMode == kModeOccluded) tl.any_t[my] = -1.0f;
                else tl.hits[my] = make_float4(-1.0f, __int_as_float(-1), 0.0f, 0.0f);
            } else {
                start_ray(mk3(r0.x, r0.y, r0.z), mk3(r1.x, r1.y, r1.z), r0.w, r1.w);
                active = true;
            }
        } else if (kMode == kModeBatch) {
            // work item -> job (binary search over the job prefix),
            // then sample and path inside the job
            int lo = 0, hi = bl.n_jobs;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (bl.work_begin[mid] <= my) lo = mid; else hi = mid;
            }
            const BatchJobDevice& job = bl.jobs[lo];
            const uint32_t local = my - bl.work_begin[lo];
            const uint32_t sample = local / job.entries;
            const uint32_t path = local - sample * job.entries;
            const uint32_t tile = path >> 6, tl_lane = path & 63u;
            const int mx = (tl_lane & 1) | ((tl_lane >> 1) & 2) | ((tl_lane >> 2) & 4);
            const int my_ = ((tl_lane >> 1) & 1) | ((tl_lane >> 2) & 2) | ((tl_lane >> 3) & 4);
            const int x = (int)(tile % (uint32_t)job.tiles_x) * 8 + mx;
            const int y = (int)(tile / (uint32_t)job.tiles_x) * 8 + my_;
            if (x < job.width && y < job.height) {
                pixel = x + y * job.width;
                const SceneDevice jsc = bl.scenes[job.scene];
                scene_id = job.scene;
                nodes = global_view(jsc.nodes);
                tris = global_view(jsc.tris);
                prim_ids = global_view(jsc.prim_ids);
                sample_out = bl.samples + job.sample_base +
                             (size_t)sample * (size_t)(job.width * job.height) + pixel;
                max_depth = job.max_depth;
                albedo = job.albedo;
                rng = sampler_seed(job.pass0 + (int)sample, pixel);
                const float u1 = sampler_next(rng);
                const float u2 = sampler_next(rng);
                const float l1 = sampler_next(rng);  // lens 2D
                const float l2 = sampler_next(rng);
                f3 org, dir;
                camera_ray(job.cam, ((float)x + u1) * job.inv_w, ((float)y + u2) * job.inv_h, l1, l2,
                           org, dir);
                start_ray(org, dir, 0.0f, 3.402823466e38f);
                depth = 0;
                lw = 1.0f;
                active = true;
            }
        } else if (kLookMode && look && !spec_claim && my >= lk_F) {
            // a path that the previous call stopped at a bounce
            // (or in the middle of a ray): its next ray
            const uint4* q = pl.q_in[0] + kLookItem * (size_t)(my - lk_res[0]);
            level = 0;
#pragma unroll
            for (int l = 1; l < kLookLevels; ++l)
                if (my >= lk_res[l]) {
                    q = pl.q_in[l] + kLookItem * (size_t)(my - lk_res[l]);
                    level = l;
                }
            const uint4 e0 = q[0], e1 = q[1], e2 = q[2];
            pixel = (int32_t)e0.w;
            rng = e1.w;
            depth = (int)e2.x;
            lw = as_f(e2.y);
            if (kMode == kModeDiffuse2) {
                const uint4 e3 = q[3], e4 = q[4];
                lsum = as_f(e2.z);
                shadow = e2.w != 0;
                eo = mk3(as_f(e3.x), as_f(e3.y), as_f(e3.z));
                ed = mk3(as_f(e3.w), as_f(e4.x), as_f(e4.y));
            }
            start_ray(mk3(as_f(e0.x), as_f(e0.y), as_f(e0.z)), mk3(as_f(e1.x), as_f(e1.y), as_f(e1.z)),
                      0.0f, 3.402823466e38f);
            active = true;
        } else {
            // camera ray of path `my`: 8x8 tiles, Morton order inside
            // a tile (image/morton.cpp:22), as the wavefront raygen
            uint32_t path = my;
            path_pass = pl.pass;
            if (kLookMode && look) {
                level = 0;
                path = lk_S[0] + my;
                if (spec_claim) {
#pragma unroll
                    for (int l = 1; l <= kLookLevels; ++l)
                        if (my >= lk_spec[l]) {
                            level = l;
                            path = lk_S[l] + (my - lk_spec[l]);
                        }
                }
                path_pass = pl.pass + level;
            }
            if (kMode == kModeAdjoint || (kMode == kModeRgb && pl.rgb_planes)) {
                const uint32_t sample = my / pl.entries;
                path = my - sample * pl.entries;
                path_pass = pl.pass + (int)sample;
            }
            const uint32_t tile = path >> 6, tl_lane = path & 63u;
            const int mx = (tl_lane & 1) | ((tl_lane >> 1) & 2) | ((tl_lane >> 2) & 4);
            const int my_ = ((tl_lane >> 1) & 1) | ((tl_lane >> 2) & 2) | ((tl_lane >> 3) & 4);
            const int x = (int)(tile % (uint32_t)pl.tiles_x) * 8 + mx;
            const int y = (int)(tile / (uint32_t)pl.tiles_x) * 8 + my_;
            if (x < pl.width && y < pl.height) {
                pixel = x + y * pl.width;
                rng = sampler_seed(path_pass, pixel);
                const float u1 = sampler_next(rng);
                const float u2 = sampler_next(rng);
                const float l1 = sampler_next(rng);  // lens 2D
                const float l2 = sampler_next(rng);
                f3 org, dir;
                camera_ray(pl.cam, ((float)x + u1) * pl.inv_w, ((float)y + u2) * pl.inv_h, l1, l2, org,
                           dir);
                start_ray(org, dir, 0.0f, 3.402823466e38f);
                depth = 0;
                lw = lg = lb = 1.0f;
                lsum = 0.0f;
                shadow = false;
                active = true;
                if (kMode == kModeAdjoint) {
                    replay = false;
                    // one per lane; a group's paths use their first lane's
                    hit_slot = blockIdx.x * (uint32_t)kBlock + (uint32_t)(pl.coop == kCoopSpread ? tid & ~7 : tid);
                    pr = pg = pb = 1.0f;
                    zeros = 0;
                    const float* g = pl.dldi + 3 * (size_t)pixel;
                    gw_r = g[0] * pl.inv_spp;
                    gw_g = g[1] * pl.inv_spp;
                    gw_b = g[2] * pl.inv_spp;
                    if (gw_r == 0.0f && gw_g == 0.0f && gw_b == 0.0f) active = tracing = false;
                }
            }
        }
    };

    // Adjoint: adds a hit's gradient, dL_c/da_c(t) = product of the path's other
    // albedos.  The lanes here hand their triangles and three sums to each other
    // through LDS, so that three lanes next to each other add the channels of
    // one triangle: one request of 12 bytes to the memory instead of three.
    // Requests bound these adds.  Adjoint of 512x512 x 8 spp, depth 6, ms with
    // every lane adding its own three / this / no adds at all: 33.5 k triangles
    // 2.46 / 2.15 / 2.06, 2.4 k triangles 1.98 / 1.43 / 1.20.
    auto add_gradient = [&](uint32_t tri, float ar, float ag, float ab, bool add) __attribute__((always_inline)) {
        const uint32_t zr = zeros & 0xffu, zg = (zeros >> 8) & 0xffu, zb = zeros >> 16;
        const float dr = zr == 0 ? pr / ar : (zr == 1 && ar == 0.0f ? pr : 0.0f);
        const float dg = zg == 0 ? pg / ag : (zg == 1 && ag == 0.0f ? pg : 0.0f);
        const float db = zb == 0 ? pb / ab : (zb == 1 && ab == 0.0f ? pb : 0.0f);
        if (!add) return;
        uint4* const sums = grad_sums + (tid & ~63);
        const uint64_t here = __ballot(1);
        const uint32_t n = (uint32_t)__popcll(here), rank = (uint32_t)__popcll(here & lane_lt);
        sums[rank] = make_uint4(tri, __float_as_uint(gw_r * dr), __float_as_uint(gw_g * dg), __float_as_uint(gw_b * db));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (uint32_t j = 0; j < 3; ++j) {
            const uint32_t slot = j * n + rank;  // of 3 n <= 192
            const uint32_t from = (slot * 171u) >> 9, c = slot - 3u * from;  // slot / 3, exact below 256
            const uint32_t* e = reinterpret_cast<const uint32_t*>(sums + from);
            const float v = __uint_as_float(e[1 + c]);
            if (v != 0.0f) atomicAdd(pl.grad + 3 * (size_t)e[0] + c, v);
        }
        __builtin_amdgcn_wave_barrier();
    };

    // Counts a ray for the frame that its path belongs to.
    auto count_ray = [&](bool lead) __attribute__((always_inline)) {
        if (kLookMode && level > 0) {
#pragma unroll
            for (int l = 1; l <= kLookLevels; ++l)
                if (level == l && lead) ++n_ahead[l - 1];
        } else {
            n_rays += lead ? 1u : 0u;
        }
    };

    // A later frame's sample, for the call whose tag it carries.
    auto side_sample = [&](float c, bool lead) __attribute__((always_inline)) {
        const uint32_t tag = pl.look_gen + (uint32_t)level;
        if (lead)
            pl.side[(size_t)(tag % (uint32_t)kLookLevels) * (size_t)(pl.width * pl.height) + pixel] =
                make_uint2(__float_as_uint(c), tag);
    };

    // Shades the lanes whose ray has finished (active, not tracing).  lead: the
    // lane counts and writes for its path; grouped: its path is held by a group
    // of 8 lanes.
    auto shade = [&](bool lead, bool grouped) __attribute__((always_inline)) {
        if (kCount && __ballot(active && !tracing) != 0 && lane == 0) ++n_wshade;
        if (active && !tracing) do {
            if (kMode == kModeOccluded) {
                if (lead) tl.any_t[ray_idx] = best_prim >= 0 ? tbest : -1.0f;
                active = false;
                break;
            }
            if (kMode == kModeDiffuse2 && shadow) {
                // shadow ray done: light from the sky unless blocked (MIS weight 1/2)
                if constexpr (kCount) { if (lead) atomicAdd(&depth_hist[min(depth, kMaxQueueDepth - 1)], 1u); }
                count_ray(lead);
                if (best_prim < 0) lsum += lw * 0.5f;
                shadow = false;
                start_ray(eo, ed, 0.0f, 3.402823466e38f);
                break;
            }
            float t = -1.0f;
            f3 p0{}, p1{}, p2{};
            if (best_prim >= 0) {
                const PRT_GLOBAL float* tp = tris + 9 * (size_t)best_rec;
                p0 = mk3(tp[0], tp[1], tp[2]);
                p1 = mk3(tp[3], tp[4], tp[5]);
                p2 = mk3(tp[6], tp[7], tp[8]);
                t = tbest;  // plane distance of the winner (tri_test)
            }
            if (kMode == kModeTrace) {
                float bu = 0.0f, bv = 0.0f;
                if (best_prim >= 0) tri_barycentrics(wr, o, p0, p1, p2, bu, bv);
                if (lead)
                    tl.hits[ray_idx] = best_prim >= 0
                                           ? make_float4(t, __int_as_float(best_prim), bu, bv)
                                           : make_float4(-1.0f, __int_as_float(-1), 0.0f, 0.0f);
                active = false;
                break;
            }
            if constexpr (kCount && kMode != kModeBatch) { if (lead) atomicAdd(&depth_hist[min(depth, kMaxQueueDepth - 1)], 1u); }
            count_ray(lead);
            float4* acc = kMode == kModeBatch ? nullptr : pl.accum + pixel;
            if (kMode == kModeDiffuse2) {
                // extension ray done (render/diffuse2_integrator_single.h:52-85)
                bool done = false;
                if (best_prim < 0) {
                    lsum += lw * (depth > 0 ? 0.5f : 1.0f);
                    done = true;
                } else if (depth == max_depth) {
                    done = true;
                }
                if (done) {
                    active = false;
                    if (kLookMode && level > 0) {
                        side_sample(lsum, lead);
                        break;
                    }
                    const float4 a = pl.fast ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : *acc;
                    if (lead) *acc = make_float4(a.x + lsum, a.y + lsum, a.z + lsum, a.w + 1.0f);
                    break;
                }
                lw *= albedo;
                const Frame fr = hit_frame(p0, p1, p2);
                const float s1 = sampler_next(rng);
                const float s2 = sampler_next(rng);
                const float s3 = sampler_next(rng);
                const float s4 = sampler_next(rng);
                f3 so, sd;
                diffuse_bounce(o, d, t, fr, s1, s2, so, sd);
                diffuse_bounce(o, d, t, fr, s3, s4, eo, ed);
                ++depth;
                shadow = true;
                start_ray(so, sd, 0.0f, 3.402823466e38f);
                break;
            }
            if (kMode == kModePrimary) {
                f3 c = mk3(0.05f, 0.05f, 0.05f);
                if (best_prim >= 0) {
                    const f3 n = hit_frame(p0, p1, p2).n;
                    c = mk3((n.x + 1.0f) * 0.5f, (n.y + 1.0f) * 0.5f, (n.z + 1.0f) * 0.5f);
                }
                const float4 a = pl.fast ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : *acc;
                if (lead) *acc = make_float4(a.x + c.x, a.y + c.y, a.z + c.z, a.w + 1.0f);
                active = false;
                break;
            }
            if (best_prim < 0 || depth == max_depth) {
                if (kMode == kModeAdjoint) {
                    if (best_prim < 0 && pl.path_hits) {
                        // the path escaped: hand each of its recorded hits its
                        // share of the gradient (a group's lanes take turns).
                        // 4 B per hit written and read instead of a ray traced
                        // again: an albedo step of 33.5 k triangles, 512x512 x
                        // 8 spp, depth 6 (forward and adjoint) 5.44 -> 4.95 ms
                        for (int k = grouped ? gj : 0; k < depth; k += grouped ? 8 : 1) {
                            const uint32_t tri = pl.path_hits[(size_t)k * pl.path_hits_stride + hit_slot];
                            const float* a = pl.albedo_rgb + 3 * (size_t)tri;
                            add_gradient(tri, a[0], a[1], a[2], true);
                        }
                        n_rays += lead ? (uint32_t)depth + 1u : 0u;  // the replayed rays
                    } else if (!replay && best_prim < 0) {
                        // the path escaped: replay it from its seed to
                        // hand each hit its share of the gradient
                        replay = true;
                        rng = sampler_seed(path_pass, pixel);
                        const float u1 = sampler_next(rng);
                        const float u2 = sampler_next(rng);
                        const float l1 = sampler_next(rng);
                        const float l2 = sampler_next(rng);
                        f3 org, dir;
                        const int y = pixel / pl.width, x = pixel - y * pl.width;
                        camera_ray(pl.cam, ((float)x + u1) * pl.inv_w, ((float)y + u2) * pl.inv_h, l1, l2, org, dir);
                        depth = 0;
                        start_ray(org, dir, 0.0f, 3.402823466e38f);
                        continue;
                    }
                    active = false;
                    break;
                }
                const float c = best_prim < 0 ? lw : 0.0f;
                if (kMode == kModeBatch) {
                    if (lead) *sample_out = c;
                } else if (kMode == kModeRgb) {
                    const float cg = best_prim < 0 ? lg : 0.0f, cb = best_prim < 0 ? lb : 0.0f;
                    if (pl.rgb_planes) {
                        // one plane per sample; they are added in pass order afterwards
                        if (lead)
                            pl.rgb_planes[(size_t)(path_pass - pl.pass) * (size_t)(pl.width * pl.height) + pixel] =
                                make_float4(c, cg, cb, 0.0f);
                    } else {
                        const float4 a = *acc;
                        if (lead) *acc = make_float4(a.x + c, a.y + cg, a.z + cb, a.w + 1.0f);
                    }
                } else if (kLookMode && level > 0) {
                    side_sample(c, lead);
                } else {
                    const float4 a = pl.fast ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : *acc;
                    if (lead) *acc = make_float4(a.x + c, a.y + c, a.z + c, a.w + 1.0f);
                }
                active = false;
                break;
            }
            // diffuse bounce: the next ray of this path
            if (kMode == kModeRgb || kMode == kModeAdjoint) {
                const float* a = pl.albedo_rgb + 3 * (size_t)best_prim;
                const float ar = a[0], ag = a[1], ab = a[2];
                if (kMode == kModeAdjoint) {
                    if (!replay) {
                        // primal: products of the nonzero albedos, zero counts
                        if (ar != 0.0f) pr *= ar; else zeros += 1u;
                        if (ag != 0.0f) pg *= ag; else zeros += 1u << 8;
                        if (ab != 0.0f) pb *= ab; else zeros += 1u << 16;
                        if (lead && pl.path_hits)
                            pl.path_hits[(size_t)depth * pl.path_hits_stride + hit_slot] = (uint32_t)best_prim;
                    } else {
                        add_gradient((uint32_t)best_prim, ar, ag, ab, lead);
                    }
                } else {
                    lw *= ar;
                    lg *= ag;
                    lb *= ab;
                }
            } else {
                lw *= albedo;
            }
            const Frame fr = hit_frame(p0, p1, p2);
            const float s1 = sampler_next(rng);
            const float s2 = sampler_next(rng);
            f3 no, nd;
            diffuse_bounce(o, d, t, fr, s1, s2, no, nd);
            ++depth;
            if (kLookMode && level > 0 && stop) {
                o = no;
                d = nd;
                suspend = true;
                active = false;
                break;
            }
            start_ray(no, nd, 0.0f, 3.402823466e38f);
        } while (0);
    };

    // ---- cooperative traversal.  A wave out of work that holds at most 8
    // paths moves each, in the middle of its ray or between rays, to a group
    // of 8 lanes that hold its state alike.  Per step, lane j of a group tests
    // one of up to 8 pending triangles, then child j of the group's node; the
    // nearest children and the closest hit come from DPP minima inside the
    // group (no trip through the LDS crossbar).  A step then issues about a
    // third of the lane-by-lane instructions and tests up to 8 triangles at
    // once, so the dependent steps of the last paths, which set a launch's
    // end, follow each other faster.  The closest hit is the same (t, primId)
    // minimum in any order, so hits and images do not change.  8 lanes: a
    // group's lanes are the node's children.  Plain frames with it and lane by
    // lane: 1080p spheres 1.199 / 1.285 ms, 720p of 0.4 M triangles 1.146 /
    // 1.283 ms, next-event frames of 717x405 0.937 / 0.986 ms (4 workgroups
    // per CU on all).
    auto to_groups = [&](uint64_t paths) {
        const int npaths = __popcll(paths);
        const int grp = lane >> 3;
        uint64_t mm = paths;
        for (int k = 0; k < grp; ++k) mm &= mm - 1;
        const int src = mm ? __ffsll((unsigned long long)mm) - 1 : 0;
        auto mv_u = [&](uint32_t v) -> uint32_t { return (uint32_t)__shfl((int)v, src, 64); };
        auto mv_i = [&](int& v) { v = __shfl(v, src, 64); };
        auto mv_w = [&](uint32_t& v) { v = mv_u(v); };
        auto mv_f = [&](float& v) { v = __shfl(v, src, 64); };
        auto mv_3 = [&](f3& v) { mv_f(v.x); mv_f(v.y); mv_f(v.z); };
        auto mv_b = [&](bool& v) { v = __shfl(v ? 1 : 0, src, 64) != 0; };
        auto mv_p = [&](auto& v) {
            uint64_t u = (uint64_t)v;
            u = (uint64_t)mv_u((uint32_t)u) | ((uint64_t)mv_u((uint32_t)(u >> 32)) << 32);
            v = (std::remove_reference_t<decltype(v)>)u;
        };
        mv_i(sp);
        // the ray's stack (all in LDS: bottom is 0, so at most kStack entries):
        // read by the group's lanes, then written in the joined order
        const int stid = (tid & ~63) + src;
        uint32_t en[kStack / 8], et[kStack / 8];
#pragma unroll
        for (int r = 0; r < kStack / 8; ++r) {
            const int at = (8 * r + gj) * kBlock + stid;
            en[r] = st_node[at];
            et[r] = __float_as_uint(st_t[at]);
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < kStack / 8; ++r) {
            st_node[group_slot(8 * r + gj)] = en[r];
            st_t[group_slot(8 * r + gj)] = as_f(et[r]);
        }
        mv_b(active);
        mv_b(tracing);
        mv_3(o);
        mv_3(d);
        mv_f(tmin);
        mv_f(tbest);
        mv_f(inv_x);
        mv_f(inv_y);
        mv_f(inv_z);
        neg_x = inv_x < 0.0f;
        neg_y = inv_y < 0.0f;
        neg_z = inv_z < 0.0f;
        mv_i(wr.kx);
        mv_i(wr.ky);
        mv_i(wr.kz);
        mv_f(wr.sx);
        mv_f(wr.sy);
        mv_f(wr.sz);
        mv_i(best_prim);
        mv_w(best_rec);
        mv_i(node);
        mv_f(node_t);
        mv_w(pend);
        mv_w(pend_base);
        mv_w(pend2);
        mv_w(pend2_base);
        if constexpr (kRayQuery) {
            mv_w(ray_idx);
        } else {
            mv_i(pixel);
            mv_w(rng);
            mv_i(depth);
            mv_f(lw);
        }
        if constexpr (kLookMode) mv_i(level);
        if constexpr (kMode == kModeBatch) {
            mv_i(max_depth);
            mv_f(albedo);
            mv_i(scene_id);
            mv_p(nodes);
            mv_p(tris);
            mv_p(prim_ids);
            mv_p(sample_out);
        }
        if constexpr (kMode == kModeRgb || kMode == kModeAdjoint) {
            mv_f(lg);
            mv_f(lb);
            mv_i(path_pass);
        }
        if constexpr (kMode == kModeAdjoint) {
            mv_f(pr);
            mv_f(pg);
            mv_f(pb);
            mv_w(zeros);
            mv_f(gw_r);
            mv_f(gw_g);
            mv_f(gw_b);
            mv_b(replay);
            mv_w(hit_slot);
        }
        if constexpr (kMode == kModeDiffuse2) {
            mv_b(shadow);
            mv_3(eo);
            mv_3(ed);
            mv_f(lsum);
        }
        if (grp >= npaths) active = tracing = false;
    };

    // Traverses the groups' rays until half of the `groups` with a path wait
    // for shading.
    auto coop_traverse = [&](int groups) {
        const int keep = max(0, groups - max(1, groups >> 1));  // no groups: nothing to trace
        for (;;) {
            const int left = __popcll(__ballot(tracing)) >> 3;
            if (left <= keep) break;
            if (kCount) {
                if (tracing) {
                    ++n_lsteps;
                    ++n_dlsteps;
                }
                if (lane == 0) {
                    ++n_wsteps;
                    ++n_dwsteps;
                }
            }
            if (tracing && pend != 0) {
                // up to 8 pending triangles, one per lane
                const int np = __popc(pend);
                uint32_t cp = ~0u, crec = 0;
                float hit_t = __builtin_inff();
                if (gj < np) {
                    const uint32_t rec = pend_base + nth_bit(pend, (uint32_t)gj);
                    const PRT_GLOBAL float* tp = tris + 9 * (size_t)rec;
                    const f3 p0 = mk3(tp[0], tp[1], tp[2]);
                    const f3 p1 = mk3(tp[3], tp[4], tp[5]);
                    const f3 p2 = mk3(tp[6], tp[7], tp[8]);
                    if (kCount) ++n_tris;
                    if (tri_test(wr, o, d, p0, p1, p2, tmin, tbest, hit_t)) {
                        cp = (uint32_t)prim_ids[rec];
                        crec = rec;
                    }
                }
                if (np <= 8) {
                    pend = pend2;
                    pend_base = pend2_base;
                    pend2 = 0;
                } else {
                    pend &= ~0u << nth_bit(pend, 8);
                }
                if (__ballot(cp != ~0u) != 0) {
                    // the smallest (t, primId): floats ordered as unsigned
                    // integers (t is negative only where tnear is; -0 as +0)
                    const uint32_t tb = __float_as_uint(hit_t + 0.0f);
                    const uint32_t ct = cp != ~0u ? tb ^ (tb >> 31 ? 0xffffffffu : 0x80000000u) : ~0u;
                    const uint32_t mt = min8(ct);
                    const uint32_t mp = min8(ct == mt ? cp : ~0u);
                    if (mp != ~0u) {
                        const bool won = ct == mt && cp == mp;
                        const float t = __uint_as_float(or8(won ? __float_as_uint(hit_t) : 0u));
                        const uint32_t mr = or8(won ? crec : 0u);
                        if (kMode == kModeOccluded || (kMode == kModeDiffuse2 && shadow)) {
                            // any hit ends the query
                            tbest = t;
                            best_prim = 0;
                            sp = bottom = 0;
                            pend = pend2 = 0;
                            node = -1;
                        } else if (t < tbest || best_prim < 0 || (int32_t)mp < best_prim) {
                            tbest = t;
                            best_prim = (int32_t)mp;
                            best_rec = mr;
                        }
                    }
                }
            }
            if (tracing && pend == 0) {
                if (node >= 0 && node_t > tbest) node = -1;
                while (node < 0 && sp > 0) {
                    // the 8 youngest entries at once: the topmost that can
                    // still hold a closer hit
                    const int q = sp - 1 - gj;
                    uint32_t nid = 0;
                    float nt = __builtin_inff();
                    if (q >= bottom) {
                        const int slot = group_slot(q);
                        nid = st_node[slot];
                        nt = st_t[slot];
                    } else if (q >= 0) {
                        const uint2 e = g_spill[q];
                        nid = e.x;
                        nt = as_f(e.y);
                    }
                    const uint32_t ok = (uint32_t)(__ballot(q >= 0 && nt <= tbest) >> gbase) & 0xffu;
                    if (ok == 0) {
                        sp = max(sp - 8, 0);
                    } else {
                        const int f = __builtin_ctz(ok);
                        node = __shfl((int)nid, gbase + f, 64);
                        node_t = __shfl(nt, gbase + f, 64);
                        sp -= f + 1;
                    }
                    bottom = min(bottom, sp);
                }
                if (node < 0) tracing = false;
            }
            if (tracing && pend == 0) {
                // ---- child gj of the group's node
                const PRT_GLOBAL uint8_t* nb = reinterpret_cast<const PRT_GLOBAL uint8_t*>(nodes + node);
                const PRT_GLOBAL uint4* np = reinterpret_cast<const PRT_GLOBAL uint4*>(nb);
                const uint4 w0 = np[0];
                const uint2 base = reinterpret_cast<const PRT_GLOBAL uint2*>(nb)[2];
                const uint32_t mb = nb[24 + gj];
                const PRT_GLOBAL uint8_t* qb = nb + 32 + gj;
                const float qnx = (float)qb[neg_x ? 24 : 0], qfx = (float)qb[neg_x ? 0 : 24];
                const float qny = (float)qb[neg_y ? 32 : 8], qfy = (float)qb[neg_y ? 8 : 32];
                const float qnz = (float)qb[neg_z ? 40 : 16], qfz = (float)qb[neg_z ? 16 : 40];
                if (kCount && gj == 0) ++n_nodes;
                const float ax = __builtin_amdgcn_ldexpf(inv_x, (int)(int8_t)(w0.w & 0xffu));
                const float ay = __builtin_amdgcn_ldexpf(inv_y, (int)(int8_t)((w0.w >> 8) & 0xffu));
                const float az = __builtin_amdgcn_ldexpf(inv_z, (int)(int8_t)((w0.w >> 16) & 0xffu));
                const uint32_t imask = w0.w >> 24;
                const float bx = (as_f(w0.x) - o.x) * inv_x;
                const float by = (as_f(w0.y) - o.y) * inv_y;
                const float bz = (as_f(w0.z) - o.z) * inv_z;
                // slack 2^-21 (255 |a| + |b|): the roundings of b, b -/+ slack
                // and the fma, the reciprocal's ulp and the hit distance's
                // rounding sum to at most 2^-21 (128 |a| + |b|)
                const float slx = 0x1p-21f * __builtin_fmaf(255.0f, fabsf(ax), fabsf(bx));
                const float sly = 0x1p-21f * __builtin_fmaf(255.0f, fabsf(ay), fabsf(by));
                const float slz = 0x1p-21f * __builtin_fmaf(255.0f, fabsf(az), fabsf(bz));
                const float tn = fmaxf(fmaxf(fmaxf(__builtin_fmaf(qnx, ax, bx - slx), __builtin_fmaf(qny, ay, by - sly)),
                                             __builtin_fmaf(qnz, az, bz - slz)), tmin);
                const float tf = fminf(fminf(fminf(__builtin_fmaf(qfx, ax, bx + slx), __builtin_fmaf(qfy, ay, by + sly)),
                                             __builtin_fmaf(qfz, az, bz + slz)), tbest);
                const bool hit = tn <= tf;
                const bool inner = ((imask >> gj) & 1u) != 0;
                // leaf slots: one pending mask over the node's records
                pend = or8(hit && !inner ? ((1u << (mb >> 5)) - 1u) << (mb & 31u) : 0u);
                pend_base = base.y;
                // nearest internal child next, the others pushed by slot with
                // the second nearest on top (keys as lane by lane)
                const uint32_t key = hit && inner ? (__float_as_uint(tn) & 0x7ffffff8u) | (uint32_t)gj : ~0u;
                const uint32_t m1 = min8(key);
                const uint32_t m2 = min8(key == m1 ? ~0u : key);
                node = -1;
                if (m1 != ~0u) {
                    node = (int32_t)(base.x + __popc(imask & ((1u << (m1 & 7u)) - 1u)));
                    node_t = __uint_as_float(m1 & ~7u);
                    const bool push = key != ~0u && key != m1;
                    const uint32_t pm = (uint32_t)(__ballot(push && key != m2) >> gbase) & 0xffu;
                    if (m2 != ~0u) {
                        const int npush = __popc(pm) + 1;
                        bool room = true;
                        while (sp + npush - bottom > kGStack) {
                            if (bottom >= spill_cap) { if (gj == 0) raise_overflow(); room = false; break; }
                            const int bs = group_slot(bottom);
                            g_spill[bottom] = make_uint2(st_node[bs], __float_as_uint(st_t[bs]));
                            ++bottom;
                            if (kCount && gj == 0) ++n_spill;
                        }
                        if (room) {
                            if (push) {
                                const int at = sp + (key == m2 ? npush - 1 : __popc(pm & ((1u << gj) - 1u)));
                                const int slot = group_slot(at);
                                st_node[slot] = base.x + __popc(imask & ((1u << gj) - 1u));
                                st_t[slot] = tn;
                            }
                            sp += npush;
                        }
                    }
                }
            }
        }
    };

    // ---- work items.  They are dealt in runs of 64 (spread: 8) to the
    // counters (work_deal.h), and each wave starts with the run of its own number
    // without asking.  It goes on with the counter of that run and, in launches
    // of few waves, when that has run out with the next that has not
    // (kOwnCounterWaves).
    // Measured: atomics on one line take 11.5 ns each, whoever asks, so one
    // counter spends 47 us on the first items of 4096 waves and 0.7 ms on a
    // frame of 2.07 M paths, taken 34 at a time; 16 lines take 0.9 ns each.
    // 500 k any-hit rays 247 -> 217 us, lookahead frames of 2.07 M paths 1170
    // -> 1110 us, batches of eight scenes 9.8 -> 8.3 ms.  Runs kept by the wave
    // that takes them (64 to 128 items) cost as few atomics but left some waves
    // with the expensive tiles: plain frames 24 to 40 % slower.
    uint32_t* const work = kRayQuery ? tl.work : (kMode == kModeBatch ? bl.work : pl.work);
    // a small launch is traced in groups from its start (wave-uniform)
    const bool spread = kCoop && pl.coop == kCoopSpread;
    const uint32_t run_lg = spread ? 3u : 6u;
    constexpr uint32_t ctr_last = kWorkCounterLast;
    const uint32_t items = kLookMode && look ? lk_fresh_end : count;
    const uint32_t n_waves = gridDim.x * (uint32_t)(kBlock / 64);
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t my_run = spread ? blockIdx.x + gridDim.x * wave : blockIdx.x * (uint32_t)(kBlock / 64) + wave;
    uint32_t ctr = deal_counter(my_run);
    bool first_run = true, work_out = false;  // wave-uniform; work_out: all items are handed out
    // positions of counter c: the waves' first runs end at dealt(c, n_waves),
    // its items at dealt(c, runs of all items)
    auto dealt = [&](uint32_t c, uint32_t runs) -> uint32_t { return dealt_runs(c, runs) << run_lg; };
    const uint32_t n_runs = (items + (1u << run_lg) - 1u) >> run_lg;
    // Hands n items out to the lanes or groups that take part, numbered by
    // rank; false: none for this one.
    auto claim = [&](uint32_t n, uint32_t rank, uint32_t& my) -> bool {
        uint32_t base = (my_run >> kWorkCountersLg) << run_lg;
        const uint32_t end = dealt(ctr, n_runs);
        if (!first_run) {
            if (lane == 0) base = atomicAdd(work + ctr * kWorkCounterStride, n);
            base = dealt(ctr, n_waves) + (uint32_t)__builtin_amdgcn_readfirstlane((int)base);  // wave-uniform
        }
        const uint32_t at = base + rank;
        my = (deal_run(ctr, at >> run_lg) << run_lg) | (at & ((1u << run_lg) - 1u));
        const bool ok = at < end && my < items;
        const bool ended = first_run ? dealt(ctr, n_waves) >= end : base + n >= end;
        if (n_waves >= n_runs || (ended && n_waves >= kOwnCounterWaves)) {
            work_out = true;
        } else if (ended) {
            uint32_t c = (uint32_t)lane & ctr_last;
            const uint32_t used = dealt(c, n_waves) + __hip_atomic_load(work + c * kWorkCounterStride, __ATOMIC_RELAXED,
                                                                        __HIP_MEMORY_SCOPE_AGENT);
            const uint64_t open = __ballot((uint32_t)lane <= ctr_last && used < dealt(c, n_runs));
            work_out = open == 0;
            const uint64_t from = open & (~0ull << ctr);
            if (!work_out) ctr = (uint32_t)__builtin_ctzll(from ? from : open);
        }
        first_run = false;
        return ok;
    };
    while (!spread) {
        // lookahead: a wave that holds paths of this frame takes no items of
        // later frames once this frame's are handed out, and issues ahead of
        // the waves that run later frames' paths, so the frame's last paths
        // keep the pace they would have alone
        bool hold = false;
        if (kLookMode && look) {
            hold = fresh_out && __ballot(active && level == 0) != 0;
            if (live && fresh_out && !hold) look_leave();
            if (!live && !stop) {
                const uint32_t f = __hip_atomic_load(stop_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                stop = (uint32_t)__builtin_amdgcn_readfirstlane(f) == pl.look_gen;
                if (stop) exhausted = true;
            }
            // after the stop only later frames' paths are left: those in the
            // middle of a ray leave now and trace that ray again next call
            // (its origin, direction and path state are what a bounce leaves)
            if (stop && tracing) {
                suspend = true;
                tracing = false;
                active = false;
            }
            if (hold) __builtin_amdgcn_s_setprio(3);
            else __builtin_amdgcn_s_setprio(0);
        }
        // ---- shade the lanes whose ray has finished: the traversal loop hands
        // them over in groups, so this code runs for many lanes at once
        // instead of stalling every traversal step of the wave for one lane
        shade(true, false);
        if (kMode == kModeDiffuse2 && kLookMode && stop && tracing) {
            suspend = true;  // at a bounce, or between its shadow ray and its next
            tracing = false;
            active = false;
        }

        // ---- refill idle lanes (wave-uniform branch)
        const uint64_t idle = __ballot(!active);
        const int n_idle = __popcll(idle);
        if (!exhausted && !hold && n_idle >= refill) {
            const uint32_t rank = (uint32_t)__popcll(idle & lane_lt);
            const bool spec_claim = kLookMode && look && fresh_out;  // items of later frames
            uint32_t my = 0;
            bool ok, out;
            if (spec_claim) {
                uint32_t base = 0;
                if (lane == 0) base = atomicAdd(&look->spec_counter, (uint32_t)n_idle);
                base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
                my = base + rank;
                ok = my < lk_spec[kLookLevels + 1];
                out = (uint64_t)base + (uint64_t)n_idle >= lk_spec[kLookLevels + 1];
            } else {
                ok = claim((uint32_t)n_idle, rank, my);
                out = work_out;
            }
            if (!active && ok) start_item(my, spec_claim);
            if (out) {
                if (kLookMode && look && !spec_claim) {
                    fresh_out = true;
                } else {
                    exhausted = true;
                    if (kCount) t_exhausted = wall_clock64();
                }
            }
        }

        const uint64_t busy = __ballot(active);
        if (busy == 0) {
            if (exhausted) break;
            continue;
        }
        if (kCoop && coop_on && exhausted && __popcll(busy) <= 8 && __ballot(active && bottom != 0) == 0) {
            coop_paths = busy;
            break;
        }

        // ---- traverse until enough lanes wait for shading or for new work:
        // refill lanes once no more than 64 - refill trace; after the work
        // counter ran out, shade once half of the remaining lanes wait
        const int n_act = __popcll(busy);
        const int keep = !(exhausted || hold) ? 64 - refill
                                    : n_act - max(1, min(refill, n_act >> 1));
        while (tracing) {
            if (kCount) {
                const bool lead = lane == __ffsll((unsigned long long)__ballot(1)) - 1;
                ++n_lsteps;
                if (lead) ++n_wsteps;
                if (exhausted) {
                    ++n_dlsteps;
                    if (lead) ++n_dwsteps;
                }
            }
            // A step tests one pending triangle and visits one node: a lane
            // keeps descending while its leaf triangles are tested, with room
            // for one more leaf group.  The test comes first, so the node's
            // culling sees its result.
            if (pend != 0) {
                // ---- one triangle of the pending group per step, so lanes
                // with many candidate triangles do not hold up the wave
                const uint32_t rec = pend_base + (uint32_t)__builtin_ctz(pend);
                pend &= pend - 1;
                const PRT_GLOBAL float* tp = tris + 9 * (size_t)rec;
                const f3 p0 = mk3(tp[0], tp[1], tp[2]);
                const f3 p1 = mk3(tp[3], tp[4], tp[5]);
                const f3 p2 = mk3(tp[6], tp[7], tp[8]);
                if (kCount) ++n_tris;
                float ct;
                if (tri_test(wr, o, d, p0, p1, p2, tmin, tbest, ct)) {
                    if (kMode == kModeOccluded || (kMode == kModeDiffuse2 && shadow)) {
                        // any hit ends the query: drop the stack and the pending work
                        tbest = ct;
                        best_prim = 0;
                        sp = bottom = 0;
                        pend = pend2 = 0;
                        node = -1;
                    } else {
                        const int32_t prim = prim_ids[rec];
                        if (ct < tbest || best_prim < 0 || prim < best_prim) {
                            tbest = ct;
                            best_prim = prim;
                            best_rec = rec;
                        }
                    }
                }
                if (pend == 0 && pend2 != 0) {
                    pend = pend2;
                    pend_base = pend2_base;
                    pend2 = 0;
                }
            }

            if (pend2 == 0) {
                // ---- node step: the next node that can still hold a closer hit
                if (node >= 0 && node_t > tbest) node = -1;
                if (node < 0) {
                    while (sp > 0) {
                        --sp;
                        uint32_t nid;
                        float nt;
                        if (sp < bottom) {
                            const uint2 e = my_spill[sp];
                            bottom = sp;
                            nid = e.x;
                            nt = as_f(e.y);
                        } else {
                            const uint32_t off = ring_off(sp);
                            nid = ring_node(off);
                            nt = ring_t(off);
                        }
                        if (nt <= tbest) { node = (int32_t)nid; break; }
                    }
                }
            }
            if (pend2 == 0 && node < 0) {
                if (pend == 0) {
                    tracing = false;  // the ray is finished: shade it in the outer loop
                    break;
                }
            } else if (pend2 == 0) {

                // ---- visit one BVH8 node
                const PRT_GLOBAL uint4* np = reinterpret_cast<const PRT_GLOBAL uint4*>(nodes + node);
                const uint4 w0 = np[0], w1 = np[1], w2 = np[2], w3 = np[3], w4 = np[4];
                if (kCount) ++n_nodes;
                const int ex = (int)(int8_t)(w0.w & 0xffu);
                const int ey = (int)(int8_t)((w0.w >> 8) & 0xffu);
                const int ez = (int)(int8_t)((w0.w >> 16) & 0xffu);
                const uint32_t imask = w0.w >> 24;
                const float ax = __builtin_amdgcn_ldexpf(inv_x, ex);
                const float ay = __builtin_amdgcn_ldexpf(inv_y, ey);
                const float az = __builtin_amdgcn_ldexpf(inv_z, ez);
                const float bx = (as_f(w0.x) - o.x) * inv_x;
                const float by = (as_f(w0.y) - o.y) * inv_y;
                const float bz = (as_f(w0.z) - o.z) * inv_z;
                // A plane byte q enters as the half 1024 + q (two per v_perm,
                // read by v_fma_mix_f32 without a conversion), so the distance
                // is fma(1024 + q, a, c -/+ slack), c = b - 1024 a.  The
                // roundings of b, c, c -/+ slack and the fma, the reciprocal's
                // ulp and the hit distance's own rounding sum to at most
                // 2^-21 (384 |a| + |b|); slack 2^-21 (512 |a| + 2 |b|) covers
                // them.
                const float slx = __builtin_fmaf(0x1p-12f, fabsf(ax), 0x1p-20f * fabsf(bx));
                const float sly = __builtin_fmaf(0x1p-12f, fabsf(ay), 0x1p-20f * fabsf(by));
                const float slz = __builtin_fmaf(0x1p-12f, fabsf(az), 0x1p-20f * fabsf(bz));
                const float cx = __builtin_fmaf(-1024.0f, ax, bx), bxn = cx - slx, bxf = cx + slx;
                const float cy = __builtin_fmaf(-1024.0f, ay, by), byn = cy - sly, byf = cy + sly;
                const float cz = __builtin_fmaf(-1024.0f, az, bz), bzn = cz - slz, bzf = cz + slz;
                // near/far planes per axis from the direction signs
                const uint32_t nx0 = neg_x ? w3.z : w2.x, nx1 = neg_x ? w3.w : w2.y;
                const uint32_t fx0 = neg_x ? w2.x : w3.z, fx1 = neg_x ? w2.y : w3.w;
                const uint32_t ny0 = neg_y ? w4.x : w2.z, ny1 = neg_y ? w4.y : w2.w;
                const uint32_t fy0 = neg_y ? w2.z : w4.x, fy1 = neg_y ? w2.w : w4.y;
                const uint32_t nz0 = neg_z ? w4.z : w3.x, nz1 = neg_z ? w4.w : w3.y;
                const uint32_t fz0 = neg_z ? w3.x : w4.z, fz1 = neg_z ? w3.y : w4.w;
                const uint32_t meta0 = w1.z, meta1 = w1.w;
                // the halves 1024 + q of plane word w: bytes 0, 1 (lo) and 2, 3 (hi)
                auto halves = [](uint32_t w) {
                    return make_uint2(__builtin_amdgcn_perm(0x64646464u, w, 0x04010400u),
                                      __builtin_amdgcn_perm(0x64646464u, w, 0x04030402u));
                };
                const uint2 hnx0 = halves(nx0), hnx1 = halves(nx1), hfx0 = halves(fx0), hfx1 = halves(fx1);
                const uint2 hny0 = halves(ny0), hny1 = halves(ny1), hfy0 = halves(fy0), hfy1 = halves(fy1);
                const uint2 hnz0 = halves(nz0), hnz1 = halves(nz1), hfz0 = halves(fz0), hfz1 = halves(fz1);
                // 1024 + byte k of the plane word pair (h0: bytes 0-3, h1: bytes 4-7)
                auto qf = [](uint2 h0, uint2 h1, int k) -> float {
                    const uint2 h = k < 4 ? h0 : h1;
                    const uint32_t w = (k & 2) ? h.y : h.x;
                    const unsigned short bits = (unsigned short)((k & 1) ? (w >> 16) : (w & 0xffffu));
                    return (float)__builtin_bit_cast(_Float16, bits);
                };

                // branchless child tests; empty slots carry inverted boxes, and a
                // leaf slot with meta 0 holds no triangle, so no leaf mask is needed
                uint32_t hits = 0;
                float tk[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const float tnx = __builtin_fmaf(qf(hnx0, hnx1, k), ax, bxn);
                    const float tny = __builtin_fmaf(qf(hny0, hny1, k), ay, byn);
                    const float tnz = __builtin_fmaf(qf(hnz0, hnz1, k), az, bzn);
                    const float tfx = __builtin_fmaf(qf(hfx0, hfx1, k), ax, bxf);
                    const float tfy = __builtin_fmaf(qf(hfy0, hfy1, k), ay, byf);
                    const float tfz = __builtin_fmaf(qf(hfz0, hfz1, k), az, bzf);
                    const float tn = fmaxf(fmaxf(fmaxf(tnx, tny), tnz), tmin);
                    const float tf = fminf(fminf(fminf(tfx, tfy), tfz), tbest);
                    tk[k] = tn;
                    hits |= (tn <= tf ? 1u : 0u) << k;
                }
                const uint32_t hit_int = hits & imask;
                uint32_t hit_leaf = hits & ~imask;

                // ---- leaf slots: one pending mask over the node's triangle
                // records (a node owns at most 8 x kLeafMax <= 32 of them),
                // the first group if it is free, else the second
                uint32_t newp = 0;
                while (hit_leaf) {
                    const int k = __builtin_ctz(hit_leaf);
                    hit_leaf &= hit_leaf - 1;
                    const uint32_t mb = __builtin_amdgcn_perm(meta1, meta0, 0x0c0c0c00u | (uint32_t)k);
                    newp |= ((1u << (mb >> 5)) - 1u) << (mb & 31u);
                }
                if (newp != 0) {
                    if (pend == 0) {
                        pend = newp;
                        pend_base = w1.y;
                    } else {
                        pend2 = newp;
                        pend2_base = w1.y;
                    }
                }

                // ---- internal slots: the nearest is visited next, the others
                // are pushed with the second nearest on top.  Unrolled over the
                // 8 slots with per-slot predicates, so a wave pays one pass
                // whatever the number of hit children per lane.
                node = -1;
                if (hit_int) {
                    // nearest and second-nearest hit internal child by integer
                    // minimum over keys (entry distance bits with the slot in
                    // the low 3 bits; the distances are >= 0, and a -0 loses
                    // its sign bit).  Ties and distances within 8 ulps order by
                    // slot; node_t is the key's distance, at most 7 ulps below
                    // the true one, so culling with it stays conservative.
                    uint32_t key[8];
                    const uint32_t not_int = ~hit_int;
#pragma unroll
                    for (int k = 0; k < 8; ++k) {
                        // all ones unless bit k of hit_int is set (a 1-bit signed field)
                        const uint32_t miss = (uint32_t)__builtin_amdgcn_sbfe((int)not_int, (unsigned)k, 1u);
                        key[k] = (__float_as_uint(tk[k]) & 0x7ffffff8u) | (uint32_t)k | miss;
                    }
                    const uint32_t m1 = min(min(min(key[0], key[1]), min(key[2], key[3])),
                                            min(min(key[4], key[5]), min(key[6], key[7])));
                    // second smallest: no other key equals m1, so key - m1 - 1
                    // (mod 2^32) maps m1 to the largest value and keeps the
                    // order of the keys above it
                    uint32_t e[8];
#pragma unroll
                    for (int k = 0; k < 8; ++k) e[k] = key[k] + ~m1;
                    const uint32_t m2 = min(min(min(e[0], e[1]), min(e[2], e[3])), min(min(e[4], e[5]), min(e[6], e[7]))) +
                                        m1 + 1u;
                    const int k1 = (int)(m1 & 7u);
                    const int k2 = (int)(m2 & 7u);
                    const uint32_t child_base = w1.x;
                    node = (int32_t)(child_base + __popc(imask & ((1u << k1) - 1u)));
                    node_t = __uint_as_float(m1 & ~7u);
                    const uint32_t pushm = hit_int & ~(1u << k1);
                    if (pushm) {
                        const int npush = __popc(pushm);
                        // branch-free: slot k goes to sp + (pushed slots
                        // below k, k2 left out).  A slot that is not pushed
                        // (or is k2) lands on the position of the next
                        // pushed slot above it, written later, or on the
                        // top, written last with k2's entry; so every
                        // write stays inside [sp, sp + npush).  k2 is in
                        // pushm: it is the second hit internal child, on top
                        // with its key's distance (at most 7 ulps below its
                        // entry distance: conservative).
                        const uint32_t pm2 = pushm & ~(1u << k2);
                        auto push_all = [&](auto offset_of) {
#pragma unroll
                            for (int k = 0; k < 8; ++k) {
                                const int pos = __popc(pm2 & ((1u << k) - 1u));
                                const uint32_t off = offset_of(sp + pos);
                                ring_node(off) = child_base + __popc(imask & ((1u << k) - 1u));
                                ring_t(off) = tk[k];
                            }
                            const uint32_t off = offset_of(sp + npush - 1);
                            ring_node(off) = child_base + __popc(imask & ((1u << k2) - 1u));
                            ring_t(off) = __uint_as_float(m2 & ~7u);
                            sp += npush;
                        };
                        // wave-uniform: while no lane's stack reaches past the
                        // first lap of the ring, positions need no wrap
                        if (__all(sp + npush <= kStack)) {
                            push_all([&](int q) -> uint32_t { return ((uint32_t)q << kRingShift) + tid4; });
                        } else {
                            // make room in the LDS ring: move its oldest
                            // entries to the lane's global slice
                            bool ok = true;
                            while (sp + npush - bottom > kStack) {
                                if (bottom >= spill_cap) { raise_overflow(); ok = false; break; }
                                const uint32_t boff = ring_off(bottom);
                                my_spill[bottom] = make_uint2(ring_node(boff), __float_as_uint(ring_t(boff)));
                                ++bottom;
                                if (kCount) ++n_spill;
                            }
                            if (ok) push_all(ring_off);
                        }
                    }
                }
            }

            if ((int)__popcll(__ballot(1)) <= keep) break;
            // lookahead: look at the stop flag every 8 steps (its load is
            // waited for with the next node's)
            if (kLookMode && look && !live && !stop && (++poll_steps & 7u) == 0) {
                const uint32_t f = __hip_atomic_load(stop_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if ((uint32_t)__builtin_amdgcn_readfirstlane(f) == pl.look_gen) {
                    stop = true;
                    exhausted = true;
                    break;
                }
            }
        }
    }

    if (kLookMode && look && live) look_leave();

    if constexpr (kCoop) {
        if (coop_paths != 0) to_groups(coop_paths);
        while ((spread && !work_out) || __ballot(active) != 0) {
            const uint64_t idle = __ballot(!active);
            const uint32_t n = (uint32_t)__popcll(idle) >> 3;
            if (spread && !work_out && n >= 4) {
                uint32_t my;
                const bool ok = claim(n, (uint32_t)__popcll(idle & ((1ull << gbase) - 1ull)) >> 3, my);
                if (!active && ok) start_item(my, false);
            }
            coop_traverse(__popcll(__ballot(active)) >> 3);
            shade(gj == 0, true);
        }
    }

    if (kCount) {
        for (int off = 32; off > 0; off >>= 1) {
            n_nodes += __shfl_down(n_nodes, off, 64);
            n_tris += __shfl_down(n_tris, off, 64);
            n_spill += __shfl_down(n_spill, off, 64);
            n_wsteps += __shfl_down(n_wsteps, off, 64);
            n_lsteps += __shfl_down(n_lsteps, off, 64);
            n_wshade += __shfl_down(n_wshade, off, 64);
            n_dwsteps += __shfl_down(n_dwsteps, off, 64);
            n_dlsteps += __shfl_down(n_dlsteps, off, 64);
        }
        if (lane == 0) {
            unsigned long long* st = kRayQuery ? tl.stats : (kMode == kModeBatch ? bl.stats : pl.stats);
            atomicAdd(&st[0], n_nodes);
            atomicAdd(&st[1], n_tris);
            atomicAdd(&st[2], n_spill);
            atomicAdd(&st[4], n_wsteps);
            atomicAdd(&st[5], n_lsteps);
            atomicAdd(&st[6], n_wshade);
            atomicAdd(&st[7], n_dwsteps);
            atomicAdd(&st[8], n_dlsteps);
            // drain window: earliest exhaustion, latest exit (wall clock ticks)
            if (t_exhausted) atomicMin(&st[9], t_exhausted);
            atomicMax(&st[10], (unsigned long long)wall_clock64());
        }
    }
    // ---- what a block adds to shared words, it adds once, not once per wave
    // (11.5 ns each, above).  Lookahead waves all end with the frame, so theirs
    // queued up: 3 sums and up to 2 queue positions each.  Frames of 262 k paths
    // 120 -> 111 us, of 2.07 M 1110 -> 1070 us.
    if constexpr (!kRayQuery) {
        constexpr int kWaves = kBlock / 64;
        constexpr int kSums = 1 + (kLookMode ? kLookLevels : 0);
        unsigned long long* sums = reinterpret_cast<unsigned long long*>(st_node);
        auto wave_sum = [](unsigned long long r) -> unsigned long long {
            for (int off = 32; off > 0; off >>= 1) r += __shfl_down(r, off, 64);
            return r;
        };
        __syncthreads();  // the stack is free
        const unsigned long long r0 = wave_sum(n_rays);
        if (lane == 0) sums[wave] = r0;
        uint64_t left[kLookLevels];  // lookahead: the lanes whose path stopped, by level
        uint32_t* const n_left = reinterpret_cast<uint32_t*>(sums + kWaves * kSums);  // [level][wave]
        if constexpr (kLookMode) {
#pragma unroll
            for (int l = 0; l < kLookLevels; ++l) {
                const unsigned long long r = wave_sum(n_ahead[l]);
                left[l] = __ballot(suspend && level == l + 1);
                if (lane == 0) {
                    sums[(l + 1) * kWaves + wave] = r;
                    n_left[l * kWaves + wave] = (uint32_t)__popcll(left[l]);
                }
            }
        }
        __syncthreads();
        if (tid < kSums) {
            unsigned long long r = 0;
            for (int k = 0; k < kWaves; ++k) r += sums[tid * kWaves + k];
            unsigned long long* to = &(kMode == kModeBatch ? bl.stats : pl.stats)[3];
            if (kLookMode && tid > 0) to = look ? &look->rays[tid] : nullptr;
            if (r && to) atomicAdd(to, r);
        }
        if constexpr (kLookMode) {
            // queue the later frames' paths that stopped, by level
            if (look) {
                uint32_t* const q_base = n_left + kLookLevels * kWaves;
                if (tid < kLookLevels) {
                    uint32_t r = 0;
                    for (int k = 0; k < kWaves; ++k) r += n_left[tid * kWaves + k];
                    q_base[tid] = r ? atomicAdd(&look->resume_out[tid + 1], r) : 0u;
                }
                __syncthreads();
                if (suspend) {
                    uint32_t slot = q_base[level - 1];
                    for (uint32_t k = 0; k < wave; ++k) slot += n_left[(uint32_t)((level - 1) * kWaves) + k];
                    uint64_t sm = left[0];
#pragma unroll
                    for (int l = 1; l < kLookLevels; ++l)
                        if (level == l + 1) sm = left[l];
                    slot += (uint32_t)__popcll(sm & lane_lt);
                    if (slot < pl.q_cap) {
                        uint4* q = pl.q_out[level - 1] + kLookItem * (size_t)slot;
                        q[0] = make_uint4(__float_as_uint(o.x), __float_as_uint(o.y), __float_as_uint(o.z),
                                          (uint32_t)pixel);
                        q[1] = make_uint4(__float_as_uint(d.x), __float_as_uint(d.y), __float_as_uint(d.z), rng);
                        q[2] = make_uint4((uint32_t)depth, __float_as_uint(lw), __float_as_uint(lsum), shadow ? 1u : 0u);
                        if (kMode == kModeDiffuse2) {
                            q[3] = make_uint4(__float_as_uint(eo.x), __float_as_uint(eo.y), __float_as_uint(eo.z),
                                              __float_as_uint(ed.x));
                            q[4] = make_uint4(__float_as_uint(ed.y), __float_as_uint(ed.z), 0u, 0u);
                        }
                    } else {
                        atomicOr(err, 2u);
                    }
                }
            }
        }
        if constexpr (kCount && kMode != kModeBatch) {
            __syncthreads();
            if (tid < kMaxQueueDepth && depth_hist[tid])
                atomicAdd(&pl.depth_rays[tid], (unsigned long long)depth_hist[tid]);
        }
    }
}

// Persistent workgroups of a launch over `items` rays or paths.  Each wave of a
// path launch pays for the drain of its own last paths (about 50 steps at a few
// active lanes), so one that has few items per lane gains more from fewer waves
// than it loses in latency hiding.  Rays drain fast, and up to a run for every
// wave they need no counter, so their launches take all waves, except where a
// few runs would be left over for a second round.  Measured per frame or launch
// with 1 / 2 / 3 / 4 workgroups per CU (256 CUs of 256 lanes each), ms, on the
// spheres and on a mixed scene of 400 k triangles:
//   closest    70 k 0.153 0.128 0.128 0.127, 0.244 0.241 0.243 0.242;
//             260 k 0.335 0.224 0.203 0.167, 0.427 0.314 0.291 0.279;
//             300 k 0.376 0.240 0.214 0.217, 0.498 0.343 0.301 0.321;
//             2 M   2.045 1.144 0.874 0.774, 2.183 1.277 1.022 0.911
//   any hit   260 k 0.241 0.171 0.159 0.124, 0.260 0.207 0.199 0.192;
//             280 k 0.261 0.182 0.168 0.186, 0.268 0.200 0.194 0.212;
//             2 M   1.456 0.827 0.659 0.586, 1.250 0.755 0.621 0.569
//   primary   144 k 0.129 0.134 0.125 0.126, 0.179 0.186 0.177 0.177;
//             262 k 0.182 0.166 0.167 0.138, 0.252 0.205 0.193 0.177;
//             2 M   0.502 0.374 0.341 0.330, 0.738 0.503 0.457 0.433
//   diffuse   495 k 0.992 0.707 0.710 0.767, 1.415 0.984 0.998 1.098;
//             640 k 1.214 0.799 0.728 0.780, 1.739 1.194 1.055 1.130;
//             0.97 M 1.724 1.092 0.919 0.900, 2.452 1.571 1.389 1.298
//   diffuse2  495 k 1.673 1.150 1.177 1.296, 2.222 1.515 1.581 1.789;
//             640 k 2.048 1.343 1.227 1.305, 2.761 1.855 1.656 1.798;
//             1.05 M 3.068 1.907 1.601 1.545, 4.160 2.655 2.310 2.160
// With the lookahead the drain is filled with later frames' work:
//   diffuse   262 k 0.620 0.413 0.435 0.447, 0.820 0.611 0.620 0.639;
//             495 k 0.972 0.638 0.487 0.513, 1.394 0.839 0.742 0.755;
//             810 k 1.456 0.906 0.747 0.630, 2.075 1.306 1.047 0.924
// On scenes whose nodes and triangles outgrow the memory-side cache (256 MiB)
// diffuse launches run at most one below the occupancy limit: their paths take
// long, so does the drain; the albedo and query launches are faster with all.
int grid_for(const prt_hip_ctx* ctx, int mode, uint64_t items, bool look = false)
{
    int per_cu;
    if (mode == kModeTrace || mode == kModeOccluded || mode == kModePrimary)
        per_cu = items > 256u << 10 && items <= 400u << 10 ? 3 : 4;
    else if (items <= 128u << 10)
        per_cu = 1;
    else if (items <= (look ? 384u : 576u) << 10)
        per_cu = 2;
    else
        per_cu = items <= (look ? 640u : 928u) << 10 ? 3 : 4;
    int limit = ctx->trace_per_cu;
    if (mode == kModeDiffuse && limit > 1) {
        const SceneBuffers& s = ctx->scene;
        const int64_t scene_bytes =
            s.node_count * (int64_t)sizeof(Bvh8Node) + s.tri_count * (int64_t)(9 * sizeof(float) + sizeof(int32_t));
        if (scene_bytes > kLargeSceneBytes) limit -= 1;
    }
    return std::min(per_cu, limit) * ctx->num_cus;
}

// Work items of a launch; ~0 where only the device knows.
uint64_t launch_items(int mode, const TraceLaunch& t, const PathLaunch& p)
{
    if (mode == kModeTrace || mode == kModeOccluded) return t.count_ptr ? ~0ull : t.count;
    if (mode == kModeAdjoint || (mode == kModeRgb && p.rgb_planes)) return (uint64_t)p.entries * (uint64_t)p.spp;
    return p.entries;
}

uint64_t spread_limit(int mode)
{
    return mode == kModeTrace || mode == kModeOccluded || mode == kModePrimary ? kSpreadRays : kSpreadPaths;
}

// Tail mode and grid of a launch.
int launch_shape(const prt_hip_ctx* ctx, int mode, uint64_t items, int& coop)
{
    coop = ctx->tail_coop ? kCoopTail : 0;
    if (coop && items <= spread_limit(mode)) {
        coop = kCoopSpread;
        return spread_grid(ctx->num_cus, items, kTraceBlock / 64, ctx->trace_grid);
    }
    return grid_for(ctx, mode, items);
}

template <int kMode>
hipError_t launch_mode(prt_hip_ctx* ctx, const TraceLaunch& t, const PathLaunch& paths, bool instrumented)
{
    const SceneDevice sc = ctx->scene.device();
    uint32_t* err = t.err ? t.err : ctx->d_counters + 32;
    const BatchLaunch bl{};
    PathLaunch p = paths;
    const int grid = p.look ? diffuse_grid(ctx, p.entries)
                            : launch_shape(ctx, kMode, launch_items(kMode, t, p), p.coop);
    if (instrumented) {
        k_trace<true, kMode><<<grid, kTraceBlock, 0, ctx->stream>>>(
            sc, t, p, bl, ctx->d_spill, ctx->stack_entries, kRefill, err);
        return hipGetLastError();
    }
    if constexpr (kMode == kModeDiffuse || kMode == kModeDiffuse2) {
        if (p.look != nullptr) {
            k_trace<false, kMode, kTraceBlock, kStackLds, true><<<grid, kTraceBlock, 0, ctx->stream>>>(
                sc, t, p, bl, ctx->d_spill, ctx->stack_entries, kRefill, err);
            return hipGetLastError();
        }
    }
    k_trace<false, kMode><<<grid, kTraceBlock, 0, ctx->stream>>>(
        sc, t, p, bl, ctx->d_spill, ctx->stack_entries, kRefill, err);
    return hipGetLastError();
}

// Batch kernel variants the autotuner chooses from: (block size, LDS stack).
template <int kBlock, int kStack>
hipError_t launch_batch_variant(prt_hip_ctx* ctx, const BatchLaunch& bl, int blocks_per_cu, int refill,
                                bool instrumented, int* max_blocks_per_cu)
{
    if (max_blocks_per_cu) {
        int per_cu = 0;
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per_cu, k_trace<false, kModeBatch, kBlock, kStack>, kBlock, 0);
        *max_blocks_per_cu = per_cu;
        return e;
    }
    int grid = blocks_per_cu * ctx->num_cus;
    uint32_t* err = ctx->d_counters + 32;
    const SceneDevice sc{};
    const TraceLaunch t{};
    PathLaunch p{};
    p.coop = ctx->tail_coop ? kCoopTail : 0;
    // Small job sets are traced in groups from their start, as small frames are.
    // us per render lane by lane / in groups: 1 k paths 400 / 226, 16 k 525 / 310
    // and 380 / 223 (two scenes), 20 k 555 / 275; where most paths escape at once
    // 16 k 43 / 39, 20 k 44 / 43, 40 k 44 / 71, so these stop at the rays' limit.
    if (p.coop && bl.total_work <= kSpreadRays) {
        p.coop = kCoopSpread;
        grid = spread_grid(ctx->num_cus, bl.total_work, kBlock / 64, grid);
    }
    if (instrumented)
        k_trace<true, kModeBatch, kBlock, kStack><<<grid, kBlock, 0, ctx->stream>>>(
            sc, t, p, bl, ctx->d_spill, ctx->stack_entries, refill, err);
    else
        k_trace<false, kModeBatch, kBlock, kStack><<<grid, kBlock, 0, ctx->stream>>>(
            sc, t, p, bl, ctx->d_spill, ctx->stack_entries, refill, err);
    return hipGetLastError();
}

}  // namespace

int ensure_trace_resources(prt_hip_ctx* ctx)
{
    if (ctx->trace_per_cu == 0) {
        // the lookahead variants' workgroups must all be resident at once: a
        // workgroup that starts only when another ends would hold the frame's
        // stop (every wave leaves the live count) until then
        int per_cu = 0, per_cu_look = 0, per_cu_look2 = 0;
        PRT_TRY(ctx, hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_trace<false, kModeDiffuse>,
                                                                  kTraceBlock, 0));
        PRT_TRY(ctx, hipOccupancyMaxActiveBlocksPerMultiprocessor(
                         &per_cu_look, k_trace<false, kModeDiffuse, kTraceBlock, kStackLds, true>, kTraceBlock, 0));
        PRT_TRY(ctx, hipOccupancyMaxActiveBlocksPerMultiprocessor(
                         &per_cu_look2, k_trace<false, kModeDiffuse2, kTraceBlock, kStackLds, true>, kTraceBlock, 0));
        per_cu = std::min(per_cu, std::min(per_cu_look, per_cu_look2));
        if (per_cu * kTraceBlock > 2048) per_cu = 2048 / kTraceBlock;
        if (per_cu < 1) per_cu = 1;
        ctx->trace_per_cu = per_cu;
    }
    ctx->trace_grid = ctx->trace_per_cu * ctx->num_cus;
    // worst case stack: 7 pushes per level of the tree, plus slack; sized for
    // the deepest scene and for every lane a CU can hold (2048), so any
    // persistent launch shape fits
    int depth = ctx->scene.bvh_depth;
    for (const SceneBuffers& b : ctx->batch_scenes) depth = depth > b.bvh_depth ? depth : b.bvh_depth;
    // The per-lane stride only grows, so a shallower scene keeps the buffer;
    // a captured launch graph holds the buffer and stride as kernel
    // arguments, so every change bumps spill_gen, which the graph's owner
    // compares before a replay.
    int need = 7 * (depth + 1) + 8;
    if (need < kStackLds) need = kStackLds;
    if (need < ctx->stack_entries) need = ctx->stack_entries;
    const int64_t lanes = (int64_t)ctx->num_cus * 2048;
    const int64_t bytes = lanes * need * (int64_t)sizeof(uint2);
    if (bytes > ctx->spill_bytes || need != ctx->stack_entries) {
        ctx->spill_gen += 1;
        if (ctx->d_spill) { (void)hipFree(ctx->d_spill); ctx->d_spill = nullptr; }
        ctx->spill_bytes = 0;
        ctx->stack_entries = 0;
        PRT_TRY(ctx, device_alloc(ctx, &ctx->d_spill, bytes));
        ctx->spill_bytes = bytes;
        ctx->stack_entries = need;
    }
    return 0;
}

int diffuse_grid(const prt_hip_ctx* ctx, uint32_t entries) { return grid_for(ctx, kModeDiffuse, entries, true); }

hipError_t launch_trace(prt_hip_ctx* ctx, const TraceLaunch& t, bool instrumented)
{
    return launch_mode<kModeTrace>(ctx, t, PathLaunch{}, instrumented);
}

hipError_t launch_trace_scratch(prt_hip_ctx* ctx, const TraceLaunch& t, uint2* spill, int stack_entries,
                                uint32_t* err, int max_grid)
{
    PathLaunch p{};
    int grid = launch_shape(ctx, kModeTrace, t.count, p.coop);
    if (grid > max_grid) {
        // fewer workgroups than a small launch is spread over: one by one
        if (p.coop == kCoopSpread) p.coop = kCoopTail;
        grid = max_grid;
    }
    k_trace<false, kModeTrace><<<grid, kTraceBlock, 0, ctx->stream>>>(ctx->scene.device(), t, p, BatchLaunch{}, spill,
                                                                     stack_entries, kRefill, err);
    return hipGetLastError();
}

hipError_t launch_paths_rgb(prt_hip_ctx* ctx, const PathLaunch& p, bool instrumented)
{
    return launch_mode<kModeRgb>(ctx, TraceLaunch{}, p, instrumented);
}

hipError_t launch_adjoint(prt_hip_ctx* ctx, const PathLaunch& p, bool instrumented)
{
    return launch_mode<kModeAdjoint>(ctx, TraceLaunch{}, p, instrumented);
}

hipError_t launch_occluded(prt_hip_ctx* ctx, const TraceLaunch& t, bool instrumented)
{
    return launch_mode<kModeOccluded>(ctx, t, PathLaunch{}, instrumented);
}

hipError_t launch_paths(prt_hip_ctx* ctx, const PathLaunch& p, int renderer, bool instrumented)
{
    TraceLaunch t{};
    switch (renderer) {
    case PRT_RENDERER_PRIMARY: return launch_mode<kModePrimary>(ctx, t, p, instrumented);
    case PRT_RENDERER_DIFFUSE: return launch_mode<kModeDiffuse>(ctx, t, p, instrumented);
    case PRT_RENDERER_DIFFUSE2: return launch_mode<kModeDiffuse2>(ctx, t, p, instrumented);
    default: return hipErrorInvalidValue;
    }
}

const BatchKernelConfig kBatchVariants[kBatchVariantCount] = {
    {256, 16}, {256, 8}, {128, 16}, {128, 8},
};

hipError_t launch_batch(prt_hip_ctx* ctx, const BatchLaunch& bl, const BatchTuning& tu, bool instrumented,
                        int* max_blocks_per_cu)
{
    switch (tu.variant) {
    case 0: return launch_batch_variant<256, 16>(ctx, bl, tu.blocks_per_cu, tu.refill, instrumented, max_blocks_per_cu);
    case 1: return launch_batch_variant<256, 8>(ctx, bl, tu.blocks_per_cu, tu.refill, instrumented, max_blocks_per_cu);
    case 2: return launch_batch_variant<128, 16>(ctx, bl, tu.blocks_per_cu, tu.refill, instrumented, max_blocks_per_cu);
    case 3: return launch_batch_variant<128, 8>(ctx, bl, tu.blocks_per_cu, tu.refill, instrumented, max_blocks_per_cu);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace prt
