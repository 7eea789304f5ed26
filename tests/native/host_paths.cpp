// Host control flow of the library against a stand-in for the HIP runtime
// (hip/hip_runtime.h beside this file): the entry points as they are, with the
// launches replaced by what their kernels leave in memory.
//   host_paths NAME   runs one check; prints what failed and returns 1
#include <chrono>
#include <cstdio>
#include <filesystem>
#include <functional>

#include "../../embree-benchmark-protoray_amd/csrc/api.hip"
#include "../../embree-benchmark-protoray_amd/csrc/host_copy.hip"
#include "../../embree-benchmark-protoray_amd/csrc/launch_shape.h"

namespace {

int g_failed = 0;
#define EXPECT(cond)                                                        \
    do {                                                                    \
        if (!(cond)) {                                                      \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #cond);          \
            g_failed = 1;                                                   \
        }                                                                   \
    } while (0)

int g_per_cu = 4;                 // workgroups per CU that fit
prt::PathLaunch g_paths;          // the last path launch
bool g_look_valid = false;        // ... and whether the lookahead kept earlier work for it

// A ray's record: its own first origin coordinate, so that a test knows it.
prt_hit answer(const float4& r0) { return prt_hit{r0.x, 7, 0.25f, 0.5f}; }

// What a query launch writes: the waves' first runs always, the others only if
// the work counters start from zero.
hipError_t query(prt_hip_ctx* ctx, const prt::TraceLaunch& t, bool any)
{
    const uint64_t n = t.count;
    const bool spread = ctx->tail_coop && n <= prt::kSpreadRays;
    uint64_t reached = n;
    if (spread) reached = 4 * prt::kSpreadRun * (uint64_t)prt::spread_grid(ctx->num_cus, n, 4, ctx->trace_grid);
    for (int w = 0; w < prt::kWorkWords; w += prt::kWorkCounterStride)
        if (t.work[w] == 0) reached = n;
    for (uint64_t k = 0; k < std::min(n, reached); ++k) {
        if (any) t.any_t[k] = t.rays[2 * k].x;
        else reinterpret_cast<prt_hit*>(t.hits)[k] = answer(t.rays[2 * k]);
    }
    for (int w = 0; w < prt::kWorkWords; w += prt::kWorkCounterStride) t.work[w] += 12345;  // what a launch leaves
    return hipSuccess;
}

}  // namespace

namespace prt {

int ensure_trace_resources(prt_hip_ctx* ctx)
{
    ctx->trace_per_cu = g_per_cu;
    ctx->trace_grid = g_per_cu * ctx->num_cus;
    return 0;
}
int diffuse_grid(const prt_hip_ctx* ctx, uint32_t) { return ctx->trace_grid; }
hipError_t launch_trace(prt_hip_ctx* ctx, const TraceLaunch& t, bool) { return query(ctx, t, false); }
hipError_t launch_occluded(prt_hip_ctx* ctx, const TraceLaunch& t, bool) { return query(ctx, t, true); }
hipError_t launch_trace_scratch(prt_hip_ctx*, const TraceLaunch&, uint2*, int, uint32_t*, int) { return hipSuccess; }
hipError_t launch_zero_u32(uint32_t* p, int n, hipStream_t) { std::memset(p, 0, 4 * (size_t)n); return hipSuccess; }
hipError_t launch_paths(prt_hip_ctx*, const PathLaunch& p, int, bool)
{
    g_paths = p;
    return hipGetLastError();
}
hipError_t launch_look_call_begin(prt_hip_ctx*, bool valid, uint32_t)
{
    g_look_valid = valid;
    return hipGetLastError();
}
hipError_t launch_paths_rgb(prt_hip_ctx*, const PathLaunch&, bool) { return hipSuccess; }
hipError_t launch_adjoint(prt_hip_ctx*, const PathLaunch& p, bool)
{
    g_paths = p;
    return hipGetLastError();
}
const BatchKernelConfig kBatchVariants[kBatchVariantCount] = {{256, 16}, {256, 8}, {128, 16}, {128, 8}};
hipError_t launch_batch(prt_hip_ctx*, const BatchLaunch&, const BatchTuning&, bool, int* max_blocks_per_cu)
{
    if (max_blocks_per_cu) *max_blocks_per_cu = g_per_cu;
    return hipSuccess;
}
hipError_t launch_raygen(prt_hip_ctx*, int, float4*, int32_t*, uint32_t*) { return hipSuccess; }
hipError_t launch_frame_begin(prt_hip_ctx*, uint32_t) { return hipSuccess; }
hipError_t launch_shade_diffuse(prt_hip_ctx*, int, int, float, bool) { return hipSuccess; }
hipError_t launch_queue_recycle(prt_hip_ctx*, int) { return hipSuccess; }
hipError_t launch_shade_primary(prt_hip_ctx*, bool) { return hipSuccess; }
hipError_t launch_tonemap(prt_hip_ctx*) { return hipSuccess; }
hipError_t launch_batch_begin(prt_hip_ctx*) { return hipSuccess; }
hipError_t launch_accum_mean_rgb(prt_hip_ctx*, float*) { return hipSuccess; }
hipError_t launch_rgb_planes_add(prt_hip_ctx*, const float4*, int) { return hipSuccess; }
hipError_t launch_batch_finalize(prt_hip_ctx*) { return hipSuccess; }
hipError_t launch_batch_advance(prt_hip_ctx*) { return hipSuccess; }
hipError_t launch_unpack_rays(const float4*, const int32_t*, const uint32_t*, int64_t, int, int, prt_ray*, uint32_t*,
                              hipStream_t)
{
    return hipSuccess;
}
Camera to_camera(const prt_camera&) { return Camera{}; }
int build_bvh8(prt_hip_ctx*, SceneBuffers& sb, prt_build_stats*)
{
    sb.bvh_ready = true;
    sb.bvh_depth = 4;
    sb.node_count = 1;
    return 0;
}

}  // namespace prt

namespace {

struct Context {
    prt_hip_ctx* ctx = nullptr;
    explicit Context(int num_cus = 256, int per_cu = 4)
    {
        fake::state().num_cus = num_cus;
        g_per_cu = per_cu;
        EXPECT(prt_hip_create(0, &ctx) == 0);
    }
    ~Context() { EXPECT(prt_hip_destroy(ctx) == 0); }
    operator prt_hip_ctx*() const { return ctx; }
};

const int32_t kIdx[3] = {0, 1, 2};
const float kPos[9] = {0, 0, 0, 1, 0, 0, 0, 1, 0};

void with_scene(prt_hip_ctx* ctx)
{
    EXPECT(prt_hip_scene_upload(ctx, kIdx, 1, kPos, 3) == 0);
    EXPECT(prt_hip_bvh_build(ctx, nullptr) == 0);
}

// Every ray of a small host query is answered on devices of any size: the
// launch goes without work counters only where each ray has a wave.
void small_query_on_small_devices()
{
    for (int num_cus : {1, 4, 32, 64, 128, 255, 256, 304})
        for (int per_cu : {1, 2, 3, 4, 8}) {
            Context c(num_cus, per_cu);
            with_scene(c);
            float base = 1.0f;
            for (int64_t n : {1, 7, 8, 9, 31, 1000, 8191, 8192, 8193, 24577, 32767, 32768, 32769, 1}) {
                std::vector<prt_ray> rays(n);
                for (int64_t k = 0; k < n; ++k) reinterpret_cast<float*>(&rays[k])[0] = base + (float)k;
                std::vector<prt_hit> hits(n);
                std::vector<float> any(n);
                EXPECT(prt_hip_intersect_closest(c, rays.data(), hits.data(), n) == 0);
                EXPECT(prt_hip_occluded(c, rays.data(), any.data(), n) == 0);
                int64_t bad = 0;
                for (int64_t k = 0; k < n; ++k)
                    bad += reinterpret_cast<const float*>(&hits[k])[0] != base + (float)k || any[k] != base + (float)k;
                if (bad) std::printf("%d CUs, %d workgroups each, %lld rays: %lld not answered\n", num_cus, per_cu,
                                     (long long)n, (long long)bad);
                EXPECT(bad == 0);
                base += 100000.0f;
            }
        }
}

// A small query needs no pinned memory beside what the context laid out when it
// was made, and leaves the copies that use the same memory as they were.
void small_query_memory()
{
    Context c;
    with_scene(c);
    const int pinned = fake::state().pinned_calls;
    EXPECT(prt_hip_frame_init(c, 700, 700) == 0);
    std::vector<float> image((size_t)4 * 700 * 700);
    for (int64_t n : {1, 32768, 300000, 5}) {
        std::vector<prt_ray> rays(n);
        for (int64_t k = 0; k < n; ++k) reinterpret_cast<float*>(&rays[k])[0] = 2.0f + (float)k;
        std::vector<prt_hit> hits(n);
        std::vector<float> any(n);
        EXPECT(prt_hip_intersect_closest(c, rays.data(), hits.data(), n) == 0);
        EXPECT(prt_hip_occluded(c, rays.data(), any.data(), n) == 0);
        for (int64_t k : {(int64_t)0, n / 2, n - 1})
            EXPECT(reinterpret_cast<const float*>(&hits[k])[0] == 2.0f + (float)k && any[k] == 2.0f + (float)k);
        std::fill(image.begin(), image.end(), -1.0f);
        EXPECT(prt_hip_accum_read(c, image.data()) == 0);
        EXPECT(*std::min_element(image.begin(), image.end()) == 0.0f && *std::max_element(image.begin(), image.end()) == 0.0f);
    }
    EXPECT(fake::state().pinned_calls == pinned);
}

// A count that no query accepts is refused before anything is copied.
void bad_ray_counts()
{
    Context c;
    with_scene(c);
    std::vector<prt_ray> rays(4);
    std::vector<prt_hit> hits(4);
    std::vector<float> any(4);
    prt_trace_counters counters;
    const size_t copies = fake::state().copies.size();
    for (int64_t n : {(int64_t)-1, (int64_t)-2, -((int64_t)1 << 21), -((int64_t)3 << 46), -((int64_t)1 << 62), INT64_MIN,
                      (int64_t)1 << 31, (int64_t)1 << 58, INT64_MAX}) {
        EXPECT(prt_hip_intersect_closest(c, rays.data(), hits.data(), n) != 0);
        EXPECT(prt_hip_occluded(c, rays.data(), any.data(), n) != 0);
        EXPECT(prt_hip_intersect_counters(c, rays.data(), hits.data(), n, &counters) != 0);
        EXPECT(std::string(prt_hip_last_error(c)).find("bad ray count") != std::string::npos);
        EXPECT(prt_hip_intersect_closest_device(c, rays.data(), hits.data(), n) != 0);
        EXPECT(prt_hip_occluded_device(c, rays.data(), any.data(), n) != 0);
    }
    EXPECT(fake::state().copies.size() == copies);
    EXPECT(prt_hip_intersect_closest(c, rays.data(), hits.data(), 4) == 0);
}

// Without pinned memory beyond the context's own small block, every host copy and
// query still does its work.
void no_pinned_memory()
{
    fake::state().pinned_fail_from = 2;
    Context c;
    with_scene(c);
    for (int64_t n : {1, 1000, 40000, 300000}) {
        std::vector<prt_ray> rays(n);
        for (int64_t k = 0; k < n; ++k) reinterpret_cast<float*>(&rays[k])[0] = 3.0f + (float)k;
        std::vector<prt_hit> hits(n);
        std::vector<float> any(n);
        EXPECT(prt_hip_intersect_closest(c, rays.data(), hits.data(), n) == 0);
        EXPECT(prt_hip_occluded(c, rays.data(), any.data(), n) == 0);
        for (int64_t k = 0; k < n; k += n > 1 ? n - 1 : 1)
            EXPECT(reinterpret_cast<const float*>(&hits[k])[0] == 3.0f + (float)k && any[k] == 3.0f + (float)k);
    }
    for (int w : {1, 64, 700, 1500}) {
        EXPECT(prt_hip_frame_init(c, w, w) == 0);
        std::vector<float> image((size_t)4 * w * w, -1.0f);
        EXPECT(prt_hip_accum_read(c, image.data()) == 0);
        EXPECT(image.front() == 0.0f && image.back() == 0.0f);
    }
    EXPECT(hipGetLastError() == hipSuccess);   // a launch check would take it for its own
}

// Copies of every length class, one chunk, two halves, a ring that wraps, both
// ways and with two contexts on two threads at once; then copies that fail part
// way, after which the next one works.
void host_copies()
{
    constexpr size_t kChunk = size_t(2) << 20;
    auto copies = [](uint32_t seed) {
        HostCopy copy;
        for (size_t bytes : {(size_t)1, kChunk / 4, kChunk / 4 + 1, kChunk - 1, kChunk, kChunk + 1, 2 * kChunk, 2 * kChunk + 1,
                             5 * kChunk, 6 * kChunk - 3, 6 * kChunk, 6 * kChunk + 1, 13 * kChunk + 12345}) {
            std::vector<unsigned char> src(bytes), dst(bytes + 2, 0xee);
            uint32_t s = seed + (uint32_t)bytes;
            for (unsigned char& b : src) b = (unsigned char)((s = s * 1664525u + 1013904223u) >> 24);
            EXPECT(copy.to_host(dst.data() + 1, src.data(), bytes, nullptr) == hipSuccess);
            EXPECT(std::memcmp(dst.data() + 1, src.data(), bytes) == 0 && dst.front() == 0xee && dst.back() == 0xee);
            std::fill(dst.begin(), dst.end(), (unsigned char)0xee);
            EXPECT(copy.to_device(dst.data() + 1, src.data(), bytes, nullptr) == hipSuccess);
            EXPECT(std::memcmp(dst.data() + 1, src.data(), bytes) == 0 && dst.front() == 0xee && dst.back() == 0xee);
        }
    };
    std::thread other([&] { copies(99); });
    copies(1);
    other.join();
    HostCopy copy;
    std::vector<unsigned char> src(9 * kChunk + 5, 7), dst(src.size(), 0);
    for (int fail = 1; fail <= 11; ++fail)
        for (int up = 0; up < 2; ++up) {
            fake::state().copy_fail_at = fake::state().copy_calls + fail;
            const hipError_t e = up ? copy.to_device(dst.data(), src.data(), src.size(), nullptr)
                                    : copy.to_host(dst.data(), src.data(), src.size(), nullptr);
            EXPECT((e != hipSuccess) == (fail <= 10));
            fake::state().copy_fail_at = 1 << 30;
            std::fill(dst.begin(), dst.end(), (unsigned char)0);
            EXPECT(copy.to_host(dst.data(), src.data(), src.size(), nullptr) == hipSuccess && dst == src);
            (void)hipGetLastError();
        }
}

// Pinned memory of the caller is copied in one piece, straight to or from it;
// pageable memory in chunks through the ring.
void pinned_caller()
{
    HostCopy copy;
    for (size_t bytes : {(size_t)64 << 10, (size_t)1 << 20, (size_t)5 << 20, ((size_t)40 << 20) + 4}) {
        char *pinned = nullptr, *device = nullptr;
        EXPECT(hipHostMalloc(&pinned, bytes + 8, hipHostMallocDefault) == hipSuccess);
        EXPECT(hipMalloc(&device, bytes) == hipSuccess);
        std::memset(device, 5, bytes);
        auto& copies = fake::state().copies;
        copies.clear();
        EXPECT(copy.to_host(pinned + 4, device, bytes, nullptr) == hipSuccess);   // inside the allocation
        EXPECT(copies.size() == 1 && copies[0].dst == pinned + 4 && copies[0].bytes == bytes);
        EXPECT(pinned[3] == 0 && pinned[4] == 5 && pinned[3 + bytes] == 5 && pinned[4 + bytes] == 0);
        copies.clear();
        EXPECT(copy.to_device(device, pinned, bytes, nullptr) == hipSuccess);
        EXPECT(copies.size() == 1 && copies[0].src == pinned && copies[0].bytes == bytes);
        std::vector<char> pageable(bytes, 9);
        copies.clear();
        EXPECT(copy.to_device(device, pageable.data(), bytes, nullptr) == hipSuccess);
        EXPECT(bytes <= (size_t)4 << 20 || copies.size() > 2);
        EXPECT(device[0] == 9 && device[bytes - 1] == 9);
        EXPECT(hipGetLastError() == hipSuccess);
        EXPECT(hipFree(device) == hipSuccess && hipHostFree(pinned) == hipSuccess);
    }
}

int threads()
{
    int n = 0;
    for (const auto& e : std::filesystem::directory_iterator("/proc/self/task")) n += e.exists();
    return n;
}

// A context starts its copy threads with the first copy that needs them, and
// ends them with itself.
void copy_threads()
{
    const int before = threads();
    {
        Context c;
        with_scene(c);
        std::vector<prt_ray> rays(40000);
        std::vector<prt_hit> hits(40000);
        EXPECT(prt_hip_intersect_closest(c, rays.data(), hits.data(), 40000) == 0);
        EXPECT(threads() == before);
        EXPECT(prt_hip_frame_init(c, 1000, 1000) == 0);
        std::vector<float> image(4000000);
        EXPECT(prt_hip_accum_read(c, image.data()) == 0);
        EXPECT(threads() > before);
    }
    // a joined thread's entry can outlast the join by a moment
    for (int k = 0; k < 200 && threads() != before; ++k) std::this_thread::sleep_for(std::chrono::milliseconds(10));
    EXPECT(threads() == before);
}

// The deal of work items: each run belongs to one counter, in its order, and no
// column of a frame's tiles leaves more than half of its runs to one counter.
void work_deal()
{
    for (uint32_t runs : {0u, 1u, 15u, 16u, 17u, 31u, 33u, 255u, 4096u, 4097u, 70001u}) {
        std::vector<uint32_t> next(16, 0);
        for (uint32_t r = 0; r < runs; ++r) {
            const uint32_t c = deal_counter(r);
            EXPECT(c < 16 && deal_run(c, r >> 4) == r && next[c] == r >> 4);
            EXPECT(dealt_runs(c, r) == next[c]);
            ++next[c];
        }
        uint32_t all = 0;
        for (uint32_t c = 0; c < 16; ++c) {
            EXPECT(dealt_runs(c, runs) == next[c]);
            all += dealt_runs(c, runs);
        }
        EXPECT(all == runs);
    }
    // the most runs of a launch: 2^32 - 2^20 items in runs of 64
    for (uint32_t r : {67092479u, 67092478u, 67092464u, 67092463u}) EXPECT(deal_run(deal_counter(r), r >> 4) == r);
    for (uint32_t tiles = 16; tiles <= 512; tiles += 16)
        for (uint32_t rows : {16u, 64u, 135u})
            for (uint32_t x = 0; x < tiles; ++x) {
                std::vector<uint32_t> count(16, 0);
                for (uint32_t y = 0; y < rows; ++y) ++count[deal_counter(y * tiles + x)];
                EXPECT(*std::max_element(count.begin(), count.end()) <= (rows + 1) / 2);
            }
}

// Frames render where the lookahead's buffers find no room, and with it again
// once there is.
void no_room_for_the_lookahead()
{
    for (int renderer : {PRT_RENDERER_DIFFUSE, PRT_RENDERER_DIFFUSE2})
        for (size_t room : {(size_t)0, (size_t)1 << 20, (size_t)10 << 20}) {  // none, ..., the side samples alone
            Context c;
            with_scene(c);
            prt_camera cam{};
            cam.focal_distance = 1.0f;
            EXPECT(prt_hip_camera_set(c, &cam) == 0);
            EXPECT(prt_hip_frame_init(c, 717, 405) == 0);
            fake::state().device_limit = fake::state().device_bytes + room;
            for (int k = 0; k < 6; ++k) {
                EXPECT(prt_hip_render(c, renderer, 6, 0.8f, nullptr) == 0);
                EXPECT(g_paths.look == nullptr);
            }
            fake::state().device_limit = ~size_t(0);
            EXPECT(prt_hip_set_lookahead(c, 1) == 0);
            int runs = 0;
            for (int k = 0; k < 6; ++k) {
                EXPECT(prt_hip_render(c, renderer, 6, 0.8f, nullptr) == 0);
                if (g_paths.look) EXPECT(g_look_valid == (runs++ > 0));
            }
            EXPECT(runs >= 3);
        }
}

// A frame that finds no room for one of its buffers is none: what needs it is
// refused until there is one.
void half_a_frame()
{
    Context c;
    with_scene(c);
    prt_camera cam{};
    cam.focal_distance = 1.0f;
    EXPECT(prt_hip_camera_set(c, &cam) == 0);
    std::vector<float> image(4 * 512 * 512);
    std::vector<int32_t> pixels(512 * 512);
    for (size_t room : {(size_t)0, (size_t)5 << 20, (size_t)8 << 20, (size_t)20 << 20}) {  // none, image, pixels, some queues
        fake::state().device_limit = fake::state().device_bytes + room;
        EXPECT(prt_hip_frame_init(c, 512, 512) != 0);
        EXPECT(prt_hip_frame_clear(c) != 0);
        EXPECT(prt_hip_render(c, PRT_RENDERER_DIFFUSE, 6, 0.8f, nullptr) != 0);
        EXPECT(prt_hip_accum_read(c, image.data()) != 0);
        EXPECT(prt_hip_frame_read_bgr8(c, pixels.data()) != 0);
        fake::state().device_limit = ~size_t(0);
    }
    EXPECT(prt_hip_frame_init(c, 512, 512) == 0);
    EXPECT(prt_hip_render(c, PRT_RENDERER_DIFFUSE, 6, 0.8f, nullptr) == 0);
    EXPECT(prt_hip_frame_read_bgr8(c, pixels.data()) == 0);
}

// The adjoint runs where its hit record finds no room (its paths are traced again
// instead), with the record again once there is, and never beyond the depth that
// is recorded.
void no_room_for_the_hit_record()
{
    Context c;
    with_scene(c);
    prt_camera cam{};
    cam.focal_distance = 1.0f;
    EXPECT(prt_hip_camera_set(c, &cam) == 0);
    EXPECT(prt_hip_frame_init(c, 64, 64) == 0);
    const float rgb[3] = {0.5f, 0.5f, 0.5f};
    EXPECT(prt_hip_set_albedo_host(c, rgb) == 0);
    std::vector<float> dldi(3 * 64 * 64, 1.0f), grad(3, 0.0f);
    const int64_t lanes = (int64_t)c.ctx->trace_grid * kTraceBlock;
    for (int depth : {0, 1, 6, 64, 65, 6}) {
        fake::state().device_limit = fake::state().device_bytes;
        EXPECT(prt_hip_adjoint_albedo(c, 0, 1, depth, dldi.data(), grad.data(), nullptr) == 0);
        const bool kept = c.ctx->path_hits_cap >= lanes * std::max(1, depth);
        EXPECT((g_paths.path_hits != nullptr) == (kept && depth <= 64));
        fake::state().device_limit = ~size_t(0);
        EXPECT(prt_hip_adjoint_albedo(c, 0, 1, depth, dldi.data(), grad.data(), nullptr) == 0);
        EXPECT((g_paths.path_hits != nullptr) == (depth <= 64));
        EXPECT(depth > 64 || (g_paths.path_hits_stride == lanes && c.ctx->path_hits_cap >= lanes * depth));
    }
}

// Memory that a job set or a scene needs and the one before it gives up is there
// for it: a device that holds either holds one after the other.
void replaced_buffers()
{
    Context c;
    int scene = -1;
    EXPECT(prt_hip_batch_scene_add(c, kIdx, 1, kPos, 3, nullptr, &scene) == 0);
    prt_batch_job wide{}, deep{};
    wide.camera.focal_distance = deep.camera.focal_distance = 1.0f;
    wide.scene = deep.scene = scene;
    wide.width = wide.height = 2048;   // 67 MB of accumulators, 17 MB of samples
    wide.spp = 1;
    deep.width = deep.height = 1024;   // 17 and 67
    deep.spp = 16;
    const size_t before = fake::state().device_bytes;
    fake::state().device_limit = before + ((size_t)90 << 20);
    for (int k = 0; k < 4; ++k) {
        const bool ok = prt_hip_batch_set_jobs(c, k & 1 ? &deep : &wide, 1) == 0;
        if (!ok) std::printf("set %d: %s\n", k, prt_hip_last_error(c));
        EXPECT(ok);
    }
    fake::state().device_limit = ~size_t(0);
    EXPECT(prt_hip_batch_reset(c) == 0);

    // 1 M triangles of 4 vertices, then 40 k of 3 M vertices, in turn
    std::vector<int32_t> idx(3000000, 1);
    std::vector<float> pos(9000000, 0.5f);
    fake::state().device_limit = fake::state().device_bytes + ((size_t)40 << 20);
    for (int k = 0; k < 4; ++k) {
        EXPECT(prt_hip_scene_upload(c, idx.data(), k & 1 ? 40000 : 1000000, pos.data(), k & 1 ? 3000000 : 4) == 0);
        EXPECT(prt_hip_bvh_build(c, nullptr) == 0);
    }
    // a scene that finds no room leaves none behind
    fake::state().device_limit = fake::state().device_bytes;
    EXPECT(prt_hip_scene_upload(c, idx.data(), 1000000, pos.data(), 3000000) != 0);
    EXPECT(c.ctx->scene.tri_count == 0);
    fake::state().device_limit = ~size_t(0);
}

// What a context keeps between calls (build scratch, the adjoint's hit record,
// the lookahead's buffers) gives way to an allocation that finds no room.
void kept_memory()
{
    constexpr size_t kMb = (size_t)1 << 20;
    Context c;
    with_scene(c);
    prt_camera cam{};
    cam.focal_distance = 1.0f;
    EXPECT(prt_hip_camera_set(c, &cam) == 0);
    int scene = -1;
    EXPECT(prt_hip_batch_scene_add(c, kIdx, 1, kPos, 3, nullptr, &scene) == 0);
    std::vector<float> values(9000000, 0.5f), image(3 * 512 * 512);
    std::vector<int32_t> idx(3000000, 1);
    std::vector<prt_ray> rays(1000000);
    std::vector<prt_hit> hits(1000000);
    prt_batch_job job{};
    job.camera.focal_distance = 1.0f;
    job.scene = scene;
    job.width = job.height = 1024;
    job.spp = 8;
    const std::function<int()> calls[] = {
        [&] { return prt_hip_frame_init(c, 1024, 1024); },
        [&] { return prt_hip_intersect_closest(c, rays.data(), hits.data(), 1000000); },
        [&] { return prt_hip_batch_set_jobs(c, &job, 1); },
        [&] { return prt_hip_batch_scene_add(c, idx.data(), 1000000, values.data(), 3000000, nullptr, &scene); },
        [&] { return prt_hip_scene_upload(c, idx.data(), 1000000, values.data(), 3000000); },
        [&] { return prt_hip_scene_attributes(c, values.data(), values.data()); },
        [&] { return prt_hip_set_albedo_host(c, values.data()); },
        [&] { return prt_hip_bvh_build(c, nullptr) || prt_hip_render_albedo_image_host(c, 0, 16, 6, image.data(), nullptr); },
        [&] { return prt_hip_adjoint_albedo_host(c, 0, 1, 65, image.data(), values.data(), nullptr); },
    };
    for (const auto& call : calls) {
        auto room = [&](int64_t left) {   // a device with so much left, and all kept memory laid out
            fake::state().device_limit = ~size_t(0);
            EXPECT(prt_hip_bvh_build(c, nullptr) == 0);
            std::vector<float> rgb(3 * (size_t)c.ctx->scene.tri_count, 0.5f), image(3 * 512 * 512);
            EXPECT(prt_hip_set_albedo_host(c, rgb.data()) == 0);
            if (c.ctx->width != 512) EXPECT(prt_hip_frame_init(c, 512, 512) == 0);
            EXPECT(prt_hip_frame_clear(c) == 0);
            for (int k = 0; k < 6; ++k) EXPECT(prt_hip_render(c, PRT_RENDERER_DIFFUSE2, 6, 0.8f, nullptr) == 0);
            EXPECT(g_paths.look != nullptr);
            EXPECT(prt_hip_adjoint_albedo_host(c, 0, 1, 6, image.data(), rgb.data(), nullptr) == 0);
            EXPECT(c.ctx->d_path_hits != nullptr && c.ctx->d_look != nullptr);
            if (!c.ctx->d_build) EXPECT(hipMalloc(&c.ctx->d_build, c.ctx->build_bytes = 200 * kMb) == hipSuccess);
            fake::state().device_limit = fake::state().device_bytes + left;
        };
        room(0);
        const int refused = call();
        if (refused) std::printf("call %d: %s\n", (int)(&call - calls), prt_hip_last_error(c));
        EXPECT(refused == 0);
        EXPECT(hipGetLastError() == hipSuccess);
        // the frames go on, with the lookahead from its beginning
        fake::state().device_limit = ~size_t(0);
        if (!c.ctx->scene.bvh_ready) EXPECT(prt_hip_bvh_build(c, nullptr) == 0);
        EXPECT(prt_hip_frame_clear(c) == 0);
        int runs = 0;
        for (int k = 0; k < 12; ++k) {
            EXPECT(prt_hip_render(c, PRT_RENDERER_DIFFUSE2, 6, 0.8f, nullptr) == 0);
            if (g_paths.look) EXPECT(g_look_valid == (runs++ > 0));
        }
        EXPECT(runs >= 3);
    }
    // the lookahead's own buffers take the scratch's room
    EXPECT(prt_hip_frame_init(c, 512, 512) == 0);
    for (int k = 0; k < 2; ++k) EXPECT(prt_hip_render(c, PRT_RENDERER_DIFFUSE2, 6, 0.8f, nullptr) == 0);
    EXPECT(prt_hip_frame_init(c, 640, 480) == 0);
    if (!c.ctx->d_build) EXPECT(hipMalloc(&c.ctx->d_build, c.ctx->build_bytes = 200 * kMb) == hipSuccess);
    fake::state().device_limit = fake::state().device_bytes;
    for (int k = 0; k < 6; ++k) EXPECT(prt_hip_render(c, PRT_RENDERER_DIFFUSE2, 6, 0.8f, nullptr) == 0);
    EXPECT(g_paths.look != nullptr && c.ctx->d_build == nullptr);
    // refused all the same, and nothing of it left to the next call
    fake::state().device_limit = fake::state().device_bytes;
    EXPECT(prt_hip_frame_init(c, 16384, 16384) != 0);
    EXPECT(std::string(prt_hip_last_error(c)).find("out of memory") != std::string::npos);
    EXPECT(hipGetLastError() == hipSuccess);
    fake::state().device_limit = ~size_t(0);
}

const struct {
    const char* name;
    void (*run)();
} kChecks[] = {
    {"small_query_on_small_devices", small_query_on_small_devices},
    {"small_query_memory", small_query_memory},
    {"bad_ray_counts", bad_ray_counts},
    {"no_pinned_memory", no_pinned_memory},
    {"host_copies", host_copies},
    {"pinned_caller", pinned_caller},
    {"copy_threads", copy_threads},
    {"work_deal", work_deal},
    {"no_room_for_the_lookahead", no_room_for_the_lookahead},
    {"no_room_for_the_hit_record", no_room_for_the_hit_record},
    {"half_a_frame", half_a_frame},
    {"replaced_buffers", replaced_buffers},
    {"kept_memory", kept_memory},
};

}  // namespace

int main(int argc, char** argv)
{
    for (const auto& c : kChecks)
        if (argc > 1 && std::strcmp(argv[1], c.name) == 0) {
            c.run();
            return g_failed;
        }
    std::printf("no such check\n");
    return 2;
}
