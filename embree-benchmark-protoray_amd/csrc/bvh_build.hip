// bvh_build.hip -- LBVH build on the GPU, collapsed to a quantised BVH8.
//
// Replaces the closed OptiX Prime build of
// accel/optix/optix_intersector_stream_cuda.cpp:23-75 (timed buildMs / buildMprim).
//   1. centroid bounds (one partial box per block, finished by the next kernel)
//   2. 63-bit Morton codes of triangle box centres
//   3. LSD radix sort of (key, triangle id), 8 passes of 8 bits
//   4. radix tree (T. Karras, "Maximizing Parallelism in the Construction of
//      BVHs, Octrees, and k-d Trees", HPG 2012), equal keys split by index
//   5. bottom-up boxes with one arrival counter per internal node: tiles of
//      1024 leaves in LDS, the nodes above them in phases of 32 times
//      larger tiles, a workgroup each
//   6. top-down collapse to BVH8, two launches per level, 8 lanes per wide
//      node (one per slot).  Which binary nodes become the (at most 8) slots
//      of a wide node follows a surface-area cost optimum computed bottom-up
//      during the refit (S. Ylitie, T. Karras, S. Laine, "Efficient Incoherent
//      Ray Traversal on GPUs Through Compressed Wide BVHs", HPG 2017, section
//      4.1); subtrees of at most kLeafMax triangles become leaf slots.  (The
//      greedy alternative opens the widest-area internal child until 8 slots
//      are used.)  Node and record offsets are prefix sums over the level's
//      tasks, so the layout is deterministic.
//
// A build is bound by the chain of its dependent launches and loads, not by
// bandwidth: 8 k triangles move 1 MB.  So the level sizes stay on the device
// (the host looks once after the levels it expects), every pass does what the
// next one needs, and the scratch is one allocation that the context keeps.
// Build time against launches with host-sized levels, three scan launches per
// sort pass and one thread per wide node: 8 k triangles 1.21 -> 0.28 ms, 200 k
// 2.33 -> 0.58, 1.3 M 3.01 -> 1.00, 16 M 16.0 -> 7.9.
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <vector>

#include "prt_internal.h"

namespace prt {
namespace {

constexpr int kBlock = 256;
constexpr int32_t kEmptySlot = INT32_MIN;

__device__ __forceinline__ float3 vtx(const float* pos, int i)
{
    return make_float3(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]);
}

struct Box {
    float lo[3], hi[3];
};

__device__ __forceinline__ Box tri_box(const int32_t* idx, const float* pos, int t)
{
    float3 a = vtx(pos, idx[3 * t]), b = vtx(pos, idx[3 * t + 1]), c = vtx(pos, idx[3 * t + 2]);
    Box r;
    r.lo[0] = fminf(fminf(a.x, b.x), c.x);
    r.lo[1] = fminf(fminf(a.y, b.y), c.y);
    r.lo[2] = fminf(fminf(a.z, b.z), c.z);
    r.hi[0] = fmaxf(fmaxf(a.x, b.x), c.x);
    r.hi[1] = fmaxf(fmaxf(a.y, b.y), c.y);
    r.hi[2] = fmaxf(fmaxf(a.z, b.z), c.z);
    return r;
}

__device__ __forceinline__ float box_half_area(const Box& b)
{
    const float dx = b.hi[0] - b.lo[0], dy = b.hi[1] - b.lo[1], dz = b.hi[2] - b.lo[2];
    return dx * dy + dy * dz + dz * dx;
}

// ---------------------------------------------------------------- collapse cost
// cost(n, i), i = 1..7: the least surface-area cost of covering the subtree of
// binary node n with at most i slots of the parent wide node.  A slot that is
// a subtree of at most kLeafMax triangles is a leaf (area x triangles x
// c_prim); a larger one is a wide node (area x c_node plus the best split of
// its 8 slots between its two children).  Per internal node the array holds
// the 7 costs and one word of choices: bits 0-2 the left child's share of
// the wide node's 8 slots, bits 3(i-1)..3(i-1)+2 for i = 2..7 the left share
// of i slots (0: cost(n, i-1) is no worse, use fewer).
constexpr int kDpWords = 8;

struct DpCost {
    float c[7];
};

__device__ __forceinline__ DpCost dp_leaf(float area, float c_prim)
{
    DpCost r;
#pragma unroll
    for (int i = 0; i < 7; ++i) r.c[i] = area * c_prim;
    return r;
}

__device__ __forceinline__ DpCost dp_combine(const DpCost& l, const DpCost& r, float area, int size, float c_node,
                                             float c_prim, uint32_t& choice)
{
    float dist[9];
    int dk[9];
#pragma unroll
    for (int j = 2; j <= 8; ++j) {
        float best = __builtin_inff();
        int bk = 1;
#pragma unroll
        for (int k = 1; k < j; ++k) {
            if (k > 7 || j - k > 7) continue;
            const float v = l.c[k - 1] + r.c[j - k - 1];
            if (v < best) {
                best = v;
                bk = k;
            }
        }
        dist[j] = best;
        dk[j] = bk;
    }
    DpCost out;
    out.c[0] = size <= kLeafMax ? area * (float)size * c_prim : area * c_node + dist[8];
    choice = (uint32_t)dk[8];
#pragma unroll
    for (int i = 2; i <= 7; ++i) {
        if (dist[i] < out.c[i - 2]) {
            out.c[i - 1] = dist[i];
            choice |= (uint32_t)dk[i] << (3 * (i - 1));
        } else {
            out.c[i - 1] = out.c[i - 2];
        }
    }
    return out;
}

// Written and read as agent-scope atomics where a sibling's costs come from
// another thread of the workgroup through global memory.
__device__ __forceinline__ void dp_store(uint32_t* dp, int32_t node, const DpCost& c, uint32_t choice)
{
    uint32_t* d = dp + (int64_t)kDpWords * node;
#pragma unroll
    for (int i = 0; i < 7; ++i)
        __hip_atomic_store(d + i, __float_as_uint(c.c[i]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(d + 7, choice, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------- bounds
__global__ __launch_bounds__(kBlock) void k_centroid_partial(const int32_t* idx, const float* pos,
                                                             int64_t n, float* partial)
{
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kBlock) {
        Box b = tri_box(idx, pos, (int)i);
        for (int k = 0; k < 3; ++k) {
            float c = 0.5f * (b.lo[k] + b.hi[k]);
            lo[k] = fminf(lo[k], c);
            hi[k] = fmaxf(hi[k], c);
        }
    }
    __shared__ float red[6][kBlock];
    for (int k = 0; k < 3; ++k) {
        red[k][threadIdx.x] = lo[k];
        red[3 + k][threadIdx.x] = hi[k];
    }
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            for (int k = 0; k < 3; ++k) {
                red[k][threadIdx.x] = fminf(red[k][threadIdx.x], red[k][threadIdx.x + s]);
                red[3 + k][threadIdx.x] = fmaxf(red[3 + k][threadIdx.x], red[3 + k][threadIdx.x + s]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) partial[blockIdx.x * 6 + threadIdx.x] = red[threadIdx.x][0];
}

// ---------------------------------------------------------------- Morton
__device__ __forceinline__ uint64_t spread3_21(uint32_t v)
{
    uint64_t x = v & 0x1fffffu;
    x = (x | x << 32) & 0x001f00000000ffffull;
    x = (x | x << 16) & 0x001f0000ff0000ffull;
    x = (x | x << 8) & 0x100f00f00f00f00full;
    x = (x | x << 4) & 0x10c30c30c30c30c3ull;
    x = (x | x << 2) & 0x1249249249249249ull;
    return x;
}

// Every block finishes the bounds from the partial boxes (at most kBlock of
// them) itself, which is cheaper than a launch of its own.  Also clears the
// refit's arrival flags and pending counts (n_counts <= n).
__global__ __launch_bounds__(kBlock) void k_morton(const int32_t* idx, const float* pos, int64_t n,
                                                   const float* partial, int nparts, uint64_t* keys, uint32_t* vals,
                                                   uint32_t* flags, uint32_t* pending_counts, int n_counts)
{
    __shared__ float red[6][kBlock];
    for (int k = 0; k < 6; ++k)
        red[k][threadIdx.x] = (int)threadIdx.x < nparts ? partial[threadIdx.x * 6 + k] : (k < 3 ? INFINITY : -INFINITY);
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            for (int k = 0; k < 6; ++k)
                red[k][threadIdx.x] = k < 3 ? fminf(red[k][threadIdx.x], red[k][threadIdx.x + s])
                                            : fmaxf(red[k][threadIdx.x], red[k][threadIdx.x + s]);
        __syncthreads();
    }
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    flags[i] = 0u;
    if (i < n_counts) pending_counts[i] = 0u;
    Box b = tri_box(idx, pos, (int)i);
    uint32_t q[3];
    for (int k = 0; k < 3; ++k) {
        float c = 0.5f * (b.lo[k] + b.hi[k]);
        float ext = red[3 + k][0] - red[k][0];
        float u = ext > 0.0f ? (c - red[k][0]) / ext : 0.0f;
        float s = u * 2097152.0f;  // 2^21
        uint32_t qi = s <= 0.0f ? 0u : (s >= 2097151.0f ? 2097151u : (uint32_t)s);
        q[k] = qi;
    }
    keys[i] = (spread3_21(q[0]) << 2) | (spread3_21(q[1]) << 1) | spread3_21(q[2]);
    vals[i] = (uint32_t)i;
}

// ---------------------------------------------------------------- scan
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v)
{
    const int lane = threadIdx.x & 63;
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

// exclusive scan of kBlock values held one per thread; returns the block total
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t& total)
{
    __shared__ uint32_t wsum[kBlock / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t inc = wave_incl_scan(v);
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    uint32_t off = 0, tot = 0;
    for (int w = 0; w < kBlock / 64; ++w) {
        if (w < wave) off += wsum[w];
        tot += wsum[w];
    }
    __syncthreads();
    total = tot;
    return off + inc - v;
}

// ---------------------------------------------------------------- radix sort
// Per pass: digit counts per tile, one scan per digit over the tiles, a stable
// scatter.  A tile is kBlock * kItems consecutive keys, kItems chosen by the
// key count (build_bvh8): the scatter's rounds are a serial chain, so small
// sorts take short tiles.
template <int kItems>
__global__ __launch_bounds__(kBlock) void k_radix_hist(const uint64_t* keys, int64_t n, int shift,
                                                       uint32_t* counts, int nblocks)
{
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    int64_t base = (int64_t)blockIdx.x * kBlock * kItems;
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
        int64_t i = base + (int64_t)j * kBlock + threadIdx.x;
        if (i < n) atomicAdd(&h[(uint32_t)(keys[i] >> shift) & 255u], 1u);
    }
    __syncthreads();
    counts[(int64_t)threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

// One block per digit: exclusive scan of the digit's tile counts in place, and
// the digit's total (the scatter adds up the smaller digits' totals itself).
__global__ __launch_bounds__(kBlock) void k_radix_scan(uint32_t* counts, int nblocks, uint32_t* totals)
{
    uint32_t* row = counts + (int64_t)blockIdx.x * nblocks;
    uint32_t carry = 0;
    for (int base = 0; base < nblocks; base += kBlock) {
        const int i = base + (int)threadIdx.x;
        const uint32_t v = i < nblocks ? row[i] : 0u;
        uint32_t total;
        const uint32_t off = block_excl_scan(v, total);
        if (i < nblocks) row[i] = carry + off;
        carry += total;
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// Stable scatter.  A wave owns kItems * 64 consecutive keys and ranks them
// round by round against its own digit counts in LDS (lanes with equal digits
// are found with 8 ballots), so the waves meet only once, to add up the
// earlier waves' counts.
template <int kItems>
__global__ __launch_bounds__(kBlock) void k_radix_scatter(const uint64_t* kin, const uint32_t* vin,
                                                          uint64_t* kout, uint32_t* vout, int64_t n,
                                                          int shift, const uint32_t* offsets, int nblocks,
                                                          const uint32_t* totals)
{
    __shared__ uint32_t wcnt[kBlock / 64][256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint32_t all;
    const uint32_t first = block_excl_scan(totals[tid], all) + offsets[(int64_t)tid * nblocks + blockIdx.x];
    for (int w = 0; w < kBlock / 64; ++w) wcnt[w][tid] = 0;
    __syncthreads();
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int64_t base = (int64_t)blockIdx.x * kBlock * kItems + (int64_t)wave * 64 * kItems + lane;
    uint64_t key[kItems];
    uint32_t val[kItems], rank[kItems];
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const int64_t i = base + r * 64;
        key[r] = i < n ? kin[i] : 0ull;
        val[r] = i < n ? vin[i] : 0u;
    }
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        const bool valid = base + r * 64 < n;
        const uint32_t d = (uint32_t)(key[r] >> shift) & 255u;
        uint64_t peers = __ballot(valid);
        for (int b = 0; b < 8; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bb = __ballot(bit);
            peers &= bit ? bb : ~bb;
        }
        const uint32_t below = (uint32_t)__popcll(peers & lt);
        // the wave's LDS operations run in order: all lanes read the count
        // before its first peer moves it on
        const uint32_t before = wcnt[wave][d];
        rank[r] = before + below;
        __builtin_amdgcn_wave_barrier();
        if (valid && below == 0) wcnt[wave][d] = before + (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    uint32_t at = first;
    for (int w = 0; w < kBlock / 64; ++w) {
        const uint32_t c = wcnt[w][tid];
        wcnt[w][tid] = at;
        at += c;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kItems; ++r) {
        if (base + r * 64 < n) {
            const uint32_t to = wcnt[wave][(uint32_t)(key[r] >> shift) & 255u] + rank[r];
            kout[to] = key[r];
            vout[to] = val[r];
        }
    }
}

// All passes in one workgroup, which spares a small build 24 launches.  The same
// stable passes: wave w owns the w-th part of the keys, ranks them as
// k_radix_scatter does, and the keys move in LDS.  8192 keys are what its registers
// and LDS hold, and where the gain has shrunk: a pass of one workgroup takes 1 us
// and 1 us per 1000 keys.  Build time in launches / in one workgroup, us: 100
// triangles 162 / 99, 1000 189 / 127, 2000 243 / 181, 4000 262 / 204, 6000 269 /
// 227, 8192 281 / 249.
constexpr int kSmallThreads = 1024;
constexpr int kSmallItems = 8;  // most keys per thread
constexpr int kSmallSort = kSmallThreads * kSmallItems;

__global__ __launch_bounds__(kSmallThreads) void k_sort_small(uint64_t* keys, uint32_t* vals, int n)
{
    constexpr int kWaves = kSmallThreads / 64;
    __shared__ uint64_t skey[kSmallSort];
    __shared__ uint32_t sval[kSmallSort];
    __shared__ uint16_t cnt[kWaves][256];  // positions stay below 2^16
    __shared__ uint32_t wsum[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int rounds = (n + kSmallThreads - 1) / kSmallThreads;
    const int base = wave * 64 * rounds + lane;
    uint64_t key[kSmallItems];
    uint32_t val[kSmallItems], rank[kSmallItems];
#pragma unroll
    for (int r = 0; r < kSmallItems; ++r) {
        const bool valid = r < rounds && base + r * 64 < n;
        key[r] = valid ? keys[base + r * 64] : 0ull;
        val[r] = valid ? vals[base + r * 64] : 0u;
    }
    for (int shift = 0; shift < 64; shift += 8) {
        for (int k = tid; k < kWaves * 128; k += kSmallThreads) reinterpret_cast<uint32_t*>(cnt)[k] = 0u;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kSmallItems; ++r) {
            if (r >= rounds) break;
            const bool valid = base + r * 64 < n;
            const uint32_t d = (uint32_t)(key[r] >> shift) & 255u;
            uint64_t peers = __ballot(valid);
            for (int b = 0; b < 8; ++b) {
                const bool bit = (d >> b) & 1u;
                const uint64_t bb = __ballot(bit);
                peers &= bit ? bb : ~bb;
            }
            const uint32_t below = (uint32_t)__popcll(peers & lt);
            const uint32_t before = cnt[wave][d];
            rank[r] = before + below;
            __builtin_amdgcn_wave_barrier();
            if (valid && below == 0) cnt[wave][d] = (uint16_t)(before + (uint32_t)__popcll(peers));
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        // digit tid: its keys in all waves, then where each wave's begin
        uint32_t total = 0;
        if (tid < 256) {
            for (int w = 0; w < kWaves; ++w) total += cnt[w][tid];
            const uint32_t inc = wave_incl_scan(total);
            if (lane == 63) wsum[wave] = inc;
            total = inc - total;
        }
        __syncthreads();
        if (tid < 256) {
            uint32_t at = total;
            for (int w = 0; w < wave; ++w) at += wsum[w];
            for (int w = 0; w < kWaves; ++w) {
                const uint32_t c = cnt[w][tid];
                cnt[w][tid] = (uint16_t)at;
                at += c;
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kSmallItems; ++r) {
            if (r < rounds && base + r * 64 < n) {
                const uint32_t to = cnt[wave][(uint32_t)(key[r] >> shift) & 255u] + rank[r];
                skey[to] = key[r];
                sval[to] = val[r];
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kSmallItems; ++r) {
            if (r < rounds && base + r * 64 < n) {
                key[r] = skey[base + r * 64];
                val[r] = sval[base + r * 64];
            }
        }
    }
#pragma unroll
    for (int r = 0; r < kSmallItems; ++r) {
        if (r < rounds && base + r * 64 < n) {
            keys[base + r * 64] = key[r];
            vals[base + r * 64] = val[r];
        }
    }
}

// ---------------------------------------------------------------- radix tree
__device__ __forceinline__ int common_prefix(const uint64_t* k, int64_t n, int64_t i, int64_t j)
{
    if (j < 0 || j >= n) return -1;
    uint64_t a = k[i], b = k[j];
    if (a == b) return 64 + __clz((uint32_t)(i ^ j));
    return __clzll(a ^ b);
}

// Levels of the collapse, sizes on the device: level l has `tasks` wide nodes,
// whose nodes start at node_base and records at tri_base.  The emit kernel of
// level l fills in level l + 1.
struct Level {
    uint32_t tasks, node_base, tri_base, reserved;
};
constexpr int kMaxLevels = 128;         // a binary radix tree is at most 63 + 31 levels deep

// child encoding: >= 0 internal node index, < 0 leaf ~index (sorted order).
// Also sets up the collapse's first level: one task, the root.
__global__ __launch_bounds__(kBlock) void k_radix_tree(const uint64_t* keys, int64_t n, int32_t* left,
                                                       int32_t* right, int32_t* first, int32_t* last,
                                                       int32_t* iparent, int32_t* lparent,
                                                       Level* levels, Level* summary, int32_t* tasks)
{
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n - 1) return;
    int d = (common_prefix(keys, n, i, i + 1) - common_prefix(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = common_prefix(keys, n, i, i - d);
    int64_t lmax = 2;
    while (common_prefix(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int64_t l = 0;
    for (int64_t t = lmax >> 1; t >= 1; t >>= 1)
        if (common_prefix(keys, n, i, i + (l + t) * d) > dmin) l += t;
    int64_t j = i + l * d;
    int dnode = common_prefix(keys, n, i, j);
    int64_t s = 0;
    int64_t t = l;
    do {
        t = (t + 1) >> 1;
        if (common_prefix(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    int64_t gamma = i + s * d + (d < 0 ? -1 : 0);
    int64_t lo = i < j ? i : j, hi = i < j ? j : i;
    int32_t lc = (lo == gamma) ? ~(int32_t)gamma : (int32_t)gamma;
    int32_t rc = (hi == gamma + 1) ? ~(int32_t)(gamma + 1) : (int32_t)(gamma + 1);
    left[i] = lc;
    right[i] = rc;
    first[i] = (int32_t)lo;
    last[i] = (int32_t)hi;
    if (lc >= 0) iparent[lc] = (int32_t)i; else lparent[~lc] = (int32_t)i;
    if (rc >= 0) iparent[rc] = (int32_t)i; else lparent[~rc] = (int32_t)i;
    if (i == 0) {
        iparent[0] = -1;
        levels[0] = Level{1u, 0u, 0u, 0u};
        *summary = Level{1u, 0u, 0u, 0u};
        tasks[0] = 0;
    }
}

__device__ __forceinline__ float ld_coherent(const float* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_coherent(float* p, float v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ Box child_box(int32_t c, const uint32_t* sorted, const int32_t* idx,
                                         const float* pos, const float* ibox)
{
    if (c < 0) return tri_box(idx, pos, (int)sorted[~c]);
    Box b;
    for (int k = 0; k < 3; ++k) {
        b.lo[k] = ld_coherent(ibox + 6 * (int64_t)c + k);
        b.hi[k] = ld_coherent(ibox + 6 * (int64_t)c + 3 + k);
    }
    return b;
}

__device__ __forceinline__ DpCost child_cost(int32_t c, const Box& cb, const uint32_t* dp, float c_prim)
{
    if (c < 0) return dp_leaf(box_half_area(cb), c_prim);
    DpCost r;
#pragma unroll
    for (int i = 0; i < 7; ++i)
        r.c[i] = __uint_as_float(__hip_atomic_load(dp + (int64_t)kDpWords * c + i, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT));
    return r;
}

// Refit in phases over ever larger tiles of sorted leaves.  Phase 0: one
// workgroup per tile of kRefitTile leaves, one thread per leaf, finishes every
// internal node whose leaf range lies inside the tile.  A Karras node's index
// is one end of its range, so those nodes have indices inside the tile too,
// and everything a climb reads (children, parents, boxes, costs, arrival
// flags) lives in LDS: a level costs LDS round trips instead of four dependent
// global ones.  1024 leaves take 91 KB.  A climb that reaches a node crossing
// the tile border waits in the pending list of the tile of the next phase,
// kRefitFan times as large, whose workgroup goes on from there through global
// memory, until one tile holds all leaves.  Threads of a workgroup see each
// other's results through workgroup fences; device-scope ones would write back
// and invalidate the L2s at every node.
// 1.3 M triangles: phase 0 136 us, the two above 220 us (one phase over
// 4096-leaf tiles with costs in global memory 511 us, the rest with
// device-scope fences 171 us; the rest in a single workgroup 1367 us); 16 M:
// 1473 + 379 us.
constexpr int kRefitTile = 1024;
constexpr int kRefitFan = 32;

__global__ __launch_bounds__(kRefitTile) void k_refit_local(
    int64_t n, const uint32_t* sorted, const int32_t* idx, const float* pos, const int32_t* left,
    const int32_t* right, const int32_t* first, const int32_t* last, const int32_t* iparent,
    const int32_t* lparent, float* ibox, int32_t* pending, uint32_t* pending_count, uint32_t* dp, float c_node,
    float c_prim)
{
    // the pending list of this tile's next larger tile: completed subtrees are
    // disjoint, so a tile of m leaves has at most m of them
    pending += (int64_t)(blockIdx.x / kRefitFan) * ((int64_t)kRefitTile * kRefitFan);
    pending_count += blockIdx.x / kRefitFan;
    __shared__ float leaf_box[6][kRefitTile], node_box[6][kRefitTile], node_cost[7][kRefitTile];
    // parent: -2 where the node crosses the tile border
    __shared__ int32_t node_left[kRefitTile], node_right[kRefitTile], node_parent[kRefitTile];
    __shared__ uint32_t flag[kRefitTile];
    const int64_t lo = (int64_t)blockIdx.x * kRefitTile;
    const int64_t hi = (lo + kRefitTile < n ? lo + kRefitTile : n) - 1;
    const int t = threadIdx.x;
    const int64_t j = lo + t;
    flag[t] = 0u;
    if (j < n - 1) {
        const bool inside = first[j] >= lo && last[j] <= hi;
        node_left[t] = left[j];
        node_right[t] = right[j];
        node_parent[t] = inside ? iparent[j] : -2;
    }
    Box b;
    if (j <= hi) {
        b = tri_box(idx, pos, (int)sorted[j]);
        for (int a = 0; a < 3; ++a) {
            leaf_box[a][t] = b.lo[a];
            leaf_box[3 + a][t] = b.hi[a];
        }
    }
    __syncthreads();
    if (j > hi) return;
    int32_t cur = ~(int32_t)j;
    int size = 1;
    DpCost cur_cost = dp_leaf(box_half_area(b), c_prim);
    int32_t p = lparent[j];
    while (p >= 0) {
        // a parent inside the tile has its index inside it; one outside may too
        const int s = (int)(p - lo);
        if (p < lo || p > hi || node_parent[s] == -2) {
            pending[atomicAdd(pending_count, 1u)] = p;
            break;
        }
        __threadfence_block();
        if (atomicAdd(&flag[s], (uint32_t)size) == 0u) break;
        __threadfence_block();
        const int32_t l = node_left[s], r = node_right[s];
        const bool cur_left = l == cur;
        const int32_t sib = cur_left ? r : l;
        size = (int)flag[s];  // both children's leaves
        Box o;
        DpCost sib_cost;
        if (sib < 0) {
            const int q = (int)((int64_t)~sib - lo);
            for (int a = 0; a < 3; ++a) {
                o.lo[a] = leaf_box[a][q];
                o.hi[a] = leaf_box[3 + a][q];
            }
            sib_cost = dp_leaf(box_half_area(o), c_prim);
        } else {
            const int q = (int)(sib - lo);
            for (int a = 0; a < 3; ++a) {
                o.lo[a] = node_box[a][q];
                o.hi[a] = node_box[3 + a][q];
            }
#pragma unroll
            for (int i = 0; i < 7; ++i) sib_cost.c[i] = node_cost[i][q];
        }
        for (int a = 0; a < 3; ++a) {
            b.lo[a] = fminf(b.lo[a], o.lo[a]);
            b.hi[a] = fmaxf(b.hi[a], o.hi[a]);
            node_box[a][s] = b.lo[a];
            node_box[3 + a][s] = b.hi[a];
            ibox[6 * (int64_t)p + a] = b.lo[a];
            ibox[6 * (int64_t)p + 3 + a] = b.hi[a];
        }
        if (dp) {
            uint32_t choice;
            const float area = box_half_area(b);
            cur_cost = cur_left ? dp_combine(cur_cost, sib_cost, area, size, c_node, c_prim, choice)
                                : dp_combine(sib_cost, cur_cost, area, size, c_node, c_prim, choice);
#pragma unroll
            for (int i = 0; i < 7; ++i) node_cost[i][s] = cur_cost.c[i];
            uint4* d = reinterpret_cast<uint4*>(dp + (int64_t)kDpWords * p);
            d[0] = make_uint4(__float_as_uint(cur_cost.c[0]), __float_as_uint(cur_cost.c[1]),
                              __float_as_uint(cur_cost.c[2]), __float_as_uint(cur_cost.c[3]));
            d[1] = make_uint4(__float_as_uint(cur_cost.c[4]), __float_as_uint(cur_cost.c[5]),
                              __float_as_uint(cur_cost.c[6]), choice);
        }
        cur = p;
        p = node_parent[s];
    }
}

constexpr int kCrossThreads = 512;

// One phase above phase 0: tile blockIdx.x of `tile` leaves.
__global__ __launch_bounds__(kCrossThreads) void k_refit_crossing(
    int64_t n, int64_t tile, const int32_t* pending_in, const uint32_t* count_in, int32_t* pending_out,
    uint32_t* count_out, const uint32_t* sorted, const int32_t* idx, const float* pos, const int32_t* left,
    const int32_t* right, const int32_t* first, const int32_t* last, const int32_t* iparent, float* ibox,
    uint32_t* flags, uint32_t* dp, float c_node, float c_prim)
{
    const int64_t lo = (int64_t)blockIdx.x * tile;
    const int64_t hi = (lo + tile < n ? lo + tile : n) - 1;
    pending_in += lo;
    const uint32_t count = count_in[blockIdx.x];
    pending_out += (int64_t)(blockIdx.x / kRefitFan) * (tile * kRefitFan);
    count_out += blockIdx.x / kRefitFan;
    for (uint32_t k = threadIdx.x; k < count; k += kCrossThreads) {
        int32_t p = pending_in[k];
        while (p >= 0) {
            const int32_t f = first[p], e = last[p], l = left[p], r = right[p], up = iparent[p];
            if (f < lo || e > hi) {
                pending_out[atomicAdd(count_out, 1u)] = p;
                break;
            }
            __threadfence_block();
            // the first of a node's two arrivals leaves it to the second
            if (atomicAdd(&flags[p], 1u) == 0u) break;
            __threadfence_block();
            Box a = child_box(l, sorted, idx, pos, ibox);
            Box b = child_box(r, sorted, idx, pos, ibox);
            Box u;
            for (int c = 0; c < 3; ++c) {
                u.lo[c] = fminf(a.lo[c], b.lo[c]);
                u.hi[c] = fmaxf(a.hi[c], b.hi[c]);
                st_coherent(ibox + 6 * (int64_t)p + c, u.lo[c]);
                st_coherent(ibox + 6 * (int64_t)p + 3 + c, u.hi[c]);
            }
            if (dp) {
                uint32_t choice;
                const DpCost c = dp_combine(child_cost(l, a, dp, c_prim), child_cost(r, b, dp, c_prim),
                                            box_half_area(u), e - f + 1, c_node, c_prim, choice);
                dp_store(dp, p, c, choice);
            }
            p = up;
        }
    }
}

// ---------------------------------------------------------------- collapse
__device__ __forceinline__ float half_area(const float* b)
{
    float dx = b[3] - b[0], dy = b[4] - b[1], dz = b[5] - b[2];
    return dx * dy + dy * dz + dz * dx;
}

constexpr int kTaskBlock = 1024;        // threads of a collapse block: 8 lanes per task
constexpr int kBlockTasks = kTaskBlock / 8;

// Exclusive prefix of v over the block's tasks (the same v in a task's 8
// lanes); total over the block.
__device__ __forceinline__ uint32_t task_excl_scan(uint32_t v, uint32_t& total)
{
    __shared__ uint32_t wsum[kTaskBlock / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t inc = v;
    for (int o = 8; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
    }
    if (lane == 63) wsum[wave] = inc;
    __syncthreads();
    uint32_t off = 0, tot = 0;
    for (int w = 0; w < kTaskBlock / 64; ++w) {
        if (w < wave) off += wsum[w];
        tot += wsum[w];
    }
    __syncthreads();
    total = tot;
    return off + inc - v;
}

// Slots of each task's wide node.  Lane k of a task walks from the task's
// binary node to the part of the cost choices' 8-slot budget that position k
// falls in: a node with budget j owns positions [a, a + j), its left child the
// first of them.  The walk ends at a slot, owned by the lane at its first
// position; the owners in order are the slots.  Per task: the 8 slots and the
// counts of internal children (low half) and leaf triangles (high half),
// prefixed within the block; per block their sums.
__global__ __launch_bounds__(kTaskBlock) void k_collapse_plan(const Level* level, const int32_t* tasks,
                                                              const int32_t* left, const int32_t* right,
                                                              const int32_t* first, const int32_t* last,
                                                              const float* ibox, const uint32_t* dp,
                                                              int32_t* slots, uint32_t* task_prefix,
                                                              uint32_t* block_sum)
{
    const uint32_t ntasks = level->tasks;
    if (blockIdx.x * (uint32_t)kBlockTasks >= ntasks) return;
    const uint32_t t = blockIdx.x * (uint32_t)kBlockTasks + threadIdx.x / 8;
    const int k = threadIdx.x & 7;
    const int shift = threadIdx.x & 56;     // first lane of the task in its wave
    const bool valid = t < ntasks;
    int32_t c = kEmptySlot;
    bool owner = false;
    if (valid && dp) {
        c = tasks[t];
        int a = 0, j = 8;
        bool root = true;
        for (;;) {
            if (c < 0) break;
            const uint32_t ch = dp[(int64_t)kDpWords * c + 7];
            int kl;
            if (root) {
                kl = (int)(ch & 7u);
                root = false;
            } else {
                while (j > 1 && ((ch >> (3 * (j - 1))) & 7u) == 0u) --j;
                if (j == 1) break;
                kl = (int)((ch >> (3 * (j - 1))) & 7u);
            }
            if (k < a + kl) {
                c = left[c];
                j = kl;
            } else {
                c = right[c];
                a += kl;
                j -= kl;
            }
        }
        owner = k == a;
    } else if (valid) {
        // greedy: every lane of the task follows the same openings
        int32_t s[8];
        const int32_t b = tasks[t];
        s[0] = left[b];
        s[1] = right[b];
        int ns = 2;
        while (ns < 8) {
            int best = -1;
            float best_a = -1.0f;
            for (int q = 0; q < ns; ++q) {
                if (s[q] >= 0) {
                    float a = half_area(ibox + 6 * (int64_t)s[q]);
                    if (a > best_a) { best_a = a; best = q; }
                }
            }
            if (best < 0) break;
            const int32_t o = s[best];
            s[best] = left[o];
            s[ns++] = right[o];
        }
        owner = k < ns;
        if (owner) c = s[k];
    }
    const uint32_t owners = (uint32_t)(__ballot(owner) >> shift) & 0xffu;
    int size = 0;
    if (owner) size = c < 0 ? 1 : last[c] - first[c] + 1;
    const bool inner = owner && size > kLeafMax;
    const uint32_t leaf = owner && !inner ? (uint32_t)size : 0u;
    const uint32_t m_int = (uint32_t)(__ballot(inner) >> shift) & 0xffu;
    const uint32_t m_l1 = (uint32_t)(__ballot(leaf & 1u) >> shift) & 0xffu;
    const uint32_t m_l2 = (uint32_t)(__ballot(leaf & 2u) >> shift) & 0xffu;
    const uint32_t packed = (uint32_t)__popc(m_int) | ((uint32_t)(__popc(m_l1) + 2 * __popc(m_l2)) << 16);
    if (valid) {
        // owners in order, then the empty slots
        const uint32_t below = (1u << k) - 1u;
        const int at = owner ? __popc(owners & below) : __popc(owners) + __popc(~owners & 0xffu & below);
        slots[8 * (int64_t)t + at] = owner ? c : kEmptySlot;
    }
    uint32_t total;
    const uint32_t prefix = task_excl_scan(valid ? packed : 0u, total);
    if (valid && k == 0) task_prefix[t] = prefix;
    if (threadIdx.x == 0) block_sum[blockIdx.x] = total;
}

__device__ __forceinline__ void write_record(int64_t rec, int tri, const int32_t* idx, const float* pos,
                                             float* tris, int32_t* prim_ids)
{
    for (int v = 0; v < 3; ++v) {
        int vi = idx[3 * tri + v];
        tris[9 * rec + 3 * v + 0] = pos[3 * vi + 0];
        tris[9 * rec + 3 * v + 1] = pos[3 * vi + 1];
        tris[9 * rec + 3 * v + 2] = pos[3 * vi + 2];
    }
    prim_ids[rec] = tri;
}

// smallest e with 255 * 2^e >= extent (e >= -126); exact in double
__device__ __forceinline__ int quant_exponent(double extent)
{
    if (!(extent > 0.0)) return -126;
    int e = ilogb(extent) - 7;
    while (ldexp(255.0, e) < extent) ++e;
    while (e > -126 && ldexp(255.0, e - 1) >= extent) --e;
    return e < -126 ? -126 : e;
}

// Writes each task's node, leaf records and next-level tasks, one lane per
// slot.  The counts before this block come from the block sums, added up here
// (a level has at most n / 4 tasks, so a few thousand sums).
__global__ __launch_bounds__(kTaskBlock) void k_collapse_emit(
    Level* level, Level* summary, const int32_t* tasks, const int32_t* slots, const uint32_t* task_prefix,
    const uint32_t* block_sum, const int32_t* first, const int32_t* last, const float* ibox, const uint32_t* sorted,
    const int32_t* idx, const float* pos, Bvh8Node* nodes, float* tris, int32_t* prim_ids, int32_t* next_tasks)
{
    const Level lv = level[0];
    const uint32_t nblocks = (lv.tasks + kBlockTasks - 1) / kBlockTasks;
    if (blockIdx.x != 0 && blockIdx.x >= nblocks) return;
    // sums of the blocks before this one, and of all blocks (block 0 only)
    __shared__ uint32_t part[2][kTaskBlock / 64];
    const uint32_t upto = blockIdx.x == 0 ? nblocks : blockIdx.x;
    uint32_t si = 0, st = 0;
    for (uint32_t q = threadIdx.x; q < upto; q += kTaskBlock) {
        const uint32_t v = block_sum[q];
        si += v & 0xffffu;
        st += v >> 16;
    }
    for (int o = 32; o > 0; o >>= 1) {
        si += __shfl_down(si, o, 64);
        st += __shfl_down(st, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        part[0][threadIdx.x >> 6] = si;
        part[1][threadIdx.x >> 6] = st;
    }
    __syncthreads();
    uint32_t int_before = 0, tri_before = 0;
    for (int w = 0; w < kTaskBlock / 64; ++w) {
        int_before += part[0][w];
        tri_before += part[1][w];
    }
    const uint32_t next_base = lv.node_base + lv.tasks;
    if (blockIdx.x == 0) {
        if (threadIdx.x == 0) {
            level[1] = Level{int_before, next_base, lv.tri_base + tri_before, 0u};
            if (lv.tasks) *summary = Level{int_before, next_base, lv.tri_base + tri_before, summary->reserved + 1u};
        }
        int_before = tri_before = 0;
    }
    const uint32_t t = blockIdx.x * (uint32_t)kBlockTasks + threadIdx.x / 8;
    if (t >= lv.tasks) return;
    const int k = threadIdx.x & 7;
    const int shift = threadIdx.x & 56;
    const uint32_t prefix = task_prefix[t];
    const uint32_t my_int = int_before + (prefix & 0xffffu);
    const uint32_t child_base = next_base + my_int;
    const uint32_t tri_base = lv.tri_base + tri_before + (prefix >> 16);

    const int32_t b = tasks[t];
    const int32_t c = slots[8 * (int64_t)t + k];
    const bool used = c != kEmptySlot;
    const float* nb = ibox + 6 * (int64_t)b;
    Box cb{};
    int f = 0, size = 0;
    if (used && c < 0) {
        f = ~c;
        size = 1;
        cb = tri_box(idx, pos, (int)sorted[f]);
    } else if (used) {
        f = first[c];
        size = last[c] - f + 1;
        for (int a = 0; a < 3; ++a) {
            cb.lo[a] = ibox[6 * (int64_t)c + a];
            cb.hi[a] = ibox[6 * (int64_t)c + 3 + a];
        }
    }
    const bool inner = used && size > kLeafMax;
    const uint32_t leaf = used && !inner ? (uint32_t)size : 0u;
    const uint32_t below = (1u << k) - 1u;
    const uint32_t m_int = (uint32_t)(__ballot(inner) >> shift) & 0xffu;
    const uint32_t m_l1 = (uint32_t)(__ballot(leaf & 1u) >> shift) & 0xffu;
    const uint32_t m_l2 = (uint32_t)(__ballot(leaf & 2u) >> shift) & 0xffu;
    const uint32_t toff = (uint32_t)(__popc(m_l1 & below) + 2 * __popc(m_l2 & below));

    // the node's byte planes, one byte per lane and plane
    uint8_t* out = reinterpret_cast<uint8_t*>(nodes + lv.node_base + t);
    int e[3];
    for (int a = 0; a < 3; ++a) {
        e[a] = quant_exponent((double)nb[3 + a] - (double)nb[a]);
        uint8_t ql = 255, qh = 0;       // empty slots carry inverted boxes
        if (used) {
            const double inv_scale = ldexp(1.0, -e[a]), p = (double)nb[a];
            double lo = floor(((double)cb.lo[a] - p) * inv_scale);
            double hi = ceil(((double)cb.hi[a] - p) * inv_scale);
            lo = lo < 0.0 ? 0.0 : (lo > 255.0 ? 255.0 : lo);
            hi = hi < 0.0 ? 0.0 : (hi > 255.0 ? 255.0 : hi);
            ql = (uint8_t)lo;
            qh = (uint8_t)hi;
        }
        out[offsetof(Bvh8Node, qlo_x) + 8 * a + k] = ql;
        out[offsetof(Bvh8Node, qhi_x) + 8 * a + k] = qh;
    }
    out[offsetof(Bvh8Node, meta) + k] = (uint8_t)(leaf ? (leaf << 5) | toff : 0u);
    if (k == 0) {
        const uint32_t exps = (uint32_t)(uint8_t)(int8_t)e[0] | (uint32_t)(uint8_t)(int8_t)e[1] << 8 |
                              (uint32_t)(uint8_t)(int8_t)e[2] << 16 | m_int << 24;
        *reinterpret_cast<uint4*>(out) =
            make_uint4(__float_as_uint(nb[0]), __float_as_uint(nb[1]), __float_as_uint(nb[2]), exps);
        *reinterpret_cast<uint2*>(out + 16) = make_uint2(child_base, tri_base);
    }
    if (inner) {
        next_tasks[my_int + __popc(m_int & below)] = c;
    } else {
        for (uint32_t q = 0; q < leaf; ++q)
            write_record((int64_t)tri_base + toff + q, (int)sorted[f + q], idx, pos, tris, prim_ids);
    }
}

// ---------------------------------------------------------------- host side
inline int blocks_for(int64_t n, int per) { return (int)((n + per - 1) / per); }

// The build's scratch: slices of one allocation, 256-byte aligned.  Counted
// first (base null), then handed out.
struct Arena {
    char* base = nullptr;
    size_t used = 0;
    template <class T> T* take(int64_t count)
    {
        T* p = reinterpret_cast<T*>(base + used);
        used += ((size_t)std::max<int64_t>(count, 1) * sizeof(T) + 255) & ~(size_t)255;
        return p;
    }
};

struct Scratch {
    uint64_t* keys[2];
    uint32_t* vals[2];
    uint32_t *counts, *totals;
    float* partial;
    int32_t *left, *right, *first, *last, *iparent, *lparent, *pending[2];
    float* ibox;
    uint32_t *flags, *pending_counts, *dp;
    int32_t *tasks[2], *slots;
    uint32_t *task_prefix, *block_sum;
    Level* levels;   // kMaxLevels + 2, then the summary
};

// Keys per thread of a sort tile: a short chain of rounds for small sorts,
// fewer tiles to scan for large ones.  Build time with 4 / 16: 8 k triangles
// 0.282 / 0.327 ms, 500 k 0.611 / 0.646, 1.3 M 0.989 / 0.995, 16 M 8.42 / 7.83.
inline int sort_items(int64_t n) { return n <= (1 << 20) ? 4 : 16; }

// Tiles of all refit phases above phase 0, one pending count each.
int64_t refit_tiles(int64_t n)
{
    int64_t sum = 0;
    for (int64_t tile = (int64_t)kRefitTile * kRefitFan;; tile *= kRefitFan) {
        const int64_t t = (n + tile - 1) / tile;
        sum += t;
        if (t == 1) return sum + 1;  // and the (unused) list above the last
    }
}

Scratch take_scratch(Arena& a, int64_t n, bool sah)
{
    Scratch s{};
    const int64_t ni = std::max<int64_t>(1, n - 1);
    const int64_t tiles = blocks_for(n, kBlock * sort_items(n));
    // tasks of one level: disjoint subtrees of more than kLeafMax triangles
    const int64_t max_tasks = n / (kLeafMax + 1) + 1;
    for (int k = 0; k < 2; ++k) {
        s.keys[k] = a.take<uint64_t>(n);
        s.vals[k] = a.take<uint32_t>(n);
        s.tasks[k] = a.take<int32_t>(max_tasks);
    }
    s.counts = a.take<uint32_t>(256 * tiles);
    s.totals = a.take<uint32_t>(256);
    s.partial = a.take<float>(6 * kBlock);
    s.left = a.take<int32_t>(ni);
    s.right = a.take<int32_t>(ni);
    s.first = a.take<int32_t>(ni);
    s.last = a.take<int32_t>(ni);
    s.iparent = a.take<int32_t>(ni);
    s.lparent = a.take<int32_t>(n);
    for (int k = 0; k < 2; ++k) s.pending[k] = a.take<int32_t>(n);
    s.pending_counts = a.take<uint32_t>(refit_tiles(n));
    s.ibox = a.take<float>(6 * ni);
    s.flags = a.take<uint32_t>(n);
    if (sah) s.dp = a.take<uint32_t>(kDpWords * ni);
    s.slots = a.take<int32_t>(8 * max_tasks);
    s.task_prefix = a.take<uint32_t>(max_tasks);
    s.block_sum = a.take<uint32_t>(max_tasks / kBlockTasks + 1);
    s.levels = a.take<Level>(kMaxLevels + 3);
    return s;
}

template <int kItems>
void sort_pass(const Scratch& w, int cur, int64_t n, int shift, hipStream_t s)
{
    const int tiles = blocks_for(n, kBlock * kItems);
    k_radix_hist<kItems><<<tiles, kBlock, 0, s>>>(w.keys[cur], n, shift, w.counts, tiles);
    k_radix_scan<<<256, kBlock, 0, s>>>(w.counts, tiles, w.totals);
    k_radix_scatter<kItems><<<tiles, kBlock, 0, s>>>(w.keys[cur], w.vals[cur], w.keys[1 - cur], w.vals[1 - cur], n,
                                                     shift, w.counts, tiles, w.totals);
}

}  // namespace

int build_bvh8(prt_hip_ctx* ctx, SceneBuffers& sb, prt_build_stats* stats)
{
    const int64_t n = sb.tri_count;
    hipStream_t s = ctx->stream;
    if (n <= 0) return set_error(ctx, "bvh_build: scene has no triangles");
    if (n >= (int64_t)1 << 31) return set_error(ctx, "bvh_build: more than 2^31-1 triangles");

    sb.bvh_ready = false;
    const int64_t max_nodes = std::max<int64_t>(1, n - 1);
    // the last build's buffers serve again if they have room and are not over
    // four times too large
    if (!sb.d_nodes || n > sb.bvh_cap || sb.bvh_cap > std::max<int64_t>(4 * n, 1 << 18)) {
        if (sb.d_nodes) (void)hipFree(sb.d_nodes);
        if (sb.d_tris) (void)hipFree(sb.d_tris);
        if (sb.d_prim_ids) (void)hipFree(sb.d_prim_ids);
        sb.d_nodes = nullptr;
        sb.d_tris = nullptr;
        sb.d_prim_ids = nullptr;
        sb.bvh_cap = 0;
        PRT_TRY(ctx, device_alloc(ctx, &sb.d_nodes, sizeof(Bvh8Node) * max_nodes));
        PRT_TRY(ctx, device_alloc(ctx, &sb.d_tris, sizeof(float) * 9 * n));
        PRT_TRY(ctx, device_alloc(ctx, &sb.d_prim_ids, sizeof(int32_t) * n));
        sb.bvh_cap = n;
    }

    const bool sah = ctx->bvh_collapse == PRT_COLLAPSE_SAH;
    Arena arena;
    take_scratch(arena, n, sah);
    if (arena.used > ctx->build_bytes) {
        if (ctx->d_build) (void)hipFree(ctx->d_build);
        ctx->d_build = nullptr;
        ctx->build_bytes = 0;
        PRT_TRY(ctx, device_alloc(ctx, &ctx->d_build, arena.used));
        ctx->build_bytes = arena.used;
    }
    arena = Arena{static_cast<char*>(ctx->d_build), 0};
    const Scratch w = take_scratch(arena, n, sah);

    PRT_TRY(ctx, hipEventRecord(ctx->ev0, s));

    if (n == 1) {
        // one triangle: a root whose single leaf slot holds it
        Bvh8Node root{};
        std::vector<int32_t> idx(3);
        std::vector<float> pos;
        PRT_TRY(ctx, hipMemcpyAsync(idx.data(), sb.d_idx, 12, hipMemcpyDeviceToHost, s));
        PRT_TRY(ctx, hipStreamSynchronize(s));
        pos.resize(9);
        for (int v = 0; v < 3; ++v)
            PRT_TRY(ctx, hipMemcpyAsync(&pos[3 * v], sb.d_pos + 3 * (int64_t)idx[v], 12,
                                        hipMemcpyDeviceToHost, s));
        PRT_TRY(ctx, hipStreamSynchronize(s));
        float lo[3], hi[3];
        for (int a = 0; a < 3; ++a) {
            lo[a] = std::min(std::min(pos[a], pos[3 + a]), pos[6 + a]);
            hi[a] = std::max(std::max(pos[a], pos[3 + a]), pos[6 + a]);
        }
        root.px = lo[0]; root.py = lo[1]; root.pz = lo[2];
        uint8_t* ql[3] = {root.qlo_x, root.qlo_y, root.qlo_z};
        uint8_t* qh[3] = {root.qhi_x, root.qhi_y, root.qhi_z};
        uint8_t* ex[3] = {&root.ex, &root.ey, &root.ez};
        for (int a = 0; a < 3; ++a) {
            double extent = (double)hi[a] - (double)lo[a];
            int e = -126;
            if (extent > 0.0) {
                e = std::ilogb(extent) - 7;
                while (std::ldexp(255.0, e) < extent) ++e;
                while (e > -126 && std::ldexp(255.0, e - 1) >= extent) --e;
            }
            *ex[a] = (uint8_t)(int8_t)e;
            for (int k = 0; k < 8; ++k) { ql[a][k] = 255; qh[a][k] = 0; }
            ql[a][0] = 0;
            qh[a][0] = (uint8_t)std::min(255.0, std::ceil(extent * std::ldexp(1.0, -e)));
        }
        root.meta[0] = (uint8_t)(1u << 5);
        root.child_base = 1;
        root.tri_base = 0;
        int32_t zero = 0;
        PRT_TRY(ctx, hipMemcpyAsync(sb.d_nodes, &root, sizeof(root), hipMemcpyHostToDevice, s));
        PRT_TRY(ctx, hipMemcpyAsync(sb.d_tris, pos.data(), 36, hipMemcpyHostToDevice, s));
        PRT_TRY(ctx, hipMemcpyAsync(sb.d_prim_ids, &zero, 4, hipMemcpyHostToDevice, s));
        sb.node_count = 1;
        sb.bvh_depth = 1;
    } else {
        const int nred = std::min(blocks_for(n, kBlock), kBlock);
        k_centroid_partial<<<nred, kBlock, 0, s>>>(sb.d_idx, sb.d_pos, n, w.partial);
        k_morton<<<blocks_for(n, kBlock), kBlock, 0, s>>>(sb.d_idx, sb.d_pos, n, w.partial, nred, w.keys[0],
                                                          w.vals[0], w.flags, w.pending_counts,
                                                          (int)std::min<int64_t>(n, refit_tiles(n)));
        int cur = 0;
        if (n <= kSmallSort) k_sort_small<<<1, kSmallThreads, 0, s>>>(w.keys[0], w.vals[0], (int)n);
        for (int shift = 0; n > kSmallSort && shift < 64; shift += 8) {
            if (sort_items(n) == 4) sort_pass<4>(w, cur, n, shift, s);
            else sort_pass<16>(w, cur, n, shift, s);
            cur = 1 - cur;
        }
        PRT_TRY(ctx, hipGetLastError());
        const uint32_t* sv = w.vals[cur];
        Level* summary = w.levels + kMaxLevels + 2;
        k_radix_tree<<<blocks_for(n - 1, kBlock), kBlock, 0, s>>>(w.keys[cur], n, w.left, w.right, w.first, w.last,
                                                                  w.iparent, w.lparent, w.levels, summary, w.tasks[0]);
        const float c_node = 1.0f, c_prim = ctx->bvh_prim_cost;
        k_refit_local<<<blocks_for(n, kRefitTile), kRefitTile, 0, s>>>(
            n, sv, sb.d_idx, sb.d_pos, w.left, w.right, w.first, w.last, w.iparent, w.lparent, w.ibox, w.pending[0],
            w.pending_counts, w.dp, c_node, c_prim);
        uint32_t* counts_in = w.pending_counts;
        int from = 0;
        for (int64_t tile = (int64_t)kRefitTile; tile < n; from = 1 - from) {
            tile *= kRefitFan;
            const int64_t tiles = (n + tile - 1) / tile;
            k_refit_crossing<<<(unsigned)tiles, kCrossThreads, 0, s>>>(
                n, tile, w.pending[from], counts_in, w.pending[1 - from], counts_in + tiles, sv, sb.d_idx, sb.d_pos,
                w.left, w.right, w.first, w.last, w.iparent, w.ibox, w.flags, w.dp, c_node, c_prim);
            counts_in += tiles;
        }
        PRT_TRY(ctx, hipGetLastError());

        // collapse: launch the levels a tree of this size is expected to have,
        // then look, then a few at a time.  A level past the last one finds
        // no tasks.  Level l has at most 8^l tasks.
        const int64_t max_tasks = n / (kLeafMax + 1) + 1;
        int expected = 2;
        for (int64_t m = n; m > 3; m /= 4) ++expected;
        Level done{};
        int l = 0;
        for (;;) {
            const int upto = std::min(kMaxLevels, l == 0 ? expected : l + 4);
            for (; l < upto; ++l) {
                const int64_t most = l < 8 ? std::min<int64_t>((int64_t)1 << (3 * l), max_tasks) : max_tasks;
                const int nb = blocks_for(most, kBlockTasks);
                k_collapse_plan<<<nb, kTaskBlock, 0, s>>>(w.levels + l, w.tasks[l & 1], w.left, w.right, w.first,
                                                          w.last, w.ibox, w.dp, w.slots, w.task_prefix, w.block_sum);
                k_collapse_emit<<<nb, kTaskBlock, 0, s>>>(w.levels + l, summary, w.tasks[l & 1], w.slots,
                                                          w.task_prefix, w.block_sum, w.first, w.last, w.ibox, sv,
                                                          sb.d_idx, sb.d_pos, sb.d_nodes, sb.d_tris, sb.d_prim_ids,
                                                          w.tasks[(l + 1) & 1]);
            }
            PRT_TRY(ctx, hipGetLastError());
            PRT_TRY(ctx, hipMemcpyAsync(ctx->h_readback, summary, sizeof(Level), hipMemcpyDeviceToHost, s));
            PRT_TRY(ctx, hipStreamSynchronize(s));
            done = *static_cast<const Level*>(ctx->h_readback);
            if (done.tasks == 0) break;
            if (l == kMaxLevels) return set_error(ctx, "bvh_build: tree too deep");
        }
        const int64_t node_base = done.node_base, tri_base = done.tri_base;
        const int depth = (int)done.reserved;
        if (tri_base != n) return set_error(ctx, "bvh_build: triangle records do not cover the scene");
        sb.node_count = node_base;
        sb.bvh_depth = depth;
    }

    PRT_TRY(ctx, hipEventRecord(ctx->ev1, s));
    PRT_TRY(ctx, hipEventSynchronize(ctx->ev1));
    float ms = 0.0f;
    PRT_TRY(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
    // the scratch stays with the context up to a size that any scene shares
    if (ctx->build_bytes > kBuildKeepBytes) {
        (void)hipFree(ctx->d_build);
        ctx->d_build = nullptr;
        ctx->build_bytes = 0;
    }
    sb.bvh_ready = true;
    if (stats) {
        stats->build_ms = ms;
        stats->build_mprim = ms > 0.0f ? (double)n / 1000.0 / ms : 0.0;
        stats->node_count = sb.node_count;
        stats->tri_count = n;
        stats->depth = sb.bvh_depth;
        stats->reserved = 0;
    }
    return 0;
}

}  // namespace prt
