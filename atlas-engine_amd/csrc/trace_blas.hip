// BVH2 traversal kernels over one BLAS, gfx950.
//
// Reference: HitClosest / HitAny in BLAS mode (data/shader/raytracer/bvh.hsh:244-267,
// 411-433), launched one ray per invocation by traceClosest.csh:12-36.
//
// The engine-exact binary kernels without a register-topped stack (closest and
// any hit) run on the filtered walk of walk.h, in two launch shapes chosen by
// launch_walk: one group per batch of rays, or a resident grid that pulls
// chunks of 64 rays (its rules stand there).  The autotuner's other candidates
// (register-topped stack, float slab, wide nodes) and the visit counters keep
// the per-lane step functions of trace_core.h:
//  * grid: one ray per lane, the whole batch in one grid (the engine's shape);
//  * persistent: a resident grid of waves pulls rays from a global counter.
//    Whenever fewer than `refill` lanes of a wave are still traversing, the
//    idle lanes are refilled with new rays (ballot + popcount give each idle
//    lane its index from one atomicAdd per wave), so divergent incoherent
//    rays do not leave most of a wave idle.  The last wave to finish resets
//    the counter, so consecutive launches need no host-side reset.
// The stack lives in LDS rows [depth][lane] (bank-conflict free since lanes
// at different depths still sit in different banks) and spills to a global
// array sized from the tree depth.  Results equal the engine's bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <type_traits>

#include "rt_internal.h"
#include "trace_core.h"
#include "walk.h"

namespace atlas_rt {

namespace {

constexpr int kWave = 64;
// 400 - 800 measured the same on 1M - 4M incoherent rays, 200 and 1600 slower.
constexpr uint32_t kIdleSteps = 400;

template <int BLOCK, int LDS_DEPTH, bool STATS, int NODE_W = 2, bool REG = false, bool FLOAT_SLAB = false>
__global__ __launch_bounds__(BLOCK) void k_blas_closest(BlasDev B, const float4* __restrict__ rays,
                                                        float4* __restrict__ hits, int32_t* __restrict__ slots,
                                                        uint2* __restrict__ visits, uint32_t count,
                                                        int32_t* __restrict__ spill, uint32_t cap,
                                                        uint32_t* __restrict__ ctl) {
    __shared__ int32_t lds[LDS_DEPTH * BLOCK];
    const uint32_t gid = blockIdx.x * BLOCK + threadIdx.x;
    if (gid >= count) return;
    const float4 r0 = rays[2 * size_t(gid)];
    const float4 r1 = rays[2 * size_t(gid) + 1];
    LaneState L;
    L.slot = -1;
    uint32_t n_nodes = 0, n_tris = 0;
    if (!any_nan3(r1.x, r1.y, r1.z)) {
        lane_begin(L, B, r0, r1, NODE_W > 2);
        const LaneStack<BLOCK, LDS_DEPTH> S{lds, spill, threadIdx.x, gid, gridDim.x * BLOCK};
        int r;
        do {
            r = step_variant<NODE_W, REG, BLOCK, LDS_DEPTH, STATS, FLOAT_SLAB>(B, L, S, cap, n_nodes, n_tris);
        } while (r == kContinue);
        if (r == kOverflow) {
            atomicOr(&ctl[2], 1u);
            L.slot = -1;
        }
    }
    hits[gid] = lane_hit_record(B, L, r1.w);
    if (slots) slots[gid] = L.slot;
    if (STATS) visits[gid] = make_uint2(n_nodes, n_tris);
}

// LEAF_DIV > 0: leaf-batched waves (wave_step).
template <int BLOCK, int LDS_DEPTH, int NODE_W = 2, bool REG = false, bool FLOAT_SLAB = false, int LEAF_DIV = 0>
__global__ __launch_bounds__(BLOCK) void k_blas_closest_persistent(BlasDev B, const float4* __restrict__ rays,
                                                                   float4* __restrict__ hits,
                                                                   int32_t* __restrict__ slots, uint32_t count,
                                                                   int32_t* __restrict__ spill, uint32_t cap,
                                                                   uint32_t* __restrict__ ctl, uint32_t refill) {
    __shared__ int32_t lds[LDS_DEPTH * BLOCK];
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const LaneStack<BLOCK, LDS_DEPTH> S{lds, spill, threadIdx.x, blockIdx.x * BLOCK + threadIdx.x, gridDim.x * BLOCK};
    LaneState L;
    L.slot = -1;
    bool active = false;
    bool exhausted = false;
    uint32_t idx = 0;
    float tmax = 0.0f;
    bool pending = false;  // the lane's ray has ended; its hit record is not written yet
    RangePull rp;  // rays from kPullRanges ranges, counters ctl[kRangeWord * (r + 1)]
    rp.init(count);
    for (;;) {
        // The hit records of the rays that ended since the last refill, all
        // at once: the FP64 refinement (refine_tuv) then runs once per refill
        // round instead of in every traversal iteration in which some lane
        // of the wave ended its ray.
        if (pending) {
            hits[idx] = lane_hit_record(B, L, tmax);
            if (slots) slots[idx] = L.slot;
            pending = false;
        }
        if (!exhausted) {
            const uint64_t idle = __ballot(!active);
            if (idle) {
                const uint32_t n = __popcll(idle);
                uint32_t base = 0, end = 0;
                if (lane == 0) rp.take(ctl + kRangeWord, kRangeWord, count, n, base, end);
                base = __shfl(base, 0);
                end = __shfl(end, 0);
                rp.broadcast(0);
                if (rp.dry >= kPullRanges) exhausted = true;
                if (!active) {
                    idx = base + __popcll(idle & ((1ull << lane) - 1));
                    if (idx < end) {
                        const float4 r0 = rays[2 * size_t(idx)];
                        const float4 r1 = rays[2 * size_t(idx) + 1];
                        tmax = r1.w;
                        if (any_nan3(r1.x, r1.y, r1.z)) {
                            hits[idx] = make_float4(tmax, 0.0f, 0.0f, __int_as_float(-1));
                            if (slots) slots[idx] = -1;
                        } else {
                            lane_begin(L, B, r0, r1, NODE_W > 2);
                            active = true;
                        }
                    }
                }
            }
        }
        if (!__any(active)) {
            if (exhausted) break;
            continue;
        }
        const uint32_t threshold = exhausted ? 1u : refill;
        for (;;) {
            const int r = wave_step<NODE_W, REG, BLOCK, LDS_DEPTH, FLOAT_SLAB, LEAF_DIV>(B, L, S, cap, active);
            if (r != kContinue) {
                if (r == kOverflow) {
                    atomicOr(&ctl[2], 1u);
                    L.slot = -1;
                }
                pending = true;
                active = false;
            }
            if (uint32_t(__popcll(__ballot(active))) < threshold) break;
        }
    }
    // Every wave has taken its last ray; the last one out resets the counters.
    // Its atomics need no fence: a wave's adds to the counters have returned
    // before it adds to ctl[1] (and a device-scope fence writes back the L2,
    // once per wave).
    if (lane == 0) {
        const uint32_t waves = gridDim.x * (BLOCK / kWave);
        if (atomicAdd(&ctl[1], 1u) == waves - 1) {
            for (uint32_t r = 0; r < kPullRanges; r++) atomicExch(&ctl[kRangeWord * (r + 1)], 0u);
            atomicExch(&ctl[1], 0u);
        }
    }
}

// Words of the flag block that the walk kernels use: the chunk counters of
// ChunkPull, and whether the launch's rays were found coherent.
constexpr uint32_t kChunkWord = 8;  // sequence r's at word kRangeWord * (r + 1) + kChunkWord
constexpr uint32_t kCoherentWord = 3;

// Chunks of 64 rays in a launch of `count` (not 0) rays, up to 2^32 - 1.
__device__ __forceinline__ uint32_t chunks_of(uint32_t count) { return (count - 1) / 64u + 1; }

// Whether the wave's rays start and run close together: most lanes within a
// few degrees of the lane beside them, and within a sixteenth of the tree's
// box.
__device__ __forceinline__ bool coherent_rays(const BlasDev& B, bool valid, float4 r0, float4 r1) {
    if (!B.node_count) return true;
    const float4 a = ldg4(B.nodes), b = ldg4(B.nodes + 1), c = ldg4(B.nodes + 2);
    const float reach = 0.0625f * fmaxf(fmaxf(fmaxf(a.w, c.y) - fminf(a.x, b.z), fmaxf(b.x, c.z) - fminf(a.y, b.w)),
                                        fmaxf(b.y, c.w) - fminf(a.z, c.x));
    const auto beside = [](float v) {
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1 /* quad_perm 1 0 3 2 */, 0xf, 0xf, true));
    };
    const float nx = beside(r1.x), ny = beside(r1.y), nz = beside(r1.z);
    const float dot = r1.x * nx + r1.y * ny + r1.z * nz;
    const float dd = (r1.x * r1.x + r1.y * r1.y + r1.z * r1.z) * (nx * nx + ny * ny + nz * nz);
    const float gap = fmaxf(fmaxf(fabsf(r0.x - beside(r0.x)), fabsf(r0.y - beside(r0.y))), fabsf(r0.z - beside(r0.z)));
    // a NaN direction ends at once: it may run anywhere
    const bool apart = dot < 0.0f || dot * dot < 0.94f * dd || gap > reach;
    return uint32_t(__popcll(mask_of(valid && apart))) * 4 < uint32_t(__popcll(mask_of(valid)));
}

// Before a walk of resident waves: clears their chunk counters and, with
// `choose`, samples 64 chunks of 64 rays over the batch and notes whether
// most of them are coherent.
constexpr uint32_t kBeginBlock = 1024;
__global__ __launch_bounds__(kBeginBlock) void k_walk_begin(BlasDev B, const float4* __restrict__ rays, uint32_t count,
                                                            uint32_t* __restrict__ ctl, bool choose) {
    __shared__ uint32_t coherent;
    const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    if (tid < kPullRanges) ctl[kRangeWord * (tid + 1) + kChunkWord] = 0;
    if (!choose) return;
    if (tid == 0) coherent = 0;
    __syncthreads();
    constexpr uint32_t kWaves = kBeginBlock / kWave, kEach = 64 / kWaves;
    const uint32_t chunks = chunks_of(count);
    uint32_t found = 0;
    for (uint32_t i = 0; i < kEach; i++) {
        const uint32_t k = uint32_t(uint64_t(wave * kEach + i) * chunks / 64u) * 64u + lane;
        const bool valid = k < count;
        float4 r0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), r1 = r0;
        if (valid) {
            r0 = rays[2 * size_t(k)];
            r1 = rays[2 * size_t(k) + 1];
        }
        found += coherent_rays(B, valid, r0, r1) ? 1u : 0u;
    }
    if (lane == 0 && found) atomicAdd(&coherent, found);
    __syncthreads();
    if (tid == 0) ctl[kCoherentWord] = coherent * 2 >= 64u ? 1u : 0u;
}

// Engine-order binary walks (walk.h), by shape:
//   kOnce   one set of `per_wave` rays per wave;
//   kPull   resident waves take chunks of 64 rays and refill their idle lanes
//           from them.
// chosen: run only if k_walk_begin found the rays coherent (kOnce) or not
// (kPull); a large batch launches both.  Coherent rays share their nodes'
// cache lines and end together: a wave per chunk, started in the rays' order
// by the hardware, loads each node once for many lanes and balances best
// (kernel time of 1920 x 1080 camera rays over 1.0M triangles: 0.26 ms against
// 0.39 resident).  Incoherent rays end one by one, so lanes are refilled, and their
// node records go through LDS (NodeStage) while there is work; the last rays,
// few in each wave, load their nodes directly (1M rays in a random soup of
// 65,536 triangles: 0.62 ms against 0.90 once).
//
// When to refill.  A wave waits until its idle lanes have cost kIdleSteps
// lane-steps since its last refill, about what a refill costs.  The rays of a
// refill load beside the hit records of the rays they replace.
enum class Shape { kOnce, kPull };

template <int BLOCK, int ROWS, int OWN, bool ANY, Shape SHAPE, int LEAF_DIV>
__global__ __launch_bounds__(BLOCK, SHAPE == Shape::kPull && ROWS > 14 ? 3 : 5) void k_blas_walk(BlasDev B, const float4* __restrict__ rays,
                                                        void* __restrict__ out, int32_t* __restrict__ slots,
                                                        uint32_t count, int32_t* __restrict__ spill, uint32_t cap,
                                                        uint32_t* __restrict__ ctl, uint32_t per_wave, bool chosen) {
    constexpr bool kPulls = SHAPE == Shape::kPull;
    if (chosen && (ctl[kCoherentWord] != 0) == kPulls) return;
    __shared__ int32_t lds[ROWS * BLOCK];
    __shared__ __align__(16) char staged[kPulls ? (BLOCK / kWave) * NodeStage::kBytes : 16];
    const NodeStage stage(staged);
    using Stack = WalkStack<BLOCK, ROWS, OWN>;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    int32_t own[OWN ? OWN : 1];
    const Stack S(lds, own, spill, blockIdx.x * BLOCK + threadIdx.x, gridDim.x * BLOCK, cap);
    constexpr uint32_t kNone = 0xFFFFFFFFu;
    Walk w;
    w.node = kEnd;
    uint32_t idx = kNone;  // the lane's ray, until its result is written
    float tmax = 0.0f;
    ChunkPull pull;
    uint32_t from = 0, to = 0;   // rays this wave holds and has not started
    if (kPulls) {
        pull.init();
    } else {
        from = (blockIdx.x * (BLOCK / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave)) * per_wave;
        to = min(count, from + per_wave);
    }
    for (;;) {
        if (kPulls && from >= to && !pull.dry) {
            uint32_t chunk;
            if (pull.take(ctl + kRangeWord + kChunkWord, kRangeWord, chunks_of(count), chunk)) {
                from = chunk * 64u;
                to = from + min(64u, count - from);
            }
        }
        const uint64_t idle = mask_of(w.node == kEnd);
        const uint32_t k = from + __popcll(idle & ((1ull << lane) - 1));
        const bool start = w.node == kEnd && k < to;
        float4 r0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), r1 = r0;
        if (start) {
            r0 = rays[2 * size_t(k)];
            r1 = rays[2 * size_t(k) + 1];
        }
        from += uint32_t(__popcll(mask_of(start)));
        // The results of the rays that ended since the last refill, all at
        // once: the FP64 refinement runs once per refill round.
        if (w.node == kEnd && idx != kNone) {
            if (ANY) {
                reinterpret_cast<uint32_t*>(out)[idx] = w.slot >= 0 ? 1u : 0u;
            } else {
                reinterpret_cast<float4*>(out)[idx] = walk_hit_record(w, B.tris, B.vtx, tmax);
                if (slots) slots[idx] = w.slot;
            }
            idx = kNone;
        }
        if (start) {
            idx = k;
            tmax = r1.w;
            walk_begin(w, B.node_count, r0, r1, Stack::bottom(threadIdx.x));
            if (any_nan3(r1.x, r1.y, r1.z)) w.node = kEnd;
        }
        const bool more = from < to || (kPulls && !pull.dry);
        if (!more && mask_of(idx != kNone) == 0) break;
        const auto walk = [&](auto through_lds) {
            uint32_t wasted = 0;
            uint64_t live = mask_of(w.node != kEnd);
            while (live != 0 && wasted <= kIdleSteps) {
                // node steps until enough lanes wait at a leaf
                uint64_t inner = mask_of(w.node >= 0);
                while (LEAF_DIV ? uint32_t(__popcll(live ^ inner)) * LEAF_DIV < uint32_t(__popcll(live)) : inner != 0) {
                    int32_t below = 0;
                    bool checked = false;
                    if (through_lds) {
                        if (w.node >= 0) checked = walk_stack(w, S, below);
                        stage.fetch(B.nodes, w.node, inner);
                    }
                    if (w.node >= 0) {
                        if (through_lds)
                            stage.wait();
                        else
                            checked = walk_stack(w, S, below);
                        const NodeRec n = through_lds ? stage.read() : load_node(B.nodes, w.node);
                        const uint64_t over = walk_node(w, n, checked, below, S, ANY ? ~0ull : 0ull);
                        if (__builtin_expect(over != 0, 0)) {
                            atomicOr(&ctl[2], 1u);
                            if (lane_in(over)) w.slot = -1;
                        }
                    }
                    if (more) wasted += kWave - uint32_t(__popcll(live));
                    live = mask_of(w.node != kEnd);
                    inner = mask_of(w.node >= 0);
                    if (LEAF_DIV == 0 || wasted > kIdleSteps) break;
                }
                if (w.node < 0 && w.node != kEnd) walk_leaf(w, B.tris, S, ANY);
                live = mask_of(w.node != kEnd);
            }
        };
        if (kPulls && more)
            walk(std::true_type{});
        else
            walk(std::false_type{});
    }
}

constexpr int kBlock = 128;
constexpr int kLdsDepth = 32;
constexpr int kPBlock = 256;
constexpr int kPLdsDepth = 24;

BlasDev blas_dev(const atlas_rt_blas& b) {
    BlasDev d;
    d.nodes = b.d_nodes;
    d.tris = b.d_tris;
    d.vtx = b.d_vtx;
    d.nodes4 = b.d_nodes4;
    d.nodes8 = b.d_nodes8;
    d.node_count = uint32_t(b.nodes.size());
    d.tri_count = uint32_t(b.tris.size());
    return d;
}

}  // namespace

int device_cu_count() {
    static int cached = -1;
    if (cached < 0) {
        int dev = 0;
        hipDeviceProp_t p;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess &&
            p.multiProcessorCount > 0)
            cached = p.multiProcessorCount;
        else
            cached = 256;
    }
    return cached;
}

// Leaf batching: triangle steps once a quarter of a wave's live lanes wait at
// a leaf.
constexpr int kLeafDiv = 4;

// The counters and the overflow word, zero between launches.
static atlas_rt_status ensure_flags(atlas_rt_blas& blas) {
    if (blas.flags.ptr) return ATLAS_RT_OK;
    atlas_rt_status st = blas.flags.ensure(kFlagBytes);
    if (st != ATLAS_RT_OK) return st;
    ATLAS_HIP_TRY(hipMemset(blas.flags.ptr, 0, kFlagBytes));
    return ATLAS_RT_OK;
}

constexpr int kWalkBlock = 256;
// LDS stack rows: with the staged nodes, five groups of resident waves fit
// one CU (14 KB + 16.3 KB each); of the waves that run once, as many as the
// registers allow, 20 and, for any hit, 28 (LDS is allocated in pieces of
// 1,280 B: 7,680 and 5,120 B per wave; with 22 rows only 25 waves fit, and
// 877,536 shadow rays over 2.1M triangles take 125 us, not 118).
constexpr int kWalkRows = 14;
template <bool ANY>
constexpr int kOnceRows = ANY ? 20 : 30;
constexpr uint32_t kWalkGroups = 5;

// Launches below this many rays run once, with as many rays per wave as give
// every CU eight waves: a wave's step takes as long as its slowest lane's
// memory access, and all of its lanes' accesses after one another (5,003 rays
// 0.111 -> 0.093 ms, 16,384 rays 0.194 -> 0.166 ms against 64 per wave).
constexpr uint32_t kChooseRays = 65536;
inline uint32_t rays_per_wave(uint32_t count) { return std::min(64u, (count - 1) / 2048u + 1); }

// Whether any-hit rays may be worth refilling.  Their walks are short, and the
// shorter the smaller the tree, so that refills cost more than the idle lanes
// do until there are many rays.  Incoherent rays, refilled / once, us: 1,500
// triangles 91 / 43 at 131,072 rays, 575 / 591 at 4 M; 5,000: 330 / 283 at 1 M,
// 481 / 526 at 2 M; 20,011: 270 / 177 at 300,000, 330 / 320 at 600,000, 434 /
// 502 at 1 M; 65,536: 347 / 297 at 300,000, 441 / 523 at 600,000.
inline bool pays_any(uint32_t count, uint32_t nodes) {
    return uint64_t(count) * std::min(nodes, 16384u) >= uint64_t(1) << 33;
}

struct WalkArgs {
    BlasDev B;
    const float4* rays;
    void* out;
    int32_t* slots;
    uint32_t count;
    int32_t* spill;
    uint32_t cap;
    uint32_t* ctl;
    hipStream_t stream;
};

// Without own stack rows where the tree is shallow enough: a kernel that has
// scratch memory takes 0.2 to 0.4 us longer to launch (37 rays on 1,024
// triangles: 24.1 us, not 23.9; launches of 36.8 us: 37.3).
template <bool ANY>
static void walk_once(const WalkArgs& a, uint32_t groups, uint32_t per_wave, bool chosen) {
    const auto launch = [&](auto own) {
        hipLaunchKernelGGL((k_blas_walk<64, kOnceRows<ANY>, decltype(own)::value, ANY, Shape::kOnce, 0>), dim3(groups),
                           dim3(64), 0, a.stream, a.B, a.rays, a.out, a.slots, a.count, a.spill, a.cap, a.ctl, per_wave,
                           chosen);
    };
    if (a.cap < uint32_t(kOnceRows<ANY>))
        launch(std::integral_constant<int, 0>{});
    else
        launch(std::integral_constant<int, kOwnRows>{});
}

template <bool ANY, int ROWS = kWalkRows, int OWN = kOwnRows>
static void walk_pull(const WalkArgs& a, bool leaf_batch, uint32_t groups, bool chosen) {
    if (leaf_batch)
        hipLaunchKernelGGL((k_blas_walk<kWalkBlock, ROWS, OWN, ANY, Shape::kPull, kLeafDiv>), dim3(groups), dim3(kWalkBlock),
                           0, a.stream, a.B, a.rays, a.out, a.slots, a.count, a.spill, a.cap, a.ctl, 64u, chosen);
    else
        hipLaunchKernelGGL((k_blas_walk<kWalkBlock, ROWS, OWN, ANY, Shape::kPull, 0>), dim3(groups), dim3(kWalkBlock), 0,
                           a.stream, a.B, a.rays, a.out, a.slots, a.count, a.spill, a.cap, a.ctl, 64u, chosen);
}

static void walk_begin_launch(const WalkArgs& a, bool choose) {
    hipLaunchKernelGGL(k_walk_begin, dim3(1), dim3(kBeginBlock), 0, a.stream, a.B, a.rays, a.count, a.ctl, choose);
}

enum class WalkPlan { kAuto, kOnce, kPull, kPullLeafBatch };

template <bool ANY>
static atlas_rt_status launch_walk(atlas_rt_blas& blas, const TraceLaunch& L, WalkPlan plan) {
    const uint32_t cap = limit_cap(blas.max_depth + 1, blas.stack_limit);
    // a tree so deep that a wave per 64 rays would need spill rows keeps to the
    // resident shape, whose lanes are fewer than a large batch's rays; so do
    // more rays than a grid can have threads
    const bool deep = walk_spill_bytes(cap, kOnceRows<ANY> + kOwnRows, 1) != 0;
    const bool large = plan == WalkPlan::kAuto && L.count >= kChooseRays &&
                       (!ANY || deep || pays_any(L.count, uint32_t(blas.nodes.size())));
    const bool choose = large && L.count <= UINT32_MAX - 63 && !deep;
    const bool pull = large || plan == WalkPlan::kPull || plan == WalkPlan::kPullLeafBatch;
    const bool once = choose || !pull;
    const uint32_t per_wave = once && !choose && plan == WalkPlan::kAuto ? rays_per_wave(L.count) : 64u;
    const uint32_t once_groups = (L.count - 1) / per_wave + 1;
    const uint32_t pull_groups = uint32_t(device_cu_count()) * kWalkGroups;
    const size_t spill_bytes =
        std::max(once ? walk_spill_bytes(cap, kOnceRows<ANY> + kOwnRows, size_t(once_groups) * 64) : 0,
                 pull ? walk_spill_bytes(cap, kWalkRows + kOwnRows, size_t(pull_groups) * kWalkBlock) : 0);
    atlas_rt_status st = ATLAS_RT_OK;
    if (spill_bytes) st = blas.spill.ensure(spill_bytes);
    if (st == ATLAS_RT_OK) st = ensure_flags(blas);
    if (st == ATLAS_RT_OK) st = blas.timing.begin(L.stream);
    if (st != ATLAS_RT_OK) return st;
    const WalkArgs a{blas_dev(blas),
                     reinterpret_cast<const float4*>(L.rays),
                     L.hits,
                     L.slots,
                     L.count,
                     reinterpret_cast<int32_t*>(blas.spill.ptr),
                     cap,
                     reinterpret_cast<uint32_t*>(blas.flags.ptr),
                     L.stream};
    if (pull) walk_begin_launch(a, choose);
    if (once) walk_once<ANY>(a, once_groups, per_wave, choose);
    if (pull) walk_pull<ANY>(a, plan != WalkPlan::kPull, pull_groups, choose);
    ATLAS_HIP_TRY(hipGetLastError());
    return blas.timing.end(L.stream);
}

static atlas_rt_status prepare(atlas_rt_blas& blas, uint32_t threads, uint32_t lds_depth, uint32_t& cap,
                               int node_w = 2) {
    // The binary stack never holds more entries than the deepest leaf's
    // depth; the wide bounds come from the collapse.
    cap = limit_cap(variant_cap(node_w, blas.max_depth + 1, blas.cap4, blas.cap8), blas.stack_limit);
    if (cap > lds_depth) {
        const size_t need = size_t(cap - lds_depth) * threads * sizeof(int32_t);
        atlas_rt_status st = blas.spill.ensure(need);
        if (st != ATLAS_RT_OK) return st;
    }
    return ensure_flags(blas);
}

template <int NODE_W, bool REG, bool FLOAT_SLAB = false, int LEAF_DIV = 0>
static void launch_persistent(const BlasDev& B, const TraceLaunch& L, uint32_t groups, int32_t* spill, uint32_t cap,
                              uint32_t* ctl) {
    hipLaunchKernelGGL((k_blas_closest_persistent<kPBlock, kPLdsDepth, NODE_W, REG, FLOAT_SLAB, LEAF_DIV>), dim3(groups),
                       dim3(kPBlock), 0,
                       L.stream, B, reinterpret_cast<const float4*>(L.rays), reinterpret_cast<float4*>(L.hits),
                       L.slots, L.count, spill, cap, ctl, L.refill ? L.refill : 40u);
}

atlas_rt_status launch_blas_closest(atlas_rt_blas& blas, const TraceLaunch& L) {
    if (L.count == 0) return ATLAS_RT_OK;
    const BlasDev B = blas_dev(blas);
    uint32_t* ctl = reinterpret_cast<uint32_t*>(blas.flags.ptr);
    const int base = L.kernel & ATLAS_RT_KERNEL_VARIANT_MASK;
    const bool reg = (L.kernel & ATLAS_RT_KERNEL_STACK_REGISTER) != 0;
    const bool fslab = (L.kernel & ATLAS_RT_KERNEL_SLAB_FLOAT) != 0;
    const bool leaf_batch = (L.kernel & ATLAS_RT_KERNEL_LEAF_BATCH) != 0;
    const bool persistent = !L.visits && base >= ATLAS_RT_KERNEL_BVH2_PERSISTENT;
    if (!L.visits && !reg && !fslab && base <= ATLAS_RT_KERNEL_BVH2_PERSISTENT)
        return launch_walk<false>(blas, L,
                                  base == ATLAS_RT_KERNEL_AUTO ? WalkPlan::kAuto
                                  : !persistent                ? WalkPlan::kOnce
                                  : leaf_batch                 ? WalkPlan::kPullLeafBatch
                                                               : WalkPlan::kPull);
    const int node_w = base == ATLAS_RT_KERNEL_BVH4 ? 4 : (base == ATLAS_RT_KERNEL_BVH8 ? 8 : 2);
    atlas_rt_status st;
    uint32_t cap = 0;
    if (persistent) {
        // Resident grid: four 256-lane groups per CU (fewer resident waves
        // keep more of the tree in each XCD's L2).
        const uint32_t groups = uint32_t(device_cu_count()) * 4u;
        st = prepare(blas, groups * kPBlock, kPLdsDepth, cap, node_w);
        if (st != ATLAS_RT_OK) return st;
        ctl = reinterpret_cast<uint32_t*>(blas.flags.ptr);
        st = blas.timing.begin(L.stream);
        if (st != ATLAS_RT_OK) return st;
        int32_t* spill = reinterpret_cast<int32_t*>(blas.spill.ptr);
        if (node_w == 2 && leaf_batch) {
            if (fslab)
                reg ? launch_persistent<2, true, true, kLeafDiv>(B, L, groups, spill, cap, ctl)
                    : launch_persistent<2, false, true, kLeafDiv>(B, L, groups, spill, cap, ctl);
            else
                launch_persistent<2, true, false, kLeafDiv>(B, L, groups, spill, cap, ctl);
        } else if (node_w == 2 && fslab)
            reg ? launch_persistent<2, true, true>(B, L, groups, spill, cap, ctl)
                : launch_persistent<2, false, true>(B, L, groups, spill, cap, ctl);
        else if (node_w == 2)
            launch_persistent<2, true>(B, L, groups, spill, cap, ctl);
        else if (node_w == 4 && leaf_batch && fslab)
            reg ? launch_persistent<4, true, true, kLeafDiv>(B, L, groups, spill, cap, ctl)
                : launch_persistent<4, false, true, kLeafDiv>(B, L, groups, spill, cap, ctl);
        else if (node_w == 4 && leaf_batch)
            reg ? launch_persistent<4, true, false, kLeafDiv>(B, L, groups, spill, cap, ctl)
                : launch_persistent<4, false, false, kLeafDiv>(B, L, groups, spill, cap, ctl);
        else if (node_w == 4 && fslab)
            reg ? launch_persistent<4, true, true>(B, L, groups, spill, cap, ctl)
                : launch_persistent<4, false, true>(B, L, groups, spill, cap, ctl);
        else if (node_w == 4)
            reg ? launch_persistent<4, true>(B, L, groups, spill, cap, ctl)
                : launch_persistent<4, false>(B, L, groups, spill, cap, ctl);
        else
            reg ? launch_persistent<8, true>(B, L, groups, spill, cap, ctl)
                : launch_persistent<8, false>(B, L, groups, spill, cap, ctl);
    } else if ((reg || fslab) && !L.visits) {
        const uint32_t grid = (L.count + kBlock - 1) / kBlock;
        st = prepare(blas, grid * kBlock, kLdsDepth, cap);
        if (st != ATLAS_RT_OK) return st;
        ctl = reinterpret_cast<uint32_t*>(blas.flags.ptr);
        st = blas.timing.begin(L.stream);
        if (st != ATLAS_RT_OK) return st;
        const auto* rays = reinterpret_cast<const float4*>(L.rays);
        auto* hits = reinterpret_cast<float4*>(L.hits);
        int32_t* spill = reinterpret_cast<int32_t*>(blas.spill.ptr);
        if (reg && fslab)
            hipLaunchKernelGGL((k_blas_closest<kBlock, kLdsDepth, false, 2, true, true>), dim3(grid), dim3(kBlock), 0,
                               L.stream, B, rays, hits, L.slots, nullptr, L.count, spill, cap, ctl);
        else if (reg)
            hipLaunchKernelGGL((k_blas_closest<kBlock, kLdsDepth, false, 2, true>), dim3(grid), dim3(kBlock), 0,
                               L.stream, B, rays, hits, L.slots, nullptr, L.count, spill, cap, ctl);
        else
            hipLaunchKernelGGL((k_blas_closest<kBlock, kLdsDepth, false, 2, false, true>), dim3(grid), dim3(kBlock), 0,
                               L.stream, B, rays, hits, L.slots, nullptr, L.count, spill, cap, ctl);
    } else {
        const uint32_t grid = (L.count + kBlock - 1) / kBlock;
        st = prepare(blas, grid * kBlock, kLdsDepth, cap);
        if (st != ATLAS_RT_OK) return st;
        ctl = reinterpret_cast<uint32_t*>(blas.flags.ptr);
        st = blas.timing.begin(L.stream);
        if (st != ATLAS_RT_OK) return st;
        hipLaunchKernelGGL((k_blas_closest<kBlock, kLdsDepth, true>), dim3(grid), dim3(kBlock), 0, L.stream, B,
                           reinterpret_cast<const float4*>(L.rays), reinterpret_cast<float4*>(L.hits), L.slots,
                           reinterpret_cast<uint2*>(L.visits), L.count, reinterpret_cast<int32_t*>(blas.spill.ptr),
                           cap, ctl);
    }
    ATLAS_HIP_TRY(hipGetLastError());
    return blas.timing.end(L.stream);
}

// ---------------------------------------------------------------------------
// Closest hit without allocation: the persistent kernels' counters, overflow
// flag and stack spill live in one file-scope device array instead of the
// BLAS's scratch, so a trace never calls hipMalloc.  Every call on a device
// shares that device's copy; calls that overlap on one device race.
// ---------------------------------------------------------------------------
namespace {

constexpr size_t kNoAllocCtlBytes = 2048;
static_assert(kFlagBytes <= kNoAllocCtlBytes, "the flag block fits the control bytes");
constexpr size_t kNoAllocSpillBytes = size_t(16) << 20;

__device__ __align__(256) uint8_t scratch[kNoAllocCtlBytes + kNoAllocSpillBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The device address of the current device's `scratch`, looked up once per
// device with that device current.
atlas_rt_status scratch_address(void** out) {
    int dev = 0;
    ATLAS_HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(ATLAS_RT_E_UNSUPPORTED, "no-alloc trace: device index out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
        if (!p) return fail(ATLAS_RT_E_HIP, "hipGetSymbolAddress(scratch) returned NULL");
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return ATLAS_RT_OK;
}

__global__ void k_zero_words(uint32_t* __restrict__ w, uint32_t n) {
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) w[i] = 0u;
}

}  // namespace

atlas_rt_status launch_blas_closest_noalloc(const atlas_rt_blas& blas, const TraceLaunch& L0) {
    TraceLaunch L = L0;
    if (L.kernel == ATLAS_RT_KERNEL_AUTO) L.kernel = ATLAS_RT_KERNEL_BVH2_PERSISTENT | ATLAS_RT_KERNEL_LEAF_BATCH;
    const int base = L.kernel & ATLAS_RT_KERNEL_VARIANT_MASK;
    if (base != ATLAS_RT_KERNEL_BVH2_PERSISTENT)
        return fail(ATLAS_RT_E_UNSUPPORTED, "atlas_rt_trace_closest_rays_noalloc: only the binary persistent kernels "
                                            "(ATLAS_RT_KERNEL_BVH2_PERSISTENT with the register-stack, float-slab and "
                                            "leaf-batch bits, or AUTO)");
    void* sp = nullptr;
    atlas_rt_status st = scratch_address(&sp);
    if (st != ATLAS_RT_OK) return st;
    if (L.count == 0) return ATLAS_RT_OK;
    const uint32_t groups = uint32_t(device_cu_count()) * 4;
    const size_t lanes = size_t(groups) * kPBlock;
    const uint32_t cap = limit_cap(blas.max_depth + 1, blas.stack_limit);
    const size_t max_cap = kPLdsDepth + kNoAllocSpillBytes / (lanes * sizeof(int32_t));
    if (cap > max_cap)
        return fail(ATLAS_RT_E_STACK_OVERFLOW, "atlas_rt_trace_closest_rays_noalloc: the tree needs " +
                                                   std::to_string(cap) + " stack entries per ray; the fixed scratch "
                                                   "holds " + std::to_string(max_cap) +
                                                   " (use atlas_rt_trace_closest_rays)");
    uint32_t* ctl = reinterpret_cast<uint32_t*>(sp);
    int32_t* spill = reinterpret_cast<int32_t*>(static_cast<uint8_t*>(sp) + kNoAllocCtlBytes);
    // the counters and the overflow flag start at zero
    hipLaunchKernelGGL(k_zero_words, dim3(1), dim3(256), 0, L.stream, ctl, uint32_t(kNoAllocCtlBytes / 4));
    const BlasDev B = blas_dev(blas);
    const bool reg = (L.kernel & ATLAS_RT_KERNEL_STACK_REGISTER) != 0;
    const bool fslab = (L.kernel & ATLAS_RT_KERNEL_SLAB_FLOAT) != 0;
    const bool leaf_batch = (L.kernel & ATLAS_RT_KERNEL_LEAF_BATCH) != 0;
    if (!reg && !fslab) {
        // 24 stack rows leave room for three groups per CU; their spill rows
        // (one more than the persistent kernels' above) fit the scratch
        const WalkArgs a{B,      reinterpret_cast<const float4*>(L.rays), L.hits, L.slots, L.count,
                         spill,  cap,                                    ctl,    L.stream};
        static_assert(kPLdsDepth == 24, "the refusal above is the spill bound");
        const uint32_t walk_groups = uint32_t(device_cu_count()) * 3;
        walk_pull<false, kPLdsDepth, 0>(a, leaf_batch, walk_groups, false);
    } else if (leaf_batch) {
        if (fslab)
            reg ? launch_persistent<2, true, true, kLeafDiv>(B, L, groups, spill, cap, ctl)
                : launch_persistent<2, false, true, kLeafDiv>(B, L, groups, spill, cap, ctl);
        else
            launch_persistent<2, true, false, kLeafDiv>(B, L, groups, spill, cap, ctl);
    } else if (fslab) {
        reg ? launch_persistent<2, true, true>(B, L, groups, spill, cap, ctl)
            : launch_persistent<2, false, true>(B, L, groups, spill, cap, ctl);
    } else {
        launch_persistent<2, true>(B, L, groups, spill, cap, ctl);
    }
    ATLAS_HIP_TRY(hipGetLastError());
    return ATLAS_RT_OK;
}

atlas_rt_status launch_blas_any(atlas_rt_blas& blas, const TraceLaunch& L) {
    if (L.count == 0) return ATLAS_RT_OK;
    return launch_walk<true>(blas, L, WalkPlan::kAuto);
}

}  // namespace atlas_rt
