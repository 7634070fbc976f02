// Two-level (TLAS + instanced BLAS) traversal kernels, gfx950.
//
// Reference: HitClosest / HitAny with CheckInstance (data/shader/raytracer/bvh.hsh:172-273,
// 359-441).  One stack serves both levels; `tlas_index` (the engine's tlasIndex)
// records the stack depth at which the current instance was entered, so
// popping below it returns to the TLAS with the world-space ray restored.
// Entering an instance transforms the ray with the instance's inverse matrix
// as a row vector times mat3x4 (unnormalised direction, so t stays in world
// units, bvh.hsh:177-180) and selects that instance's BLAS.
//
// Opaque walks run on the filtered two-level walk of world_walk.h, the
// transparent ones on the step functions of trace_world_core.h; both give the
// engine's results bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "alpha.h"
#include "rt_internal.h"
#include "trace_world_core.h"
#include "world_walk.h"

namespace atlas_rt {

namespace {

// Stack rows in LDS of the walk kernels, one wave of 64 per group: as many as
// 20 groups per CU, all that the registers allow, leave room for.  Worlds that
// need no more run without own rows: a kernel that has scratch memory takes
// 0.2 to 0.4 us longer to launch.
constexpr int kWalkRows = 30;

// The lane's ray of a group that takes `per_wave` rays, or ~0.
__device__ __forceinline__ uint32_t lane_ray(uint32_t per_wave, uint32_t count) {
    const uint32_t k = blockIdx.x * per_wave + threadIdx.x;
    return threadIdx.x < per_wave && k < count ? k : ~0u;
}

// Compact ray in (32 B) -> refined hit (16 B) + caller instance index.
template <int ROWS, int OWN>
__global__ __launch_bounds__(64, 5) void k_world_closest_rays(WorldDev W, const float4* __restrict__ rays,
                                                              float4* __restrict__ hits, int32_t* __restrict__ inst_out,
                                                              uint32_t count, uint32_t mask,
                                                              int32_t* __restrict__ spill, uint32_t cap,
                                                              uint32_t* __restrict__ ctl, uint32_t per_wave) {
    __shared__ int32_t lds[ROWS * 64];
    using Stack = WalkStack<64, ROWS, OWN>;
    int32_t own[OWN ? OWN : 1];
    const Stack S(lds, own, spill, blockIdx.x * 64 + threadIdx.x, gridDim.x * 64, cap);
    const uint32_t ray = lane_ray(per_wave, count);
    float4 r0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), r1 = r0;
    if (ray != ~0u) {
        r0 = rays[2 * size_t(ray)];
        r1 = rays[2 * size_t(ray) + 1];
    }
    WorldWalk k;
    world_walk_begin(k, W, r0, r1, Stack::bottom(threadIdx.x));
    if (ray == ~0u || any_nan3(r1.x, r1.y, r1.z)) k.w.node = kEnd;
    NoCount none;
    if (world_walk<true>(k, W, S, 0ull, mask, none)) atomicOr(&ctl[2], 1u);
    if (ray == ~0u) return;
    float4 out = make_float4(r1.w, 0.0f, 0.0f, __int_as_float(-1));
    int32_t caller_inst = -1;
    if (k.w.slot >= 0) {
        const float4* im = W.instances + 4 * size_t(k.inst);
        const BlasDev B = ld_blas(W.blases + __float_as_int(im[3].x));
        const float4* vp = B.vtx + 3 * size_t(k.w.slot);
        float o[3], d[3], t, u, v;
        object_ray(k, W, k.inst, o, d);
        refine_tuv(o[0], o[1], o[2], d[0], d[1], d[2], ldg4(vp), ldg4(vp + 1), ldg4(vp + 2), t, u, v);
        out = make_float4(t, u, v, ldg4(B.tris + 3 * size_t(k.w.slot)).w);
        caller_inst = W.inst_order[k.inst];
    }
    hits[ray] = out;
    if (inst_out) inst_out[ray] = caller_inst;
}

template <int ROWS, int OWN, bool RESTORE_ALWAYS>
__global__ __launch_bounds__(64, 5) void k_world_any_rays(WorldDev W, const float4* __restrict__ rays,
                                                          uint32_t* __restrict__ out, uint32_t count, uint32_t mask,
                                                          int32_t* __restrict__ spill, uint32_t cap,
                                                          uint32_t* __restrict__ ctl, uint32_t per_wave) {
    __shared__ int32_t lds[ROWS * 64];
    using Stack = WalkStack<64, ROWS, OWN>;
    int32_t own[OWN ? OWN : 1];
    const Stack S(lds, own, spill, blockIdx.x * 64 + threadIdx.x, gridDim.x * 64, cap);
    const uint32_t ray = lane_ray(per_wave, count);
    float4 r0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), r1 = r0;
    if (ray != ~0u) {
        r0 = rays[2 * size_t(ray)];
        r1 = rays[2 * size_t(ray) + 1];
    }
    WorldWalk k;
    world_walk_begin(k, W, r0, r1, Stack::bottom(threadIdx.x));
    if (ray == ~0u || any_nan3(r1.x, r1.y, r1.z)) k.w.node = kEnd;
    NoCount none;
    if (world_walk<RESTORE_ALWAYS>(k, W, S, ~0ull, mask, none)) atomicOr(&ctl[2], 1u);
    if (ray != ~0u) out[ray] = k.w.slot >= 0 ? 1u : 0u;
}

// Engine-shaped PackedRay kernels (traceClosest.csh:12-36).  The live ray
// count is read on the device.
template <int ROWS, int OWN>
__global__ __launch_bounds__(64, 5) void k_world_closest_packed(WorldDev W, const float4* __restrict__ in,
                                                                float4* __restrict__ out,
                                                                const uint32_t* __restrict__ d_count,
                                                                uint32_t max_count, float tmin, float tmax,
                                                                uint32_t mask, int32_t* __restrict__ spill,
                                                                uint32_t cap, uint32_t* __restrict__ ctl,
                                                                uint32_t per_wave) {
    __shared__ int32_t lds[ROWS * 64];
    using Stack = WalkStack<64, ROWS, OWN>;
    int32_t own[OWN ? OWN : 1];
    const Stack S(lds, own, spill, blockIdx.x * 64 + threadIdx.x, gridDim.x * 64, cap);
    const uint32_t ray = lane_ray(per_wave, d_count ? min(*d_count, max_count) : max_count);
    float4 p0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), p1 = p0, p2 = p0;
    if (ray != ~0u) {
        p0 = in[3 * size_t(ray)];
        p1 = in[3 * size_t(ray) + 1];
        p2 = in[3 * size_t(ray) + 2];
    }
    const bool valid = ray != ~0u && __float_as_int(p0.w) >= 0;
    WorldWalk k;
    world_walk_begin(k, W, make_float4(p0.x, p0.y, p0.z, tmin), make_float4(p1.x, p1.y, p1.z, tmax),
                     Stack::bottom(threadIdx.x));
    if (!valid || any_nan3(p1.x, p1.y, p1.z)) k.w.node = kEnd;
    NoCount none;
    const uint64_t over = world_walk<true>(k, W, S, 0ull, mask, none);
    if (over) atomicOr(&ctl[2], 1u);
    if (ray == ~0u) return;
    const bool hit = k.w.slot >= 0;
    const float distance = !valid ? 0.0f : (lane_in(over) ? tmax : k.w.t);
    out[3 * size_t(ray)] = p0;
    out[3 * size_t(ray) + 1] = p1;
    out[3 * size_t(ray) + 2] = make_float4(distance, __int_as_float(hit ? k.w.slot : -1),
                                           hit ? __int_as_float(k.inst) : p2.z, p2.w);
}

template <int ROWS, int OWN, bool RESTORE_ALWAYS>
__global__ __launch_bounds__(64, 5) void k_world_any_packed(WorldDev W, const float4* __restrict__ in,
                                                            uint32_t* __restrict__ out,
                                                            const uint32_t* __restrict__ d_count, uint32_t max_count,
                                                            float tmin, float tmax, uint32_t mask,
                                                            int32_t* __restrict__ spill, uint32_t cap,
                                                            uint32_t* __restrict__ ctl, uint32_t per_wave) {
    __shared__ int32_t lds[ROWS * 64];
    using Stack = WalkStack<64, ROWS, OWN>;
    int32_t own[OWN ? OWN : 1];
    const Stack S(lds, own, spill, blockIdx.x * 64 + threadIdx.x, gridDim.x * 64, cap);
    const uint32_t ray = lane_ray(per_wave, d_count ? min(*d_count, max_count) : max_count);
    float4 p0 = make_float4(0.0f, 0.0f, 0.0f, 0.0f), p1 = p0;
    if (ray != ~0u) {
        p0 = in[3 * size_t(ray)];
        p1 = in[3 * size_t(ray) + 1];
    }
    WorldWalk k;
    world_walk_begin(k, W, make_float4(p0.x, p0.y, p0.z, tmin), make_float4(p1.x, p1.y, p1.z, tmax),
                     Stack::bottom(threadIdx.x));
    if (ray == ~0u || any_nan3(p1.x, p1.y, p1.z)) k.w.node = kEnd;
    NoCount none;
    if (world_walk<RESTORE_ALWAYS>(k, W, S, ~0ull, mask, none)) atomicOr(&ctl[2], 1u);
    if (ray != ~0u) out[ray] = k.w.slot >= 0 ? 1u : 0u;
}

// Opacity-aware PackedRay traces: out_rays != null runs
// HitClosestTransparency (written like k_world_closest_packed), otherwise
// HitAnyTransparency writes the transparency left along each ray.
template <int BLOCK, int LDS_DEPTH>
__global__ __launch_bounds__(BLOCK) void k_world_alpha_packed(WorldDev W, pt::AlphaArgs A, const float4* __restrict__ in,
                                                              float4* __restrict__ out_rays,
                                                              float* __restrict__ out_trans,
                                                              const uint32_t* __restrict__ d_count, uint32_t max_count,
                                                              float tmin, float tmax, uint32_t mask,
                                                              int32_t* __restrict__ spill, uint32_t cap,
                                                              uint32_t* __restrict__ ctl) {
    __shared__ int32_t lds[LDS_DEPTH * BLOCK];
    const uint32_t gid = blockIdx.x * BLOCK + threadIdx.x;
    const uint32_t count = d_count ? min(*d_count, max_count) : max_count;
    if (gid >= count) return;
    const float4 p0 = in[3 * size_t(gid)];
    const float4 p1 = in[3 * size_t(gid) + 1];
    const pt::TriOpacity op{W, A};
    const LaneStack<BLOCK, LDS_DEPTH> S{lds, spill, threadIdx.x, gid, gridDim.x * BLOCK};
    if (!out_rays) {
        float trans = 1.0f;
        if (!any_nan3(p1.x, p1.y, p1.z)) {
            WorldLane L;
            world_begin(L, make_float4(p0.x, p0.y, p0.z, tmin), make_float4(p1.x, p1.y, p1.z, tmax));
            int r;
            do {
                r = world_step_transparency<BLOCK, LDS_DEPTH>(L, W, mask, tmax, S, cap, op);
            } while (r == kContinue);
            if (r == kOverflow) atomicOr(&ctl[2], 1u);
            trans = L.trans;
        }
        out_trans[gid] = trans;
        return;
    }
    const float4 p2 = in[3 * size_t(gid) + 2];
    const int32_t id = __float_as_int(p0.w);
    float hitDistance = 0.0f;
    int32_t hitID = -1;
    int32_t hitInstance = __float_as_int(p2.z);
    if (id >= 0) {
        hitDistance = tmax;
        if (!any_nan3(p1.x, p1.y, p1.z)) {
            WorldLane L;
            world_begin(L, make_float4(p0.x, p0.y, p0.z, tmin), make_float4(p1.x, p1.y, p1.z, tmax));
            const pt::AcceptOpaque acc{op};
            int r;
            do {
                r = world_step_closest<BLOCK, LDS_DEPTH>(L, W, mask, S, cap, acc);
            } while (r == kContinue);
            if (r == kOverflow) {
                atomicOr(&ctl[2], 1u);
            } else {
                hitDistance = L.hitT;
                if (L.slot >= 0) {
                    hitID = L.slot;
                    hitInstance = L.inst;
                }
            }
        }
    }
    out_rays[3 * size_t(gid)] = p0;
    out_rays[3 * size_t(gid) + 1] = p1;
    out_rays[3 * size_t(gid) + 2] = make_float4(hitDistance, __int_as_float(hitID), __int_as_float(hitInstance), p2.w);
}

constexpr int kBlock = 128;
constexpr int kLdsDepth = 32;

}  // namespace

static atlas_rt_status world_prepare(atlas_rt_world& w, uint32_t threads, uint32_t& cap) {
    cap = w.stack_cap();
    if (cap > uint32_t(kLdsDepth)) {
        atlas_rt_status st = w.spill.ensure(size_t(cap - kLdsDepth) * threads * sizeof(int32_t));
        if (st != ATLAS_RT_OK) return st;
    }
    if (!w.flags.ptr) {
        atlas_rt_status st = w.flags.ensure(256);
        if (st != ATLAS_RT_OK) return st;
        ATLAS_HIP_TRY(hipMemset(w.flags.ptr, 0, 256));
    }
    return ATLAS_RT_OK;
}

namespace {

// Small launches spread over the chip, as those of a single mesh do.
uint32_t rays_per_wave(uint32_t count) { return std::min(64u, (count - 1) / 2048u + 1); }

atlas_rt_status walk_prepare(atlas_rt_world& w, uint32_t count, uint32_t& per_wave, uint32_t& grid, uint32_t& cap) {
    if (count > UINT32_MAX - 63)
        return fail(ATLAS_RT_E_INVALID_ARG, "world trace: more rays than a launch has threads");
    per_wave = rays_per_wave(count);
    grid = (count - 1) / per_wave + 1;
    uint32_t old_cap;
    atlas_rt_status st = world_prepare(w, 0, old_cap);  // the flag block
    cap = w.stack_cap();
    if (const size_t bytes = walk_spill_bytes(cap, kWalkRows + kOwnRows, size_t(grid) * 64); bytes && st == ATLAS_RT_OK)
        st = w.spill.ensure(bytes);
    return st;
}

}  // namespace

atlas_rt_status launch_world_closest_rays(atlas_rt_world& w, const void* rays, void* hits, int32_t* inst,
                                          uint32_t count, uint32_t mask, hipStream_t stream) {
    if (!count) return ATLAS_RT_OK;
    uint32_t per_wave, grid, cap;
    atlas_rt_status st = walk_prepare(w, count, per_wave, grid, cap);
    if (st != ATLAS_RT_OK) return st;
    st = w.timing.begin(stream);
    if (st != ATLAS_RT_OK) return st;
    const auto kernel = cap < uint32_t(kWalkRows) ? k_world_closest_rays<kWalkRows, 0>
                                                  : k_world_closest_rays<kWalkRows, kOwnRows>;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64), 0, stream, w.dev(),
                       reinterpret_cast<const float4*>(rays), reinterpret_cast<float4*>(hits), inst, count, mask,
                       reinterpret_cast<int32_t*>(w.spill.ptr), cap, reinterpret_cast<uint32_t*>(w.flags.ptr), per_wave);
    ATLAS_HIP_TRY(hipGetLastError());
    return w.timing.end(stream);
}

atlas_rt_status launch_world_any_rays(atlas_rt_world& w, const void* rays, uint32_t* out, uint32_t count,
                                      uint32_t mask, uint32_t flags, hipStream_t stream) {
    if (!count) return ATLAS_RT_OK;
    uint32_t per_wave, grid, cap;
    atlas_rt_status st = walk_prepare(w, count, per_wave, grid, cap);
    if (st != ATLAS_RT_OK) return st;
    const bool restore = (flags & ATLAS_RT_ANY_RESTORE_ALWAYS) != 0;
    const auto kernel = cap < uint32_t(kWalkRows)
                            ? (restore ? k_world_any_rays<kWalkRows, 0, true> : k_world_any_rays<kWalkRows, 0, false>)
                            : (restore ? k_world_any_rays<kWalkRows, kOwnRows, true>
                                       : k_world_any_rays<kWalkRows, kOwnRows, false>);
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64), 0, stream, w.dev(), reinterpret_cast<const float4*>(rays), out,
                       count, mask, reinterpret_cast<int32_t*>(w.spill.ptr), cap,
                       reinterpret_cast<uint32_t*>(w.flags.ptr), per_wave);
    ATLAS_HIP_TRY(hipGetLastError());
    return ATLAS_RT_OK;
}

atlas_rt_status launch_world_closest_packed(atlas_rt_world& w, const void* in, void* out, const uint32_t* d_count,
                                            uint32_t max_count, float tmin, float tmax, uint32_t mask,
                                            hipStream_t stream) {
    if (!max_count) return ATLAS_RT_OK;
    uint32_t per_wave, grid, cap;
    atlas_rt_status st = walk_prepare(w, max_count, per_wave, grid, cap);
    if (st != ATLAS_RT_OK) return st;
    const auto kernel = cap < uint32_t(kWalkRows) ? k_world_closest_packed<kWalkRows, 0>
                                                  : k_world_closest_packed<kWalkRows, kOwnRows>;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64), 0, stream, w.dev(),
                       reinterpret_cast<const float4*>(in), reinterpret_cast<float4*>(out), d_count, max_count, tmin,
                       tmax, mask, reinterpret_cast<int32_t*>(w.spill.ptr), cap,
                       reinterpret_cast<uint32_t*>(w.flags.ptr), per_wave);
    ATLAS_HIP_TRY(hipGetLastError());
    return ATLAS_RT_OK;
}

atlas_rt_status launch_world_alpha_packed(atlas_rt_world& w, const void* in, void* out_rays, float* out_trans,
                                          const uint32_t* d_count, uint32_t max_count, float tmin, float tmax,
                                          uint32_t mask, hipStream_t stream) {
    if (!max_count) return ATLAS_RT_OK;
    // per-BLAS shading and uv pointers, refreshed when a BLAS's buffers change
    const size_t nb = w.blas_handles.size();
    std::vector<const void*> tab(2 * nb);
    for (size_t k = 0; k < nb; k++) {
        if (!w.blas_handles[k]->d_shade)
            return fail(ATLAS_RT_E_INVALID_ARG, "opacity-aware trace: a BLAS has no shading data");
        tab[k] = w.blas_handles[k]->d_shade;
        tab[nb + k] = w.blas_handles[k]->d_uv;
    }
    if (tab != w.alpha_tab_host) {
        atlas_rt_status st = w.alpha_tab.ensure(tab.size() * sizeof(void*));
        if (st != ATLAS_RT_OK) return st;
        ATLAS_HIP_TRY(hipStreamSynchronize(stream));
        ATLAS_HIP_TRY(hipMemcpy(w.alpha_tab.ptr, tab.data(), tab.size() * sizeof(void*), hipMemcpyHostToDevice));
        w.alpha_tab_host = tab;
    }
    const float4* const* dtab = reinterpret_cast<const float4* const*>(w.alpha_tab.ptr);
    const pt::AlphaArgs A{dtab, dtab + nb, nullptr, nullptr, nullptr, 0u, 0u};
    const uint32_t grid = (max_count + kBlock - 1) / kBlock;
    uint32_t cap;
    atlas_rt_status st = world_prepare(w, grid * kBlock, cap);
    if (st != ATLAS_RT_OK) return st;
    hipLaunchKernelGGL((k_world_alpha_packed<kBlock, kLdsDepth>), dim3(grid), dim3(kBlock), 0, stream, w.dev(), A,
                       reinterpret_cast<const float4*>(in), reinterpret_cast<float4*>(out_rays), out_trans, d_count,
                       max_count, tmin, tmax, mask, reinterpret_cast<int32_t*>(w.spill.ptr), cap,
                       reinterpret_cast<uint32_t*>(w.flags.ptr));
    ATLAS_HIP_TRY(hipGetLastError());
    return ATLAS_RT_OK;
}

atlas_rt_status launch_world_any_packed(atlas_rt_world& w, const void* in, uint32_t* out, const uint32_t* d_count,
                                        uint32_t max_count, float tmin, float tmax, uint32_t mask, uint32_t flags,
                                        hipStream_t stream) {
    if (!max_count) return ATLAS_RT_OK;
    uint32_t per_wave, grid, cap;
    atlas_rt_status st = walk_prepare(w, max_count, per_wave, grid, cap);
    if (st != ATLAS_RT_OK) return st;
    const bool restore = (flags & ATLAS_RT_ANY_RESTORE_ALWAYS) != 0;
    const auto kernel = cap < uint32_t(kWalkRows)
                            ? (restore ? k_world_any_packed<kWalkRows, 0, true> : k_world_any_packed<kWalkRows, 0, false>)
                            : (restore ? k_world_any_packed<kWalkRows, kOwnRows, true>
                                       : k_world_any_packed<kWalkRows, kOwnRows, false>);
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64), 0, stream, w.dev(), reinterpret_cast<const float4*>(in), out,
                       d_count, max_count, tmin, tmax, mask, reinterpret_cast<int32_t*>(w.spill.ptr), cap,
                       reinterpret_cast<uint32_t*>(w.flags.ptr), per_wave);
    ATLAS_HIP_TRY(hipGetLastError());
    return ATLAS_RT_OK;
}

}  // namespace atlas_rt
