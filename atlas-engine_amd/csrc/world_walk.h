// Engine-exact walk of a world (TLAS, instances, BLASes) by whole waves, on
// the steps of walk.h: shared by the world and frame kernels.
//
// Reference: HitClosest / HitAny with CheckInstance (data/shader/raytracer/bvh.hsh:172-273,
// 359-441).  One stack serves both levels; a lane that enters an instance
// notes its stack position, and a pop below it brings the lane back to the
// TLAS with its world ray.  Both levels' inner nodes are one step, so lanes
// in the TLAS and lanes in different instances step together; triangles and
// instance entries, which a few lanes wait for at a time, run once a quarter
// of the wave's live lanes wait for either.
//
// Which lanes are inside an instance is a wave mask: keeping, testing and
// updating it is scalar work.
#pragma once

#include <hip/hip_runtime.h>

#include "walk.h"
#include "world.h"

namespace atlas_rt {

struct WorldWalk {
    Walk w;                              // ray of the current level
    float ox, oy, oz, dx, dy, dz;        // world ray
    const float4* nodes;                 // of the current level
    const float4* tris;                  // of the current instance
    uint32_t entry;                      // stack position where it was entered
    int32_t cur;                         // its slot
    int32_t inst;                        // instance slot of the best hit
};

__device__ __forceinline__ void world_walk_begin(WorldWalk& k, const WorldDev& W, float4 r0, float4 r1,
                                                 uint32_t bottom) {
    walk_begin(k.w, 1u, r0, r1, bottom);
    k.ox = r0.x;
    k.oy = r0.y;
    k.oz = r0.z;
    k.dx = r1.x;
    k.dy = r1.y;
    k.dz = r1.z;
    k.nodes = W.tlas;
    k.inst = -1;
}

__device__ __forceinline__ float row4(float x, float y, float z, float w, float4 m) {
    return ((x * m.x + y * m.y) + z * m.z) + w * m.w;
}

// The world ray in instance `inst`'s space (CheckInstance).
__device__ __forceinline__ void object_ray(const WorldWalk& k, const WorldDev& W, int32_t inst, float (&o)[3],
                                           float (&d)[3]) {
    const float4* m = W.instances + 4 * size_t(uint32_t(inst));
    const float4 c0 = ldg4(m), c1 = ldg4(m + 1), c2 = ldg4(m + 2);
    o[0] = row4(k.ox, k.oy, k.oz, 1.0f, c0);
    o[1] = row4(k.ox, k.oy, k.oz, 1.0f, c1);
    o[2] = row4(k.ox, k.oy, k.oz, 1.0f, c2);
    d[0] = row4(k.dx, k.dy, k.dz, 0.0f, c0);
    d[1] = row4(k.dx, k.dy, k.dz, 0.0f, c1);
    d[2] = row4(k.dx, k.dy, k.dz, 0.0f, c2);
}

struct NoCount {
    __device__ __forceinline__ void node() {}
    __device__ __forceinline__ void triangle() {}
    __device__ __forceinline__ void instance() {}
};

// Walks every lane of the wave to the end (node == kEnd); lanes that do not
// take part come in ended.  The whole wave calls it.
//   any      lanes whose walk ends at its first accepted triangle;
//   mask     the instances a lane may enter;
//   RESTORE  an instance the mask rejects leaves the world ray in place
//            (HitClosest, HitAnyTransparency); otherwise the TLAS walk goes
//            on with that instance's object-space ray until it returns from
//            an entered one (HitAny, bvh.hsh:382-387).
// Returns the lanes that ran out of stack; their slot is -1.
template <bool RESTORE, class STK, class Count>
__device__ __forceinline__ uint64_t world_walk(WorldWalk& k, const WorldDev& W, const STK& S, uint64_t any,
                                               uint32_t mask, Count& count) {
    constexpr uint32_t kWaitDiv = 4;
    Walk& w = k.w;
    uint64_t inside = 0;  // lanes in an instance
    uint64_t over = 0;
    // lanes whose pop left their instance: the TLAS again, with the world ray
    const auto leave = [&]() {
        const uint64_t out = inside & mask_of(w.at < k.entry);
        if (out) {
            if (lane_in(out)) {
                walk_ray(w.R, k.ox, k.oy, k.oz, k.dx, k.dy, k.dz, w.tmin);
                k.nodes = W.tlas;
            }
            inside &= ~out;
        }
    };
    uint64_t live = mask_of(w.node != kEnd);
    while (live) {
        uint64_t inner = mask_of(w.node >= 0);
        while (uint32_t(__popcll(live ^ inner)) * kWaitDiv < uint32_t(__popcll(live))) {
            bool out_of_stack = false;
            if (w.node >= 0) {
                int32_t below;
                count.node();
                const bool checked = walk_stack(w, S, below);
                const NodeRec n = load_node(k.nodes, w.node);
                out_of_stack = lane_in(walk_node(w, n, checked, below, S, any));
            }
            over |= mask_of(out_of_stack);
            leave();
            live = mask_of(w.node != kEnd);
            inner = mask_of(w.node >= 0);
        }
        const uint64_t leaf = live & ~inner;
        const uint64_t tri = leaf & inside, ins = leaf & ~inside;
        if (tri) {
            if (lane_in(tri)) {
                count.triangle();
                if (walk_leaf(w, k.tris, S, lane_in(any))) k.inst = k.cur;
            }
            leave();
        }
        if (ins) {
            bool admit = false;
            if (lane_in(ins)) {
                count.instance();
                int32_t below;
                walk_stack(w, S, below);
                const int32_t slot = ~w.node;
                const float4 meta = ldg4(W.instances + 4 * size_t(uint32_t(slot)) + 3);
                admit = (uint32_t(__float_as_int(meta.w)) & mask) > 0;
                if (admit || !RESTORE) {
                    float o[3], d[3];
                    object_ray(k, W, slot, o, d);
                    walk_ray(w.R, o[0], o[1], o[2], d[0], d[1], d[2], w.tmin);
                }
                if (admit) {
                    const BlasView B = blas_view(W.blases + __float_as_int(meta.x));
                    k.nodes = B.nodes;
                    k.tris = B.tris;
                    k.cur = slot;
                    k.entry = w.at;
                    w.node = B.node_count ? 0 : ~0;
                } else {
                    w.node = w.top;
                    w.top = below;
                    w.at -= STK::kRow;
                }
            }
            inside |= mask_of(admit);
        }
        live = mask_of(w.node != kEnd);
    }
    if (over) {
        if (lane_in(over)) w.slot = -1;
    }
    return over;
}

}  // namespace atlas_rt
