// Engine-exact walk of binary trees: the per-lane steps shared by the BLAS,
// batched, world and frame kernels.
//
// Every decision (which child boxes are hit, which child is nearer, which
// triangle is accepted) is the one the engine's arithmetic gives
// (slab_dist, tri_uvt in rt_device.h); only the way to it differs.
//
// Box tests.  The engine's slab distances are correctly rounded quotients
// T = RN((b - o) / d), which cost a conversion to double, a product and a
// conversion back per plane: on gfx950 13.6 cycles per wave, against 2.6 for
// a float product (add, mul and fma of VGPRs issue in 2.5 cycles per wave,
// everything else, FP64 and conversions included, in 4.2 - 4.6).  Here
// t = fl((b - o) * r) with r within 1 ulp of 1 / d, so t is within
// 2^-22 (relative) of T, and a comparison of two such values whose gap is
// over 2^-20 has the engine's outcome.  Values closer than that are settled
// in two further stages, taken by a wave only when one of its lanes needs
// them:
//   1. the ties that real geometry is full of: a flat box (both planes of an
//      axis the same distance away, so entry = exit there by construction)
//      and planes shared by both children (the same operands give the same
//      T), by comparing the other axes;
//   2. the engine's own arithmetic.
// Share of node visits that reach stage 1 / stage 2, counted on the host:
// random soup 7e-4 / 5e-6, heightfield 3.3e-2 / 3e-4, displaced sphere
// 2e-2 / 2e-3, axis-aligned boxes 1.1e-1 / 2e-2.
// Rays outside the bounds' premises (a direction component that is
// subnormal or over 2^126, a negative or NaN tmin) take stage 2 always.
//
// Stack.  The top entry lives in a register, the others in LDS rows
// [row][lane] (row 0 is padding), deeper ones in the lane's own array and then
// in global spill rows (WalkStack).  A node step stores the old top and loads
// the entry below it before the node arrives, whichever it will need, so
// neither waits and neither branches; only when some lane nears the end of the
// LDS rows (or of the stack limit) does the wave take the checked path.  The
// bottom of the stack is kEnd, which ends the walk when popped.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rt_device.h"
#include "rt_internal.h"

namespace atlas_rt {

// What a walk needs of a BLAS record, read from a table in global memory.
struct BlasView {
    const float4* nodes;
    const float4* tris;
    const float4* vtx;
    uint32_t node_count;
};

__device__ __forceinline__ BlasView blas_view(const BlasDev* p) {
    const __attribute__((address_space(1))) BlasDev* g = (const __attribute__((address_space(1))) BlasDev*)p;
    return BlasView{g->nodes, g->tris, g->vtx, g->node_count};
}

constexpr int32_t kEnd = INT32_MIN;   // node of a lane whose walk has ended

struct WalkRay {
    float ox, oy, oz;
    float dx, dy, dz;
    float rx, ry, rz;  // 1 / d within 1 ulp
    float floor;       // absolute part of the margin; NaN: always exact
};

__device__ __forceinline__ bool subnormal(float d) { return __builtin_isfpclass(d, 0x0090); }

__device__ __forceinline__ void walk_ray(WalkRay& R, float ox, float oy, float oz, float dx, float dy, float dz,
                                         float tmin) {
    R.ox = ox;
    R.oy = oy;
    R.oz = oz;
    R.dx = dx;
    R.dy = dy;
    R.dz = dz;
    R.rx = __builtin_amdgcn_rcpf(dx);
    R.ry = __builtin_amdgcn_rcpf(dy);
    R.rz = __builtin_amdgcn_rcpf(dz);
    const bool ok = fmaxf(fabsf(dx), fmaxf(fabsf(dy), fabsf(dz))) <= 8.507059173023462e+37f /* 2^126 */ &&
                    !subnormal(dx) && !subnormal(dy) && !subnormal(dz) && tmin >= 0.0f;
    R.floor = ok ? 7.888609052210118e-31f /* 2^-100 */ : __builtin_nanf("");
}

// v raised by the margin: certainly above the engine's value when v >= 0.
__device__ __forceinline__ float above(const WalkRay& R, float v) {
    return __builtin_fmaf(v, 1.00000095367431640625f /* 1 + 2^-20 */, R.floor);
}

__device__ __forceinline__ float max3(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }
__device__ __forceinline__ float min3(float a, float b, float c) { return fminf(fminf(a, b), c); }

// Conditions as wave masks: their logic runs on the scalar unit, beside the
// other waves' vector work.
__device__ __forceinline__ uint64_t mask_of(bool b) { return __builtin_amdgcn_ballot_w64(b); }
__device__ __forceinline__ bool lane_in(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// Both child boxes of a node record (a, b, c) against [tmin, t], as the
// engine decides them: the lanes that hit the left / right box, and of those
// that hit one or both the lanes that go left.  A closest-hit lane goes left
// when dist left <= dist right, where the dist of a missed box is t: the
// nearer box, ties left, and left too when only the right box is hit, exactly
// at t (nearer than t in every case that is settled before the engine's own
// arithmetic).  A lane of `any` goes left when the left box is hit.  Active
// lanes only.
__device__ __forceinline__ void test_children(const WalkRay& R, const float4& a, const float4& b, const float4& c,
                                              float tmin, float t, uint64_t any, uint64_t& hl, uint64_t& hr,
                                              uint64_t& go_left) {
    const float l0x = (a.x - R.ox) * R.rx, l0y = (a.y - R.oy) * R.ry, l0z = (a.z - R.oz) * R.rz;
    const float l1x = (a.w - R.ox) * R.rx, l1y = (b.x - R.oy) * R.ry, l1z = (b.y - R.oz) * R.rz;
    const float r0x = (b.z - R.ox) * R.rx, r0y = (b.w - R.oy) * R.ry, r0z = (c.x - R.oz) * R.rz;
    const float r1x = (c.y - R.ox) * R.rx, r1y = (c.z - R.oy) * R.ry, r1z = (c.w - R.oz) * R.rz;
    const float nlx = fminf(l0x, l1x), nly = fminf(l0y, l1y), nlz = fminf(l0z, l1z);
    const float flx = fmaxf(l0x, l1x), fly = fmaxf(l0y, l1y), flz = fmaxf(l0z, l1z);
    const float nrx = fminf(r0x, r1x), nry = fminf(r0y, r1y), nrz = fminf(r0z, r1z);
    const float frx = fmaxf(r0x, r1x), fry = fmaxf(r0y, r1y), frz = fmaxf(r0z, r1z);
    const float sl = max3(nlx, nly, nlz), sr = max3(nrx, nry, nrz);
    const float il = fmaxf(tmin, sl), ir = fmaxf(tmin, sr);                              // entry
    const float el = fminf(t, min3(flx, fly, flz)), er = fminf(t, min3(frx, fry, frz));  // exit
    const float irA = above(R, ir);
    const uint64_t pl = mask_of(!(above(R, el) < il)), pr = mask_of(!(above(R, er) < ir));  // possibly hit
    hl = mask_of(above(R, il) <= el);                                                       // certainly hit
    hr = mask_of(irA <= er);
    const uint64_t first = mask_of(above(R, sl) <= ir), second = mask_of(irA < il);  // certainly (not) left first
    go_left = hl & (any | first | ~hr);
    const uint64_t unsettled = (pl ^ hl) | (pr ^ hr) | (hl & hr & ~(any | first | second));
    if (__builtin_expect(unsettled != 0, 0)) {
        if ((pl ^ hl) | (pr ^ hr)) {
            const uint64_t hl1 = mask_of(above(R, tmin) <= el) & mask_of(above(R, nlx) <= min3(fly, flz, t)) &
                                 mask_of(above(R, nly) <= min3(flx, flz, t)) &
                                 mask_of(above(R, nlz) <= min3(flx, fly, t));
            const uint64_t hr1 = mask_of(above(R, tmin) <= er) & mask_of(above(R, nrx) <= min3(fry, frz, t)) &
                                 mask_of(above(R, nry) <= min3(frx, frz, t)) &
                                 mask_of(above(R, nrz) <= min3(frx, fry, t));
            hl |= pl & hl1;
            hr |= pr & hr1;
        }
        const uint64_t nx = mask_of(R.rx < 0.0f), ny = mask_of(R.ry < 0.0f), nz = mask_of(R.rz < 0.0f);
        const uint64_t sx = mask_of(nlx == nrx) & ((nx & mask_of(a.w == c.y)) | (~nx & mask_of(a.x == b.z)));
        const uint64_t sy = mask_of(nly == nry) & ((ny & mask_of(b.x == c.z)) | (~ny & mask_of(a.y == b.w)));
        const uint64_t sz = mask_of(nlz == nrz) & ((nz & mask_of(b.y == c.w)) | (~nz & mask_of(a.z == c.x)));
        const uint64_t first1 = (sx | mask_of(above(R, nlx) <= ir)) & (sy | mask_of(above(R, nly) <= ir)) &
                                (sz | mask_of(above(R, nlz) <= ir));
        go_left = hl & (any | first | (first1 & ~second) | ~hr);
        const uint64_t exact = (pl & ~hl) | (pr & ~hr) | (hl & hr & ~(any | first | second | first1));
        if (__builtin_expect(exact != 0, 0)) {
            DevRay D;
            D.ox = R.ox;
            D.oy = R.oy;
            D.oz = R.oz;
            D.rx = 1.0 / (double)R.dx;
            D.ry = 1.0 / (double)R.dy;
            D.rz = 1.0 / (double)R.dz;
            D.tmin = tmin;
            float dl, dr;
            hl = mask_of(slab_dist(D, a.x, a.y, a.z, a.w, b.x, b.y, t, dl));
            hr = mask_of(slab_dist(D, b.z, b.w, c.x, c.y, c.z, c.w, t, dr));
            go_left = (mask_of(dl <= dr) & ~any) | (hl & any);
        }
    }
}

// One lane's stack column.  `at` is the byte offset of row `depth` in the
// lane's LDS column (depth = entries below the register top, the engine's
// stack count).
//
// Rows past the LDS rows: the first OWN of them are an array of the lane's own
// (declared by the kernel; it lives in the scratch memory that the runtime
// keeps per queue), the others rows of `spill`, which the launch allocates
// (walk_spill_bytes).  With 32 own rows behind 14 in LDS, traces of trees of
// up to 44 levels allocate nothing, whatever their ray count.  With spill rows
// only, 1M rays on a tree of 19 levels took 29 MB, and the first 5,003 rays on a
// mesh of 20,011 triangles 0.26 ms, not 0.15; repeated traces take the same.
constexpr int kOwnRows = 32;

// Bytes of the spill rows of `lanes` lanes whose walks hold up to `cap`
// entries: rows 1 .. cap, of which the first are `rows` (LDS and own) less
// row 0.
inline size_t walk_spill_bytes(uint32_t cap, uint32_t rows, size_t lanes) {
    return cap >= rows ? size_t(cap + 1 - rows) * lanes * sizeof(int32_t) : 0;
}

template <int BLOCK, int ROWS, int OWN>
struct WalkStack {
    using Lds = __attribute__((address_space(3))) int32_t*;
    static constexpr uint32_t kRow = BLOCK * sizeof(int32_t);
    Lds lds;           // row 0 of the group
    int32_t* own;      // rows ROWS ... ROWS + OWN - 1
    int32_t* spill;    // row ROWS + OWN + k at spill[k * stride + column]
    uint32_t column, stride;
    uint32_t cap;      // entries a walk may hold
    uint32_t checked;  // offset from which a lane takes the checked path

    __device__ __forceinline__ WalkStack(int32_t* l, int32_t* ow, int32_t* sp, uint32_t col, uint32_t str, uint32_t c)
        : lds((Lds)l), own(ow), spill(sp), column(col), stride(str), cap(c),
          checked(min(uint32_t(ROWS - 1), c) * kRow) {}
    static __device__ __forceinline__ uint32_t bottom(uint32_t tid) { return tid * uint32_t(sizeof(int32_t)); }
    static __device__ __forceinline__ uint32_t depth(uint32_t at) { return at / kRow; }
    __device__ __forceinline__ Lds word(uint32_t at) const {
        return (Lds)((__attribute__((address_space(3))) char*)lds + at);
    }
    __device__ __forceinline__ int32_t load(uint32_t row, uint32_t at) const {
        if (row < ROWS) return *word(at);
        if (OWN && row < ROWS + OWN) return own[row - ROWS];
        return spill[size_t(row - ROWS - OWN) * stride + column];
    }
    __device__ __forceinline__ void store(uint32_t row, uint32_t at, int32_t v) const {
        if (row < ROWS)
            *word(at) = v;
        else if (OWN && row < ROWS + OWN)
            own[row - ROWS] = v;
        else
            spill[size_t(row - ROWS - OWN) * stride + column] = v;
    }
};

struct Walk {
    WalkRay R;
    float tmin;
    float t;        // current hit distance (any-hit walks: tmax)
    int32_t node;   // >= 0 inner node, < 0: ~(current triangle slot), kEnd: ended
    int32_t top;    // top of the stack
    uint32_t at;    // stack position (WalkStack)
    int32_t slot;   // best hit slot (-1 none)
};

__device__ __forceinline__ void walk_begin(Walk& w, uint32_t node_count, float4 r0, float4 r1, uint32_t bottom) {
    walk_ray(w.R, r0.x, r0.y, r0.z, r1.x, r1.y, r1.z, r0.w);
    w.tmin = __builtin_canonicalizef(r0.w);
    w.t = r1.w;
    w.node = node_count ? 0 : ~0;
    w.top = kEnd;
    w.at = bottom;
    w.slot = -1;
}

// What a step may need of the stack, fetched before its tree records arrive:
// the entry below the top, and the top stored where a push would leave it.
// Returns whether some lane is near the end of the rows or of the limit
// (wave-uniform).
template <class STK>
__device__ __forceinline__ bool walk_stack(const Walk& w, const STK& S, int32_t& below) {
    if (__builtin_expect(mask_of(w.at >= S.checked) != 0, 0)) {
        const uint32_t row = STK::depth(w.at);
        below = S.load(row, w.at);
        if (row < S.cap) S.store(row + 1, w.at + STK::kRow, w.top);
        return true;
    }
    below = *S.word(w.at);
    *S.word(w.at + STK::kRow) = w.top;
    return false;
}

// A node record: the child boxes (a, b, c) and pointers.
struct NodeRec {
    float4 a, b, c;
    int32_t left, right;
};

__device__ __forceinline__ NodeRec load_node(const float4* nodes, int32_t node) {
    const float4* np = nodes + 4 * size_t(uint32_t(node));
    NodeRec n;
    n.a = ldg4(np);
    n.b = ldg4(np + 1);
    n.c = ldg4(np + 2);
    const float4 d = ldg4(np + 3);
    n.left = __float_as_int(d.x);
    n.right = __float_as_int(d.y);
    return n;
}

// Node records through LDS.  A lane that loads its own 64 B record takes four
// accesses to the vector cache, one per 16 B, each of them alone in its cache
// line; the cache looks up one line per cycle, and between the four the lines
// of the CU's other waves may evict it.  Here the four lanes of a quad load
// one record together, one access in one instruction, straight into LDS, the
// quad's four records one after the other, and every lane reads its own back
// from there.  The four instructions' blocks of 1 KB lie 16 B more apart, so
// that the lanes that read together fall on different banks.
struct NodeStage {
    static constexpr uint32_t kStep = 64 * 16 + 16;
    static constexpr uint32_t kBytes = 4 * kStep;  // per wave
    using Lds = __attribute__((address_space(3))) char*;
    Lds base;

    __device__ __forceinline__ explicit NodeStage(char* all)
        : base((Lds)all + __builtin_amdgcn_readfirstlane(threadIdx.x / 64) * kBytes) {}

    template <int K>
    __device__ __forceinline__ void quad(uint32_t lo, uint32_t hi) const {
        constexpr int perm = K | (K << 2) | (K << 4) | (K << 6);
        const uint32_t l = uint32_t(__builtin_amdgcn_mov_dpp(int(lo), perm, 0xf, 0xf, true));
        const uint32_t h = uint32_t(__builtin_amdgcn_mov_dpp(int(hi), perm, 0xf, 0xf, true));
        // a record starts on a multiple of 64 B
        const uint64_t p = uint64_t(h) << 32 | (l | (threadIdx.x & 3u) * 16u);
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p,
                                         (__attribute__((address_space(3))) void*)(base + K * kStep), 16, 0, 0);
    }
    // Fetches the records of the lanes in `inner` (not empty), with every
    // lane of the wave active; the others fetch the first of them.
    __device__ __forceinline__ void fetch(const float4* nodes, int32_t node, uint64_t inner) const {
        const uint64_t p = uint64_t(nodes) + uint64_t(uint32_t(node)) * 64u;
        const int first = __builtin_ctzll(inner);
        const uint32_t lo = uint32_t(p), hi = uint32_t(p >> 32);
        const uint32_t lo1 = uint32_t(__builtin_amdgcn_readlane(int(lo), first));
        const uint32_t hi1 = uint32_t(__builtin_amdgcn_readlane(int(hi), first));
        const bool own = lane_in(inner);
        const uint32_t l = own ? lo : lo1, h = own ? hi : hi1;
        quad<0>(l, h);
        quad<1>(l, h);
        quad<2>(l, h);
        quad<3>(l, h);
    }
    __device__ __forceinline__ NodeRec read() const {
        using V4 = float __attribute__((ext_vector_type(4)));
        using I2 = int32_t __attribute__((ext_vector_type(2)));
        const uint32_t lane = threadIdx.x & 63u;
        const Lds p = base + (lane & 3u) * kStep + (lane >> 2) * 64u;
        const V4 a = *(const __attribute__((address_space(3))) V4*)p;
        const V4 b = *(const __attribute__((address_space(3))) V4*)(p + 16);
        const V4 c = *(const __attribute__((address_space(3))) V4*)(p + 32);
        const I2 d = *(const __attribute__((address_space(3))) I2*)(p + 48);
        return NodeRec{make_float4(a.x, a.y, a.z, a.w), make_float4(b.x, b.y, b.z, b.w),
                       make_float4(c.x, c.y, c.z, c.w), d.x, d.y};
    }
    // Waits until what fetch() asked for has arrived.
    __device__ __forceinline__ void wait() const {
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
        asm volatile("" ::: "memory");
    }
};

// Inner-node step (w.node >= 0) with its record and the entry below the top
// (walk_stack), any: lanes of any-hit walks.  Returns the lanes that ran out
// of stack (their walk has ended).
template <class STK>
__device__ __forceinline__ uint64_t walk_node(Walk& w, const NodeRec& n, bool checked, int32_t below, const STK& S,
                                              uint64_t any) {
    uint64_t hl, hr, left;
    test_children(w.R, n.a, n.b, n.c, w.tmin, w.t, any, hl, hr, left);
    uint64_t over = 0;
    if (__builtin_expect(checked, 0)) {
        over = hl & hr & mask_of(STK::depth(w.at) >= S.cap);
        hl &= ~over;  // neither pushed nor followed
        hr &= ~over;
    }
    const bool both = lane_in(hl & hr), hit = lane_in(hl | hr), go_left = lane_in(left);
    const int32_t near = go_left ? n.left : n.right, far = go_left ? n.right : n.left;
    w.node = hit ? near : w.top;
    w.top = both ? far : (hit ? w.top : below);
    w.at += both ? STK::kRow : (hit ? 0u : 0u - STK::kRow);
    if (__builtin_expect(over != 0, 0)) {
        if (lane_in(over)) w.node = kEnd;
    }
    return over;
}

__device__ __forceinline__ bool walk_triangle(const WalkRay& R, const float4& a, const float4& b, const float4& c,
                                              float& t, float& u, float& v) {
    DevRay D;
    D.ox = R.ox;
    D.oy = R.oy;
    D.oz = R.oz;
    D.dx = R.dx;
    D.dy = R.dy;
    D.dz = R.dz;
    return tri_uvt(D, a.x, a.y, a.z, b.x, b.y, b.z, c.x, c.y, c.z, t, u, v);
}

// Triangle step (w.node < 0 and not kEnd); any: the first accepted triangle
// ends the walk.  Returns whether the triangle was accepted.
template <class STK>
__device__ __forceinline__ bool walk_leaf(Walk& w, const float4* tris, const STK& S, bool any) {
    const int32_t slot = ~w.node;
    const float4* tr = tris + 3 * size_t(uint32_t(slot));
    int32_t below;
    walk_stack(w, S, below);
    const float4 a = ldg4(tr), b = ldg4(tr + 1), c = ldg4(tr + 2);
    float t, u, v;
    const bool geo = walk_triangle(w.R, a, b, c, t, u, v);
    const bool hit = geo && t > w.tmin && t < w.t;
    w.t = hit ? t : w.t;
    w.slot = hit ? slot : w.slot;
    const bool last = b.w > 0.0f;  // end of leaf: pop (the entry below kEnd is row 0, the padding)
    w.node = hit && any ? kEnd : (last ? w.top : w.node - 1 /* ~(slot + 1) */);
    w.top = last ? below : w.top;
    w.at -= last ? STK::kRow : 0u;
    return hit;
}

// Final hit record (t, u, v, caller index) of the compact 16 B hit format.
__device__ __forceinline__ float4 walk_hit_record(const Walk& w, const float4* tris, const float4* vtx, float tmax) {
    if (w.slot < 0) return make_float4(tmax, 0.0f, 0.0f, __int_as_float(-1));
    const float4* vp = vtx + 3 * size_t(uint32_t(w.slot));
    float t, u, v;
    refine_tuv(w.R.ox, w.R.oy, w.R.oz, w.R.dx, w.R.dy, w.R.dz, ldg4(vp), ldg4(vp + 1), ldg4(vp + 2), t, u, v);
    return make_float4(t, u, v, ldg4(tris + 3 * size_t(uint32_t(w.slot))).w);
}

}  // namespace atlas_rt
