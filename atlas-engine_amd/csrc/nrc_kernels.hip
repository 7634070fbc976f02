// Radiance-cache kernels for gfx950: fused hash-grid encoding + MLP
// inference, fused forward/backward training with per-block weight-gradient
// sums in registers, and the Adam updates.  Layouts and the lane/unit mapping are
// described in nrc.h.
#include <hip/hip_runtime.h>

#include "nrc.h"

namespace atlas_rt {
namespace nrc {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kBeta1 = 0.9f;
constexpr float kBeta2 = 0.99f;
constexpr float kEps = 1e-15f;
constexpr float kLossFloor = 0.01f;
constexpr int kStride = 40;              // bf16 per staged row: 32 queries + 8 pad (80 B)
constexpr int kStage = 64 * kStride;     // one staged 64-unit x 32-query matrix

__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
}

// Round to nearest even (finite inputs).
__device__ __forceinline__ uint32_t bf16_bits(float f) {
    uint32_t u = __float_as_uint(f);
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) { return bf16_bits(lo) | (bf16_bits(hi) << 16); }
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ u32x4 pack_frag(f32x4 a, f32x4 b) {
    return u32x4{pack_bf16(a[0], a[1]), pack_bf16(a[2], a[3]), pack_bf16(b[0], b[1]), pack_bf16(b[2], b[3])};
}
__device__ __forceinline__ f32x4 relu4(f32x4 a) {
    return f32x4{fmaxf(a[0], 0.0f), fmaxf(a[1], 0.0f), fmaxf(a[2], 0.0f), fmaxf(a[3], 0.0f)};
}
__device__ __forceinline__ float half_to_float(uint32_t bits16) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16);
}
__device__ __forceinline__ uint16_t float_to_half(float f) { return __builtin_bit_cast(uint16_t, (_Float16)f); }

__device__ __forceinline__ u32x4 load_frag(const uint16_t* base, int frag, int lane) {
    return *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(base + (size_t)frag * 512) + (uint32_t)lane * 16u);
}

// ---------------------------------------------------------------------------
// Hash-grid encoding
// ---------------------------------------------------------------------------

// The 8 corners of the cell around normalised position (x, y, z) at `lev`:
// table entry index (level-major) and trilinear weight.
__device__ __forceinline__ void level_corners(const NrcDev& P, int lev, float x, float y, float z, uint32_t (&idx)[8],
                                              float (&w)[8]) {
    const float R = P.res[lev];
    const float sx = x * R, sy = y * R, sz = z * R;
    const float cx = fminf(floorf(sx), R - 1.0f), cy = fminf(floorf(sy), R - 1.0f), cz = fminf(floorf(sz), R - 1.0f);
    const float fx = sx - cx, fy = sy - cy, fz = sz - cz;
    const uint32_t ix = (uint32_t)cx, iy = (uint32_t)cy, iz = (uint32_t)cz;
    const uint32_t T = 1u << P.log2_t;
    const bool dense = (P.dense_mask >> lev) & 1u;
    const uint32_t R1 = (uint32_t)R + 1u;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const uint32_t px = ix + (c & 1), py = iy + ((c >> 1) & 1), pz = iz + (c >> 2);
        const uint32_t h = dense ? px + R1 * (py + R1 * pz) : ((px ^ (py * 2654435761u) ^ (pz * 805459861u)) & (T - 1u));
        idx[c] = (uint32_t)lev * T + h;
        const float wx = (c & 1) ? fx : 1.0f - fx;
        const float wy = (c & 2) ? fy : 1.0f - fy;
        const float wz = (c & 4) ? fz : 1.0f - fz;
        w[c] = (wx * wy) * wz;
    }
}

__device__ __forceinline__ float clamp01(float v) { return fminf(fmaxf(v, 0.0f), 1.0f); }

// Level held in feature slot j (features 2j, 2j+1 of the lane's 8) by lane
// group g, or -1 when the slot holds direction/normal/roughness inputs.
__device__ __forceinline__ int slot_level(int g, int j) {
    if (j < 2) return 2 * g + j;
    return g < 2 ? 8 + 2 * g + (j - 2) : -1;
}

// The 8 input features lane group g feeds to K slots i = 0..7 for query qi:
// features 4g + 0..3 and 16 + 4g + 0..3 of the 32-input vector.
__device__ __forceinline__ void lane_features(const NrcDev& P, const float4* __restrict__ q, uint32_t qi, bool valid,
                                              int g, float (&f)[8]) {
#pragma unroll
    for (int k = 0; k < 8; k++) f[k] = 0.0f;
    if (!valid) return;
    const float4 a = q[3 * (size_t)qi], b = q[3 * (size_t)qi + 1], c = q[3 * (size_t)qi + 2];
    const float x = clamp01((a.x - P.bmin[0]) * P.binv[0]);
    const float y = clamp01((a.y - P.bmin[1]) * P.binv[1]);
    const float z = clamp01((a.z - P.bmin[2]) * P.binv[2]);
    const uint32_t* tab = reinterpret_cast<const uint32_t*>(P.table);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int lev = slot_level(g, j);
        if (lev < 0 || lev >= (int)P.levels) continue;
        uint32_t idx[8];
        float w[8];
        level_corners(P, lev, x, y, z, idx, w);
        float f0 = 0.0f, f1 = 0.0f;
#pragma unroll
        for (int cc = 0; cc < 8; cc++) {
            const uint32_t e = tab[idx[cc]];
            f0 += w[cc] * half_to_float(e & 0xffffu);
            f1 += w[cc] * half_to_float(e >> 16);
        }
        f[2 * j] = f0;
        f[2 * j + 1] = f1;
    }
    if (g == 2) {
        f[4] = b.x;
        f[5] = b.y;
        f[6] = b.z;
        f[7] = c.x;
    } else if (g == 3) {
        f[4] = c.y;
        f[5] = c.z;
        f[6] = a.w;
        f[7] = 1.0f;
    }
}

// Scatter d(loss)/d(feature) of a wave's 32 queries into the FP32 table
// gradient.  The atomics are bound by the memory requests they make, about 20
// a nanosecond over the chip wherever they go, not by their number: one lane
// per feature with its corners in turn makes one request per atomic.  Here 16
// lanes take the 8 corners and both features of one query's cell, the two
// corners along x and their features in four adjacent lanes: 16 adjacent
// bytes at a dense level, mostly one cache line at a hashed one (x enters the
// hash unmultiplied), so a request carries about four atomics.
//   df:  [32 queries][kDfStride] feature gradients, level-major pairs
//   pos: [32 queries][3] positions in [0, 1]
constexpr int kDfStride = 25;
__device__ __forceinline__ void wave_table_grad(const NrcDev& P, const float* df, const float* pos, uint32_t queries,
                                                int lane, float* __restrict__ grad) {
    const int f = lane & 1, cx = (lane >> 1) & 1, cy = (lane >> 2) & 1, cz = (lane >> 3) & 1;
    const uint32_t T = 1u << P.log2_t;
    for (uint32_t lev = 0; lev < P.levels; lev++) {
        const float R = P.res[lev];
        const bool dense = (P.dense_mask >> lev) & 1u;
        const uint32_t R1 = (uint32_t)R + 1u;
#pragma unroll 4
        for (int step = 0; step < 8; step++) {
            const uint32_t q = 4 * step + (lane >> 4);
            if (q >= queries) continue;
            const float d = df[q * kDfStride + 2 * lev + f];
            if (d == 0.0f) continue;
            // the corner's entry and weight, as level_corners gives them
            const float sx = pos[3 * q] * R, sy = pos[3 * q + 1] * R, sz = pos[3 * q + 2] * R;
            const float x0 = fminf(floorf(sx), R - 1.0f), y0 = fminf(floorf(sy), R - 1.0f),
                        z0 = fminf(floorf(sz), R - 1.0f);
            const float fx = sx - x0, fy = sy - y0, fz = sz - z0;
            const uint32_t px = (uint32_t)x0 + cx, py = (uint32_t)y0 + cy, pz = (uint32_t)z0 + cz;
            const uint32_t h =
                dense ? px + R1 * (py + R1 * pz) : ((px ^ (py * 2654435761u) ^ (pz * 805459861u)) & (T - 1u));
            const float w = ((cx ? fx : 1.0f - fx) * (cy ? fy : 1.0f - fy)) * (cz ? fz : 1.0f - fz);
            atomicAdd(grad + 2 * ((size_t)lev * T + h) + f, w * d);
        }
    }
}

// ---------------------------------------------------------------------------
// MLP building blocks (all lanes of the wave active)
// ---------------------------------------------------------------------------

// z[t][q] = W_L^T x for output tiles t, query tiles q.
template <int L, int QT>
__device__ __forceinline__ void fwd_layer(const uint16_t* __restrict__ wn, const u32x4 (&x)[kK[L] / 32][QT],
                                          f32x4 (&z)[kNp[L] / 16][QT], int lane) {
    constexpr int S = kK[L] / 32, T = kNp[L] / 16;
    const uint16_t* w = wn + wn_offset(L);
    asm volatile("" : "+s"(w));  // a scalar base per layer, not a register pair per fragment kept over the loop
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int q = 0; q < QT; q++) z[t][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < S; s++)
#pragma unroll
        for (int t = 0; t < T; t++) {
            const u32x4 a = load_frag(w, t * S + s, lane);
#pragma unroll
            for (int q = 0; q < QT; q++) z[t][q] = mfma(a, x[s][q], z[t][q]);
        }
}

// dx[t][q] = W_L dz for input tiles t.
template <int L, int QT>
__device__ __forceinline__ void bwd_layer(const uint16_t* __restrict__ wk, const u32x4 (&dz)[nk_cols(L) / 32][QT],
                                          f32x4 (&dx)[kK[L] / 16][QT], int lane) {
    constexpr int S = nk_cols(L) / 32, T = kK[L] / 16;
    const uint16_t* w = wk + wk_offset(L);
    asm volatile("" : "+s"(w));  // a scalar base per layer, not a register pair per fragment kept over the loop
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int q = 0; q < QT; q++) dx[t][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < S; s++)
#pragma unroll
        for (int t = 0; t < T; t++) {
            const u32x4 a = load_frag(w, t * S + s, lane);
#pragma unroll
            for (int q = 0; q < QT; q++) dx[t][q] = mfma(a, dz[s][q], dx[t][q]);
        }
}

template <int QT>
__device__ __forceinline__ void relu_pack(const f32x4 (&z)[4][QT], u32x4 (&h)[2][QT]) {
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int q = 0; q < QT; q++) h[s][q] = pack_frag(relu4(z[2 * s][q]), relu4(z[2 * s + 1][q]));
}

__device__ __forceinline__ float gate(uint32_t bits_word, bool hi, float v) {
    const float h = hi ? bf16_hi(bits_word) : bf16_lo(bits_word);
    return h > 0.0f ? v : 0.0f;
}

// dz = dx * relu'(z) with the gate read from the packed forward activations.
template <int QT>
__device__ __forceinline__ void gate_pack(const f32x4 (&dx)[4][QT], const u32x4 (&h)[2][QT], u32x4 (&dz)[2][QT]) {
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int q = 0; q < QT; q++) {
            const u32x4 hv = h[s][q];
            const f32x4 a = dx[2 * s][q], b = dx[2 * s + 1][q];
            const f32x4 ga{gate(hv[0], false, a[0]), gate(hv[0], true, a[1]), gate(hv[1], false, a[2]),
                           gate(hv[1], true, a[3])};
            const f32x4 gb{gate(hv[2], false, b[0]), gate(hv[2], true, b[1]), gate(hv[3], false, b[2]),
                           gate(hv[3], true, b[3])};
            dz[s][q] = pack_frag(ga, gb);
        }
}

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Transpose B-operand fragments (units P(s,g,i) x query 16 q + r) into a
// [unit][query] bf16 matrix in LDS.
template <int S, int QT>
__device__ __forceinline__ void stage(uint16_t* st, const u32x4 (&x)[S][QT], int g, int r) {
#pragma unroll
    for (int s = 0; s < S; s++)
#pragma unroll
        for (int q = 0; q < QT; q++)
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint32_t w = x[s][q][i >> 1];
                const uint16_t v = (i & 1) ? (uint16_t)(w >> 16) : (uint16_t)(w & 0xffffu);
                const int n = 32 * s + 16 * (i >> 2) + 4 * g + (i & 3);
                st[n * kStride + 16 * q + r] = v;
            }
}

// The block's waves share out the 16 x 16 tiles of each layer's weight
// gradient: each takes kDwTiles neighbours along the outputs.
constexpr int kTrainWaves = kTrainBlock / 64;
template <int L>
constexpr int kDwTiles = (kK[L] / 16) * (kNp[L] / 16) / kTrainWaves;
template <int L>
__device__ __forceinline__ int dw_in_tile(int wv) { return wv * kDwTiles<L> / (kNp[L] / 16); }
template <int L>
__device__ __forceinline__ int dw_out_tile(int wv) { return wv * kDwTiles<L> % (kNp[L] / 16); }

// acc += the wave's tiles of X_L^T dZ_L over the block's 128 queries: every
// wave stages its queries' activations and gradients (K of the product), then
// all of them are read back.  Ends with the staging rows in use.
template <int L, int S, int QT>
__device__ __forceinline__ void dw_step(uint16_t (*staging)[2][kStage], const u32x4 (&x)[kK[L] / 32][QT],
                                        const u32x4 (&dz)[S][QT], f32x4 (&acc)[kDwTiles<L>], int wv, int g, int r) {
    constexpr int NT = kNp[L] / 16;
    static_assert(kDwTiles<L> * kTrainWaves == (kK[L] / 16) * NT && (kDwTiles<L> <= NT && NT % kDwTiles<L> == 0),
                  "whole tiles of one input row per wave");
    __syncthreads();  // the rows' last readers are done
    stage<kK[L] / 32, QT>(staging[wv][0], x, g, r);
    stage<S, QT>(staging[wv][1], dz, g, r);
    __syncthreads();
    const int ti = dw_in_tile<L>(wv), to = dw_out_tile<L>(wv);
#pragma unroll 1  // unrolled, the loads of all steps raise the register count: 331 us, not 327
    for (int c = 0; c < kTrainWaves; c++) {
        const u32x4 a = *reinterpret_cast<const u32x4*>(&staging[c][0][(16 * ti + r) * kStride + 8 * g]);
#pragma unroll
        for (int j = 0; j < kDwTiles<L>; j++) {
            const u32x4 b = *reinterpret_cast<const u32x4*>(&staging[c][1][(16 * (to + j) + r) * kStride + 8 * g]);
            acc[j] = mfma(a, b, acc[j]);
        }
    }
}

// Writes the wave's tiles of layer L into the block's weight gradient.
template <int L>
__device__ __forceinline__ void dw_store(const f32x4 (&acc)[kDwTiles<L>], float* dst, int wv, int g, int r) {
    constexpr int N = kN[L];
#pragma unroll
    for (int j = 0; j < kDwTiles<L>; j++) {
        const int out = 16 * (dw_out_tile<L>(wv) + j) + r;
        if (out < N) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                dst[master_offset(L) + (16 * dw_in_tile<L>(wv) + 4 * g + i) * N + out] = acc[j][i];
        }
    }
}

// ---------------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------------

constexpr int kInferQT = kInferQueriesPerWave / 16;
constexpr int kTrainQT = kTrainQueriesPerWave / 16;
static_assert(kTrainQT == 2, "the weight-gradient product takes K = 32 queries per chunk");
static_assert(kStage * sizeof(uint16_t) >= 32 * kDfStride * sizeof(float), "the staging rows hold the feature gradients");

// The two features of level `lev` at (x, y, z), as lane_features sums them.
__device__ __forceinline__ uint32_t level_feature(const NrcDev& P, int lev, float x, float y, float z) {
    uint32_t idx[8];
    float w[8];
    level_corners(P, lev, x, y, z, idx, w);
    const uint32_t* tab = reinterpret_cast<const uint32_t*>(P.table);
    uint32_t e[8];
    if ((P.dense_mask >> lev) & 1u) {  // the two corners along x are neighbours
#pragma unroll
        for (int c = 0; c < 8; c += 2) __builtin_memcpy(&e[c], tab + idx[c], 8);
    } else {
#pragma unroll
        for (int c = 0; c < 8; c++) e[c] = tab[idx[c]];
    }
    float f0 = 0.0f, f1 = 0.0f;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        f0 += w[c] * half_to_float(e[c] & 0xffffu);
        f1 += w[c] * half_to_float(e[c] >> 16);
    }
    return pack_bf16(f0, f1);
}

// Inference, TILES tiles of 64 queries per wave; count = *d_count when
// d_count is set (device-resident counts), else n.
//
// The gathers from the hash table bound it: 12 levels x 8 corners per query,
// mostly one cache line per two corners.  Taken query by query they spread
// over the whole table (25 MB at 12 x 2^19 entries), and most of the lines
// come from outside the XCD's 4 MB L2.  Here a wave takes one level for all
// of its queries before the next, one query per lane; the waves of the chip
// start together and move through the levels at about the same pace, so the
// level in use (2 MB) mostly stays in every L2.  The features wait in LDS as
// the BF16 pairs that the network's first layer reads.  One wave per block
// spreads any count evenly over the CUs; two waves per SIMD leave the network
// its registers, with four (128 registers, spilled) 460,001 queries take
// 170 us.  460,001 queries: 230 -> 137 us, 100,000: 69 -> 40,
// 1,000: 26 -> 15.
//
// FEW: at most 16 queries, one of the network's four tiles, gathered by four
// lanes each that share out the levels: 7.5 us, level by level 14.7.
template <int TILES, bool FEW>
__global__ __launch_bounds__(64, 2) void k_nrc_infer(NrcDev P, const float4* __restrict__ q, float4* __restrict__ out,
                                                      const uint32_t* __restrict__ d_count, uint32_t n) {
    constexpr int QT = kInferQT;
    constexpr int kRow = kMaxLevels + 1;  // dwords per query: odd, so that lanes fall on different banks
    __shared__ uint32_t features[TILES][64 * kRow];
    const int lane = threadIdx.x, g = lane >> 4, r = lane & 15;
    const uint32_t count = d_count ? min(*d_count, n) : n;
    // the tiles that are there, spread over the whole grid
    if (count == 0) return;
    const uint32_t per_wave = (count - 1) / (64 * gridDim.x) + 1;  // at most TILES
    const uint32_t first = blockIdx.x * per_wave * 64;
    if (first >= count) return;  // wave-uniform
    float x[TILES], y[TILES], z3[TILES];
#pragma unroll
    for (int t = 0; t < TILES; t++) {
        const uint32_t qi = min(first + 64 * min((uint32_t)t, per_wave - 1) + lane, count - 1);
        const float4 a = q[3 * (size_t)qi];
        x[t] = clamp01((a.x - P.bmin[0]) * P.binv[0]);
        y[t] = clamp01((a.y - P.bmin[1]) * P.binv[1]);
        z3[t] = clamp01((a.z - P.bmin[2]) * P.binv[2]);
    }
#pragma unroll 1
    for (int lev = 0; lev < kMaxLevels && !FEW; lev++) {
#pragma unroll
        for (int t = 0; t < TILES; t++)
            if (t == 0 || t < (int)per_wave)  // wave-uniform
                features[t][lane * kRow + lev] = lev < (int)P.levels ? level_feature(P, lev, x[t], y[t], z3[t]) : 0u;
    }
    wave_sync();
    for (uint32_t tile = 0; tile < per_wave; tile++) {
        const uint32_t base = first + 64 * tile;
        if (base >= count) break;  // wave-uniform
        u32x4 x0[1][QT];
        if (FEW) {
            float f[8];
            lane_features(P, q, r, (uint32_t)r < count, g, f);
            x0[0][0] =
                u32x4{pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]), pack_bf16(f[4], f[5]), pack_bf16(f[6], f[7])};
        }
#pragma unroll
        for (int t = 0; t < QT; t++) {
            if (FEW) {
                if (t > 0) x0[0][t] = u32x4{0u, 0u, 0u, 0u};
                continue;
            }
            const uint32_t qi = min(base + 16 * t + r, count - 1);
            const uint32_t* row = &features[tile][(16 * t + r) * kRow];
            u32x4 v{row[2 * g], row[2 * g + 1], row[8 + 2 * (g & 1)], row[9 + 2 * (g & 1)]};
            if (g >= 2) {  // directions, normal, roughness and the constant input
                const float4 a = q[3 * (size_t)qi], b = q[3 * (size_t)qi + 1], c = q[3 * (size_t)qi + 2];
                v[2] = g == 2 ? pack_bf16(b.x, b.y) : pack_bf16(c.y, c.z);
                v[3] = g == 2 ? pack_bf16(b.z, c.x) : pack_bf16(a.w, 1.0f);
            }
            x0[0][t] = v;
        }
        f32x4 z[4][QT];
        u32x4 h[2][QT];
        fwd_layer<0, QT>(P.wn, x0, z, lane);
        relu_pack<QT>(z, h);
        fwd_layer<1, QT>(P.wn, h, z, lane);
        relu_pack<QT>(z, h);
        fwd_layer<2, QT>(P.wn, h, z, lane);
        relu_pack<QT>(z, h);
        fwd_layer<3, QT>(P.wn, h, z, lane);
        relu_pack<QT>(z, h);
        fwd_layer<4, QT>(P.wn, h, z, lane);
        relu_pack<QT>(z, h);
        f32x4 o[1][QT];
        fwd_layer<5, QT>(P.wn, h, o, lane);
        if (g == 0) {
#pragma unroll
            for (int t = 0; t < QT; t++) {
                const uint32_t qi = base + 16 * t + r;
                if (qi < count) out[qi] = make_float4(o[0][t][0], o[0][t][1], o[0][t][2], 0.0f);
            }
        }
    }
}

// Trains on slice `slice` of `slices` equal slices of the samples; the
// sample count is *d_count when d_count is set (at most n), else n.  32
// queries per wave and step.
//
// The activations that the backward pass needs, its accumulators and the
// wave's tiles of the weight gradient fill the registers of one wave per SIMD
// (at 256, two waves, they spill: a training step of 65,536 queries takes
// 344 us and not 327).  The scatter into the table is the largest part, 175 of
// the kernel's 256 us.  Adding each step's weight gradient into LDS with atomics took a
// third of the kernel: the step 486 -> 327 us, 1,024 queries 159 -> 69,
// 300,000 queries 1,950 -> 1,150.
__global__ __launch_bounds__(kTrainBlock, 1) void k_nrc_train(NrcDev P, const float4* __restrict__ q,
                                                               const float4* __restrict__ tgt,
                                                               const uint32_t* __restrict__ d_count, uint32_t n,
                                                               uint32_t slice, uint32_t slices,
                                                               float* __restrict__ partial,
                                                               float* __restrict__ grad_table, float* loss) {
    constexpr int QT = kTrainQT;
    const uint32_t total = d_count ? min(*d_count, n) : n;
    const uint32_t first = uint32_t(uint64_t(total) * slice / slices);
    const uint32_t count = uint32_t(uint64_t(total) * (slice + 1) / slices) - first;
    const float inv_norm = count ? 1.0f / (3.0f * float(count)) : 0.0f;
    q += 3 * size_t(first);
    tgt += first;
    __shared__ __align__(16) uint16_t staging[kTrainWaves][2][kStage];

    const int lane0 = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t chunks = (count + kTrainQueriesPerWave - 1) / kTrainQueriesPerWave;
    float lane_loss = 0.0f;
    f32x4 w0[kDwTiles<0>]{}, w1[kDwTiles<1>]{}, w2[kDwTiles<2>]{}, w3[kDwTiles<3>]{}, w4[kDwTiles<4>]{},
        w5[kDwTiles<5>]{};

    for (uint32_t c = blockIdx.x * kTrainWaves; c < chunks; c += gridDim.x * kTrainWaves) {  // block-uniform
        // not loop-invariant to the compiler, which would otherwise keep every
        // address that follows from the lane in registers, and spill
        int lane = lane0;
        asm volatile("" : "+v"(lane));
        const int g = lane >> 4, r = lane & 15;
        const uint32_t base = (c + wv) * kTrainQueriesPerWave;  // may lie past the end: no query, no gradient
        // forward, keeping every layer's input as packed bf16
        u32x4 x0[1][QT], h0[2][QT], h1[2][QT], h2[2][QT], h3[2][QT], h4[2][QT];
#pragma unroll
        for (int t = 0; t < QT; t++) {
            const uint32_t qi = base + 16 * t + r;
            float f[8];
            lane_features(P, q, qi, qi < count, g, f);
            x0[0][t] =
                u32x4{pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]), pack_bf16(f[4], f[5]), pack_bf16(f[6], f[7])};
        }
        f32x4 z[4][QT];
        fwd_layer<0, QT>(P.wn, x0, z, lane);
        relu_pack<QT>(z, h0);
        fwd_layer<1, QT>(P.wn, h0, z, lane);
        relu_pack<QT>(z, h1);
        fwd_layer<2, QT>(P.wn, h1, z, lane);
        relu_pack<QT>(z, h2);
        fwd_layer<3, QT>(P.wn, h2, z, lane);
        relu_pack<QT>(z, h3);
        fwd_layer<4, QT>(P.wn, h3, z, lane);
        relu_pack<QT>(z, h4);
        f32x4 y[1][QT];
        fwd_layer<5, QT>(P.wn, h4, y, lane);

        // relative L2 loss and its gradient (outputs live in lanes g == 0)
        u32x4 dz5[1][QT];
#pragma unroll
        for (int t = 0; t < QT; t++) {
            const uint32_t qi = base + 16 * t + r;
            f32x4 d{0.0f, 0.0f, 0.0f, 0.0f};
            if (g == 0 && qi < count) {
                const float4 tv = tgt[qi];
                const float tt[3] = {tv.x, tv.y, tv.z};
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    const float yv = y[0][t][i];
                    const float den = yv * yv + kLossFloor;
                    const float diff = yv - tt[i];
                    lane_loss += diff * diff / den * inv_norm;
                    d[i] = 2.0f * diff / den * inv_norm;
                }
            }
            dz5[0][t] = pack_frag(d, f32x4{0.0f, 0.0f, 0.0f, 0.0f});
        }

        // backward
        f32x4 dx[4][QT];
        u32x4 dz[2][QT];
        dw_step<5, 1, QT>(staging, h4, dz5, w5, wv, g, r);
        bwd_layer<5, QT>(P.wk, dz5, dx, lane);
        gate_pack<QT>(dx, h4, dz);
        dw_step<4, 2, QT>(staging, h3, dz, w4, wv, g, r);
        bwd_layer<4, QT>(P.wk, dz, dx, lane);
        gate_pack<QT>(dx, h3, dz);
        dw_step<3, 2, QT>(staging, h2, dz, w3, wv, g, r);
        bwd_layer<3, QT>(P.wk, dz, dx, lane);
        gate_pack<QT>(dx, h2, dz);
        dw_step<2, 2, QT>(staging, h1, dz, w2, wv, g, r);
        bwd_layer<2, QT>(P.wk, dz, dx, lane);
        gate_pack<QT>(dx, h1, dz);
        dw_step<1, 2, QT>(staging, h0, dz, w1, wv, g, r);
        bwd_layer<1, QT>(P.wk, dz, dx, lane);
        gate_pack<QT>(dx, h0, dz);
        dw_step<0, 2, QT>(staging, x0, dz, w0, wv, g, r);
        f32x4 dx0[2][QT];
        bwd_layer<0, QT>(P.wk, dz, dx0, lane);

        // input-feature gradients -> hash table, through the staging rows
        float* df = reinterpret_cast<float*>(staging[wv][0]);
        float* pos = reinterpret_cast<float*>(staging[wv][1]);
        __syncthreads();
#pragma unroll
        for (int t = 0; t < QT; t++) {
            const float d8[8] = {dx0[0][t][0], dx0[0][t][1], dx0[0][t][2], dx0[0][t][3],
                                 dx0[1][t][0], dx0[1][t][1], dx0[1][t][2], dx0[1][t][3]};
            const int qn = 16 * t + r;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int lev = slot_level(g, j);
                if (lev < 0) continue;
                df[qn * kDfStride + 2 * lev] = d8[2 * j];
                df[qn * kDfStride + 2 * lev + 1] = d8[2 * j + 1];
            }
            if (g == 0 && base + qn < count) {
                const float4 a = q[3 * (size_t)(base + qn)];
                pos[3 * qn] = clamp01((a.x - P.bmin[0]) * P.binv[0]);
                pos[3 * qn + 1] = clamp01((a.y - P.bmin[1]) * P.binv[1]);
                pos[3 * qn + 2] = clamp01((a.z - P.bmin[2]) * P.binv[2]);
            }
        }
        wave_sync();
        wave_table_grad(P, df, pos, base < count ? min(count - base, (uint32_t)kTrainQueriesPerWave) : 0u, lane,
                        grad_table);
        wave_sync();
    }

    // loss: one atomic per wave
    for (int m = 32; m >= 1; m >>= 1) lane_loss += __shfl_xor(lane_loss, m, 64);
    const int lane = lane0, g = lane >> 4, r = lane & 15;
    if (lane == 0 && lane_loss != 0.0f) atomicAdd(loss, lane_loss);
    float* dst = partial + (size_t)blockIdx.x * kMasterSize;
    dw_store<0>(w0, dst, wv, g, r);
    dw_store<1>(w1, dst, wv, g, r);
    dw_store<2>(w2, dst, wv, g, r);
    dw_store<3>(w3, dst, wv, g, r);
    dw_store<4>(w4, dst, wv, g, r);
    dw_store<5>(w5, dst, wv, g, r);
}

// Stores weight j at its places in the forward and the backward fragments
// (k_pack's inverse; the padding stays as k_pack wrote it).
__device__ __forceinline__ void put_weight(uint32_t j, uint16_t w, uint16_t* wn, uint16_t* wk) {
    int L = 0;
#pragma unroll
    for (int l = 1; l < kLayers; l++)
        if (j >= (uint32_t)master_offset(l)) L = l;
    uint32_t fwd = 0, bwd = 0, local = j;
#pragma unroll
    for (int l = 1; l < kLayers; l++)
        if (L == l) {
            fwd = wn_offset(l);
            bwd = wk_offset(l);
            local = j - master_offset(l);
        }
    const uint32_t in = local / kN[L], out = local % kN[L];
    // value 4 (p / 16) + p % 4 of lane group (p % 16) / 4 is unit p of a K step
    const auto place = [](uint32_t frag, uint32_t p, uint32_t r) {
        return (frag * 64 + 16 * ((p & 15) >> 2) + r) * 8 + 4 * (p >> 4) + (p & 3);
    };
    wn[fwd + place((out >> 4) * (kK[L] / 32) + (in >> 5), in & 31, out & 15)] = w;
    wk[bwd + place((in >> 4) * (nk_cols(L) / 32) + (out >> 5), out & 31, in & 15)] = w;
}

// Sums the blocks' weight gradients, 64 weights per group: wave w of four adds
// every fourth block's (coalesced, eight loads in flight), then the first
// adds the four sums.  One thread per weight instead walks all the blocks on
// a quarter of the chip (256 blocks: 62 us against 6).
constexpr uint32_t kReduceWeights = 64, kReduceWaves = 4;
__global__ __launch_bounds__(kReduceWeights * kReduceWaves) void k_mlp_reduce(
    const float* __restrict__ partial, uint32_t blocks, float* __restrict__ grad_out, float* __restrict__ master,
    float* __restrict__ m, float* __restrict__ v, uint16_t* __restrict__ wn, uint16_t* __restrict__ wk, float lr_t) {
    __shared__ float part[kReduceWaves][kReduceWeights];
    const uint32_t lane = threadIdx.x % kReduceWeights, wave = threadIdx.x / kReduceWeights;
    const uint32_t j = blockIdx.x * kReduceWeights + lane;
    static_assert(kMasterSize % kReduceWeights == 0, "every lane has a weight");
    float t = 0.0f;
#pragma unroll 8
    for (uint32_t b = wave; b < blocks; b += kReduceWaves) t += partial[(size_t)b * kMasterSize + j];
    part[wave][lane] = t;
    __syncthreads();
    if (wave != 0) return;
    const float s = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
    if (m == nullptr) {
        grad_out[j] = s;
        return;
    }
    const float mj = kBeta1 * m[j] + (1.0f - kBeta1) * s;
    const float vj = kBeta2 * v[j] + (1.0f - kBeta2) * s * s;
    m[j] = mj;
    v[j] = vj;
    const float w = master[j] - lr_t * mj / (sqrtf(vj) + kEps);
    master[j] = w;
    put_weight(j, (uint16_t)bf16_bits(w), wn, wk);
}

__global__ void k_table_adam(float* __restrict__ t32, uint16_t* __restrict__ t16, float* __restrict__ m,
                             float* __restrict__ v, float* __restrict__ grad, uint32_t n, float lr_t) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const float gj = grad[j];
    if (gj == 0.0f) return;
    grad[j] = 0.0f;
    const float mj = kBeta1 * m[j] + (1.0f - kBeta1) * gj;
    const float vj = kBeta2 * v[j] + (1.0f - kBeta2) * gj * gj;
    m[j] = mj;
    v[j] = vj;
    const float p = t32[j] - lr_t * mj / (sqrtf(vj) + kEps);
    t32[j] = p;
    t16[j] = float_to_half(p);
}

__device__ __forceinline__ uint16_t bf16_of(float f) { return (uint16_t)bf16_bits(f); }

__global__ void k_pack(const float* __restrict__ master, uint16_t* __restrict__ wn, uint16_t* __restrict__ wk) {
    const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    const bool fwd = e < (uint32_t)kWnSize;
    if (e >= (uint32_t)(kWnSize + kWkSize)) return;
    uint32_t local = fwd ? e : e - kWnSize;
    int L = 0;
#pragma unroll
    for (int l = 0; l < kLayers; l++) {
        const uint32_t off = fwd ? (uint32_t)wn_offset(l) : (uint32_t)wk_offset(l);
        if (local >= off) L = l;
    }
    local -= fwd ? (uint32_t)wn_offset(L) : (uint32_t)wk_offset(L);
    const int K = kK[L], N = kN[L];
    const int i = local & 7, lane = (local >> 3) & 63, frag = local >> 9;
    const int g = lane >> 4, r = lane & 15;
    int in, out;
    if (fwd) {
        const int S = K / 32;
        const int t = frag / S, s = frag % S;
        in = 32 * s + 16 * (i >> 2) + 4 * g + (i & 3);
        out = 16 * t + r;
    } else {
        const int S = nk_cols(L) / 32;
        const int t = frag / S, s = frag % S;
        in = 16 * t + r;
        out = 32 * s + 16 * (i >> 2) + 4 * g + (i & 3);
    }
    const uint16_t v = out < N ? bf16_of(master[master_offset(L) + in * N + out]) : (uint16_t)0;
    if (fwd)
        wn[e] = v;
    else
        wk[e - kWnSize] = v;
}

__global__ void k_fill(float* p, uint32_t n, float value) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) p[j] = value;
}

__global__ void k_f32_to_f16(const float* __restrict__ a, uint16_t* __restrict__ b, uint32_t n) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) b[j] = float_to_half(a[j]);
}

__global__ void k_f16_to_f32(const uint16_t* __restrict__ a, float* __restrict__ b, uint32_t n) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) b[j] = half_to_float(a[j]);
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------

static inline uint32_t blocks_for(uint32_t n, uint32_t per) { return (n + per - 1) / per; }

hipError_t launch_infer(const NrcDev& d, const float4* queries, float4* out, const uint32_t* d_count, uint32_t count,
                        hipStream_t stream) {
    if (count == 0) return hipSuccess;
    // as many tiles per wave as let the whole batch be resident (8 waves per
    // CU), so that its waves take the levels together: 1 tile per wave at
    // 460,001 queries takes 221 us, 4 take 137.  A batch of more than that
    // starts a wave at the first level while others are at the last; six, all
    // that LDS holds, then gather the most per line: 2,000,000 queries take
    // 590 us, 675 with four.
    const uint32_t waves = (uint32_t)device_cu_count() * 8u;
    const uint32_t tiles = blocks_for(count, 64);
    const uint32_t per_wave = tiles <= waves ? 1u : (tiles <= 2 * waves ? 2u : (tiles <= 4 * waves ? 4u : 6u));
    const dim3 grid(blocks_for(tiles, per_wave)), block(64);
    if (count <= 16)
        hipLaunchKernelGGL((k_nrc_infer<1, true>), grid, block, 0, stream, d, queries, out, d_count, count);
    else if (per_wave == 1)
        hipLaunchKernelGGL((k_nrc_infer<1, false>), grid, block, 0, stream, d, queries, out, d_count, count);
    else if (per_wave == 2)
        hipLaunchKernelGGL((k_nrc_infer<2, false>), grid, block, 0, stream, d, queries, out, d_count, count);
    else if (per_wave == 4)
        hipLaunchKernelGGL((k_nrc_infer<4, false>), grid, block, 0, stream, d, queries, out, d_count, count);
    else
        hipLaunchKernelGGL((k_nrc_infer<6, false>), grid, block, 0, stream, d, queries, out, d_count, count);
    return hipGetLastError();
}

hipError_t launch_train(const NrcDev& d, const float4* queries, const float4* targets, const uint32_t* d_count,
                        uint32_t count, uint32_t slice, uint32_t slices, float* partial, uint32_t max_blocks,
                        float* grad_table, float* loss, uint32_t* blocks, hipStream_t stream) {
    hipLaunchKernelGGL(k_fill, dim3(1), dim3(64), 0, stream, loss, 1u, 0.0f);
    // with a device-resident count the grid covers the largest slice
    const uint32_t most = d_count ? blocks_for(count, slices) : count;
    const uint32_t chunks = blocks_for(most, kTrainQueriesPerWave);
    uint32_t nb = blocks_for(chunks, kTrainWaves);
    if (nb > max_blocks) nb = max_blocks;
    if (nb == 0) nb = 1;  // an empty slice still writes zero partials
    *blocks = nb;
    hipLaunchKernelGGL(k_nrc_train, dim3(nb), dim3(kTrainBlock), 0, stream, d, queries, targets, d_count, count, slice,
                       slices, partial, grad_table, loss);
    return hipGetLastError();
}

hipError_t launch_mlp_reduce(const float* partial, uint32_t blocks, float* grad_out, float* master, float* m, float* v,
                             uint16_t* wn, uint16_t* wk, float lr_t, hipStream_t stream) {
    hipLaunchKernelGGL(k_mlp_reduce, dim3(kMasterSize / kReduceWeights), dim3(kReduceWeights * kReduceWaves), 0, stream,
                       partial, blocks, grad_out, master, m, v, wn, wk, lr_t);
    return hipGetLastError();
}

hipError_t launch_table_adam(float* table32, uint16_t* table16, float* m, float* v, float* grad, uint32_t n,
                             float lr_t, hipStream_t stream) {
    hipLaunchKernelGGL(k_table_adam, dim3(blocks_for(n, 256)), dim3(256), 0, stream, table32, table16, m, v, grad, n,
                       lr_t);
    return hipGetLastError();
}

hipError_t launch_pack(const float* master, uint16_t* wn, uint16_t* wk, hipStream_t stream) {
    hipLaunchKernelGGL(k_pack, dim3(blocks_for(kWnSize + kWkSize, 256)), dim3(256), 0, stream, master, wn, wk);
    return hipGetLastError();
}

hipError_t launch_fill(float* p, uint32_t n, float value, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill, dim3(blocks_for(n, 256)), dim3(256), 0, stream, p, n, value);
    return hipGetLastError();
}

hipError_t launch_table_from_f32(const float* t32, uint16_t* t16, uint32_t n, hipStream_t stream) {
    hipLaunchKernelGGL(k_f32_to_f16, dim3(blocks_for(n, 256)), dim3(256), 0, stream, t32, t16, n);
    return hipGetLastError();
}

hipError_t launch_table_from_f16(const uint16_t* t16, float* t32, uint32_t n, hipStream_t stream) {
    hipLaunchKernelGGL(k_f16_to_f32, dim3(blocks_for(n, 256)), dim3(256), 0, stream, t16, t32, n);
    return hipGetLastError();
}

}  // namespace nrc
}  // namespace atlas_rt
