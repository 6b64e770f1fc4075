// Device bodies of the dense random-block steps, shared by the single-tensor kernels
// (conef_randblock.hip) and the one-launch-per-bucket kernels (conef_randblock_batch.hip).
// A body covers the workgroups [0, gx) of one tensor; `bx` is the workgroup's index among them.
#pragma once
#include "conef_device.h"

// The tensor goes by tiles of 1024 consecutive elements a quad of every thread, all of a tile's quads
// requested before the first is used.  A tile that holds none of the block - at the ratios that compress, nine
// in ten - takes no test per element; in the others the block is two ranges of the tile, and a quad inside one
// of them moves as a quad.  Pure streaming (dense error: 16 bytes an element, unbiased: 4), bounded by memory.
// The dense step reads and writes, and workgroups that do one after the other overlap best when they are many and
// short: with 1, 2 and 4 quads a thread 23.6, 24.8 and 28.1 us for 6.5 M elements, 171, 173 and 185 us for the
// step of an LSTM (33278 x 650), 159, 157 and 163 us for WRN-28-10's.  The unbiased step only writes.
constexpr int kRbEfQuads = 1, kRbUnbiasedQuads = 4;
constexpr int conef_rb_tile(int quads) { return 256 * 4 * quads; }

// The block's ranges [lo, hi) and [0, rest) relative to the tile at f0, and where in the payload the
// tile's element 0 would sit as part of the one and of the other.
template <int QUADS>
struct RbTile {
    static constexpr int kTile = conef_rb_tile(QUADS);
    int lo, hi, rest;
    int64_t at, at_rest;
    __device__ __forceinline__ RbTile(const ConefBlock& b, int64_t f0)
    {
        const int64_t l = b.start - f0, h = b.end - f0, r = b.rest - f0;
        lo = l < 0 ? 0 : l > kTile ? kTile : (int)l;
        hi = h < 0 ? 0 : h > kTile ? kTile : (int)h;
        rest = r < 0 ? 0 : r > kTile ? kTile : (int)r;
        at = f0 - b.start;
        at_rest = b.end - b.start + f0;
    }
    __device__ __forceinline__ bool touched() const { return hi > lo || rest > 0; }
    __device__ __forceinline__ bool inside(int e) const { return (e >= lo && e < hi) || e < rest; }
    __device__ __forceinline__ int64_t pos(int e) const { return (e < rest ? at_rest : at) + e; }
    // all four elements from e on in one of the ranges
    __device__ __forceinline__ bool whole(int e) const { return (e >= lo && e + 4 <= hi) || e + 4 <= rest; }
    __device__ __forceinline__ bool outside(int e) const { return (e + 4 <= lo || e >= hi) && e >= rest; }
};

// x = g + e;  selected: payload = x, out = x, e' = 0;  not selected: out = 0, e' = x.
// (RandomBlock_hook.py:182-184,222,228,237,240,276-280)
__device__ __forceinline__ void
conef_randblock_ef_body(float* __restrict__ x, float* __restrict__ err, float* __restrict__ payload, int64_t numel,
                        ConefBlock blk, int bx, int gx)
{
    constexpr int kTile = conef_rb_tile(kRbEfQuads);
    const int64_t tiles = (numel + kTile - 1) / kTile;
    const float zero[4] = {0.f, 0.f, 0.f, 0.f};
    for (int64_t t = bx; t < tiles; t += gx) {
        const int64_t f0 = t * kTile;
        float* xt = x + f0;
        float* et = err + f0;
        const RbTile<kRbEfQuads> in(blk, f0);
        if (f0 + kTile <= numel) {
            float g[kRbEfQuads][4], e[kRbEfQuads][4];
#pragma unroll
            for (int u = 0; u < kRbEfQuads; ++u) {
                const int i = 4 * (threadIdx.x + 256 * u);
                conef_ld4u(xt + i, g[u]);
                conef_ld4u(et + i, e[u]);
            }
            const bool touched = in.touched();
#pragma unroll
            for (int u = 0; u < kRbEfQuads; ++u) {
                const int i = 4 * (threadIdx.x + 256 * u);
                float xq[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) xq[k] = __fadd_rn(g[u][k], e[u][k]);
                if (!touched || in.outside(i)) {
                    conef_st4u(xt + i, zero);
                    conef_st4u(et + i, xq);
                } else if (in.whole(i)) {
                    conef_st4u(xt + i, xq);
                    conef_st4u(et + i, zero);
                    conef_st4u(payload + in.pos(i), xq);
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const bool sel = in.inside(i + k);
                        if (sel) payload[in.pos(i + k)] = xq[k];
                        xt[i + k] = sel ? xq[k] : 0.f;
                        et[i + k] = sel ? 0.f : xq[k];
                    }
                }
            }
        } else {
            const int left = (int)(numel - f0);
            for (int i = threadIdx.x; i < left; i += 256) {
                const float xq = __fadd_rn(xt[i], et[i]);
                const bool sel = in.inside(i);
                if (sel) payload[in.pos(i)] = xq;
                xt[i] = sel ? xq : 0.f;
                et[i] = sel ? 0.f : xq;
            }
        }
    }
}

// selected: payload = x / prob, out = payload;  not selected: out = 0 (written, never read)
// (UnbiasedRandomBlock_hook.py:155,161-167,200-204)
__device__ __forceinline__ void
conef_randblock_unbiased_body(float* __restrict__ x, float* __restrict__ payload, int64_t numel, ConefBlock blk,
                              float prob, int bx, int gx)
{
    constexpr int kTile = conef_rb_tile(kRbUnbiasedQuads);
    const int64_t tiles = (numel + kTile - 1) / kTile;
    const float zero[4] = {0.f, 0.f, 0.f, 0.f};
    for (int64_t t = bx; t < tiles; t += gx) {
        const int64_t f0 = t * kTile;
        float* xt = x + f0;
        const RbTile<kRbUnbiasedQuads> in(blk, f0);
        if (f0 + kTile <= numel) {
            if (!in.touched()) {
#pragma unroll
                for (int u = 0; u < kRbUnbiasedQuads; ++u) conef_st4u(xt + 4 * (threadIdx.x + 256 * u), zero);
                continue;
            }
            float g[kRbUnbiasedQuads][4];
#pragma unroll
            for (int u = 0; u < kRbUnbiasedQuads; ++u) conef_ld4u(xt + 4 * (threadIdx.x + 256 * u), g[u]);
#pragma unroll
            for (int u = 0; u < kRbUnbiasedQuads; ++u) {
                const int i = 4 * (threadIdx.x + 256 * u);
                if (in.whole(i)) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) g[u][k] = __fdiv_rn(g[u][k], prob);
                    conef_st4u(payload + in.pos(i), g[u]);
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        if (in.inside(i + k)) {
                            g[u][k] = __fdiv_rn(g[u][k], prob);
                            payload[in.pos(i + k)] = g[u][k];
                        } else {
                            g[u][k] = 0.f;
                        }
                    }
                }
                conef_st4u(xt + i, g[u]);
            }
        } else {
            const int left = (int)(numel - f0);
            for (int i = threadIdx.x; i < left; i += 256) {
                float o = 0.f;
                if (in.inside(i)) {
                    o = __fdiv_rn(xt[i], prob);
                    payload[in.pos(i)] = o;
                }
                xt[i] = o;
            }
        }
    }
}

// workgroups of a tensor of `numel` elements
inline int conef_rb_groups(int64_t numel, int quads)
{
    const int64_t g = (numel + conef_rb_tile(quads) - 1) / conef_rb_tile(quads);
    return (int)(g < 1 ? 1 : g > 16384 ? 16384 : g);
}
