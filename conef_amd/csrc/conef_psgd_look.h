// X = M + alpha * unsketch(cs) formed where it is read (ranks 9 to 32, rounds whose last launch sketches the residual):
// the products and the residual read M as the gradient came, with the sketch's cells, and X is never written.  Laid out by a
// launch of its own it cost 12 bytes an element where the first product needs 4: 17.7 + 14.3 us a BERT bucket at rank 32, now
// 18.9 (14 with M in the Infinity Cache; written by the first product instead 22).  The other two look the cells up at
// their own cost: Q = X^T P gathers them from global memory (a lane has four columns of a row: 11.1 us -> 13.3), the residual's
// tile holds them in LDS anyway.
#pragma once
#include "conef_device.h"
#include "conef_psgd_mfma.h"

// ------------------------------------------------------------------ P = X Q ----
// psgd_mfma_mq_body with X formed from M, G column splits of a row tile to a workgroup (a group of kMfmaWaves waves
// each, its splits, blocks and sums those of a workgroup there: the same bits).  The 32 rows' cells wait in LDS, rows of an odd number of floats: the
// lanes of a half read the same bucket of 32 rows.
constexpr int look_cells_stride(int w) { return w | 1; }

template <bool EXACT, int G>
__device__ __forceinline__ void
psgd_mfma_look_mq_body(const float* __restrict__ x, const float* __restrict__ cs, const uint32_t* __restrict__ pktab,
                       const float* __restrict__ q, float* __restrict__ out, int64_t n, int m, int r, int w, int cols_per_split, int splits,
                       float alpha, int bx, int by)
{
    extern __shared__ float look_lds[];                 // [32][stride], then [G][kMfmaWaves][16][64]
    constexpr int T = G * kMfmaThreads;
    const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / kMfmaThreads);
    const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) % kMfmaWaves), lane = threadIdx.x & 63;
    const int lrow = lane & 31, half = lane >> 5;
    const int64_t row0 = (int64_t)bx * 32;
    const int64_t row = row0 + lrow < n ? row0 + lrow : n - 1;     // clamped: the sums of the others are not stored
    const int split = by * G + group;
    const int c_begin = split < splits ? split * cols_per_split : m;
    const int c_end = c_begin + cols_per_split < m ? c_begin + cols_per_split : m;
    const bool rank_ok = lrow < r;
    const int stride = look_cells_stride(w);
    const float* xrow = x + row * m;
    // A stage is half a block of 32 columns.  With whole blocks, 64-bit addresses of every lane's and tests of every quad an
    // encoder of 1024 took 441 us a step at rank 16, now 425, the LSTM 362 and 346, BERT's shapes at rank 32 749 and 726.
    constexpr int U = 2;
    struct Stage {
        float xv[U][4], qv[U][4];
        uint32_t pk[U][4];
    };
    // A stage is the wave's, so its place is a scalar, and a lane adds bytes that fit 32 bits (rows with a plan of row lists are
    // short); a whole stage has no columns to leave out.
    const char* xtile = reinterpret_cast<const char*>(x + row0 * m);
    const uint32_t xo = ((uint32_t)(row - row0) * (uint32_t)m + 4u * half) * 4u, po = 16u * half;
    const uint32_t qo = (4u * half * (uint32_t)r + (rank_ok ? (uint32_t)lrow : 0u)) * 4u;
    auto load = [&](Stage& st, int cb) {
        if (cb + 8 * U <= c_end) {
            const char* xb = xtile + 4 * (int64_t)cb;
            const char* pb = reinterpret_cast<const char*>(pktab + cb);
            const char* qb = reinterpret_cast<const char*>(q + (int64_t)cb * r);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                conef_ld4u(reinterpret_cast<const float*>(xb + 32 * u + xo), st.xv[u]);
                conef_ld4u(reinterpret_cast<const uint32_t*>(pb + 32 * u + po), st.pk[u]);
#pragma unroll
                for (int j = 0; j < 4; ++j) st.qv[u][j] = *reinterpret_cast<const float*>(qb + 4 * (8 * u + j) * (int64_t)r + qo);
            }
            return;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = cb + 8 * u + 4 * half;
            const int ce = c < c_end ? c : c_begin;     // past the end: a valid quad, its products are zeroed
            const int cc = EXACT || ce + 4 <= m ? ce : m - 4;
            conef_ld4u(xrow + cc, st.xv[u]);
            conef_ld4u(pktab + cc, st.pk[u]);
#pragma unroll
            for (int j = 0; j < 4; ++j) st.qv[u][j] = q[(int64_t)(cc + j) * r + (rank_ok ? lrow : 0)];
        }
    };
    conef_f16v acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    auto compute = [&](Stage& st, int cb) {
        if (cb + 8 * U <= c_end) {                      // (columns of Q from r on are some other's: what they make is not stored)
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float a = __fadd_rn(st.xv[u][j], conef_query_term(look_lds[lrow * stride + (st.pk[u][j] & 0x7fffffffu)],
                                                                            st.pk[u][j], alpha));
                    acc = conef_mfma32(a, st.qv[u][j], acc);
                }
            return;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = cb + 8 * u + 4 * half;
            const bool ok = c < c_end;
            const int dup = !EXACT && ok && c + 4 > m ? c - (m - 4) : 0;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                st.xv[u][j] = __fadd_rn(st.xv[u][j], conef_query_term(look_lds[lrow * stride + (st.pk[u][j] & 0x7fffffffu)],
                                                                      st.pk[u][j], alpha));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float a = ok && (EXACT || j >= dup) ? st.xv[u][j] : 0.f;
                float b = (ok && rank_ok) ? st.qv[u][j] : 0.f;
                acc = conef_mfma32(a, b, acc);
            }
        }
    };
    constexpr int kStep = kMfmaWaves * 32;
    int cb = c_begin + wave * 32;
    Stage s0, s1;
    if (cb < c_end) load(s0, cb);                       // travels with the cells
    {
        const int rows = n - row0 < 32 ? (int)(n - row0) : 32;
        const float* src = cs + row0 * w;
        const int count = rows * w;
        constexpr int kPark = 8;
        for (int i0 = threadIdx.x; i0 < count; i0 += kPark * T) {
            float t[kPark];
#pragma unroll
            for (int u = 0; u < kPark; ++u) t[u] = src[i0 + u * T < count ? i0 + u * T : count - 1];
#pragma unroll
            for (int u = 0; u < kPark; ++u) {
                const int i = i0 + u * T, a = i / w;
                if (i < count) look_lds[a * stride + (i - a * w)] = t[u];
            }
        }
        for (int i = count + threadIdx.x; i < 32 * w; i += T) look_lds[i / w * stride + i % w] = 0.f;      // rows past the end
    }
    __syncthreads();
    if (cb < c_end) {
        while (true) {
            const int nb = cb + kStep, hb = cb + 8 * U;
            if (hb < c_end) load(s1, hb);
            compute(s0, cb);
            if (nb < c_end) load(s0, nb);
            if (hb < c_end) compute(s1, hb);
            if (nb >= c_end) break;
            cb = nb;
        }
    }
    __syncthreads();                                    // the cells' place is free
    float* red = look_lds + group * kMfmaWaves * 16 * 64;
#pragma unroll
    for (int v = 0; v < 16; ++v) red[(wave * 16 + v) * 64 + lane] = acc[v];
    __syncthreads();
    if (split >= splits) return;
    float* dst = out + (int64_t)split * n * r;
    for (int e = threadIdx.x % kMfmaThreads; e < 16 * 64; e += kMfmaThreads) {
        const int v = e >> 6, l = e & 63;
        float s = (red[e] + red[16 * 64 + e]) + (red[2 * 16 * 64 + e] + red[3 * 16 * 64 + e]);
        const int64_t i = row0 + conef_mfma_row(v, l);
        const int j = l & 31;
        if (i < n && j < r) dst[i * r + j] = s;
    }
}
