// PowerSGD products at rank 16..32 on the matrix cores (v_mfma_f32_32x32x2f32: true fp32 inputs and
// accumulation, so the 1e-5 parity bar of the rank 1..8 streaming kernels holds here too).
//
// At these ranks a thread-per-column-quad kernel re-reads 4*r floats of Q (or P) for every 16 bytes
// of M it streams: the L2 -> CU traffic is 8..16 times the HBM traffic and the kernels fall to a
// twentieth of the HBM rate.  An MFMA tile shares one operand over 32 rows (or columns) of M
// instead, and the products are HBM-bound again: 2*r flops per 4 bytes of M is 16 flop/byte at
// r = 32, just below the fp32 ridge of the machine (157 TFLOP/s over 8 TB/s).
//
// Operand layout of v_mfma_f32_32x32x2f32 (D[32x32] += A[32x2] * B[2x32], one float per lane):
//   A: lane l holds A[l % 32][l / 32]          B: lane l holds B[l / 32][l % 32]
//   D: lane l, register v holds D[8 * (v / 4) + 4 * (l / 32) + v % 4][l % 32]
// The two k of a step only have to agree between A and B, not to be adjacent in memory, so a lane
// may feed consecutive steps from one 16-byte load: the kernels below pick k per lane half that way.
#pragma once
#include "conef_device.h"
#include "conef_sketch_core.h"
#include <type_traits>

typedef float conef_f16v __attribute__((ext_vector_type(16)));

__device__ __forceinline__ conef_f16v conef_mfma32(float a, float b, conef_f16v c)
{
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ int conef_mfma_row(int v, int lane) { return 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3); }

constexpr int kMfmaWaves = 4;
constexpr int kMfmaThreads = 64 * kMfmaWaves;

// ------------------------------------------------------------------ P = X Q ----
// MODE 0: X = M.  MODE 1: X = M + E, written back.  MODE 2: X = M + alpha * unsketch(cs), written
// back (the sketch rows of the tile's 32 matrix rows are parked in LDS).
// A workgroup owns 32 rows and the column range [blockIdx.y * cols_per_split, +cols_per_split); its
// four waves take 32-column blocks of that range in turn.  Lane (row = l % 32, half = l / 32) loads
// X[row][c .. c+3] with c = block + 8u + 4 * half for u = 0..3 and feeds step (u, j) with component j;
// the matching B operand is Q[c + j][l % 32].  The waves' tiles meet in LDS in a fixed order; with
// more than one column split the tile goes to a partial buffer [split][n][r] that a second kernel
// adds up in split order.  Rows of any length from four up and any alignment: a row's last quad is
// moved back to end with the row (conef_quad_col), its columns that are the quad's before it count
// as zeros.  EXACT: m % 4 == 0, no quad is moved (the tests for one cost 0.5 of 13.1 us on BERT's buckets
// at rank 32).
template <int MODE, bool EXACT>
__device__ __forceinline__ void
psgd_mfma_mq_body(float* __restrict__ x, const float* __restrict__ err, const float* __restrict__ cs,
                  const uint32_t* __restrict__ pktab, const float* __restrict__ q, float* __restrict__ out, int64_t n,
                  int m, int r, int cols_per_split, ConefMod mod, float alpha, ConefSeeds hs, int bx, int by)
{
    extern __shared__ float mfma_lds[];
    float* red = mfma_lds;                              // [kMfmaWaves][16][64]
    float* cells = mfma_lds + kMfmaWaves * 16 * 64;     // [32][w], MODE 2 only
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int lrow = lane & 31, half = lane >> 5;
    const int64_t row0 = (int64_t)bx * 32;
    const int64_t row = row0 + lrow < n ? row0 + lrow : n - 1;     // clamped for loads, stores are guarded
    const bool row_ok = row0 + lrow < n;
    const int w = (int)mod.w;
    if (MODE == 2) {
        for (int e = threadIdx.x; e < 32 * w; e += kMfmaThreads) {
            int a = e / w;
            int64_t rr = row0 + a < n ? row0 + a : n - 1;
            cells[e] = cs[rr * w + (e - a * w)];
        }
        __syncthreads();
    }
    const int c_begin = by * cols_per_split;
    const int c_end = c_begin + cols_per_split < m ? c_begin + cols_per_split : m;
    const bool rank_ok = lrow < r;
    conef_f16v acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float* xrow = x + row * m;
    const float* erow = MODE == 1 ? err + row * m : nullptr;
    // One stage = half a 32-column block: every load of a stage is issued before the previous stage's
    // products, so a wave always has a stage's worth of loads in flight while it multiplies.  A stage is the wave's, so its
    // place is a scalar; a whole one has no columns to leave out.  (Whole blocks with an address and a test a load: an encoder
    // of 1024 with dense errors 571 us a step at rank 16, now 557, the LSTM 554 and 536, WRN-16-5 95.5 and 90.4.)
    // MODE 2 looks up cells between its loads and its products and stays with whole blocks: half blocks and these, us, rank 32,
    // with a plan and without, sketches of a tenth: [30522,1024] 101.2 and 89.4, 110.7 and 106.9; [33278,650] 88.5 and 76.9, 103.7
    // and 87.9; [17000,1001] 78.1 and 73.7, 81.8 and 79.1 ([100000,130], a block and two columns, 36.5 and 40.4, 47.7 and 55.8).
    constexpr int U = MODE == 2 ? 4 : 2;
    struct Stage {
        float xv[U][4], ev[MODE == 1 ? U : 1][4], qv[U][4];
        uint32_t pk[MODE == 2 ? U : 1][4];
    };
    const uint32_t qo = (4u * half * (uint32_t)r + (rank_ok ? (uint32_t)lrow : 0u)) * 4u;
    auto load = [&](Stage& st, int cb) {
        if (MODE != 2 && cb + 8 * U <= c_end) {
            const char* qb = reinterpret_cast<const char*>(q + (int64_t)cb * r);
            const float* xl = xrow + 4 * half + cb;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                conef_ld4u(xl + 8 * u, st.xv[u]);
                if constexpr (MODE == 1) conef_ld4u(erow + 4 * half + cb + 8 * u, st.ev[u]);
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
            if constexpr (MODE == 1) conef_ld4u(erow + cc, st.ev[u]);
            if constexpr (MODE == 2) {
                if (pktab) {
                    conef_ld4u(pktab + cc, st.pk[u]);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) st.pk[u][j] = conef_bucket_sign(cc + j, mod, hs.a, hs.b, hs.sa, hs.sb);
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) st.qv[u][j] = q[(int64_t)(cc + j) * r + (rank_ok ? lrow : 0)];
        }
    };
    auto compute = [&](Stage& st, int cb) {
        if (MODE != 2 && cb + 8 * U <= c_end) {         // (columns of Q from r on are some other's: what they make is not stored)
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if constexpr (MODE == 1) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) st.xv[u][j] = __fadd_rn(st.xv[u][j], st.ev[u][j]);
                    if (row_ok) conef_st4u(xrow + 4 * half + cb + 8 * u, st.xv[u]);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) acc = conef_mfma32(st.xv[u][j], st.qv[u][j], acc);
            }
            return;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = cb + 8 * u + 4 * half;
            const bool ok = c < c_end;
            const int dup = !EXACT && ok && c + 4 > m ? c - (m - 4) : 0;
            if constexpr (MODE == 1) {
#pragma unroll
                for (int j = 0; j < 4; ++j) st.xv[u][j] = __fadd_rn(st.xv[u][j], st.ev[u][j]);
            }
            if constexpr (MODE == 2) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    st.xv[u][j] = __fadd_rn(st.xv[u][j], conef_query_term(cells[lrow * w + (st.pk[u][j] & 0x7fffffffu)],
                                                                          st.pk[u][j], alpha));
            }
            if (MODE != 0 && ok && row_ok) conef_st4_own(xrow + c - dup, st.xv[u], dup);
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
    if (cb < c_end) {
        Stage s0, s1;
        load(s0, cb);
        while (true) {
            const int nb = cb + (MODE == 2 ? 2 : 1) * kStep, hb = cb + (MODE == 2 ? kStep : 8 * U);
            if (hb < c_end) load(s1, hb);
            compute(s0, cb);
            if (nb < c_end) load(s0, nb);
            if (hb < c_end) compute(s1, hb);
            if (nb >= c_end) break;
            cb = nb;
        }
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) red[(wave * 16 + v) * 64 + lane] = acc[v];
    __syncthreads();
    float* dst = out + (int64_t)by * n * r;
    for (int e = threadIdx.x; e < 16 * 64; e += kMfmaThreads) {
        const int v = e >> 6, l = e & 63;
        float s = (red[e] + red[16 * 64 + e]) + (red[2 * 16 * 64 + e] + red[3 * 16 * 64 + e]);
        const int64_t i = row0 + conef_mfma_row(v, l);
        const int j = l & 31;
        if (i < n && j < r) dst[i * r + j] = s;
    }
}

template <int MODE>
__global__ void __launch_bounds__(kMfmaThreads)
psgd_mfma_mq_kernel(float* __restrict__ x, const float* __restrict__ err, const float* __restrict__ cs,
                    const uint32_t* __restrict__ pktab, const float* __restrict__ q, float* __restrict__ out, int64_t n,
                    int m, int r, int cols_per_split, ConefMod mod, float alpha, ConefSeeds hs)
{
    psgd_mfma_mq_body<MODE, false>(x, err, cs, pktab, q, out, n, m, r, cols_per_split, mod, alpha, hs, (int)blockIdx.x,
                            (int)blockIdx.y);
}

// -------------------------------------------------------------- Q = X^T P ----
// D[c][j] = sum_i X[i][c] P[i][j]: A[c][k] = X[i0 + k][c] is a row of X read along its columns, so
// the loads are contiguous as they come.  A wave owns 32 * V columns (V floats per lane: lane
// (q = l % 32, half) reads X[i][c0 + V*q .. + V) of row i = pair + half) and keeps V tiles, tile t
// for the columns c0 + V*q + t; a step consumes two rows.  The four waves of a workgroup split the
// rows of the slab, meet in LDS, and the slab's tile is stored (one slab) or left as a partial.
// Any alignment, any m >= V: the last run of V columns is moved back to end with the row (columns
// two lanes then hold come out of both the same).
// LOOK: X = M + alpha * unsketch(cs), formed here (conef_psgd_look.h).
// red: the workgroup's place in LDS for the waves' tiles, given by the kernel: one that takes every V has one for all.
struct MfmaLook {
    const float* cs;         // [n, w]
    const uint32_t* pk;      // bucket and sign of every column
    int w;
    float alpha;
};

template <int V, bool LOOK = false>
__device__ __forceinline__ void
psgd_mfma_mtp_body(float (*red)[16][64], const float* __restrict__ x, const float* __restrict__ p, float* __restrict__ out, int64_t n,
                   int m, int r, int rows_per_slab, int bx, int by, MfmaLook look = {})
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int lq = lane & 31, half = lane >> 5;
    const int c0 = bx * 32 * V;
    const int c = c0 + V * lq;
    const bool col_ok = c < m;
    const int cc = col_ok ? (c + V <= m ? c : m - V) : 0;
    // Rows are counted from the slab's first, in 32 bits: a wave's place is a scalar, and 64-bit compares and selections of scalars
    // are chains of instructions, ahead of a stage's loads.  Rank 32, us, with 64 bits and so: [1024,1024] 7.3 and 6.9, [300,9000]
    // 11.6 and 11.0, [4096,4096] 24.5 and 23.5, [30522,1024] 39.3 and 37.6 (a lane's own 64-bit place: 6.9, 11.0, 25.3, 40.7).
    const int64_t i0 = (int64_t)by * rows_per_slab;
    const int rows = i0 + rows_per_slab < n ? rows_per_slab : (int)(n - i0);
    x += i0 * m;
    p += i0 * r;
    const float* const slab_cells = LOOK ? look.cs + i0 * look.w : nullptr;
    const bool rank_ok = lq < r;
    conef_f16v acc[V];
#pragma unroll
    for (int t = 0; t < V; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[t][v] = 0.f;
    // A wave takes 2 UC rows, then those 2 UC kMfmaWaves on; a stage is half of them, which with the tiles of four column runs
    // and LOOK's cells fits the registers of four workgroups a CU (124 and 126 of 128 at ranks 16 and 32).
    constexpr int UC = V == 4 ? 4 : 8, U = UC / 2;
    struct Stage {
        float xv[U][V], pv[U], cv[U][LOOK ? V : 1];
    };
    uint32_t pk[V];
    if constexpr (LOOK) {
#pragma unroll
        for (int t = 0; t < V; ++t) pk[t] = look.pk[cc + t];
    }
    // A pair of rows is the wave's, so its place is a scalar; a lane adds where it reads from there (rows with a plan of
    // row lists, which LOOK asks for, are short: 32 bits do).
    using Offset = std::conditional_t<LOOK, uint32_t, int64_t>;
    const Offset xo = (Offset)half * (Offset)m + (Offset)cc, po = (Offset)half * (Offset)r + (Offset)(rank_ok ? lq : 0);
    auto load = [&](Stage& st, int ib) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // past the slab: a valid row, its products are zeroed
            const int i = ib + 2 * u < rows ? ib + 2 * u : 0;
            const bool second = i + 1 < rows;
            const float* src = x + (int64_t)i * m + (second ? xo : (Offset)cc);
            if constexpr (V == 4) {
                conef_ld4u(src, st.xv[u]);
            } else if constexpr (V == 2) {
                conef_f2u t = *reinterpret_cast<const conef_f2u*>(src);
                st.xv[u][0] = t.x; st.xv[u][1] = t.y;
            } else {
                st.xv[u][0] = *src;
            }
            st.pv[u] = (p + (int64_t)i * r)[second ? po : (Offset)(rank_ok ? lq : 0)];
            if constexpr (LOOK) {
                const float* cells = slab_cells + (int64_t)i * look.w;
                const uint32_t below = second && half ? (uint32_t)look.w : 0u;
#pragma unroll
                for (int t = 0; t < V; ++t) st.cv[u][t] = cells[(pk[t] & 0x7fffffffu) + below];
            }
        }
    };
    auto compute = [&](Stage& st, int ib) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool ok = ib + 2 * u + half < rows;
            if constexpr (LOOK) {
#pragma unroll
                for (int t = 0; t < V; ++t) st.xv[u][t] = __fadd_rn(st.xv[u][t], conef_query_term(st.cv[u][t], pk[t], look.alpha));
            }
            const float b = (ok && rank_ok) ? st.pv[u] : 0.f;
#pragma unroll
            for (int t = 0; t < V; ++t) acc[t] = conef_mfma32((ok && col_ok) ? st.xv[u][t] : 0.f, b, acc[t]);
        }
    };
    constexpr int kStep = 2 * kMfmaWaves * UC;
    int ib = 2 * wave * UC;
    if (ib < rows) {
        Stage s0, s1;
        load(s0, ib);
        while (true) {
            const int nb = ib + kStep, hb = ib + 2 * U;
            if (hb < rows) load(s1, hb);
            compute(s0, ib);
            if (nb < rows) load(s0, nb);
            if (hb < rows) compute(s1, hb);
            if (nb >= rows) break;
            ib = nb;
        }
    }
    float* dst = out + (int64_t)by * m * r;
#pragma unroll
    for (int t = 0; t < V; ++t) {
        if (t) __syncthreads();
#pragma unroll
        for (int v = 0; v < 16; ++v) red[wave][v][lane] = acc[t][v];
        __syncthreads();
        for (int e = threadIdx.x; e < 16 * 64; e += kMfmaThreads) {
            const int v = e >> 6, l = e & 63;
            const float* rr = &red[0][0][0];
            float s = (rr[e] + rr[16 * 64 + e]) + (rr[2 * 16 * 64 + e] + rr[3 * 16 * 64 + e]);
            const int cq = c0 + V * conef_mfma_row(v, l);                // the lane's run of columns, as it was loaded
            const int col = (cq + V <= m ? cq : m - V) + t;
            const int j = l & 31;
            if (cq < m && j < r) dst[(int64_t)col * r + j] = s;
        }
    }
}

template <int V>
__global__ void __launch_bounds__(kMfmaThreads)
psgd_mfma_mtp_kernel(const float* __restrict__ x, const float* __restrict__ p, float* __restrict__ out, int64_t n, int m,
                     int r, int rows_per_slab)
{
    __shared__ float red[kMfmaWaves][16][64];
    psgd_mfma_mtp_body<V>(red, x, p, out, n, m, r, rows_per_slab, (int)blockIdx.x, (int)blockIdx.y);
}

// ------------------------------------------------------------ M = P Q^T ----
// D[i][c] = sum_k P[i][k] Q[c][k] with K = R (16 or 32): R/2 steps per 32x32 tile.  Lane
// (t = l % 32, half) supplies k = half * R/2 + s at step s for both operands, so its slice of a
// row of P (and of Q) is R/2 consecutive floats: 16-byte loads.  A wave keeps the Q operand of its
// 32 columns in registers and walks the row tiles of its slab; a half-wave stores 128 contiguous
// bytes of a row of M.  MODE 1 also writes the residual E = X - M (X = what M held on entry).
template <int R, int MODE>
__device__ __forceinline__ void
psgd_mfma_pqt_body(float* __restrict__ x, float* __restrict__ err, const float* __restrict__ p,
                   const float* __restrict__ q, int64_t n, int m, int rows_per_slab, int bx, int by)
{
    constexpr int KS = R / 2;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int lt = lane & 31, half = lane >> 5;
    const int c = (bx * kMfmaWaves + wave) * 32 + lt;
    if ((bx * kMfmaWaves + wave) * 32 >= m) return;        // whole wave past the edge (no barriers below)
    const bool col_ok = c < m;
    float qb[KS];
    {
        const float* src = q + (int64_t)(col_ok ? c : m - 1) * R + half * KS;
#pragma unroll
        for (int s = 0; s < KS; s += 4) {
            conef_ld4u(src + s, qb + s);
        }
    }
    const int64_t i0 = (int64_t)by * rows_per_slab;
    const int64_t i1 = i0 + rows_per_slab < n ? i0 + rows_per_slab : n;
    for (int64_t ib = i0; ib < i1; ib += 32) {
        float pa[KS], xv[16];
        {
            const int64_t i = ib + lt < n ? ib + lt : n - 1;
            const float* src = p + i * R + half * KS;
#pragma unroll
            for (int s = 0; s < KS; s += 4) {
                conef_ld4u(src + s, pa + s);
            }
        }
        if (MODE == 1) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int64_t i = ib + conef_mfma_row(v, lane);
                xv[v] = x[(i < i1 ? i : i1 - 1) * m + (col_ok ? c : m - 1)];
            }
        }
        conef_f16v acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; ++s) acc = conef_mfma32(pa[s], qb[s], acc);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int64_t i = ib + conef_mfma_row(v, lane);
            if (i < i1 && col_ok) {
                if (MODE == 1) __builtin_nontemporal_store(__fsub_rn(xv[v], acc[v]), err + i * m + c);
                __builtin_nontemporal_store(acc[v], x + i * m + c);
            }
        }
    }
}

template <int R, int MODE>
__global__ void __launch_bounds__(kMfmaThreads)
psgd_mfma_pqt_kernel(float* __restrict__ x, float* __restrict__ err, const float* __restrict__ p,
                     const float* __restrict__ q, int64_t n, int m, int rows_per_slab)
{
    psgd_mfma_pqt_body<R, MODE>(x, err, p, q, n, m, rows_per_slab, (int)blockIdx.x, (int)blockIdx.y);
}
