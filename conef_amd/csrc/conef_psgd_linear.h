// The products of a PowerSGD round with a count-sketched error, without the error laid out (gfx950).
//
// The corrected gradient is X = M + alpha U(cs), U the unsketch (CountSketch.py:40-47): column j of row i gets
// s_j cs[i, h_j].  Both products are linear in it (powerSGD_hook.py:409,498,532):
//
//   P  = X Q    = M Q + alpha cs F(Q)        F(Q)[b] = sum over the columns j of bucket b of s_j Q[j]
//   Q' = X^T P  = M^T P + alpha (row h_j of cs^T P, times s_j)
//
// So M is only read until P Q'^T replaces it in the last pass, which forms X again from M and the old cells for
// the residual, term by term as before: the first product used to write X back into M (54 MB for a 27 MB bucket)
// and was bound by that.  The order of the sums is fixed: no atomics, the same result on every run.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "conef_device.h"
#include "conef_rowlist.h"
#include "conef_psgd_stream.h"

// ------------------------------------------------------------------ F(Q) ----
// RP floats of a row of F(Q) from a row-major Q with rows of `stride` floats, a bucket's columns in ascending
// order, U rows of Q requested together and the next U entries of the list with them.
template <int RP, int U>
__device__ __forceinline__ void conef_fold_row(const float* q, int stride, const uint16_t* ent, uint32_t e0, uint32_t e1, float* out)
{
    double f[RP];            // rounded once
#pragma unroll
    for (int c = 0; c < RP; ++c) f[c] = 0.;
    uint32_t next[U];
#pragma unroll
    for (int u = 0; u < U; ++u) next[u] = e0 < e1 ? ent[e0 + u < e1 ? e0 + u : e1 - 1] : 0u;
    for (uint32_t e = e0; e < e1; e += U) {
        uint32_t en[U];
        float v[U][RP];
#pragma unroll
        for (int u = 0; u < U; ++u) en[u] = next[u];
#pragma unroll
        for (int u = 0; u < U; ++u) next[u] = ent[e + U + u < e1 ? e + U + u : e1 - 1];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float* src = q + (int64_t)(en[u] & 0x7fffu) * stride;
            if constexpr (RP % 4 == 0) {
#pragma unroll
                for (int c = 0; c < RP; c += 4) conef_ld4u(src + c, v[u] + c);
            } else {
#pragma unroll
                for (int c = 0; c < RP; ++c) v[u][c] = src[c];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (e + u < e1) {
#pragma unroll
                for (int c = 0; c < RP; ++c) f[c] += (double)((en[u] & 0x8000u) ? v[u][c] : -v[u][c]);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < RP; ++c) out[c] = (float)f[c];
}

struct FoldItem {
    const float* q;          // [m, RP]
    const uint32_t* csr;
    const uint16_t* ent;
    float* f;                // [w, RP]
    int w;
};

// -------------------------------------------------------------- P = X Q ----
struct LinMqItem {
    const float* x;
    const float* cs;
    const float* q;
    const float* qi;         // not null: q laid out by quads (conef_load_slices)
    const float* fold;       // F(Q), [w, RP]
    const float* tmat;       // not null: the column steps that orthogonalise q (b_ij, then 1 / d_i), applied to the rows of P
    float* p;
    double* gram;            // workgroup g leaves its rows' share of P^T P at gram[g * RP (RP + 1) / 2]
    int n, m, w, r;          // r: the rank, at most RP
    int gw, rows;            // threads of a group; rows of a tile
};

struct LinMqShape {
    int T;                   // threads of a workgroup
    size_t lds;
    int64_t wgs;
};

inline int lin_mq_slabs(int64_t m, int w, int gw)
{
    const int64_t m4 = (m + 3) >> 2, a = (m4 + gw - 1) / gw, b = ((int64_t)w + gw - 1) / gw;
    return (int)(a > b ? a : b);
}

// LDS of a workgroup: the tile, its cells, the waves' sums, Q's steps, the tile's rows of P
inline size_t lin_mq_lds(int64_t m, int w, int gw, int rows, int T, int rp)
{
    const int groups = T / gw, per = ((rows + groups - 1) / groups + 1) & ~1;
    return (((size_t)rows * m + 7) & ~(size_t)3) * 4 + (((size_t)rows * w + 3) & ~(size_t)3) * 4 +
           (size_t)lin_mq_slabs(m, w, gw) * per * (T / 64) * rp * 4 + (size_t)rows * rp * 8 + (size_t)(rp + 1) * rp * 4 + 8;
}

// Fills in gw and rows of every item of one launch.  A tile holds about 8192 values of M (32 KB: four
// workgroups of 256 threads a CU, each with its whole tile requested at once), less where the launch
// would have fewer than 512 tiles.  Rows of more than 2048 columns take 512 threads.
inline bool lin_mq_plan(LinMqItem* items, int count, int rp, LinMqShape* s)
{
    s->T = 256;
    for (int k = 0; k < count; ++k)
        if (items[k].m > 2048) s->T = 512;
    for (int64_t target = 8192;; target >>= 1) {
        s->lds = 0;
        s->wgs = 0;
        for (int k = 0; k < count; ++k) {
            LinMqItem& it = items[k];
            it.gw = mqs_group_width(it.m, s->T);
            const int groups = s->T / it.gw;
            int64_t rows = target / it.m;
            rows = rows >= 2 * groups ? rows / (2 * groups) * (2 * groups) : 2 * groups;
            if (rows > 64) rows = 64;
            while (rows > 1 && lin_mq_lds(it.m, it.w, it.gw, (int)rows, s->T, rp) > 80 * 1024) rows >>= 1;
            it.rows = (int)rows;
            const size_t need = lin_mq_lds(it.m, it.w, it.gw, it.rows, s->T, rp);
            if (need > kConefRowlistLdsLimit) return false;
            if (need > s->lds) s->lds = need;
        }
        // Every workgroup of the launch takes the LDS of the largest.  Where few of those fit a CU, taller tiles for the
        // others, as long as no fewer do: [640, 5760] and [640, 2880] as 480 workgroups instead of 640, two a CU
        // either way, 11.2 against 14.9 us.
        const size_t room = kConefRowlistLdsLimit / (kConefRowlistLdsLimit / s->lds);
        for (int k = 0; k < count; ++k) {
            LinMqItem& it = items[k];
            while (room > 48 * 1024 && (int64_t)it.rows * 2 * it.m <= 12288 && it.rows * 2 <= 64 &&
                   lin_mq_lds(it.m, it.w, it.gw, it.rows * 2, s->T, rp) <= room)
                it.rows *= 2;
            const size_t need = lin_mq_lds(it.m, it.w, it.gw, it.rows, s->T, rp);
            if (need > s->lds) s->lds = need;
            s->wgs += (it.n + it.rows - 1) / it.rows;
        }
        if (s->wgs >= 512 || target <= 2048) return s->wgs <= 0x7fffffff;
    }
}

template <int RP, int T>
__device__ __forceinline__ void psgd_lin_mq_body(const LinMqItem& it, float alpha, int bx)
{
    constexpr int WAVES = T / 64;
    extern __shared__ __attribute__((aligned(16))) float lin_lds[];
    const int m = it.m, m4 = (m + 3) >> 2, w = it.w, gw = it.gw;
    const int groups = T / gw, per = (it.rows + groups - 1) / groups, per2 = (per + 1) & ~1;
    const int nslab = (m4 + gw - 1) / gw;
    const int cslab = (w + gw - 1) / gw, slabs = nslab > cslab ? nslab : cslab;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int64_t row0 = (int64_t)bx * it.rows;
    const int rows = it.n - row0 < it.rows ? (int)(it.n - row0) : it.rows;
    // The tile is one contiguous run.  Up to three leading elements bring it to a 16-byte boundary of memory;
    // in LDS it starts that far before one, so that both sides of the copy move 16 bytes.
    const float* base = it.x + row0 * m;
    const int total = rows * m;
    int lead = (int)(((16u - (unsigned)(reinterpret_cast<uintptr_t>(base) & 15u)) & 15u) >> 2);
    if (lead > total) lead = total;
    const int total4 = (total - lead) >> 2;
    float* vals = lin_lds + ((4 - lead) & 3);
    float* cells = lin_lds + ((it.rows * m + 7) & ~3);
    float* red = cells + ((it.rows * w + 3) & ~3);                  // [slabs][per2][WAVES][RP]
    float* t_l = red + (size_t)slabs * per2 * WAVES * RP;           // the column steps of Q
    double* prow = reinterpret_cast<double*>(t_l + ((RP * (RP + 1) + 1) & ~1));      // [rows][RP]

    // Everything is requested before anything is used, straight into LDS: the tile, its cells, Q's column steps.
    for (int q = tid; q < total4; q += T) conef_to_lds16(base + lead + 4 * q, vals + lead + 4 * (q - lane));
    const float* cell_src = it.cs + row0 * w;
    const int ncells = rows * w;
    for (int i = tid; i < ncells; i += T) conef_to_lds4(cell_src + i, cells + (i - lane));
    if (it.tmat && tid < RP * RP + RP) conef_to_lds4(it.tmat + tid, t_l + (tid - lane));
    const int rest = total - (total4 << 2);                // leading and trailing elements, at most six
    if (tid < rest) {
        const int e = tid < lead ? tid : tid + (total4 << 2);
        vals[e] = base[e];
    }
    // The products: a group of gw threads takes its rows a few at a time, a thread a column quad and a column of
    // the cells in every slab.  red[slab][row of the group][wave][rank] receives a wave's sums.
    const int g = tid / gw < groups ? tid / gw : groups - 1;
    const bool idle = tid / gw >= groups;                  // threads past the last whole group
    {
        constexpr int B = 2, NV = B * RP;
        constexpr int kShift = NV >= 32 ? 1 : NV >= 16 ? 2 : NV >= 8 ? 3 : NV >= 4 ? 4 : 5;   // 6 - log2 NV
        const int gt = tid - g * gw;
        const int wave_q = __builtin_amdgcn_readfirstlane(gt & ~63);       // the wave's first quad of a slab
        const bool aligned = (m & 3) == 0 && lead == 0;    // rows start on 16 bytes of LDS
        float qreg[4 * RP], fold[RP];
        auto request = [&](int slab) {
            const int j = slab * gw + gt < m4 ? slab * gw + gt : m4 - 1;
            conef_load_slices<RP>(conef_quad_slices<RP>(it.q, it.qi, j, conef_quad_col(j, m), m), qreg);
            const int e = slab * gw + gt < w ? slab * gw + gt : w - 1;
            if constexpr (RP % 4 == 0) {
#pragma unroll
                for (int c = 0; c < RP; c += 4) conef_ld4u(it.fold + (int64_t)e * RP + c, fold + c);
            } else {
#pragma unroll
                for (int c = 0; c < RP; ++c) fold[c] = it.fold[(int64_t)e * RP + c];
            }
        };
        request(0);
        conef_wait_lds();
        __syncthreads();
        for (int slab = 0; slab < slabs; ++slab) {
            const bool has_x = slab < nslab;
            const int qj = slab * gw + gt, j = qj < m4 ? qj : m4 - 1, col = conef_quad_col(j, m), dup = 4 * j - col;
            if (slab > 0) request(slab);
            if (idle || qj >= m4 || dup) {                 // another thread's columns add nothing here
#pragma unroll
                for (int k = 0; k < 4 * RP; ++k)
                    if (idle || qj >= m4 || k / RP < dup) qreg[k] = 0.f;
            }
            const bool has_c = !idle && qj < w;
            const int e = qj < w ? qj : w - 1;
            for (int b = 0; b < per; b += B) {
                float acc[NV];
                int lr[B];
#pragma unroll
                for (int a = 0; a < B; ++a) {
                    lr[a] = g * per + b + a;
                    if (lr[a] >= rows) lr[a] = rows - 1;
#pragma unroll
                    for (int c = 0; c < RP; ++c) acc[a * RP + c] = 0.f;
                }
                if (has_x) {
                    float xv[B][4];
#pragma unroll
                    for (int a = 0; a < B; ++a) {
                        const float* src = vals + lr[a] * m + col;
                        if (aligned) {
                            const float4 v = *reinterpret_cast<const float4*>(src);
                            xv[a][0] = v.x; xv[a][1] = v.y; xv[a][2] = v.z; xv[a][3] = v.w;
                        } else {
#pragma unroll
                            for (int k = 0; k < 4; ++k) xv[a][k] = src[k];
                        }
                    }
#pragma unroll
                    for (int a = 0; a < B; ++a)
#pragma unroll
                        for (int c = 0; c < RP; ++c)
#pragma unroll
                            for (int k = 0; k < 4; ++k) acc[a * RP + c] = fmaf(xv[a][k], qreg[k * RP + c], acc[a * RP + c]);
                }
                if (slab * gw + wave_q < w) {              // uniform over the wave; the larger terms last: they round once
#pragma unroll
                    for (int a = 0; a < B; ++a) {
                        const float cell = __fmul_rn(alpha, cells[lr[a] * w + e]);
#pragma unroll
                        for (int c = 0; c < RP; ++c) acc[a * RP + c] = fmaf(cell, has_c ? fold[c] : 0.f, acc[a * RP + c]);
                    }
                }
                mqs_wave_reduce<NV>(acc, lane);
                const int o = lane >> kShift, a = o / RP, c = o - a * RP;
                if ((lane & ((1 << kShift) - 1)) == 0) red[(((size_t)slab * per2 + b + a) * WAVES + wave) * RP + c] = acc[0];
            }
        }
    }
    __syncthreads();

    // P and the tile's share of P^T P, by one wave
    if (wave == 0) {
        const int wpg = gw >> 6;                           // waves of a group
        for (int o = lane; o < rows * RP; o += 64) {
            const int r = o / RP, c = o - r * RP;
            const int gg = groups == 1 ? 0 : r / per, rr = r - gg * per;
            double s = 0.;                                 // (few terms: exact but for the last rounding)
            for (int slab = 0; slab < slabs; ++slab) {
                const float* src = red + (((size_t)slab * per2 + rr) * WAVES + gg * wpg) * RP + c;
#pragma unroll 4
                for (int v = 0; v < wpg; ++v) s += (double)src[v * RP];
            }
            prow[o] = s;
        }
        auto settle = [] {                                 // LDS of one lane for the others of the wave
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        };
        settle();
        if (lane < rows) {
            double x[RP];
            float out[RP];
#pragma unroll
            for (int c = 0; c < RP; ++c) x[c] = prow[lane * RP + c];
            if (it.tmat) {
#pragma unroll
                for (int i = 0; i < RP; ++i) {
#pragma unroll
                    for (int k = i + 1; k < RP; ++k) x[k] = fma(-(double)t_l[i * RP + k], x[i], x[k]);
                    x[i] *= (double)t_l[RP * RP + i];
                }
            }
#pragma unroll
            for (int c = 0; c < RP; ++c) {
                out[c] = it.tmat && c >= it.r ? 0.f : (float)x[c];      // the steps of columns that are not there divide by zero
                prow[lane * RP + c] = (double)out[c];
            }
            store_row<RP>(it.p + (row0 + lane) * RP, out);
        }
        settle();
        constexpr int NG = RP * (RP + 1) / 2;
        if (lane < NG) {
            int i = 0, e0 = 0;                             // entry `lane` of the row-major upper triangle is (i, j)
            while (lane >= e0 + RP - i) {
                e0 += RP - i;
                ++i;
            }
            const int j = i + (lane - e0);
            double s = 0.;
#pragma unroll 8
            for (int r = 0; r < rows; ++r) s = fma(prow[r * RP + i], prow[r * RP + j], s);
            it.gram[(size_t)bx * NG + lane] = s;
        }
    }
}
