// P = X Q for ranks up to 8, streaming form (gfx950).
//
// X is the matrix M as stored (MODE 0), M + E with a dense error (MODE 1) or M + alpha * unsketch(cs)
// (MODE 2: DenseCS.query fused, CountSketch.py:40-47); in modes 1 and 2 X is written back into M.
// Reference semantics: powerSGD_hook.py:596-640 (error added, P = M Q by bmm).
//
// A workgroup of T threads is split into groups of `gw` threads (a multiple of 64, at least a
// quarter of the matrix's columns).  A group owns S consecutive rows; a thread owns the column
// quads slab * gw + t and keeps their 4 x RP block of Q, and their buckets and signs, in registers
// for all rows of a slab.  Rows go four at a time, the next four requested before the current four
// are used.  The 4 x RP sums of a thread are reduced over the wave by a butterfly that halves the
// number of values with every exchange (4 RP exchanges instead of 6 for each of the 4 RP values),
// the waves' results are parked in LDS and added in a fixed order at the end: no atomics, the same
// result on every run.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "conef_device.h"

struct MqsItem {
    float* x;
    const float* err;
    const float* cs;
    const uint32_t* pktab;   // bucket | sign << 31 per column, or null: hashed
    const float* q;
    float* p;
    int64_t n;
    int m, w;
    int gw, S;               // threads of a group, rows of a group (multiple of 4)
    ConefMod mod;
    // not null: workgroup g of the matrix also leaves the upper triangle of (its rows of P)^T (its
    // rows of P), RP (RP + 1) / 2 doubles, at gram[g * RP (RP + 1) / 2]: the shares of P^T P
    double* gram;
    const float* qi;         // not null: q laid out by quads (conef_load_slices)
};

// threads of a group for a matrix of m columns in a workgroup of T threads
inline int mqs_group_width(int64_t m, int T)
{
    const int64_t m4 = (m + 3) >> 2;
    const int64_t nslab = (m4 + T - 1) / T;
    int64_t gw = ((m4 + nslab - 1) / nslab + 63) / 64 * 64;
    if (gw < 64) gw = 64;
    // a group width that does not divide T leaves threads idle: take the next one that does when that is cheaper
    if (T % gw != 0) {
        int64_t up = gw;
        while (T % up != 0) up += 64;
        if (up - gw < T % gw) gw = up;
    }
    return (int)gw;
}

inline int64_t mqs_workgroups(int64_t n, int gw, int S, int T)
{
    const int64_t rows = (int64_t)(T / gw) * S;
    return (n + rows - 1) / rows;
}

inline size_t mqs_lds_bytes(int64_t m, int w, int gw, int S, int T, int rp, bool sketch, bool gram = false)
{
    const int64_t m4 = (m + 3) >> 2;
    const int64_t niter = (m4 + gw - 1) / gw * (S >> 2);
    return (size_t)niter * (T / 64) * 4 * rp * 4 + (sketch ? (size_t)(T / gw) * S * w * 4 : 0) +
           (gram ? (size_t)(T / gw) * S * rp * 4 : 0);
}

// Workgroup size and rows per group for one launch over `count` matrices.  Wide matrices need the
// threads of a large workgroup side by side; rows per group are as many as still leave the launch
// enough workgroups, and as the parked sketch rows leave room for in LDS.  False: no geometry fits,
// or the matrices are too small for this kernel to pay.
inline bool mqs_plan_launch(const MqsItem* items, int count, int rp, bool sketch, int* T_out, int* S_out, size_t* lds_out,
                            bool gram = false)
{
    int T = 256;
    for (int k = 0; k < count; ++k)
        if (((items[k].m + 3) >> 2) > 512) T = 1024;
    const int want = T == 256 ? 384 : 160;
    for (int S = T == 256 ? 16 : 8; S >= 4; S >>= 1) {
        int64_t wgs = 0;
        size_t lds = 0;
        for (int k = 0; k < count; ++k) {
            const int gw = mqs_group_width(items[k].m, T);
            wgs += mqs_workgroups(items[k].n, gw, S, T);
            const size_t need = mqs_lds_bytes(items[k].m, items[k].w, gw, S, T, rp, sketch, gram);
            if (need > lds) lds = need;
        }
        if (lds > 64 * 1024) continue;
        // a launch that cannot give every CU a workgroup's worth of threads is better served by the
        // row-block kernel, whose workgroups are a row or four each
        // (not where the caller wants the shares of P^T P: those save it more launches than that)
        if (S == 4 && wgs * T < 256 * 256 && !gram) return false;
        if (wgs >= want || S == 4) {
            *T_out = T;
            *S_out = S;
            *lds_out = lds;
            return true;
        }
    }
    return false;
}

// x_k -= b_ik x_i (k > i), x_i *= 1 / d_i for i = 0 .. r - 1: the reference's column steps
// (powerSGD_hook.py:21-43) on one row, coefficients from t_l as gram_solve_lds leaves them
template <int RP>
__device__ __forceinline__ void gram_apply_row(float* x, const float* t_l)
{
#pragma unroll
    for (int i = 0; i < RP; ++i) {
#pragma unroll
        for (int k = i + 1; k < RP; ++k) x[k] = fmaf(-t_l[i * RP + k], x[i], x[k]);
        x[i] = __fmul_rn(x[i], t_l[RP * RP + i]);
    }
}

template <int RP>
__device__ __forceinline__ void load_row(const float* p, float* x)
{
    if (RP >= 4) {
#pragma unroll
        for (int c = 0; c < RP; c += 4) conef_ld4u(p + c, x + c);
    } else {
#pragma unroll
        for (int c = 0; c < RP; ++c) x[c] = p[c];
    }
}

template <int RP>
__device__ __forceinline__ void store_row(float* p, const float* x)
{
    if (RP >= 4) {
#pragma unroll
        for (int c = 0; c < RP; c += 4) conef_st4u(p + c, x + c);
    } else {
#pragma unroll
        for (int c = 0; c < RP; ++c) p[c] = x[c];
    }
}

// The value of lane l ^ mask, by the crossing that mask has of its own (no index to form, and LDS for mask 4
// alone).
template <int MASK>
__device__ __forceinline__ float mqs_xor(float v)
{
    const int x = __float_as_int(v);
    if constexpr (MASK == 1) return __int_as_float(__builtin_amdgcn_mov_dpp(x, 0xb1, 0xf, 0xf, true));         // quad_perm [1, 0, 3, 2]
    else if constexpr (MASK == 2) return __int_as_float(__builtin_amdgcn_mov_dpp(x, 0x4e, 0xf, 0xf, true));    // quad_perm [2, 3, 0, 1]
    else if constexpr (MASK == 4) return __int_as_float(__builtin_amdgcn_ds_swizzle(x, (4 << 10) | 0x1f));
    else if constexpr (MASK == 8) return __int_as_float(__builtin_amdgcn_mov_dpp(x, 0x128, 0xf, 0xf, true));   // row_ror 8
    else return __shfl_xor(v, MASK, 64);
}

// One exchange of the butterfly: lanes with the mask's bit keep the upper N / 2 values, the others the lower,
// each with its partner's added.  Across half waves and rows of 16 lanes an instruction swaps the two
// values' halves, and the sum of what comes out is both lanes' result.
template <int N, int MASK>
__device__ __forceinline__ void mqs_halve(float* v, int lane)
{
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
        if constexpr (MASK >= 16) {
            const unsigned lo = __float_as_uint(v[i]), hi = __float_as_uint(v[N / 2 + i]);
            const auto t = MASK == 32 ? __builtin_amdgcn_permlane32_swap(lo, hi, false, false)
                                      : __builtin_amdgcn_permlane16_swap(lo, hi, false, false);
            v[i] = __uint_as_float(t[0]) + __uint_as_float(t[1]);
        } else {
            const bool up = (lane & MASK) != 0;
            const float keep = up ? v[N / 2 + i] : v[i];
            const float send = up ? v[i] : v[N / 2 + i];
            v[i] = keep + mqs_xor<MASK>(send);
        }
    }
}

// Sums NV values over the 64 lanes.  Afterwards lane l holds in v[0] the sum of value
// l >> (6 - log2 NV); every lane of that run holds the same number.
template <int NV>
__device__ __forceinline__ void mqs_wave_reduce(float* v, int lane)
{
    constexpr int kTop = NV >= 32 ? 32 : NV >= 16 ? 16 : NV >= 8 ? 8 : NV >= 4 ? 4 : 2;
    mqs_halve<kTop, 32>(v, lane);
    if constexpr (kTop >= 4) mqs_halve<kTop / 2, 16>(v, lane);
    if constexpr (kTop >= 8) mqs_halve<kTop / 4, 8>(v, lane);
    if constexpr (kTop >= 16) mqs_halve<kTop / 8, 4>(v, lane);
    if constexpr (kTop >= 32) mqs_halve<kTop / 16, 2>(v, lane);
    // the lanes that still differ
    if constexpr (kTop < 4) v[0] += mqs_xor<16>(v[0]);
    if constexpr (kTop < 8) v[0] += mqs_xor<8>(v[0]);
    if constexpr (kTop < 16) v[0] += mqs_xor<4>(v[0]);
    if constexpr (kTop < 32) v[0] += mqs_xor<2>(v[0]);
    v[0] += mqs_xor<1>(v[0]);
}

template <int RP, int MODE, int T>
__device__ __forceinline__ void
psgd_mqs_body(const MqsItem& it, float alpha, ConefSeeds hs, int bx)
{
    constexpr int NV = 4 * RP;
    constexpr int WAVES = T / 64;
    constexpr int kShift = NV >= 32 ? 1 : NV >= 16 ? 2 : NV >= 8 ? 3 : NV >= 4 ? 4 : 5;   // 6 - log2 NV
    extern __shared__ float mqs_lds[];
    const int m = it.m, m4 = (m + 3) >> 2, w = it.w, gw = it.gw, S = it.S;
    const int64_t n = it.n;
    const int groups = T / gw;
    const int nslab = (m4 + gw - 1) / gw;
    const int nblk = S >> 2;
    const int niter = nslab * nblk;
    float* red = mqs_lds;                                  // [niter][WAVES][NV]
    float* cells = mqs_lds + (size_t)niter * WAVES * NV;   // [groups * S][w], MODE 2 only
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    int g = tid / gw;
    const int gt = tid - g * gw;
    const bool idle = g >= groups;                         // threads past the last whole group
    if (idle) g = groups - 1;
    const int64_t wg_row0 = (int64_t)bx * groups * S;
    const int rows_here = n - wg_row0 < (int64_t)groups * S ? (int)(n - wg_row0) : groups * S;   // >= 1
    // local row of (block b, row a of the block), clamped to the last row this workgroup has
    auto local_row = [&](int b, int a) {
        const int lr = g * S + 4 * b + a;
        return lr < rows_here ? lr : rows_here - 1;
    };
    auto quad_of = [&](int slab) {
        const int j = slab * gw + gt;
        return j < m4 ? j : m4 - 1;
    };
    float xn[4][4], en[4][4];
    auto request = [&](int iter) {
        const int slab = iter / nblk, b = iter - slab * nblk;
        const int j = quad_of(slab);
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const int64_t off = (wg_row0 + local_row(b, a)) * m + conef_quad_col(j, m);
            conef_ld4u(it.x + off, xn[a]);
            if (MODE == 1) conef_ld4u(it.err + off, en[a]);
        }
    };
    // a slab's slice of Q and its columns' buckets.  With sketch rows to wait for, the first slab's travel with them;
    // without, the registers they would hold that long cost more than the wait (MODE 1 at rank 8: 926 against 915 us
    // over BERT's buckets)
    float qreg[4 * RP];
    uint32_t pk[4] = {0u, 0u, 0u, 0u};
    auto request_slab = [&](int slab) {
        const int j = quad_of(slab), c = conef_quad_col(j, m);
        conef_load_slices<RP>(conef_quad_slices<RP>(it.q, it.qi, j, c, m), qreg);
        if (MODE == 2 && it.pktab) conef_ld4u(it.pktab + c, pk);
    };
    request(0);
    if (MODE == 2) {
        request_slab(0);
        // the workgroup's sketch rows, eight requests a thread at a time: one by one, as a plain loop, each was
        // a trip to memory, 7 of the 16 us of a [640, 5760] launch with 1152 cells a row
        const float* src = it.cs + wg_row0 * w;
        const int count = rows_here * w;
        for (int i0 = tid; i0 < count; i0 += 8 * T) {
            float t[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (i0 - tid + u * T < count) t[u] = src[i0 + u * T < count ? i0 + u * T : count - 1];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (i0 + u * T < count) cells[i0 + u * T] = t[u];
        }
        __syncthreads();
    }
    bool valid = false;
    int col = 0, dup = 0;
    for (int iter = 0; iter < niter; ++iter) {
        const int slab = iter / nblk, b = iter - slab * nblk;
        if (b == 0) {
            const int j = quad_of(slab);
            col = conef_quad_col(j, m);
            dup = 4 * j - col;
            valid = !idle && slab * gw + gt < m4;
            if (MODE != 2 || slab > 0) request_slab(slab);
            if (!valid || dup) {        // another thread's columns (the last quad a second time, a moved quad's first ones): they add nothing
#pragma unroll
                for (int t = 0; t < 4 * RP; ++t)
                    if (!valid || t / RP < dup) qreg[t] = 0.f;
            }
            if (MODE == 2) {
                if (!it.pktab) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) pk[k] = conef_bucket_sign(col + k, it.mod, hs.a, hs.b, hs.sa, hs.sb);
                }
            }
        }
        float xv[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                xv[a][k] = xn[a][k];
                if (MODE == 1) xv[a][k] = __fadd_rn(xv[a][k], en[a][k]);
            }
        if (iter + 1 < niter) request(iter + 1);
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const int lr = g * S + 4 * b + a;
            if (MODE == 2) {
                const float* crow = cells + (size_t)(lr < rows_here ? lr : rows_here - 1) * w;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    xv[a][k] = __fadd_rn(xv[a][k], conef_query_term(crow[pk[k] & 0x7fffffffu], pk[k], alpha));
            }
            if (MODE != 0 && valid && lr < rows_here) conef_st4_own(it.x + (wg_row0 + lr) * m + col, xv[a], dup);
        }
        float acc[NV];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int c = 0; c < RP; ++c) {
                float s = 0.f;
#pragma unroll
                for (int k = 0; k < 4; ++k) s = fmaf(xv[a][k], qreg[k * RP + c], s);
                acc[a * RP + c] = s;
            }
        mqs_wave_reduce<NV>(acc, lane);
        if ((lane & ((1 << kShift) - 1)) == 0) red[((size_t)iter * WAVES + wave) * NV + (lane >> kShift)] = acc[0];
    }
    __syncthreads();
    const int wpg = gw >> 6;                               // waves of a group
    float* prow = cells + (MODE == 2 ? (size_t)groups * S * w : 0);   // [groups * S][RP], only with it.gram
    for (int o = tid; o < rows_here * RP; o += T) {
        const int lr = o / RP, c = o - lr * RP;
        const int gg = lr / S, rr = lr - gg * S;
        const int b = rr >> 2, idx = (rr & 3) * RP + c;
        float s = 0.f;
        for (int slab = 0; slab < nslab; ++slab) {
            const float* base = red + ((size_t)(slab * nblk + b) * WAVES + gg * wpg) * NV + idx;
#pragma unroll 4
            for (int v = 0; v < wpg; ++v) s += base[(size_t)v * NV];
        }
        it.p[(wg_row0 + lr) * RP + c] = s;
        if (it.gram) prow[o] = s;
    }
    if (it.gram) {
        constexpr int NG = RP * (RP + 1) / 2;
        __syncthreads();
        if (tid < NG) {
            int i = 0, e0 = 0;                             // entry tid of the row-major upper triangle is (i, j)
            while (tid >= e0 + RP - i) {
                e0 += RP - i;
                ++i;
            }
            const int j = i + (tid - e0);
            double s = 0.;
#pragma unroll 8
            for (int lr = 0; lr < rows_here; ++lr) s = fma((double)prow[lr * RP + i], (double)prow[lr * RP + j], s);
            it.gram[(size_t)bx * NG + tid] = s;
        }
    }
}

// ------------------------------------------------------------ M = P Q^T ----
// MODE 0: write M.  MODE 1: also write the dense residual E = X - M (X = what M held on entry).
// Factors of rank RP exactly (rows of RP floats, 16-byte aligned), rows of at least four columns of
// any alignment.  A thread owns a column quad, whose 4 x RP slice of Q stays in registers, and walks
// rows four at a time with their loads in flight together.  A workgroup is cut into groups of
// `lanes` threads that cover a row (or 1024 columns of it) and take rows in turn; lanes is a multiple
// of 64 wherever a row has more than 64 quads, so that a wave's row of P is uniform and comes through
// the scalar cache.
struct PqtItem {
    float* x;
    float* err;
    const float* p;
    const float* q;
    int64_t n;
    int m, r, rows_per_slab, col_tiles;
    int lanes;
    const float* qi;         // not null: q laid out by quads (conef_load_slices)
};

typedef __attribute__((address_space(4))) float conef_cfloat;      // constant memory: uniform loads are scalar

inline int pqt_lanes(int64_t m)
{
    const int64_t m4 = (m + 3) / 4;
    return (int)(m4 >= 256 ? 256 : m4 > 64 ? (m4 + 63) / 64 * 64 : m4);
}

template <int RP, int MODE, bool UNIFORM>
__device__ __forceinline__ void
psgd_pqt_rows(float* __restrict__ x, float* __restrict__ err, const float* __restrict__ p, const float* __restrict__ q,
              const float* __restrict__ qi, const PqtItem& it, int bx, int by)
{
    const int m = it.m, groups = 256 / it.lanes;
    int grp = (int)threadIdx.x / it.lanes;
    const int quad = bx * 256 + (int)threadIdx.x - grp * it.lanes;
    if (UNIFORM) grp = __builtin_amdgcn_readfirstlane(grp);
    if (grp >= groups || 4 * quad >= m) return;
    const int col = conef_quad_col(quad, m), dup = 4 * quad - col;
    const int64_t i0 = (int64_t)by * it.rows_per_slab;
    const int64_t i1 = i0 + it.rows_per_slab < it.n ? i0 + it.rows_per_slab : it.n;
    float qf[4 * RP];
    conef_load_slices<RP>(conef_quad_slices<RP>(q, qi, quad, col, m), qf);
    auto walk = [&](auto store) {
        for (int64_t ib = i0 + grp; ib < i1; ib += 4 * groups) {
            float xv[4][4];
            if (MODE == 1) {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int64_t i = ib + u * groups < i1 ? ib + u * groups : ib;
                    conef_ld4u(x + i * m + col, xv[u]);
                }
            }
            // The four rows of P: through constant memory where they are uniform.  (The pointers come out of a table:
            // nothing else tells the compiler that the stores leave P alone, and the rows became vector loads
            // behind them.)
            float pv[4][RP];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int64_t i = ib + u * groups < i1 ? ib + u * groups : ib;
                if (UNIFORM) {
                    const conef_cfloat* ps = (const conef_cfloat*)(uintptr_t)(p + i * RP);
#pragma unroll
                    for (int c = 0; c < RP; ++c) pv[u][c] = ps[c];
                } else {
#pragma unroll
                    for (int c = 0; c < RP; ++c) pv[u][c] = p[i * RP + c];
                }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int64_t i = ib + u * groups;
                if (i >= i1) break;
                float mh[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < RP; ++c) {
                    const float pc = pv[u][c];
#pragma unroll
                    for (int k = 0; k < 4; ++k) mh[k] = fmaf(pc, qf[k * RP + c], mh[k]);
                }
                if (MODE == 1) {
                    float ev[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) ev[k] = __fsub_rn(xv[u][k], mh[k]);
                    store(err + i * m + col, ev);
                }
                store(x + i * m + col, mh);
            }
        }
    };
    // (rows of whole quads have a loop without the moved quad's test; uniform)
    if (m % 4 == 0) walk([](float* at, const float* v) { conef_st4u(at, v); });
    else walk([&](float* at, const float* v) { conef_st4_own(at, v, dup); });
}
