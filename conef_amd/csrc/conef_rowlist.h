// Row-list sketch accumulation: the count-sketch update without atomics for rows that fit LDS.
//
// The bucket and sign of a column depend on the column alone, so every row of an [n,d] tensor
// scatters the same way.  A plan built once per sketch lists, per bucket, the columns that fall
// into it (ascending).  A workgroup then takes a tile of `rb` consecutive rows:
//
//   (the bucket lists and their offsets, d + w small integers, are requested first and parked in
//   LDS once the tile is staged)
//   stage   the values to be sketched are produced in column order with 16-byte accesses and
//           parked in LDS; whatever the fused step has to do in column order (payload, writing
//           the decompressed gradient, the low-rank product) happens here;
//   gather  a thread walks a bucket's list for a row or two, picks its values out of LDS
//           and adds the terms in ascending column order, several entries a trip; buckets are
//           handed out in the order of falling list length (a table of the plan), so that the
//           lanes of a wave have lists of about the same length to walk.
//
// No atomics, one read of the tensor, deterministic, and the order of the adds is the CPU
// oracle's, so the sketch comes out bit for bit.  cs_out may be cs_in: a tile reads its rows'
// old cells before it writes them and no other tile touches those rows.
#pragma once
#include "conef_device.h"
#include "conef_sketch_core.h"
#include <algorithm>
#include <type_traits>

constexpr int kConefRowlistThreads = 256;
constexpr int64_t kConefRowlistMaxCols = 24576;       // 4 B value + 2 B list entry per column in LDS
constexpr size_t kConefRowlistLdsLimit = 160 * 1024;   // LDS of a gfx950 CU

struct ConefRowlistView {
    const uint32_t* csr;   // [w+1] first list entry of bucket j
    const uint16_t* ent;   // [d] column | sign bit << 15, buckets ascending, columns ascending
    const uint32_t* pk;    // [d] bucket | sign bit << 31 of every column
    const uint16_t* order; // [w] the buckets by falling list length
};

struct ConefRowlistShape {
    int rb;          // rows per tile
    size_t lds;      // bytes of dynamic LDS
    int64_t tiles;
    bool pk_lds;     // the column table (bucket and sign per column) has room in LDS behind the cells
};

// Fronts that read the old cells while they stage look up every column's bucket there too.
inline size_t conef_rowlist_pk_bytes(int64_t d) { return (((size_t)d + 3) & ~(size_t)3) * 4; }

inline size_t conef_rowlist_lds(int rb, int64_t d, int32_t w, bool cells)
{
    size_t vals = (((size_t)rb * d + 3) & ~(size_t)3) * 4;
    size_t ent = (((size_t)d + 7) & ~(size_t)7) * 2;
    size_t csr = (((size_t)w + 1 + 3) & ~(size_t)3) * 4;
    size_t ord = (((size_t)w + 7) & ~(size_t)7) * 2;
    (void)cells;      // every front parks the tile's old sketch rows in LDS
    return vals + ent + csr + ord + (size_t)rb * w * 4;
}

// A front with kCompact has the offsets in 16 bits and nothing between the tables.
inline size_t conef_rowlist_lds_compact(int rb, int64_t d, int32_t w)
{
    const size_t vals = (((size_t)rb * d + 3) & ~(size_t)3) * 4, ent = (((size_t)d + 7) & ~(size_t)7) * 2;
    return vals + ent + (((size_t)2 * w + 1 + 1) & ~(size_t)1) * 2 + (size_t)rb * w * 4;
}

// Rows per tile: about 32 KB of values (several tiles per CU), but no more than leaves a
// thousand tiles for the 256 CUs.
// `companions`: matrices of about this size that share the launch (a batch leaves enough tiles
// for the machine with taller tiles per matrix); 0: full-height tiles whatever the count (for a
// batch whose caller has checked that it has tiles enough that way).
inline bool conef_rowlist_shape(int64_t n, int64_t d, int32_t w, bool cells, bool halves, ConefRowlistShape* s,
                                int companions = 1)
{
    if (d < 1 || d > kConefRowlistMaxCols || n < 1 || w < 1 || w > 0xffff) return false;
    int64_t rb = 8192 / d;
    // tiles to spare, in a front that asks for it (Front::halves): half-height ones, twice as many resident per
    // CU (a quarter was slower again)
    if (halves && rb >= 2 && n / rb >= 2048) rb = (rb + 1) / 2;
    if (companions > 0 && rb > n * companions / 1024) rb = n * companions / 1024;
    if (rb > 16) rb = 16;
    if (rb < 1) rb = 1;
    // the column table goes to LDS where a tile has at least two rows to use it for (a launch takes
    // the LDS of its largest tile for every tile, and a one-row tile would double that for nothing)
    const size_t pk = cells && rb >= 2 ? conef_rowlist_pk_bytes(d) : 0;
    while (rb > 1 && conef_rowlist_lds((int)rb, d, w, cells) + pk > 64 * 1024) --rb;
    // rows that are not a whole number of 16-byte quads: tiles of 2 (4) rows start on a quad again,
    // and the fronts then read a tile as one flat run of quads
    if (d % 4 == 2 && rb > 1) rb &= ~(int64_t)1;
    else if (d % 2 == 1 && rb >= 4) rb &= ~(int64_t)3;
    size_t lds = conef_rowlist_lds((int)rb, d, w, cells);
    if (lds > kConefRowlistLdsLimit) return false;
    s->pk_lds = pk > 0 && rb >= 2 && lds + pk <= kConefRowlistLdsLimit;
    if (s->pk_lds) lds += pk;
    s->rb = (int)rb;
    s->lds = lds;
    s->tiles = (n + rb - 1) / rb;
    return s->tiles <= 0x7fffffff;
}

// Taller tiles for matrices of few or of long rows (the shapes above give those one row a tile), and the threads of a
// workgroup: sixteen waves a CU with as many tiles as its LDS holds or the launch has, and at least `least` values each.
// A tile is a chain - its rows, then the lists - that a CU with one or two of them in it waits for, and a thread that walks a
// list for two rows reads it once.  One row by 256 threads against this, us, sketches of 0.1 and of 0.4:
//                        update, half cells            update                        random-block step
//   [300,1000]           4.8   4.6    4.6   4.4        4.6   4.3    4.6   4.3        6.1   6.2    6.0   6.2
//   [2000,2000]          8.4   6.0   11.3   8.6        7.9   6.1   11.1   8.2       14.8  10.3   17.8  11.7
//   [900,5700]           9.5   8.1   17.9   9.9        8.6   7.9   16.8  10.0       17.9  17.4   29.9  19.1
//   [4096,5700]         41.1  29.0   71.3  44.5       38.7  28.1   68.3  40.9       63.7  46.8  115.4  72.3
//   [2000,9000]         37.4  25.9   95.8  48.1       37.1  25.3   95.7  46.7       68.1  47.7  153.8  64.4
//   [2000,12000]        71.4  34.8  124.2  73.7       71.3  34.2  124.8  71.5      138.6  60.3  194.7  93.5
// Over 354 such shapes (rows of 600 to 20000, 64 to 4096 of them) a third less on average, one 7 % more (0.5 us).
// A random-block step (cells) whose tiles have two rows stays as it is: its old cells and the column table lie in LDS too, and four
// rows of a long matrix leave a CU too few tiles.  Two or three rows and four, us, buffers out of the caches, sketches of 0.1 and of 0.4:
//   [2600,650]    9.4   9.5   10.2  10.8      three of them  19.9  21.0   21.4  24.4
//   [2600,1000]  11.4  12.4   12.3  13.4      [2048,2502]    17.3  19.4   21.0  20.8
//   [3400,800]   11.4  13.9   13.3  15.8      [16000,1500]   56.9  71.4   87.6  93.0
// (Over 110 shapes of 2048 to 16000 rows 3 % less than four rows, against one workgroup size for all 7 % less and 5 % more at
// worst, where four rows were 26 % more.  Updates of such shapes by four rows are 3 % faster.)
inline void conef_rowlist_taller(int64_t n, int64_t d, int32_t w, bool cells, ConefRowlistShape* s)
{
    if (cells && s->rb >= 2) return;
    for (int rb = 4; rb >= 2; rb -= 2) {
        if (s->rb >= rb) return;
        // (cells, rows of more than 2048 columns: two rows of [640,5760] 15.8 us, one row by 512 threads 14.2, [640,4096] 12.2 and
        // 11.2, [260,4096] 9.3 and 8.2; three [640,2880] in a launch 18.2 and 20.0, [640,9000] 21.1 and 24.0)
        if (n < (int64_t)rb * (cells && (rb == 4 || d > 2048) ? 400 : rb == 4 ? 200 : 128)) continue;
        const size_t lds = conef_rowlist_lds(rb, d, w, cells), pk = cells ? conef_rowlist_pk_bytes(d) : 0;
        if (lds > kConefRowlistLdsLimit) continue;
        s->rb = rb;
        // (the column table stays out where it would leave a CU fewer tiles: [2000,7000] 35.0 us without, 37.7 with)
        s->pk_lds = cells && lds + pk <= kConefRowlistLdsLimit && kConefRowlistLdsLimit / (lds + pk) == kConefRowlistLdsLimit / lds;
        s->lds = s->pk_lds ? lds + pk : lds;
        s->tiles = (n + rb - 1) / rb;
        return;
    }
}

inline int conef_rowlist_workgroup(size_t lds, int64_t tiles, double values, int least)
{
    const int64_t per_cu = std::min<int64_t>((int64_t)(kConefRowlistLdsLimit / std::max<size_t>(lds, 1)), (tiles + 255) / 256);
    int threads = per_cu <= 1 ? 1024 : per_cu <= 3 ? 512 : 256;
    while (threads > 256 && values < (double)least * threads * (double)tiles) threads /= 2;
    return threads;
}

// ------------------------------------------------------------------ fronts ----
// A front fills vals[row_in_tile * d + col] for the tile's rows.  `cells` (only when
// kNeedsCells) holds the tile's old sketch rows, [rows][w]; a front with kParksCells puts them there itself
// while it stages.

// DenseCS.update: the value is the dense tensor itself.
template <int T>
struct ConefListVecT {
    const float* vec;
    bool vec_ok;           // base 16-byte aligned and d % 4 == 0 (the tile copy works either way)
    static constexpr bool kNeedsCells = false, kParksCells = false, kCompact = false;
    static constexpr int kThreads = T, kLeastValues = 8;
    // whether a tensor with tiles to spare goes by half-height ones.  Full against half height: [50000,512] 40.2
    // and 29.9 us, [20000,2048] 49.0 and 45.9, [30522,1024] 37.0 and 36.2, [33278,650] 26.2 and 26.0, [60000,300]
    // and [33278,200] within 1 % either way.
    static bool halves(int64_t) { return true; }
    struct Regs {};
    __device__ __forceinline__ void stage(int64_t row0, int rows, int d, int, float* vals, const float*,
                                          const uint32_t*) const
    {
        const float* base = vec + row0 * d;
        const int total = rows * d;
        // A tile is one contiguous run: up to three leading elements bring it to a 16-byte
        // boundary, 16-byte loads from there (eight in flight per thread; indices past the end are
        // clamped, not branched around), the last few elements one by one.
        int lead = (int)(((16u - (unsigned)(reinterpret_cast<uintptr_t>(base) & 15u)) & 15u) >> 2);
        if (lead > total) lead = total;
        const int total4 = (total - lead) >> 2;
        const float4* src4 = reinterpret_cast<const float4*>(base + lead);
        for (int q0 = threadIdx.x; q0 < total4; q0 += 8 * T) {
            float4 t[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                int q = q0 + u * T;
                t[u] = src4[q < total4 ? q : total4 - 1];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                int q = q0 + u * T;
                if (q < total4) {
                    if (lead == 0) {
                        reinterpret_cast<float4*>(vals)[q] = t[u];
                    } else {
                        float* o = vals + lead + (q << 2);
                        o[0] = t[u].x; o[1] = t[u].y; o[2] = t[u].z; o[3] = t[u].w;
                    }
                }
            }
        }
        const int rest = total - (total4 << 2);          // leading and trailing elements, at most 6
        if ((int)threadIdx.x < rest) {
            const int e = (int)threadIdx.x < lead ? (int)threadIdx.x : (int)threadIdx.x + (total4 << 2);
            vals[e] = base[e];
        }
    }
};
using ConefListVec = ConefListVecT<kConefRowlistThreads>;

// RandomBlock + ConEF (reference: communication/RandomBlock_hook.py:190,216-243,272-280 at world
// size 1): xq = x + alpha * unsketch(old cells); inside the wrap-around block xq goes to the
// payload and stays in x and a zero is sketched, outside x becomes zero and xq is sketched.
//
// The tile is one flat run of quads (up to three leading elements bring it to a 16-byte boundary,
// the last few go one by one).  The first kQuads quads of a thread are requested before the old
// cells and the column table are parked in LDS (`request`), so that the tile travels with them;
// `stage` then works from LDS: row and column of a quad advance with it (no division per quad),
// the block is a pair of tile-relative ranges, and a tile that does not touch the block at all -
// most of them - runs without any of that.
template <int T>
struct ConefListRandBlockT {
    float* x;
    float* payload;
    ConefBlock blk;
    float alpha;
    static constexpr bool kNeedsCells = true, kParksCells = false, kCompact = false;
    static constexpr int kThreads = T, kLeastValues = 3;
    static bool halves(int64_t) { return true; }      // (the column table sits in LDS next to the tiles)
    static constexpr int kQuads = 4;
    struct Regs {          // a thread's first kQuads quads, by name: no array for the compiler to keep in memory
        float4 g0, g1, g2, g3;
    };

    __device__ __forceinline__ float finish(int64_t f, float g, float cell, uint32_t pk, float* out) const
    {
        float xq = __fadd_rn(g, conef_query_term(cell, pk, alpha));
        int64_t pos = conef_payload_pos(f, blk);
        if (pos >= 0) {
            payload[pos] = xq;
            *out = xq;
            return 0.f;
        }
        *out = 0.f;
        return xq;
    }

    static __device__ __forceinline__ int lead_of(const float* base, int total)
    {
        int lead = (int)(((16u - (unsigned)(reinterpret_cast<uintptr_t>(base) & 15u)) & 15u) >> 2);
        return lead > total ? total : lead;
    }

    __device__ __forceinline__ Regs request(int64_t row0, int rows, int d) const
    {
        const float* base = x + row0 * d;
        const int total = rows * d, lead = lead_of(base, total), total4 = (total - lead) >> 2;
        const float4* base4 = reinterpret_cast<const float4*>(base + lead);
        Regs r;
        r.g0 = r.g1 = r.g2 = r.g3 = make_float4(0.f, 0.f, 0.f, 0.f);
        if (total4 > 0) {
            const int q = threadIdx.x, last = total4 - 1;      // past the end: a valid address, result unused
            r.g0 = base4[q < last ? q : last];
            r.g1 = base4[q + T < last ? q + T : last];
            r.g2 = base4[q + 2 * T < last ? q + 2 * T : last];
            r.g3 = base4[q + 3 * T < last ? q + 3 * T : last];
        }
        return r;
    }

    // One quad: element e of the tile onwards, which sits in column `col` of the row whose cells
    // start at `roff`.  pk_l: the column table, in LDS or (rows too long for that) in global memory.
    template <bool BLOCK>
    __device__ __forceinline__ void quad(float4 g, int q, int e, int col, int roff, float4* base4, int64_t f0,
                                         int lead, int d, int w, float* vals, const float* cells,
                                         const uint32_t* pk_l, int lo, int hi, int rest) const
    {
        const float gv[4] = {g.x, g.y, g.z, g.w};
        float o[4], v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            int c = col + k, ro = roff;
            if (c >= d) {
                c -= d;
                ro += w;
                if (d < 4)                     // a quad may then cross several rows
                    while (c >= d) {
                        c -= d;
                        ro += w;
                    }
            }
            const uint32_t p = pk_l[c];
            const float xq = __fadd_rn(gv[k], conef_query_term(cells[ro + (p & 0x7fffffffu)], p, alpha));
            const int ek = e + k;
            if (BLOCK && ((ek >= lo && ek < hi) || ek < rest)) {
                payload[conef_payload_pos(f0 + ek, blk)] = xq;
                o[k] = xq;
                v[k] = 0.f;
            } else {
                o[k] = 0.f;
                v[k] = xq;
            }
        }
        base4[q] = make_float4(o[0], o[1], o[2], o[3]);
        if (lead == 0) {
            reinterpret_cast<float4*>(vals)[q] = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) vals[e + k] = v[k];
        }
    }

    template <bool BLOCK>
    __device__ __forceinline__ void quads(Regs r, float* base, int64_t f0, int lead, int total4, int d, int w,
                                          float* vals, const float* cells, const uint32_t* pk_l, int lo, int hi,
                                          int rest) const
    {
        float4* base4 = reinterpret_cast<float4*>(base + lead);
        constexpr int kStep = 4 * T;          // elements between a thread's quads
        const int drow = kStep / d, dcol = kStep - drow * d;
        int q = threadIdx.x;
        int e = lead + (q << 2);
        int col = e % d;
        int roff = (e / d) * w;
        auto one = [&](float4 g) {
            if (q < total4) quad<BLOCK>(g, q, e, col, roff, base4, f0, lead, d, w, vals, cells, pk_l, lo, hi, rest);
            q += T;
            e += kStep;
            col += dcol;
            roff += drow * w;
            if (col >= d) {
                col -= d;
                roff += w;
            }
        };
        one(r.g0);
        one(r.g1);
        one(r.g2);
        one(r.g3);
        while (q < total4) {                 // taller tiles: four more quads a trip
            const int last = total4 - 1;
            const float4 g0 = base4[q];
            const float4 g1 = base4[q + T < last ? q + T : last];
            const float4 g2 = base4[q + 2 * T < last ? q + 2 * T : last];
            const float4 g3 = base4[q + 3 * T < last ? q + 3 * T : last];
            one(g0);
            one(g1);
            one(g2);
            one(g3);
        }
    }

    __device__ __forceinline__ void stage(Regs r, int64_t row0, int rows, int d, int w, float* vals,
                                          const float* cells, const uint32_t* pk_l) const
    {
        const int64_t f0 = row0 * d;
        float* base = x + f0;
        const int total = rows * d, lead = lead_of(base, total), total4 = (total - lead) >> 2;
        // the block's two ranges, [start,end) and [0,rest), relative to the tile
        const int64_t a0 = blk.start - f0, a1 = blk.end - f0, a2 = blk.rest - f0;
        const int lo = a0 < 0 ? 0 : a0 > total ? total : (int)a0;
        const int hi = a1 < 0 ? 0 : a1 > total ? total : (int)a1;
        const int rest = a2 < 0 ? 0 : a2 > total ? total : (int)a2;
        if (hi > lo || rest > 0) quads<true>(r, base, f0, lead, total4, d, w, vals, cells, pk_l, lo, hi, rest);
        else quads<false>(r, base, f0, lead, total4, d, w, vals, cells, pk_l, 0, 0, 0);
        const int tail = total - (total4 << 2);      // leading and trailing elements, at most 6
        if ((int)threadIdx.x < tail) {
            const int e = (int)threadIdx.x < lead ? (int)threadIdx.x : (int)threadIdx.x + (total4 << 2);
            const int row = e / d, col = e - row * d;
            const uint32_t p = pk_l[col];
            float o;
            vals[e] = finish(f0 + e, base[e], cells[row * w + (p & 0x7fffffffu)], p, &o);
            base[e] = o;
        }
    }
};
using ConefListRandBlock = ConefListRandBlockT<kConefRowlistThreads>;

// ------------------------------------------------------------------ kernel ----
// count >= 1 words from global memory to LDS, eight loads in flight per thread
template <int T>
__device__ __forceinline__ void conef_copy_words_to_lds(uint32_t* dst, const uint32_t* __restrict__ src, int count)
{
    for (int i0 = threadIdx.x; i0 < count; i0 += 8 * T) {
        uint32_t t[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            int i = i0 + u * T;
            t[u] = src[i < count ? i : count - 1];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            int i = i0 + u * T;
            if (i < count) dst[i] = t[u];
        }
    }
}

template <typename CsT, typename Front>
__device__ __forceinline__ void
conef_rowlist_body(const Front& front, ConefRowlistView plan, const CsT* cs_in, CsT* cs_out, int64_t n, int d, int w,
                   int rb, double one_minus_beta, int bx, bool pk_lds = false)
{
    // Requests past the end of a table are left out where the cells are floats (a uniform test each; rows there
    // are often short, and a request past the end is a request all the same: [33278,650] 25.6 us against 26.0,
    // [30522,1024] 34.8 against 36.2, a pair [4096,1024] + [1024,4096] 16.9 against 16.7) and made where they are
    // halves ([640,5760] 10.3 us without the tests, 11.2 with them; [33278,650] 25.5 and 27.8).
    constexpr int T = Front::kThreads;
    constexpr bool sparing = sizeof(CsT) == sizeof(float);
    extern __shared__ float conef_rl[];
    float* vals = conef_rl;
    uint16_t* ent_l = reinterpret_cast<uint16_t*>(vals + ((rb * d + 3) & ~3));
    constexpr bool compact = Front::kCompact;
    using Offset = std::conditional_t<compact, uint16_t, uint32_t>;
    Offset* csr_l = reinterpret_cast<Offset*>(ent_l + ((d + 7) & ~7));
    uint16_t* ord_l = reinterpret_cast<uint16_t*>(csr_l + (compact ? w + 1 : (w + 1 + 3) & ~3));
    float* cells = reinterpret_cast<float*>(compact ? ent_l + ((d + 7) & ~7) + ((2 * w + 1 + 1) & ~1) : ord_l + ((w + 7) & ~7));
    const int64_t row0 = (int64_t)bx * rb;
    const int rows = n - row0 < rb ? (int)(n - row0) : rb;

    // The bucket lists (two entries per load; the table is padded to a multiple of 256 bytes) and
    // their offsets are only needed by the walk: the first words of both are requested now and
    // parked after the tile has been staged, so that they travel while the tile does.
    constexpr int kPreE = 8, kPreC = 2;
    const int ent_words = (d + 1) >> 1, csr_words = w + 1, ord_words = (w + 1) >> 1;
    const uint32_t* ent_src = reinterpret_cast<const uint32_t*>(plan.ent);
    const uint32_t* ord_src = reinterpret_cast<const uint32_t*>(plan.order);
    uint32_t ent_pre[kPreE], csr_pre[kPreC];
    const uint32_t ord_pre = ord_src[(int)threadIdx.x < ord_words ? (int)threadIdx.x : ord_words - 1];
#pragma unroll
    for (int u = 0; u < kPreE; ++u) {
        const int i = threadIdx.x + u * T;
        if (!sparing || u * T < ent_words) ent_pre[u] = ent_src[i < ent_words ? i : ent_words - 1];
    }
#pragma unroll
    for (int u = 0; u < kPreC; ++u) {
        const int i = threadIdx.x + u * T;
        if (!sparing || u * T < csr_words) csr_pre[u] = plan.csr[i < csr_words ? i : csr_words - 1];
    }
    typename Front::Regs regs;
    uint32_t* pk_l = reinterpret_cast<uint32_t*>(cells + rb * w);
    if constexpr (Front::kNeedsCells) {
        // The tile's first quads, its rows' old cells and the column table are requested together;
        // cells and table are parked in LDS, the quads wait in registers.
        regs = front.request(row0, rows, d);
        const CsT* src = cs_in + row0 * w;
        const int count = rows * w;
        constexpr int kPark = 4;
        float ct[kPark];
        uint32_t pt[kPark];
#pragma unroll
        for (int u = 0; u < kPark; ++u) {
            const int i = threadIdx.x + u * T;
            if (!sparing || u * T < count) ct[u] = conef_ld(src + (i < count ? i : count - 1));
            if (!sparing || (pk_lds && u * T < d)) pt[u] = plan.pk[i < d ? i : d - 1];
        }
#pragma unroll
        for (int u = 0; u < kPark; ++u) {
            const int i = threadIdx.x + u * T;
            if (i < count) cells[i] = ct[u];
            if (pk_lds && i < d) pk_l[i] = pt[u];
        }
        for (int i = threadIdx.x + kPark * T; i < count; i += T)
            cells[i] = conef_ld(src + i);
        if (pk_lds)
            for (int i = threadIdx.x + kPark * T; i < d; i += T)
                pk_l[i] = plan.pk[i];
        __syncthreads();
    }
    // The tile's cells are rows * w consecutive values; thread t owns cells t, t + 256, ...  Fronts
    // that do not need the old rows for staging request their cells now, so that the values arrive
    // while the tile is staged, and park them in LDS before the barrier.
    const int total = rows * w;
    constexpr int kPre = 8;
    float aux_pre[kPre];
    if constexpr (!Front::kNeedsCells && !Front::kParksCells) {
#pragma unroll
        for (int u = 0; u < kPre; ++u) {
            const int p = threadIdx.x + u * T;
            if (!sparing || u * T < total) aux_pre[u] = conef_ld(cs_in + row0 * w + (p < total ? p : total - 1));
        }
    }
    if constexpr (Front::kNeedsCells) {
        if (pk_lds) front.stage(regs, row0, rows, d, w, vals, cells, pk_l);
        else front.stage(regs, row0, rows, d, w, vals, cells, plan.pk);
    }
    else front.stage(row0, rows, d, w, vals, cells, plan.pk);
    {
        uint32_t* ent_w = reinterpret_cast<uint32_t*>(ent_l);
#pragma unroll
        for (int u = 0; u < kPreE; ++u) {
            const int i = threadIdx.x + u * T;
            if (i < ent_words) ent_w[i] = ent_pre[u];
        }
#pragma unroll
        for (int u = 0; u < kPreC; ++u) {
            const int i = threadIdx.x + u * T;
            if (i < csr_words) csr_l[i] = (Offset)csr_pre[u];
        }
        if constexpr (compact) {
            for (int i = threadIdx.x; i < ord_words; i += T) {
                const uint32_t two = i == (int)threadIdx.x ? ord_pre : ord_src[i];
                ord_l[2 * i] = (uint16_t)two;
                if (2 * i + 1 < w) ord_l[2 * i + 1] = (uint16_t)(two >> 16);
            }
            for (int i = threadIdx.x + kPreC * T; i < csr_words; i += T) csr_l[i] = (Offset)plan.csr[i];
        } else {
            uint32_t* ord_w = reinterpret_cast<uint32_t*>(ord_l);
            if ((int)threadIdx.x < ord_words) ord_w[threadIdx.x] = ord_pre;
            if (ord_words > T)
                conef_copy_words_to_lds<T>(ord_w + T, ord_src + T,
                                        ord_words - T);
            if (csr_words > kPreC * T)
                conef_copy_words_to_lds<T>(csr_l + kPreC * T, plan.csr + kPreC * T,
                                        csr_words - kPreC * T);
        }
        if (ent_words > kPreE * T)
            conef_copy_words_to_lds<T>(ent_w + kPreE * T, ent_src + kPreE * T,
                                    ent_words - kPreE * T);
    }
    if constexpr (!Front::kNeedsCells && !Front::kParksCells) {
#pragma unroll
        for (int u = 0; u < kPre; ++u) {
            const int p = threadIdx.x + u * T;
            if (p < total) cells[p] = aux_pre[u];
        }
        for (int p = threadIdx.x + kPre * T; p < total; p += T)
            cells[p] = conef_ld(cs_in + row0 * w + p);
    }
    __syncthreads();

    // One thread per (bucket, row), buckets in the order of falling list length and the rows of a
    // bucket on neighbouring lanes: the lanes of a wave walk lists of about the same length (a wave
    // takes as many trips as its longest list).
    constexpr int kWalk = 4;
    // (halves: update of [3000,200] with 80 buckets by 4 rows 4.6 us either way, [640,5760] by 2 rows 8.4 and 7.5)
    // A tile with more (bucket, row) pairs than threads: a thread walks a bucket's list for two rows, an entry
    // is taken apart once for both.  Update and random-block step, one row and two rows a thread: [33278,650]
    // 24.0 and 22.5, 38.5 and 37.3 us; [30522,1024] 33.1 and 31.9, 54.0 and 52.6; [6144,1024] 10.9 and 10.2, 17.5 and
    // 16.8; [9000,333] with 166 buckets 9.9 and 8.7, 13.3 and 12.2.  Four rows were slower than two everywhere
    // ([33278,650] 25.4), and two lose where they leave threads without work ([20000,300] with 15 buckets 9.0
    // and 9.7).
    if (rows >= 2 && total > T) {
        constexpr int kTrip = 2;
        const int per = (rows + 1) >> 1, items = per * w;
        int jj = threadIdx.x / per, rg = threadIdx.x - jj * per;
        const int sjj = T / per, srg = T - sjj * per;
        for (int p = threadIdx.x; p < items; p += T) {
            const int j = ord_l[jj], ra = 2 * rg, rb2 = ra + 1 < rows ? ra + 1 : ra;
            const uint32_t e0 = csr_l[j], e1 = csr_l[j + 1];
            const float *va = vals + ra * d, *vb = vals + rb2 * d;
            float acc_a = cells[ra * w + j], acc_b = cells[rb2 * w + j];
            const double decay_a = __dmul_rn(one_minus_beta, (double)acc_a), decay_b = __dmul_rn(one_minus_beta, (double)acc_b);
            for (uint32_t e = e0; e < e1; e += kTrip) {
                uint32_t en[kTrip];
                float ta[kTrip], tb[kTrip];
#pragma unroll
                for (int u = 0; u < kTrip; ++u) en[u] = ent_l[e + u < e1 ? e + u : e1 - 1];
#pragma unroll
                for (int u = 0; u < kTrip; ++u) {
                    const uint32_t at = en[u] & 0x7fffu, flip = ((~en[u]) & 0x8000u) << 16;      // sign bit clear (-1): flip the float's sign
                    ta[u] = (float)__dsub_rn((double)__uint_as_float(__float_as_uint(va[at]) ^ flip), decay_a);
                    tb[u] = (float)__dsub_rn((double)__uint_as_float(__float_as_uint(vb[at]) ^ flip), decay_b);
                }
#pragma unroll
                for (int u = 0; u < kTrip; ++u)
                    if (e + u < e1) {
                        acc_a = __fadd_rn(acc_a, ta[u]);
                        acc_b = __fadd_rn(acc_b, tb[u]);
                    }
            }
            conef_st(cs_out + (row0 + ra) * w + j, acc_a);
            if (rb2 != ra) conef_st(cs_out + (row0 + rb2) * w + j, acc_b);
            jj += sjj;
            rg += srg;
            if (rg >= per) {
                rg -= per;
                ++jj;
            }
        }
        return;
    }
    int jj = threadIdx.x / rows, row = threadIdx.x - jj * rows;
    const int sjj = T / rows, srow = T - sjj * rows;
    for (int p = threadIdx.x; p < total; p += T) {
        const int j = ord_l[jj];
        const int cell = row * w + j;
        const uint32_t e0 = csr_l[j], e1 = csr_l[j + 1];
        const float aux = cells[cell];
        const double decay = __dmul_rn(one_minus_beta, (double)aux);
        const float* vr = vals + row * d;
        float acc = aux;
        // kWalk entries a trip: their list words and values are requested together and the terms
        // formed side by side; only the adds onto the cell are a chain.  Slots past the end of the
        // list read its last entry and are not added.
        for (uint32_t e = e0; e < e1; e += kWalk) {
            uint32_t en[kWalk];
            float term[kWalk];
#pragma unroll
            for (int u = 0; u < kWalk; ++u) en[u] = ent_l[e + u < e1 ? e + u : e1 - 1];
#pragma unroll
            for (int u = 0; u < kWalk; ++u) {
                uint32_t flip = ((~en[u]) & 0x8000u) << 16;      // sign bit clear (-1): flip the float's sign
                double sv = (double)__uint_as_float(__float_as_uint(vr[en[u] & 0x7fffu]) ^ flip);
                term[u] = (float)__dsub_rn(sv, decay);
            }
#pragma unroll
            for (int u = 0; u < kWalk; ++u)
                if (e + u < e1) acc = __fadd_rn(acc, term[u]);
        }
        conef_st(cs_out + row0 * w + cell, acc);
        jj += sjj;
        row += srow;
        if (row >= rows) {
            row -= rows;
            ++jj;
        }
    }
}

template <typename CsT, typename Front>
__global__ void __launch_bounds__(Front::kThreads)
conef_rowlist_kernel(Front front, ConefRowlistView plan, const CsT* cs_in, CsT* cs_out, int64_t n, int d, int w,
                     int rb, double one_minus_beta, bool pk_lds)
{
    conef_rowlist_body<CsT, Front>(front, plan, cs_in, cs_out, n, d, w, rb, one_minus_beta, (int)blockIdx.x, pk_lds);
}

template <typename CsT, typename Front>
int conef_launch_rowlist_shape(Front front, const ConefRowlistShape& shape, ConefRowlistView plan, const CsT* cs_in, CsT* cs_out,
                               int64_t n, int64_t d, int32_t w, float beta, hipStream_t s)
{
    auto k = conef_rowlist_kernel<CsT, Front>;
    hipError_t e = conef_allow_lds((const void*)k, shape.lds);
    if (e != hipSuccess) return (int)e;
    const double omb = 1. - (double)beta;   // (1. - beta) with beta an fp32 value, CountSketch.py:38,63
    conef_launch(k, dim3((unsigned)shape.tiles), dim3(Front::kThreads), shape.lds, s, front, plan, cs_in,
                       cs_out, n, (int)d, (int)w, shape.rb, omb, shape.pk_lds);
    return (int)hipGetLastError();
}

template <typename CsT, typename Front>
int conef_launch_rowlist(Front front, ConefRowlistView plan, const CsT* cs_in, CsT* cs_out, int64_t n, int64_t d,
                         int32_t w, float beta, hipStream_t s)
{
    ConefRowlistShape shape;
    if (!conef_rowlist_shape(n, d, w, Front::kNeedsCells, Front::halves(d), &shape)) return CONEF_ERR_INVALID;
    return conef_launch_rowlist_shape(front, shape, plan, cs_in, cs_out, n, d, w, beta, s);
}

// The same for a front of any workgroup size, made by make(std::integral_constant<int, threads>).
template <template <int> class FrontT, typename CsT, typename Make>
int conef_launch_rowlist_any(Make make, ConefRowlistView plan, const CsT* cs_in, CsT* cs_out, int64_t n, int64_t d, int32_t w, float beta,
                             hipStream_t s)
{
    using Front = FrontT<kConefRowlistThreads>;
    ConefRowlistShape shape;
    if (!conef_rowlist_shape(n, d, w, Front::kNeedsCells, Front::halves(d), &shape)) return CONEF_ERR_INVALID;
    conef_rowlist_taller(n, d, w, Front::kNeedsCells, &shape);
    auto go = [&](auto threads) { return conef_launch_rowlist_shape(make(threads), shape, plan, cs_in, cs_out, n, d, w, beta, s); };
    switch (conef_rowlist_workgroup(shape.lds, shape.tiles, (double)n * (double)d, Front::kLeastValues)) {
        case 256: return go(std::integral_constant<int, 256>());
        case 512: return go(std::integral_constant<int, 512>());
        default: return go(std::integral_constant<int, 1024>());
    }
}
