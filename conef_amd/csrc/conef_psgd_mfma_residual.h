// The last launch of a round with a sketched error at ranks 9 to 32: M = P Q^T on the matrix cores, the residual
// sketched where it is formed.
//
// The dense form of these ranks writes the residual (psgd_mfma_pqt_body, MODE 1) for a row-list launch to read: 8 of
// the 16 bytes an element the two move.  A row-list tile is a few rows (8192 values: 8 of 1024 columns, 2 of 4096), which
// a 32 x 32 tile of the matrix cores would waste three quarters of and more.  v_mfma_f32_4x4x1 with its first operand
// broadcast to all sixteen blocks is a 4-row tile instead: D[4][64] += A[4][1] B[1][64], lane l holds column l of B and
// of D, register v of D is row v.  A lane so owns a column; its RP entries of Q stay in registers for the rows of the
// tile, and two registers (one at rank 16) hold P of four rows: lane 4 b + i has P[i][b], and the step that wants k = b
// names block b.
//
// Two groups of four rows side by side: a chain of 32 dependent steps is what one alone waits for.  What is left is the sum of
// three phases that the tiles of a CU overlap in part: [30522,1024] at rank 32 takes 65 us, 45 without the products and
// 51 without the walk (40 without either and Q loaded once: 6.8 TB/s).  In a BERT step at rank 32 the two launches
// it replaces took 25 + 14 us a bucket, it takes 20 to 24.
//
// Both instructions are chains of fused multiply-adds, 32x32x2 its two k in order (compared over 2e5 entries), so the
// steps here go k = 0, RP/2, 1, RP/2 + 1, .. as psgd_mfma_pqt_body's do and M comes out the same to the bit.
#pragma once
#include "conef_device.h"
#include "conef_psgd_mfma.h"
#include "conef_rowlist.h"
#include <utility>

typedef float conef_f4v __attribute__((ext_vector_type(4)));

// G groups of four rows, their chains side by side.
template <int RP, int G, int... S>
__device__ __forceinline__ void conef_mfma_rows4(const float (*a)[RP / 16], const float* q, conef_f4v* acc, std::integer_sequence<int, S...>)
{
    constexpr int KS = RP / 2;
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g] = {0.f, 0.f, 0.f, 0.f};
    auto step = [&](auto k) {
        constexpr int K = decltype(k)::value;
#pragma unroll
        for (int g = 0; g < G; ++g) acc[g] = __builtin_amdgcn_mfma_f32_4x4x1f32(a[g][K / 16], q[K], acc[g], 4, K % 16, 0);
    };
    ((step(std::integral_constant<int, S>()), step(std::integral_constant<int, KS + S>())), ...);
}

// Q [m, RP] by pieces of four floats of a row, one column's after the other's, then the next piece: a wave's load of a
// piece is one run of 1 KB (from the row-major factor 64 lines of 128 bytes).
__host__ __device__ __forceinline__ int64_t conef_piece_at(int64_t m, int piece, int64_t col) { return (piece * m + col) * 4; }

// Front of the row-list kernel (conef_rowlist.h).  LOOK: M lies as the gradient came, and X is formed here
// (conef_psgd_look.h); the tile's old cells go to their place in LDS first.
template <int RP, bool LOOK, int T>
struct ListMfmaResidual {
    float* x;
    const float* p;          // [n, RP]
    const float* qp;         // Q by pieces
    MfmaLook look;
    static constexpr bool kNeedsCells = false, kParksCells = LOOK, kCompact = true;
    static constexpr int kThreads = T;
    struct Regs {};
    __device__ __forceinline__ void stage(int64_t row0, int rows, int d, int w, float* vals, float* cells, const uint32_t*) const
    {
        constexpr int H = RP / 16, W = T / 64;
        constexpr int kRows = 8, G = kRows / 4;            // rows of a column that are requested together
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        float* base = x + row0 * d;
        const int blocks = (d + 63) >> 6;
        // Units of (eight rows, block of 64 columns), blocks first.  More waves than blocks: the waves of a block
        // take turns at its rows.
        const int split = blocks < W ? W / blocks : 1, bstep = split > 1 ? blocks : W;
        const int part = wave / bstep;
        const int block0 = wave - part * bstep;
        int r = part < split ? kRows * part : rows, block = block0;
        float q[RP], qn[RP], xn[kRows], a[G][H], an[G][H];
        uint32_t pkn = 0;
        auto request = [&](bool rows_too, float* qd) {     // what the unit (r, block) reads
            const int c = block * 64 + lane < d ? block * 64 + lane : d - 1;
#pragma unroll
            for (int v = 0; v < RP / 4; ++v) conef_ld4u(qp + conef_piece_at(d, v, c), qd + 4 * v);
            if constexpr (LOOK) pkn = look.pk[c];
            const float* src = base + (int64_t)r * d + c;
#pragma unroll
            for (int u = 0; u < kRows; ++u)
                if (r + u < rows) xn[u] = src[(int64_t)u * d];                     // uniform
            if (rows_too) {
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const int i = r + 4 * g + (lane & 3);
                    const float* pi = p + (row0 + (i < rows ? i : rows - 1)) * RP + (lane >> 2);
#pragma unroll
                    for (int h = 0; h < H; ++h) an[g][h] = pi[16 * h];
                }
            }
        };
        bool have = r < rows && block < blocks, fresh = true;
        if (have) request(true, qn);
        if constexpr (LOOK) {                              // they travel together
            const float* src = look.cs + row0 * w;
            const int count = rows * w;
            constexpr int kPark = 4;
            for (int i0 = threadIdx.x; i0 < count; i0 += kPark * T) {
                float t[kPark];
#pragma unroll
                for (int u = 0; u < kPark; ++u) t[u] = src[i0 + u * T < count ? i0 + u * T : count - 1];
#pragma unroll
                for (int u = 0; u < kPark; ++u)
                    if (i0 + u * T < count) cells[i0 + u * T] = t[u];
            }
            __syncthreads();
        }
        while (have) {
            const int cur = block, first = r;
            float xv[kRows];
#pragma unroll
            for (int u = 0; u < kRows; ++u) {
                xv[u] = xn[u];
                if constexpr (LOOK)
                    if (first + u < rows)
                        xv[u] = __fadd_rn(xv[u], conef_query_term(cells[(first + u) * w + (int)(pkn & 0x7fffffffu)], pkn, look.alpha));
            }
#pragma unroll
            for (int t = 0; t < RP; ++t) q[t] = qn[t];
            if (fresh) {
#pragma unroll
                for (int g = 0; g < G; ++g)
#pragma unroll
                    for (int h = 0; h < H; ++h) a[g][h] = an[g][h];
            }
            block += bstep;
            fresh = block >= blocks;
            if (fresh) {
                block = block0;
                r += kRows * split;
            }
            have = r < rows;
            if (have) request(fresh, qn);
            const int c = cur * 64 + lane;
            conef_f4v acc[G];
            if (first + 4 < rows) conef_mfma_rows4<RP, G>(a, q, acc, std::make_integer_sequence<int, RP / 2>());      // uniform
            else conef_mfma_rows4<RP, 1>(a, q, acc, std::make_integer_sequence<int, RP / 2>());
            if (c < d) {
#pragma unroll
                for (int u = 0; u < kRows; ++u)
                    if (first + u < rows) {
                        const float mh = acc[u >> 2][u & 3];
                        base[(int64_t)(first + u) * d + c] = mh;
                        vals[(first + u) * d + c] = __fsub_rn(xv[u], mh);
                    }
            }
        }
    }
};

template <int RP, bool LOOK, int T>
struct MfmaResidualItem {
    ListMfmaResidual<RP, LOOK, T> front;
    ConefRowlistView plan;
    const float* cs_in;
    float* cs_out;
    int64_t n;
    int d, w, rb;
};
