// One foreign call per bucket for the random-block hooks: every >= 2-D tensor of a bucket goes
// through its fused step from a table of items, instead of one call per tensor from the hook's
// Python loop (reference loops: RandomBlock_hook.py:215-245, UnbiasedRandomBlock_hook.py:150-170).
//
// The dense steps (unbiased block, dense error feedback) of all tensors share one launch: the table
// travels by value, a workgroup finds its tensor from the running workgroup count and then does
// what it would do in a launch of its own.  Sketched steps on row-list plans share one launch the
// same way; a sketched step on a binned plan (a few long rows) or without a plan is issued by its
// single-tensor launcher from inside this call.  Same kernels' arithmetic on the same values: the
// results are bit-identical to the single-tensor entry points.
#include <vector>

#include "conef_plan.h"
#include "conef_randblock_core.h"
#include "conef_hip.h"

namespace {

// Tensors a launch takes: as many as its arguments have room for (4 KB).  The arguments of a launch
// are copied into memory the GPU reads whatever part of them is used, 3 us for 3 KB: buckets of up
// to four tensors (a layer, an LSTM's) take a table of four.
template <typename Item>
constexpr int rb_batch_max() { return sizeof(Item) <= 64 ? 48 : 32; }
constexpr int kRbFew = 4;

template <typename Item, int CAP = rb_batch_max<Item>()>
struct RbBatch {
    Item item[CAP];
    int first[CAP + 1];   // first workgroup of item i; first[count] = workgroups in all
    int count;
};

template <typename Item, int CAP>
__device__ __forceinline__ int rb_locate(const RbBatch<Item, CAP>& b, int* local, int* width)
{
    int i = 0, last = b.count - 1;                // the last item that starts at or before this workgroup
    while (i < last) {
        const int mid = (i + last + 1) >> 1;
        if (b.first[mid] <= (int)blockIdx.x) i = mid;
        else last = mid - 1;
    }
    *local = (int)blockIdx.x - b.first[i];
    *width = b.first[i + 1] - b.first[i];
    return i;
}

struct DenseItem {
    float* x;
    float* err;        // dense error (mode 1), unused otherwise
    float* payload;
    int64_t numel;
    ConefBlock blk;
    float prob;        // mode 0
};

template <int CAP>
__global__ void __launch_bounds__(256) randblock_unbiased_batch_kernel(RbBatch<DenseItem, CAP> b)
{
    int local, width;
    const DenseItem& it = b.item[rb_locate(b, &local, &width)];
    conef_randblock_unbiased_body(it.x, it.payload, it.numel, it.blk, it.prob, local, width);
}

template <int CAP>
__global__ void __launch_bounds__(256) randblock_ef_batch_kernel(RbBatch<DenseItem, CAP> b)
{
    int local, width;
    const DenseItem& it = b.item[rb_locate(b, &local, &width)];
    conef_randblock_ef_body(it.x, it.err, it.payload, it.numel, it.blk, local, width);
}

struct ListItem {
    float* x;
    float* payload;
    ConefBlock blk;
    float alpha;
    ConefRowlistView plan;
    const float* cs_in;
    float* cs_out;
    int64_t n;
    int d, w, rb;
    bool pk_lds;
};

template <int CAP, int T>
__global__ void __launch_bounds__(T)
randblock_rowlist_batch_kernel(RbBatch<ListItem, CAP> b, double one_minus_beta)
{
    int local, width;
    const ListItem& it = b.item[rb_locate(b, &local, &width)];
    const ConefListRandBlockT<T> front = {it.x, it.payload, it.blk, it.alpha};
    conef_rowlist_body<float, ConefListRandBlockT<T>>(front, it.plan, it.cs_in, it.cs_out, it.n, it.d, it.w, it.rb,
                                                      one_minus_beta, local, it.pk_lds);
}

template <typename Item, int CAP, typename Go>
int rb_run_cap(const std::vector<Item>& table, const std::vector<int>& blocks, Go go)
{
    size_t k = 0;
    while (k < table.size()) {
        RbBatch<Item, CAP> b;
        int nb = 0, total = 0;
        while (k < table.size() && nb < CAP) {
            b.item[nb] = table[k];
            b.first[nb] = total;
            total += blocks[k];
            ++nb;
            ++k;
        }
        b.first[nb] = total;
        b.count = nb;
        if (total > 0) go(b, total);
    }
    return (int)hipGetLastError();
}

// go(batch, workgroups) for the table in runs; `go` is generic over the batch's capacity
template <typename Item, typename Go>
int rb_run(const std::vector<Item>& table, const std::vector<int>& blocks, Go go)
{
    if (table.size() <= (size_t)kRbFew) return rb_run_cap<Item, kRbFew>(table, blocks, go);
    return rb_run_cap<Item, rb_batch_max<Item>()>(table, blocks, go);
}

inline bool by_row_list(const ConefRandBlockItem& it)
{
    const ConefPlanHeader* hp = (const ConefPlanHeader*)it.plan_host;
    return hp && hp->kind == kConefPlanRowlist;
}

// How a launch takes the tensors on row lists of a sketched step.
struct ListTiles {
    std::vector<ConefRowlistShape> shapes;      // of those tensors, in order
    size_t lds;
    int threads;
};

inline bool list_tiles(const ConefRandBlockItem* items, int count, ListTiles* lt)
{
    std::vector<ConefRowlistShape> taller;
    std::vector<double> values;
    size_t lds = 0;
    for (int k = 0; k < count; ++k) {
        const ConefRandBlockItem& it = items[k];
        if (!by_row_list(it)) continue;
        ConefRowlistShape shape;
        if (!conef_rowlist_shape(it.n, it.m, it.w, ConefListRandBlock::kNeedsCells, ConefListRandBlock::halves(it.m), &shape)) return false;
        lt->shapes.push_back(shape);
        conef_rowlist_taller(it.n, it.m, it.w, ConefListRandBlock::kNeedsCells, &shape);
        taller.push_back(shape);
        values.push_back((double)it.n * (double)it.m);
        lds = std::max(lds, shape.lds);
    }
    // A launch gives every tile the LDS of its largest: taller ones where half the values are in tiles of half of that.
    // Steps with one row by 256 threads and so, us: WRN-28-10 with sketches of 0.05 and 0.5 192 and 172, 325 and 242,
    // an LSTM of 500 and one of 300 66 and 53, 34 and 21, an encoder of 1024 with 0.2 327 and 302.
    double all = 0., large = 0.;
    for (size_t k = 0; k < values.size(); ++k) {
        all += values[k];
        if (2 * taller[k].lds >= lds) large += values[k];
    }
    if (2. * large >= all) lt->shapes = taller;
    lt->lds = 0;
    int64_t tiles = 0;
    for (const ConefRowlistShape& t : lt->shapes) {
        tiles += t.tiles;
        lt->lds = std::max(lt->lds, t.lds);
    }
    lt->threads = values.empty() ? 0 : conef_rowlist_workgroup(lt->lds, tiles, all, ConefListRandBlock::kLeastValues);
    return true;
}

}  // namespace

extern "C" {

int conef_randblock_step_batch_f32(const ConefRandBlockItem* items, int32_t count, int32_t mode, float alpha,
                                   float beta, int32_t a, int32_t b, void* stream)
{
    if (count < 0 || (count > 0 && !items) || mode < 0 || mode > 2) return CONEF_ERR_INVALID;
    if (count == 0) return CONEF_OK;
    // everything is checked before anything is enqueued
    for (int k = 0; k < count; ++k) {
        const ConefRandBlockItem& it = items[k];
        if (it.n < 1 || it.m < 1 || (mode == 2 && it.m > 0x7fffffffLL) || !it.x || !it.payload) return CONEF_ERR_INVALID;
        const int64_t numel = it.n * it.m;
        if (!(it.start >= 0 && it.start < numel && it.block >= 1 && it.block <= numel)) return CONEF_ERR_INVALID;
        if (mode == 1 && !it.err) return CONEF_ERR_INVALID;
        if (mode == 2) {
            if (!it.cs_in || !it.cs_out || it.w < 1 || it.w > (1 << 30)) return CONEF_ERR_INVALID;
            if (it.plan_host) {
                const ConefPlanHeader* hp = (const ConefPlanHeader*)it.plan_host;
                if (!conef_plan_matches(hp, it.n, it.m, it.w, a, b) || !it.plan_dev) return CONEF_ERR_INVALID;
                if (hp->kind == kConefPlanBinned && (!it.staging || it.cs_in == it.cs_out)) return CONEF_ERR_INVALID;
            }
        }
    }
    hipStream_t s = (hipStream_t)stream;
    if (mode == 0 || mode == 1) {
        std::vector<DenseItem> table;
        std::vector<int> blocks;
        for (int k = 0; k < count; ++k) {
            const ConefRandBlockItem& it = items[k];
            const int64_t numel = it.n * it.m;
            DenseItem d;
            d.x = it.x;
            d.err = it.err;
            d.payload = it.payload;
            d.numel = numel;
            d.blk = conef_make_block(numel, it.start, it.block);
            // the reference divides by the Python double block / numel, which reaches the tensor as fp32
            d.prob = (float)((double)it.block / (double)numel);
            table.push_back(d);
            blocks.push_back(conef_rb_groups(numel, mode == 0 ? kRbUnbiasedQuads : kRbEfQuads));
        }
        if (mode == 0)
            return rb_run(table, blocks, [&](const auto& bt, int grid) {
                conef_launch((randblock_unbiased_batch_kernel<sizeof(bt.item) / sizeof(bt.item[0])>), dim3((unsigned)grid), dim3(256), 0, s, bt);
            });
        return rb_run(table, blocks, [&](const auto& bt, int grid) {
            conef_launch((randblock_ef_batch_kernel<sizeof(bt.item) / sizeof(bt.item[0])>), dim3((unsigned)grid), dim3(256), 0, s, bt);
        });
    }
    // sketched error: row-list plans share launches, the rest go one by one
    std::vector<ListItem> table;
    for (int k = 0; k < count; ++k) {
        const ConefRandBlockItem& it = items[k];
        if (!by_row_list(it)) continue;
        table.push_back(ListItem{it.x, it.payload, conef_make_block(it.n * it.m, it.start, it.block), alpha,
                                 conef_rowlist_view((const ConefPlanHeader*)it.plan_host, it.plan_dev), it.cs_in, it.cs_out, it.n,
                                 (int)it.m, it.w, 0, false});
    }
    ListTiles tiles;
    if (!list_tiles(items, count, &tiles)) return CONEF_ERR_INVALID;
    if (!table.empty()) {
        const size_t lds = tiles.lds;
        std::vector<int> blocks;
        for (size_t k = 0; k < table.size(); ++k) {
            table[k].rb = tiles.shapes[k].rb;
            table[k].pk_lds = tiles.shapes[k].pk_lds;
            blocks.push_back((int)tiles.shapes[k].tiles);
        }
        const double omb = 1. - (double)beta;
        auto with = [&](auto threads) {
            constexpr int T = decltype(threads)::value;
            hipError_t e = hipSuccess;
            const int rc = rb_run(table, blocks, [&](const auto& bt, int grid) {
                auto kern = randblock_rowlist_batch_kernel<sizeof(bt.item) / sizeof(bt.item[0]), T>;
                e = conef_allow_lds((const void*)kern, lds);
                if (e == hipSuccess) conef_launch(kern, dim3((unsigned)grid), dim3(T), lds, s, bt, omb);
            });
            return e != hipSuccess ? (int)e : rc;
        };
        int rc;
        switch (tiles.threads) {
            case 256: rc = with(std::integral_constant<int, 256>()); break;
            case 512: rc = with(std::integral_constant<int, 512>()); break;
            default: rc = with(std::integral_constant<int, 1024>()); break;
        }
        if (rc != CONEF_OK) return rc;
    }
    for (int k = 0; k < count; ++k) {
        const ConefRandBlockItem& it = items[k];
        if (by_row_list(it)) continue;
        int rc;
        if (it.plan_host)
            rc = conef_randblock_conef_step_planned_f32(it.x, it.cs_in, it.cs_out, it.payload, it.plan_host, it.plan_dev,
                                                        it.staging, it.n, it.m, it.w, it.start, it.block, alpha, beta, a,
                                                        b, stream);
        else
            rc = conef_randblock_conef_step_f32(it.x, it.cs_in, it.cs_out, it.payload, it.n, it.m, it.w, it.start,
                                                it.block, alpha, beta, a, b, stream);
        if (rc != CONEF_OK) return rc;
    }
    return CONEF_OK;
}

// Host only.
int conef_randblock_step_tiles(const ConefRandBlockItem* items, int32_t count, int32_t a, int32_t b, int32_t* rows, int32_t* threads)
{
    if (count < 0 || (count > 0 && (!items || !rows)) || !threads) return CONEF_ERR_INVALID;
    for (int k = 0; k < count; ++k) {
        const ConefRandBlockItem& it = items[k];
        if (it.n < 1 || it.m < 1 || it.m > 0x7fffffffLL || it.w < 1 || it.w > (1 << 30)) return CONEF_ERR_INVALID;
        if (it.plan_host && !conef_plan_matches((const ConefPlanHeader*)it.plan_host, it.n, it.m, it.w, a, b)) return CONEF_ERR_INVALID;
    }
    ListTiles tiles;
    if (!list_tiles(items, count, &tiles)) return CONEF_ERR_INVALID;
    size_t at = 0;
    for (int k = 0; k < count; ++k) rows[k] = by_row_list(items[k]) ? tiles.shapes[at++].rb : 0;
    *threads = tiles.threads;
    return CONEF_OK;
}

}  // extern "C"
