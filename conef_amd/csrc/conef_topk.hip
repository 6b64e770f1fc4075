// Magnitude top-k sparsifier (gfx950) for the dense error kept by the hPowerSGD hook.
//
// Reference semantics: communication/hPowerSGD_hook.py:90-97 - keep the k entries of largest
// magnitude, zero everything else, in place.  The reference asks torch.topk for unsorted
// positions and so leaves ties open; here ties on the threshold magnitude keep the lowest flat
// indices, which makes the result a function of the input alone.
//
// Selection is a most-significant-digit radix select on the 31 magnitude bits (a non-negative
// float orders like its bit pattern) in three histogram passes of 11, 11 and 9 bits.  Choosing the
// digit that holds the k-th largest key is not a launch of its own: every workgroup of the next
// pass does it from the finished histogram before it starts (2048 counters, one suffix scan).
// The filter keeps every key at or above the threshold.  If more keys equal the threshold than may
// be kept (two equal magnitudes at the threshold turn up in a few percent of million-element
// gradients; at a zero threshold it makes no difference which zeros stay), the filter's workgroups
// also note where those keys sit, and the workgroup that finishes last ranks the noted indices
// and clears the ties past the first `remaining` of them.  More than 1024 such ties (a tensor of
// repeated values) are settled by one workgroup walking the tensor in index order instead: exact,
// slow, and of no practical concern.  Nothing returns to the host between passes.
#include <mutex>

#include "conef_device.h"
#include "conef_hip.h"

namespace {

constexpr int kPasses = 3;
constexpr int kDigitBits[kPasses] = {11, 11, 9};
constexpr int kDigitShift[kPasses] = {20, 9, 0};
constexpr int kBins = 2048;          // bins of the widest digit
constexpr int kFilterChunk = 1024;   // elements per workgroup iteration in the ordered walk
constexpr int kTieMax = 1024;        // surplus ties up to this many are ranked from a list, more by a walk

struct TopkState {
    uint32_t k;
    uint32_t prefix[kPasses];       // prefix[p]: selected digits of passes 0..p, written by pass p + 1
    uint32_t remaining[kPasses];    // how many keys to take among those matching prefix[p]
    uint32_t ties[kPasses];         // keys that match prefix[p] exactly in their high digits
    uint32_t done;                  // workgroups of the filter that have finished (surplus ties only)
    uint32_t tie_count;             // indices recorded in tie_idx so far
    uint32_t final_count;           // keys gathered in final_idx so far (selection through a candidate list)
    uint32_t pad[3];
    uint32_t hist[kPasses][kBins];
    uint32_t tie_idx[kTieMax];      // where the keys equal to the threshold sit, in no order
};

__device__ __forceinline__ uint32_t mag_key(float v) { return __float_as_uint(v) & 0x7fffffffu; }

// Several tensors per launch (the dense errors of a bucket's matrices, each with its own k and its
// own state): the table travels by value, a workgroup finds its tensor from the running workgroup
// count (`first`, the same for every pass) and then
// does what it would do in a launch of its own.  The arguments of a launch are copied into memory the GPU
// reads whatever part of them is used (3 us for 3 KB): up to eight tensors, most buckets of a large model,
// take a table of eight, more of them one of 48 (2.9 KB).
constexpr int kTopkBatchFew = 8, kTopkBatchMax = 48;

struct TopkItem {
    float* x;
    int64_t numel;
    TopkState* st;
    uint32_t k;
    uint32_t cap;               // candidates a workgroup's segment holds
    uint32_t* counts;           // [workgroups] candidates found, or kTopkOverflow
    uint2* list;                // [workgroups][cap] (index, magnitude key)
    uint32_t* final_idx;        // [kTopkFinal] the keys that share two digits with the threshold, then their keys
};

template <int CAP>
struct TopkBatch {
    TopkItem item[CAP];
    int first[CAP + 1];
    int count;
};

__device__ __forceinline__ int topk_locate(const int* first, int count, int* local, int* width)
{
    int i = 0;
    while (i + 1 < count && (int)blockIdx.x >= first[i + 1]) ++i;
    *local = (int)blockIdx.x - first[i];
    *width = first[i + 1] - first[i];
    return i;
}

__device__ __forceinline__ void topk_init_body(TopkState* st, uint32_t k)
{
    for (int i = threadIdx.x; i < kPasses * kBins; i += blockDim.x) (&st->hist[0][0])[i] = 0u;
    if (threadIdx.x == 0) {
        st->k = k;
        st->done = 0u;
        st->tie_count = 0u;
        st->final_count = 0u;
    }
}

__global__ void topk_init_kernel(TopkState* st, uint32_t k) { topk_init_body(st, k); }

template <int CAP>
__global__ void topk_init_batch_kernel(TopkBatch<CAP> b) { topk_init_body(b.item[blockIdx.x].st, b.item[blockIdx.x].k); }

// The bin that holds the want-th largest of the keys counted in 256 * per bins, thread t holding the counts
// of bins t * per .. in cnt: (bin, how many are wanted of it, how many it holds), the same in every
// thread of a 256-thread workgroup.
__device__ __forceinline__ void topk_pick(const uint32_t (&cnt)[8], int per, uint32_t want, uint32_t* bin, uint32_t* wanted,
                                          uint32_t* held)
{
    __shared__ uint32_t wave_sum[4];
    __shared__ uint32_t picked[3];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint32_t mine = 0;
    for (int b = 0; b < per; ++b) mine += cnt[b];
    // suffix sums over threads: keys in bins above mine
    uint32_t incl = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        uint32_t t = __shfl_down(incl, off, 64);
        if (lane + off < 64) incl += t;
    }
    if (lane == 0) wave_sum[wave] = incl;
    __syncthreads();
    uint32_t above = incl - mine;
    for (int wv = wave + 1; wv < 4; ++wv) above += wave_sum[wv];
    // exactly one (thread, bin) satisfies above < want <= above + count
    for (int b = per - 1; b >= 0; --b) {
        if (above < want && want <= above + cnt[b]) {
            picked[0] = (uint32_t)(threadIdx.x * per + b);
            picked[1] = want - above;
            picked[2] = cnt[b];
        }
        above += cnt[b];
    }
    __syncthreads();
    *bin = picked[0];
    *wanted = picked[1];
    *held = picked[2];
    __syncthreads();
}

// What pass `p` selected, from its finished histogram: the digit holding the k-th largest key
// among those matching the earlier digits.  Every thread of a 256-thread workgroup returns the
// same (prefix, remaining, ties); workgroup 0 (bx) of the tensor also leaves them in the state for
// the next kernel.
__device__ __forceinline__ void topk_resolve(TopkState* st, int p, uint32_t* prefix, uint32_t* remaining, uint32_t* ties,
                                             int bx)
{
    const uint32_t before_prefix = p == 0 ? 0u : st->prefix[p - 1];
    const uint32_t before_remaining = p == 0 ? st->k : st->remaining[p - 1];
    const int per = (1 << kDigitBits[p]) / 256;          // 8, 8, 2 bins per thread
    uint32_t cnt[8];
    for (int b = 0; b < per; ++b) cnt[b] = st->hist[p][threadIdx.x * per + b];
    uint32_t digit;
    topk_pick(cnt, per, before_remaining, &digit, remaining, ties);
    *prefix = (before_prefix << kDigitBits[p]) | digit;
    if (bx == 0 && threadIdx.x == 0) {
        st->prefix[p] = *prefix;
        st->remaining[p] = *remaining;
        st->ties[p] = *ties;
    }
}

// REP copies of every bin, copy = lane % REP, laid out [bin][copy]: the keys of a gradient crowd
// into a few dozen bins of the first digit (one exponent and three mantissa bits), and lanes of a
// wave that meet in a bin then add to different LDS banks instead of queueing on one address.
// `kept` (a state that stays with its tensor from call to call, zero-filled before the first): no
// launch clears the state; the first workgroup of pass 0 clears what the later passes count into,
// and the filter's, or the settling pass's, clears what pass 0 of the next call counts into.
template <int REP, int T = 256>
__device__ __forceinline__ void
topk_hist_body(const float* __restrict__ x, int64_t numel, TopkState* st, int pass, int bx, int gx, bool kept = false,
               uint32_t k = 0)
{
    __shared__ uint32_t bins[kBins * REP];
    uint32_t prefix = 0, remaining = 0, ties = 0;
    if (pass > 0) topk_resolve(st, pass - 1, &prefix, &remaining, &ties, bx);
    if (kept && pass == 0 && bx == 0) {
        for (int i = threadIdx.x; i < (kPasses - 1) * kBins; i += T) (&st->hist[1][0])[i] = 0u;
        if (threadIdx.x == 0) {
            st->k = k;
            st->done = 0u;
            st->tie_count = 0u;
            st->final_count = 0u;
        }
    }
    const int nb = 1 << kDigitBits[pass];
    for (int i = threadIdx.x; i < nb * REP; i += T) bins[i] = 0u;
    __syncthreads();
    const int shift = kDigitShift[pass], hi = shift + kDigitBits[pass];
    const uint32_t mask = (uint32_t)nb - 1u;
    const int copy = (int)(threadIdx.x & (REP - 1));
    const int64_t quads = numel >> 2;
    const bool vec = (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
    const int64_t stride = (int64_t)gx * T;
    if (vec) {
        // eight 16-byte loads in flight per thread: a thread's share is sixteen quads or so, and every
        // round of loads is a trip to memory
        constexpr int U = 8;
        auto count = [&](float4 v) {
            const uint32_t key[4] = {mag_key(v.x), mag_key(v.y), mag_key(v.z), mag_key(v.w)};
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (pass == 0 || (key[e] >> hi) == prefix) atomicAdd(&bins[((key[e] >> shift) & mask) * REP + copy], 1u);
        };
        // Runs of 256 quads, run c to a workgroup whose number leaves the remainder of c by eight where there are
        // that many: a pass with more threads in a workgroup then reads a run on the XCD whose L2 the next pass
        // finds it in.
        const int run = T == 256 || (gx & 7) ? bx * (T / 256) + ((int)threadIdx.x >> 8)
                                             : (bx >> 3) * (T / 32) + ((int)threadIdx.x >> 8) * 8 + (bx & 7);
        int64_t q0 = (int64_t)run * 256 + (threadIdx.x & 255);
        for (; q0 + (U - 1) * stride < quads; q0 += U * stride) {
            float4 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = reinterpret_cast<const float4*>(x)[q0 + u * stride];
#pragma unroll
            for (int u = 0; u < U; ++u) count(v[u]);
        }
        if (q0 < quads) {
            float4 v[U - 1];
#pragma unroll
            for (int u = 0; u < U - 1; ++u) {
                const int64_t q = q0 + u * stride;
                v[u] = reinterpret_cast<const float4*>(x)[q < quads ? q : q0];
            }
#pragma unroll
            for (int u = 0; u < U - 1; ++u)
                if (q0 + u * stride < quads) count(v[u]);
        }
    }
    for (int64_t i = (vec ? quads * 4 : 0) + bx * (int64_t)T + threadIdx.x; i < numel; i += stride) {
        uint32_t key = mag_key(x[i]);
        if (pass == 0 || (key >> hi) == prefix) atomicAdd(&bins[((key >> shift) & mask) * REP + copy], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nb; i += T) {
        uint32_t c = 0;
#pragma unroll
        for (int k = 0; k < REP; ++k) c += bins[i * REP + k];
        if (c) atomicAdd(&st->hist[pass][i], c);
    }
}

// pass 0 counts every key (replicated bins), the later passes only the few that match the prefix
__global__ void __launch_bounds__(256)
topk_hist_kernel(const float* __restrict__ x, int64_t numel, TopkState* st, int pass)
{
    if (pass == 0) topk_hist_body<4>(x, numel, st, 0, (int)blockIdx.x, (int)gridDim.x);
    else topk_hist_body<1>(x, numel, st, pass, (int)blockIdx.x, (int)gridDim.x);
}

template <int CAP>
__global__ void __launch_bounds__(256)
topk_hist_batch_kernel(TopkBatch<CAP> b, int pass, bool kept)
{
    int local, width;
    const TopkItem& it = b.item[topk_locate(b.first, b.count, &local, &width)];
    if (pass == 0) topk_hist_body<4>(it.x, it.numel, it.st, 0, local, width, kept, it.k);
    else topk_hist_body<1>(it.x, it.numel, it.st, pass, local, width);
}

// keys equal to the threshold, in index order: the first `keep_ties` stay, the rest are cleared.
// One workgroup of 256 threads, 1024 elements a round; once the quota is used up the rounds need
// no scan any more.
__device__ __forceinline__ void topk_order_ties(float* __restrict__ x, int64_t numel, uint32_t thr, uint32_t keep_ties)
{
    __shared__ uint32_t wave_ties[4];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint32_t running = 0;                       // ties seen in earlier rounds: the same in every thread
    for (int64_t base0 = 0; base0 < numel; base0 += kFilterChunk) {
        const int64_t base = base0 + (int64_t)threadIdx.x * 4;
        bool tie[4];
        uint32_t mine = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            tie[k] = base + k < numel && mag_key(x[base + k]) == thr;
            mine += tie[k];
        }
        if (running >= keep_ties) {             // uniform: nothing more may stay
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (tie[k]) x[base + k] = 0.f;
            continue;
        }
        uint32_t incl = mine;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            uint32_t t = __shfl_up(incl, off, 64);
            if (lane >= off) incl += t;
        }
        if (lane == 63) wave_ties[wave] = incl;
        __syncthreads();
        uint32_t rank = running + incl - mine;
        for (int wv = 0; wv < wave; ++wv) rank += wave_ties[wv];
        const uint32_t total = (wave_ties[0] + wave_ties[1]) + (wave_ties[2] + wave_ties[3]);
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (tie[k]) {
                if (rank >= keep_ties) x[base + k] = 0.f;
                ++rank;
            }
        running += total;
        __syncthreads();
    }
}

// Surplus ties on the threshold (`held` keys equal it, `keep_ties` of them stay): every workgroup comes here
// when it is through with its own share, up to kTieMax ties noted in tie_idx; the last one settles them.
__device__ __forceinline__ void topk_settle_ties(float* __restrict__ x, int64_t numel, TopkState* st, uint32_t thr,
                                                 uint32_t keep_ties, uint32_t held, int gx)
{
    __shared__ uint32_t ticket;
    __shared__ uint32_t tie_l[kTieMax];
    __syncthreads();
    if (threadIdx.x == 0) ticket = atomicAdd(&st->done, 1u);
    __syncthreads();
    if (ticket != (uint32_t)gx - 1u) return;
    __threadfence();
    if (held > (uint32_t)kTieMax) {
        topk_order_ties(x, numel, thr, keep_ties);
        return;
    }
    const int n = (int)held;
    for (int j = threadIdx.x; j < n; j += blockDim.x)
        tie_l[j] = __hip_atomic_load(&st->tie_idx[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    for (int j = threadIdx.x; j < n; j += blockDim.x) {
        const uint32_t mine = tie_l[j];
        uint32_t rank = 0;
        for (int t = 0; t < n; ++t) rank += tie_l[t] < mine;
        if (rank >= keep_ties) x[mine] = 0.f;
    }
}

// keep key >= threshold, zero the rest, settle surplus ties on the threshold by index
__device__ __forceinline__ void
topk_filter_body(float* __restrict__ x, int64_t numel, TopkState* st, int bx, int gx, bool kept = false)
{
    uint32_t thr, keep_ties, ties;
    topk_resolve(st, kPasses - 1, &thr, &keep_ties, &ties, bx);
    if (kept && bx == 0)       // nobody reads the first digit's counters any more: ready for the next call
        for (int i = threadIdx.x; i < kBins; i += 256) st->hist[0][i] = 0u;
    const bool surplus = ties != keep_ties && thr != 0u;      // a zero threshold has only zeros for ties
    const bool listed = surplus && ties <= (uint32_t)kTieMax;
    auto note = [&](int64_t i) {
        const uint32_t slot = atomicAdd(&st->tie_count, 1u);
        if (slot < (uint32_t)kTieMax) st->tie_idx[slot] = (uint32_t)i;
    };
    const int64_t quads = numel >> 2;
    const bool vec = (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
    const int64_t stride = (int64_t)gx * blockDim.x;
    if (vec) {
        // eight quads requested before the first is used (a load behind a store to the same array is
        // not moved up by the compiler: one quad a trip otherwise)
        constexpr int U = 8;
        for (int64_t q0 = bx * (int64_t)blockDim.x + threadIdx.x; q0 < quads; q0 += U * stride) {
            float4 vv[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t q = q0 + u * stride;
                vv[u] = reinterpret_cast<const float4*>(x)[q < quads ? q : q0];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t q = q0 + u * stride;
                if (q >= quads) break;
                const float4 v = vv[u];
                const uint32_t key[4] = {mag_key(v.x), mag_key(v.y), mag_key(v.z), mag_key(v.w)};
                bool k0 = key[0] >= thr, k1 = key[1] >= thr, k2 = key[2] >= thr, k3 = key[3] >= thr;
                if (!(k0 && k1 && k2 && k3))
                    reinterpret_cast<float4*>(x)[q] = make_float4(k0 ? v.x : 0.f, k1 ? v.y : 0.f, k2 ? v.z : 0.f, k3 ? v.w : 0.f);
                if (listed) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (key[e] == thr) note(4 * q + e);
                }
            }
        }
    }
    for (int64_t i = (vec ? quads * 4 : 0) + bx * (int64_t)blockDim.x + threadIdx.x; i < numel; i += stride) {
        const uint32_t key = mag_key(x[i]);
        if (key < thr) x[i] = 0.f;
        else if (listed && key == thr) note(i);
    }
    if (!surplus) return;
    // The workgroup that finishes last sees every noted index, and nobody else's 16-byte stores
    // (which rewrite a tie with its own value when a neighbour in the quad goes) can land after
    // the zeros it writes.
    __threadfence();
    topk_settle_ties(x, numel, st, thr, keep_ties, ties, gx);
}

__global__ void __launch_bounds__(256)
topk_filter_kernel(float* __restrict__ x, int64_t numel, TopkState* st)
{
    topk_filter_body(x, numel, st, (int)blockIdx.x, (int)gridDim.x);
}

template <int CAP>
__global__ void __launch_bounds__(256)
topk_filter_batch_kernel(TopkBatch<CAP> b, bool kept)
{
    int local, width;
    const TopkItem& it = b.item[topk_locate(b.first, b.count, &local, &width)];
    topk_filter_body(it.x, it.numel, it.st, local, width, kept);
}


// ---- selection through a candidate list ----
// Three histogram passes and the filter read a tensor four times.  After the first digit, though, only
// the keys that share it with the threshold are undecided - about one in twenty of a gradient's error,
// 11 bits being an exponent and three mantissa bits.  So, for a caller that lends room for lists:
//   pass 0     the first digit's histogram, as above;
//   pass 1     zeroes what lies below the digit, counts the second digit of the keys that share it
//              and notes them, (index, key), each workgroup in a segment of its own: no counter is shared;
//   pass 2     goes over the notes alone: zeroes what lies below the first two digits, counts the third of
//              the keys that share both and, if they are no more than kTopkFinal, gathers them;
//   pass 3     resolves the threshold and clears what lies below it: one workgroup over the gathered keys
//              (a few hundred of a gradient's), else every workgroup over its own notes once more.
// Two reads and one write of the tensor instead of four and one.  A workgroup whose segment runs over
// (more than a quarter of its keys share the digit) goes over its elements again instead of its notes.
// Every step is spread over all workgroups however the magnitudes are distributed, but for more than
// kTieMax keys equal to the threshold (as in the filter).  The keys that share two digits grow with the
// tensor - 2e-5 of a Gaussian's, more than kTopkFinal from 100 M elements on - and are all of a tensor
// whose magnitudes lie within 512 floats of each other.
constexpr uint32_t kTopkOverflow = 0xffffffffu;
constexpr int kTopkFinal = 2048;
constexpr int kTopkTrip = 8;             // quads a thread requests together

// f(index, key) for every element of a workgroup's share, in trips: the elements of quads first, then the rest
template <typename F>
__device__ __forceinline__ void topk_for_each(const float* x, int64_t numel, int bx, int gx, F f)
{
    const int64_t quads = numel >> 2, stride = (int64_t)gx * 256;
    for (int64_t q0 = bx * (int64_t)256 + threadIdx.x; q0 < quads; q0 += stride) {
        float v[4];
        conef_ld4u(x + 4 * q0, v);
#pragma unroll
        for (int e = 0; e < 4; ++e) f(4 * q0 + e, mag_key(v[e]));
    }
    for (int64_t i = quads * 4 + bx * (int64_t)256 + threadIdx.x; i < numel; i += stride) f(i, mag_key(x[i]));
}

__device__ __forceinline__ void topk_note_body(const TopkItem& it, int bx, int gx)
{
    __shared__ uint32_t bins[kBins];
    __shared__ uint32_t found;
    TopkState* st = it.st;
    uint32_t digit, remaining, ties;
    topk_resolve(st, 0, &digit, &remaining, &ties, bx);
    for (int i = threadIdx.x; i < kBins; i += 256) bins[i] = 0u;
    if (threadIdx.x == 0) found = 0u;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int shift = kDigitShift[0];
    uint2* seg = it.list + (size_t)bx * it.cap;
    const int64_t quads = it.numel >> 2, stride = (int64_t)gx * 256;
    const int64_t rest0 = quads * 4;
    // A thread's quads of one trip; the elements behind the last quad are a trip of single ones at the end.
    // Zeros are never noted: there is nothing to clear in them (they are counted where they share the digit).
    uint32_t zeros = 0u;
    auto note = [&](uint32_t mask, auto index_of, auto key_of) {
        const uint32_t mine = (uint32_t)__popc(mask);
        uint32_t incl = mine;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t t = __shfl_up(incl, off, 64);
            if (lane >= off) incl += t;
        }
        const uint32_t total = __shfl(incl, 63, 64);
        uint32_t base = 0;
        if (total && lane == 63) base = atomicAdd(&found, total);
        base = __shfl(base, 63, 64) + incl - mine;
        while (mask) {
            const int b = __ffs(mask) - 1;
            mask &= mask - 1;
            const uint32_t key = key_of(b);
            atomicAdd(&bins[(key >> kDigitShift[1]) & (kBins - 1)], 1u);
            if (base < it.cap) seg[base] = make_uint2(index_of(b), key);
            ++base;
        }
    };
    for (int64_t t0 = bx * (int64_t)256; t0 < quads; t0 += kTopkTrip * stride) {     // uniform: the waves scan together
        const int64_t q0 = t0 + threadIdx.x;
        float v[kTopkTrip][4];
#pragma unroll
        for (int u = 0; u < kTopkTrip; ++u) {
            const int64_t q = q0 + u * stride;
            conef_ld4u(it.x + 4 * (q < quads ? q : quads - 1), v[u]);
        }
        uint32_t mask = 0u;
#pragma unroll
        for (int u = 0; u < kTopkTrip; ++u) {
            const int64_t q = q0 + u * stride;
            if (q >= quads) continue;
            float o[4];
            bool any = false;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t key = mag_key(v[u][e]), d = key >> shift;
                o[e] = d >= digit ? v[u][e] : 0.f;
                any |= d < digit;
                if (d == digit) {
                    if (key) mask |= 1u << (4 * u + e);
                    else ++zeros;
                }
            }
            if (any) conef_st4u(it.x + 4 * q, o);
        }
        note(mask, [&](int b) { return (uint32_t)(4 * (q0 + (b >> 2) * stride) + (b & 3)); },
             [&](int b) {
                 float f = 0.f;
#pragma unroll
                 for (int u = 0; u < kTopkTrip; ++u)
#pragma unroll
                     for (int e = 0; e < 4; ++e) f = b == 4 * u + e ? v[u][e] : f;
                 return mag_key(f);
             });
    }
    for (int64_t t0 = rest0 + bx * (int64_t)256; t0 < it.numel; t0 += stride) {
        const int64_t i = t0 + threadIdx.x;
        uint32_t key = 0u;
        if (i < it.numel) {
            key = mag_key(it.x[i]);
            if ((key >> shift) < digit) it.x[i] = 0.f;
            if (digit == 0u && !key) ++zeros;
        }
        note(key && (key >> shift) == digit ? 1u : 0u, [&](int) { return (uint32_t)i; }, [&](int) { return key; });
    }
    if (zeros) atomicAdd(&bins[0], zeros);
    __syncthreads();
    if (threadIdx.x == 0) it.counts[bx] = found <= it.cap ? found : kTopkOverflow;
    for (int i = threadIdx.x; i < kBins; i += 256)
        if (bins[i]) atomicAdd(&st->hist[1][i], bins[i]);
}

constexpr int kTopkLow = 1 << kDigitBits[2];

// f(index, key) for a workgroup's notes, or for its elements that share the digit where it has none
template <typename F>
__device__ __forceinline__ void topk_for_notes(const TopkItem& it, uint32_t digit, int bx, int gx, F f)
{
    const uint32_t n = it.counts[bx];
    if (n == kTopkOverflow) {
        topk_for_each(it.x, it.numel, bx, gx, [&](int64_t i, uint32_t key) {
            if (key && (key >> kDigitShift[0]) == digit) f((uint32_t)i, key);
        });
        return;
    }
    const uint2* seg = it.list + (size_t)bx * it.cap;
    for (uint32_t j0 = threadIdx.x; j0 < n; j0 += 4 * 256) {
        uint2 c[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) c[u] = seg[j0 + u * 256 < n ? j0 + u * 256 : j0];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (j0 + u * 256 < n) f(c[u].x, c[u].y);
    }
}

// pass 2
__device__ __forceinline__ void topk_gather_body(const TopkItem& it, int bx, int gx)
{
    __shared__ uint32_t low[kTopkLow];
    TopkState* st = it.st;
    uint32_t prefix, keep, share;                        // `share` keys share both digits, `keep` of them stay
    topk_resolve(st, 1, &prefix, &keep, &share, bx);
    if (bx == 0)       // nobody reads the first digit's counters any more: ready for the next call
        for (int i = threadIdx.x; i < kBins; i += 256) st->hist[0][i] = 0u;
    for (int i = threadIdx.x; i < kTopkLow; i += 256) low[i] = 0u;
    __syncthreads();
    const bool undecided = keep < share, gathered = share <= (uint32_t)kTopkFinal;      // all of them stay otherwise
    topk_for_notes(it, prefix >> kDigitBits[1], bx, gx, [&](uint32_t i, uint32_t key) {
        const uint32_t two = key >> kDigitBits[2];
        if (two < prefix) {
            it.x[i] = 0.f;
        } else if (two == prefix && undecided) {
            atomicAdd(&low[key & (kTopkLow - 1)], 1u);
            if (gathered) {
                const uint32_t slot = atomicAdd(&st->final_count, 1u);      // below `share`
                it.final_idx[slot] = i;
                it.final_idx[kTopkFinal + slot] = key;
            }
        }
    });
    if (!undecided) return;
    __syncthreads();
    for (int i = threadIdx.x; i < kTopkLow; i += 256)
        if (low[i]) atomicAdd(&st->hist[2][i], low[i]);
}

// pass 3
__device__ __forceinline__ void topk_settle_body(const TopkItem& it, int bx, int gx)
{
    __shared__ uint32_t key_l[kTopkFinal], idx_l[kTopkFinal];
    __shared__ uint32_t total;
    TopkState* st = it.st;
    const uint32_t prefix = st->prefix[1], keep = st->remaining[1], share = st->ties[1];
    const bool gathered = share <= (uint32_t)kTopkFinal;
    if (keep >= share || (gathered && bx != 0)) return;
    // the third digit's counts: of the keys but not of the zeros that may share both digits with them
    uint32_t cnt[8], m = 0;
    if (threadIdx.x == 0) total = 0u;
    __syncthreads();
    for (int b = 0; b < kTopkLow / 256; ++b) {
        cnt[b] = st->hist[2][threadIdx.x * (kTopkLow / 256) + b];
        m += cnt[b];
    }
    if (m) atomicAdd(&total, m);
    __syncthreads();
    m = total;
    if (m <= keep) return;                               // the rest of the share are zeros
    uint32_t low, ties, held;                            // `held` keys equal the threshold, `ties` of them stay
    topk_pick(cnt, kTopkLow / 256, keep, &low, &ties, &held);
    const uint32_t thr = (prefix << kDigitBits[2]) | low;
    if (gathered) {
        for (uint32_t j = threadIdx.x; j < m; j += 256) {
            idx_l[j] = it.final_idx[j];
            key_l[j] = it.final_idx[kTopkFinal + j];
        }
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < m; j += 256) {
            const uint32_t key = key_l[j], idx = idx_l[j];
            if (key > thr || (key == thr && ties == held)) continue;
            uint32_t rank = 0;
            if (key == thr)
                for (uint32_t t = 0; t < m; ++t) rank += key_l[t] == key && idx_l[t] < idx;
            if (key < thr || rank >= ties) it.x[idx] = 0.f;
        }
        return;
    }
    const bool surplus = ties != held, listed = held <= (uint32_t)kTieMax;
    topk_for_notes(it, prefix >> kDigitBits[1], bx, gx, [&](uint32_t i, uint32_t key) {
        if ((key >> kDigitBits[2]) != prefix || key > thr) return;
        if (key < thr) {
            it.x[i] = 0.f;
        } else if (surplus && listed) {
            const uint32_t slot = atomicAdd(&st->tie_count, 1u);      // below `held`
            __hip_atomic_store(&st->tie_idx[slot], i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    });
    if (!surplus) return;
    // The noted indices went out past the caches (agent-scope stores): once they have arrived a plain count
    // tells the last workgroup that it can see them all.  A walk of its own reads only keys equal to the
    // threshold, which nobody else writes.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    topk_settle_ties(it.x, it.numel, st, thr, ties, held, gx);
}

// The first digit where the lists follow.  A histogram's workgroups end with an atomic addition for every bin they
// have counted in, all on the same few dozen counters, and those queue: 8.4 M elements take 26 us with 1024 workgroups of
// 256 threads, 19 with 512, 7.8 without the additions, and 11 with 256 workgroups of four times the threads (8 if they
// take turns on eight copies of the counters, which the next pass then has to add up: not worth a larger state).
// A bucket of BERT's errors, several tensors with counters of their own: 15.0 to 10.9 us.
constexpr int kTopkFirst = 1024;

template <int CAP>
__global__ void __launch_bounds__(kTopkFirst)
topk_first_batch_kernel(TopkBatch<CAP> b)
{
    int local, width;
    const TopkItem& it = b.item[topk_locate(b.first, b.count, &local, &width)];
    topk_hist_body<4, kTopkFirst>(it.x, it.numel, it.st, 0, local, width, true, it.k);
}

template <int CAP>
__global__ void __launch_bounds__(256)
topk_note_batch_kernel(TopkBatch<CAP> b)
{
    int local, width;
    const TopkItem& it = b.item[topk_locate(b.first, b.count, &local, &width)];
    topk_note_body(it, local, width);
}

template <int CAP>
__global__ void __launch_bounds__(256)
topk_gather_batch_kernel(TopkBatch<CAP> b)
{
    int local, width;
    const TopkItem& it = b.item[topk_locate(b.first, b.count, &local, &width)];
    topk_gather_body(it, local, width);
}

template <int CAP>
__global__ void __launch_bounds__(256)
topk_settle_batch_kernel(TopkBatch<CAP> b)
{
    int local, width;
    const TopkItem& it = b.item[topk_locate(b.first, b.count, &local, &width)];
    topk_settle_body(it, local, width);
}

// Workgroups of a pass over a tensor.  A histogram workgroup ends with one global atomic per bin
// it touched, all workgroups on the same few dozen counters, and a filter workgroup that has to
// settle ties ends with one on a single counter: fewer workgroups with longer loops (16 quads a
// thread) beat many short ones.  At most 512 where three such passes read the tensor (31 M elements 141 us,
// 164 with 1024), 1024 for the note pass, which ends with no shared counter but the second digit's, and the passes
// over its notes.  From eight on a multiple of eight, the XCDs (topk_hist_body).  (The note pass with workgroups of 1024 threads was slower, 18.0 against 16.5 us a BERT bucket.)
inline int64_t topk_groups(int64_t numel, int64_t most)
{
    const int64_t g = (numel + 255) / 256 / 64;
    return g < 1 ? 1 : g > most ? most : g < 8 ? g : g & ~(int64_t)7;
}
inline int64_t topk_hist_groups(int64_t numel) { return topk_groups(numel, 512); }
inline int64_t topk_listed_groups(int64_t numel) { return topk_groups(numel, 1024); }

// of the first pass where the lists follow: four quads a thread or more
inline int64_t topk_first_groups(int64_t numel)
{
    const int64_t g = topk_listed_groups(numel);
    return g > 256 ? 256 : g;
}


// ---- selection state of the entry point that allocates nothing ------------------------------
// One TopkState per GPU, inside the code object: every GPU the library runs on holds its own
// copy at its own address until the process ends.  `scratch` is only a host-side handle of the
// symbol; kernels (topk_init_kernel clears the state at the start of every call) need the address
// hipGetSymbolAddress returns for the device that is current, looked up once per device and kept.
constexpr size_t kScratchBytes = (sizeof(TopkState) + 255) / 256 * 256;      // 29 184 bytes
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kScratchMaxDevices = 64;
std::mutex g_scratch_lock;
void* g_scratch_ptr[kScratchMaxDevices] = {};

// Address of the current device's copy of `scratch`, or null with *err set.
inline void* topk_scratch_of_current_device(int* err)
{
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        *err = (int)e;
        return nullptr;
    }
    if (dev < 0 || dev >= kScratchMaxDevices) {
        *err = CONEF_ERR_INVALID;
        return nullptr;
    }
    std::lock_guard<std::mutex> hold(g_scratch_lock);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            *err = e != hipSuccess ? (int)e : (int)hipErrorInvalidSymbol;
            return nullptr;
        }
        g_scratch_ptr[dev] = ptr;
    }
    *err = CONEF_OK;
    return g_scratch_ptr[dev];
}

}  // namespace

extern "C" {

int64_t conef_topk_workspace_bytes(int64_t numel)
{
    if (numel < 0) return -1;
    return ((int64_t)sizeof(TopkState) + 255) / 256 * 256;      // the selection state; nothing grows with numel
}

int conef_topk_sparsify_f32(float* x, int64_t numel, int64_t k, void* workspace, int64_t workspace_bytes,
                            void* stream)
{
    if (numel < 1 || k < 1 || !x || numel > 0xffffffffLL) return CONEF_ERR_INVALID;
    if (k >= numel) return CONEF_OK;
    if (!workspace || workspace_bytes < conef_topk_workspace_bytes(numel)) return CONEF_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    TopkState* st = (TopkState*)workspace;
    const int64_t g = topk_hist_groups(numel);
    conef_launch(topk_init_kernel, dim3(1), dim3(256), 0, s, st, (uint32_t)k);
    for (int pass = 0; pass < kPasses; ++pass)
        conef_launch(topk_hist_kernel, dim3((unsigned)g), dim3(256), 0, s, x, numel, st, pass);
    conef_launch(topk_filter_kernel, dim3((unsigned)g), dim3(256), 0, s, x, numel, st);
    return (int)hipGetLastError();
}

namespace {
// candidates a workgroup of the note pass has room for: a quarter of its elements
inline int64_t topk_segment(int64_t numel)
{
    const int64_t g = topk_listed_groups(numel);
    return ((numel + g - 1) / g / 4 + 63) / 64 * 64;
}

// a tensor's part of the lists: the gathered keys, the workgroups' counts, their segments
inline int64_t topk_list_bytes(int64_t numel)
{
    const int64_t g = topk_listed_groups(numel);
    return 8 * kTopkFinal + (4 * g + 255) / 256 * 256 + g * topk_segment(numel) * 8;
}
}  // namespace

// The same for `count` tensors, every pass one launch over all of them (in runs of 48): tensor i
// is xs[i] with numels[i] elements and keeps ks[i]; tensors with ks[i] >= numels[i] are left as
// they are.  xs / numels / ks are host arrays, read before the call returns.
int64_t conef_topk_batch_workspace_bytes(const int64_t* numels, int32_t count)
{
    if (count < 0 || (count > 0 && !numels)) return -1;
    int64_t total = 0;
    for (int i = 0; i < count; ++i) {
        if (numels[i] < 0) return -1;
        total += (int64_t)kScratchBytes;
    }
    return total > 256 ? total : 256;
}

int64_t conef_topk_batch_list_bytes(const int64_t* numels, int32_t count)
{
    if (count < 0 || (count > 0 && !numels)) return -1;
    int64_t total = 0;
    for (int i = 0; i < count; ++i) {
        if (numels[i] < 0) return -1;
        total += topk_list_bytes(numels[i]);
    }
    return total > 256 ? total : 256;
}

}  // extern "C"

namespace {
enum class TopkRun { kFresh, kKept, kListed };

template <int CAP>
void topk_launch(const TopkItem* items, int nb, TopkRun run, hipStream_t s)
{
    TopkBatch<CAP> b;
    int wgs = 0;
    for (int k = 0; k < nb; ++k) {
        b.item[k] = items[k];
        b.first[k] = wgs;
        wgs += (int)(run == TopkRun::kListed ? topk_listed_groups(items[k].numel) : topk_hist_groups(items[k].numel));
    }
    b.first[nb] = wgs;
    b.count = nb;
    const dim3 grid((unsigned)wgs), threads(256);
    if (run == TopkRun::kListed) {
        TopkBatch<CAP> fb = b;
        int fw = 0;
        for (int k = 0; k < nb; ++k) {
            fb.first[k] = fw;
            fw += (int)topk_first_groups(items[k].numel);
        }
        fb.first[nb] = fw;
        conef_launch(topk_first_batch_kernel<CAP>, dim3((unsigned)fw), dim3(kTopkFirst), 0, s, fb);
        conef_launch(topk_note_batch_kernel<CAP>, grid, threads, 0, s, b);
        conef_launch(topk_gather_batch_kernel<CAP>, grid, threads, 0, s, b);
        conef_launch(topk_settle_batch_kernel<CAP>, grid, threads, 0, s, b);
        return;
    }
    const bool kept = run == TopkRun::kKept;
    if (!kept) conef_launch(topk_init_batch_kernel<CAP>, dim3((unsigned)nb), threads, 0, s, b);
    for (int pass = 0; pass < kPasses; ++pass)
        conef_launch(topk_hist_batch_kernel<CAP>, grid, threads, 0, s, b, pass, kept);
    conef_launch(topk_filter_batch_kernel<CAP>, grid, threads, 0, s, b, kept);
}

int topk_sparsify_batch(float* const* xs, const int64_t* numels, const int64_t* ks, int32_t count, void* workspace,
                        int64_t workspace_bytes, void* lists, void* stream, TopkRun run)
{
    if (count < 0 || (count > 0 && (!xs || !numels || !ks))) return CONEF_ERR_INVALID;
    for (int i = 0; i < count; ++i)
        if (numels[i] < 1 || ks[i] < 1 || !xs[i] || numels[i] > 0xffffffffLL) return CONEF_ERR_INVALID;
    if (count > 0 && (!workspace || workspace_bytes < conef_topk_batch_workspace_bytes(numels, count) ||
                      (reinterpret_cast<uintptr_t>(workspace) & 15u) != 0))
        return CONEF_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    char* room = (char*)lists;
    TopkItem table[kTopkBatchMax];
    int nb = 0;
    for (int i = 0; i < count; ++i) {
        if (ks[i] < numels[i]) {
            TopkItem& it = table[nb++];
            it = {};
            it.x = xs[i];
            it.numel = numels[i];
            it.st = (TopkState*)((char*)workspace + i * (int64_t)kScratchBytes);
            it.k = (uint32_t)ks[i];
            if (run == TopkRun::kListed) {
                it.cap = (uint32_t)topk_segment(numels[i]);
                it.final_idx = (uint32_t*)room;
                it.counts = it.final_idx + 2 * kTopkFinal;
                it.list = (uint2*)(room + 8 * kTopkFinal + (4 * topk_listed_groups(numels[i]) + 255) / 256 * 256);
                room += topk_list_bytes(numels[i]);
            }
        }
        if (nb == kTopkBatchMax || (i + 1 == count && nb > 0)) {
            if (nb <= kTopkBatchFew) topk_launch<kTopkBatchFew>(table, nb, run, s);
            else topk_launch<kTopkBatchMax>(table, nb, run, s);
            nb = 0;
        }
    }
    return (int)hipGetLastError();
}
}  // namespace

extern "C" {

int conef_topk_sparsify_batch_f32(float* const* xs, const int64_t* numels, const int64_t* ks, int32_t count,
                                  void* workspace, int64_t workspace_bytes, void* stream)
{
    return topk_sparsify_batch(xs, numels, ks, count, workspace, workspace_bytes, nullptr, stream, TopkRun::kFresh);
}

// The same for a workspace that stays with its tensors: zero-filled by the caller before its first
// use and passed to nothing but this entry point and the next, with the same xs / numels / count, afterwards.
// No launch clears the selection state then (the passes clear behind themselves): four launches a
// call instead of five.
int conef_topk_sparsify_batch_kept_f32(float* const* xs, const int64_t* numels, const int64_t* ks, int32_t count,
                                       void* workspace, int64_t workspace_bytes, void* stream)
{
    return topk_sparsify_batch(xs, numels, ks, count, workspace, workspace_bytes, nullptr, stream, TopkRun::kKept);
}

// The same again with room for candidate lists, which live inside the call only: two reads of a tensor
// instead of four.
int conef_topk_sparsify_batch_listed_f32(float* const* xs, const int64_t* numels, const int64_t* ks, int32_t count,
                                         void* workspace, int64_t workspace_bytes, void* lists, int64_t list_bytes, void* stream)
{
    if (count > 0 && numels && (!lists || list_bytes < conef_topk_batch_list_bytes(numels, count) ||
                                (reinterpret_cast<uintptr_t>(lists) & 15u) != 0))
        return CONEF_ERR_INVALID;
    return topk_sparsify_batch(xs, numels, ks, count, workspace, workspace_bytes, lists, stream, TopkRun::kListed);
}


// conef_topk_sparsify_f32 for callers that may not allocate (HIP graph capture, serving loops):
// the selection state lives in the library's own per-GPU scratch (29 184 bytes), so no workspace
// is passed.  The device the stream belongs to must be current.  Calls on one GPU share that
// scratch: calls that may overlap there (different streams, different threads) race; calls on
// one stream are safe back to back because the first kernel of a call resets the state.
int conef_topk_sparsify_noalloc_f32(float* x, int64_t numel, int64_t k, void* stream)
{
    if (numel < 1 || k < 1 || !x) return CONEF_ERR_INVALID;
    if (numel > CONEF_TOPK_NOALLOC_MAX_NUMEL) return CONEF_ERR_TOO_LARGE;
    if (k >= numel) return CONEF_OK;
    int err = CONEF_OK;
    void* ptr = topk_scratch_of_current_device(&err);
    if (!ptr) return err;
    hipStream_t s = (hipStream_t)stream;
    TopkState* st = (TopkState*)ptr;
    const int64_t g = topk_hist_groups(numel);
    conef_launch(topk_init_kernel, dim3(1), dim3(256), 0, s, st, (uint32_t)k);      // clears what the last call left
    for (int pass = 0; pass < kPasses; ++pass)
        conef_launch(topk_hist_kernel, dim3((unsigned)g), dim3(256), 0, s, x, numel, st, pass);
    conef_launch(topk_filter_kernel, dim3((unsigned)g), dim3(256), 0, s, x, numel, st);
    return (int)hipGetLastError();
}

}  // extern "C"
