// pp_topn.hip -- TopN kernels: a radix select on the IEEE bits of |c|^2 (non-negative doubles order as their bits;
// three 11-bit passes, six for a crowded boundary bin), the gather of the boundary bin's terms, and the in-place
// retain.
//
// Reference semantics (truncation/builtin.rs:73-129, :152-239): with t the n-th largest |c|^2, keep every term above
// t and the first n - above of the terms at t in canonical order (the reference's bucket ascending, then the
// lexicographic key); a NaN is never kept, and with at most n other terms every non-NaN term is kept.
#include "pp_topn.h"

namespace pp {

template <typename T>
__device__ __forceinline__ uint64_t rank_bits(const T* c, const float* score, uint64_t i) {
    return score ? score_bits(score[i]) : magnitude_bits<T>(c[i]);
}

// The state of a new selection, and (one workgroup) its histogram cleared: ApproxTopN's octave pass, which shares
// it, leaves its counts behind.
__global__ void __launch_bounds__(kBlock) k_topn_init(TopnState* s, uint64_t n, uint64_t seed, uint32_t seeded,
                                                      unsigned long long* hist, uint32_t hist_words) {
    for (uint32_t i = threadIdx.x; i < hist_words; i += kBlock) hist[i] = 0ull;
    if (threadIdx.x != 0) return;
    s->prefix = 0;
    s->mask = 0;
    s->k = n;
    s->above = 0;
    s->finite = 0;
    s->ties = 0;
    s->keep_all_finite = 0;
    s->gathered = 0;
    s->done = 0;
    s->seed = seed;
    s->seeded = seeded;
}

// The digit holding the k-th largest after pass `pass`, from the complete histogram, run by one workgroup; then the
// histogram is cleared for the next pass.  The digit is the largest d whose suffix count sum_{e >= d} hist[e]
// reaches k: each thread owns kPerThread consecutive bins, a suffix scan of the per-thread sums (in LDS) finds the
// one thread whose bins hold d, and that thread walks them.
__device__ __forceinline__ void select_digit(TopnState* s, unsigned long long* hist, int pass, uint64_t n) {
    constexpr int kPerThread = kTopnBins / kBlock;
    static_assert(kPerThread * kBlock == kTopnBins, "bins split evenly over the workgroup");
    __shared__ unsigned long long suffix[kBlock];
    __shared__ int keep_all;
    __shared__ unsigned long long k_sh;  // k as every thread must see it, read before the holder updates it
    const int t = threadIdx.x;
    const int bins = 1 << topn_bits(pass);
    unsigned long long mine[kPerThread];
    unsigned long long sum = 0;
#pragma unroll
    for (int j = 0; j < kPerThread; ++j) {
        const int d = t * kPerThread + j;
        mine[j] = 0ull;
        if (d < bins) {
#pragma unroll
            for (uint32_t c = 0; c < kHistCopies; ++c) mine[j] += hist[c * kTopnBins + d];
        }
        sum += mine[j];
    }
    suffix[t] = sum;
    __syncthreads();
    // inclusive suffix scan: suffix[t] = sum over threads u >= t
    for (int off = 1; off < kBlock; off <<= 1) {
        const unsigned long long v = t + off < kBlock ? suffix[t + off] : 0ull;
        __syncthreads();
        suffix[t] += v;
        __syncthreads();
    }
    if (t == 0) {
        int ka = s->keep_all_finite;
        if (!ka && pass == 0) {
            s->finite = suffix[0];
            if (suffix[0] <= n) {
                s->keep_all_finite = 1;
                ka = 1;
            }
        }
        keep_all = ka;
        k_sh = s->k;
    }
    __syncthreads();
    if (!keep_all) {
        const unsigned long long k = k_sh;
        const unsigned long long above_mine = t + 1 < kBlock ? suffix[t + 1] : 0ull;  // bins of higher threads
        // the thread holding the digit; with no digit reaching k (not reached in a selection) thread 0 takes bin 0
        const bool holder = (above_mine < k && above_mine + sum >= k) || (t == 0 && suffix[0] < k);
        if (holder) {
            unsigned long long acc = above_mine, at = mine[0];
            int chosen = t * kPerThread;
            bool found = false;
#pragma unroll
            for (int j = kPerThread - 1; j >= 0; --j) {
                if (!found && acc + mine[j] >= k) {
                    chosen = t * kPerThread + j;
                    at = mine[j];
                    found = true;
                }
                if (!found) acc += mine[j];
            }
            const int shift = topn_shift(pass);
            s->above += acc;
            s->k -= acc;
            s->prefix |= (unsigned long long)chosen << shift;
            s->mask |= ((1ull << topn_bits(pass)) - 1ull) << shift;
            s->ties = at;
        }
    }
    __syncthreads();
    for (uint32_t i = t; i < kHistWords; i += kBlock) hist[i] = 0;
}

// One radix pass: each workgroup histograms the digit of its buckets' terms that match the prefix found so far and
// adds its counts to the global histogram; k_topn_select picks the digit.  The workgroup walks its buckets' rows
// as one list, so that its threads' loads do not wait bucket by bucket.
// The rows of buckets [b_lo, b_lo + nb) (nb <= kHistBucketsMax) as one list: first[j] rows precede bucket j, whose
// segment starts at seg[j]; returns the rows in all.  Every thread of the workgroup calls it (two barriers).
struct RowList {
    uint32_t first[kHistBucketsMax + 1];
    uint64_t seg[kHistBucketsMax];
    uint32_t wave_rows[kWaves];
};

__device__ __forceinline__ uint32_t list_rows(const uint64_t* start, const uint32_t* len, uint32_t b_lo, uint32_t nb,
                                              RowList& l) {
    const uint32_t t = threadIdx.x;
    uint32_t v = t < nb ? len[b_lo + t] : 0u;
    if (t < nb) l.seg[t] = start[b_lo + t];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(v, d, 64);
        if (lane_id() >= (uint32_t)d) v += o;
    }
    if (lane_id() == 63) l.wave_rows[wave_id()] = v;
    __syncthreads();
    uint32_t before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        before += (uint32_t)w < wave_id() ? l.wave_rows[w] : 0u;
        total += l.wave_rows[w];
    }
    if (t < nb) l.first[t + 1] = before + v;
    if (t == 0) l.first[0] = 0;
    __syncthreads();
    return total;
}

// Column positions of list rows g0 + q * kBlock (q < N) that exist; j is the caller's bucket cursor (rows only move
// forward, so it does too).
template <int N>
__device__ __forceinline__ void list_positions(const RowList& l, uint32_t total, uint32_t g0, uint32_t& j,
                                               uint64_t (&pos)[N], bool (&in)[N]) {
#pragma unroll
    for (int q = 0; q < N; ++q) {
        const uint32_t g = g0 + (uint32_t)q * kBlock;
        in[q] = g < total;
        if (in[q]) {
            while (l.first[j + 1] <= g) ++j;
            pos[q] = l.seg[j] + (g - l.first[j]);
        }
    }
}

// One histogram workgroup's share (workgroup `block` of the selection's grid).
template <typename T>
__device__ __forceinline__ void topn_hist_body(const TopnHistArgs<T>& a, uint32_t block) {
    __shared__ uint32_t h[kTopnBins];
    __shared__ RowList list;
    const TopnState st = *a.state;
    if (st.done > (unsigned long long)a.pass) return;  // decided by a seeded first pass: the whole workgroup
    for (int i = threadIdx.x; i < kTopnBins; i += kBlock) h[i] = 0;
    const uint32_t b_lo = block * a.buckets_per_block;
    const uint32_t nb = min(a.num_buckets, b_lo + a.buckets_per_block) - b_lo;  // <= kHistBucketsMax
    const uint32_t t = threadIdx.x;
    const uint32_t total = list_rows(a.start, a.len, b_lo, nb, list);
    if (!st.keep_all_finite) {
        const int shift = topn_shift(a.pass);
        const uint64_t dmask = (1ull << topn_bits(a.pass)) - 1ull;
        // Row g of the list is row g - first[j] of bucket j; a thread's rows only move forward, so j does too.
        // Four rows per thread per step, their loads issued together.
        uint32_t j = 0;
        for (uint32_t g0 = t; g0 < total; g0 += 4 * kBlock) {
            uint64_t pos[4];
            bool in[4];
            list_positions(list, total, g0, j, pos, in);
            uint64_t u[4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (in[q]) u[q] = rank_bits<T>(a.c, a.score, pos[q]);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (!in[q]) continue;
                const bool match = (a.score || !is_nan_bits(u[q])) && (u[q] & st.mask) == st.prefix;
                if (match) atomicAdd(&h[(uint32_t)((u[q] >> shift) & dmask)], 1u);
            }
        }
    }
    __syncthreads();
    unsigned long long* const copy = a.hist + (block % kHistCopies) * kTopnBins;
    for (int i = threadIdx.x; i < kTopnBins; i += kBlock)
        if (h[i]) atomicAdd(&copy[i], (unsigned long long)h[i]);
}

template <typename T>
__global__ void __launch_bounds__(kBlock) k_topn_hist(const TopnHistArgs<T> a) {
    topn_hist_body<T>(a, blockIdx.x);
}

// The item of a batched launch whose range [block_start[i], block_start[i + 1]) of workgroups holds blockIdx.x.
__device__ __forceinline__ uint32_t batch_item(const uint32_t* block_start, uint32_t num_items) {
    uint32_t lo = 0, hi = num_items;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (block_start[mid] <= blockIdx.x) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Pass `pass` of many selections in one launch (items: each sum's histogram arguments).
template <typename T>
__global__ void __launch_bounds__(kBlock) k_topn_hist_batch(const TopnHistArgs<T>* __restrict__ items,
                                                             const uint32_t* __restrict__ block_start,
                                                             uint32_t num_items, int32_t pass) {
    const uint32_t i = batch_item(block_start, num_items);
    TopnHistArgs<T> a = items[i];
    a.pass = pass;
    topn_hist_body<T>(a, blockIdx.x - block_start[i]);
}

// One workgroup after each histogram pass (a kernel boundary, not a device-scope fence per histogram workgroup: on
// a multi-XCD device such a fence writes back the XCD's L2).
__global__ void __launch_bounds__(kBlock) k_topn_select(TopnState* s, unsigned long long* hist, int pass, uint64_t n) {
    if (s->done > (unsigned long long)pass) return;  // uniform: one load, the same for every thread
    select_digit(s, hist, pass, n);
    if (threadIdx.x == 0) s->done = (unsigned long long)pass + 1ull;
}

// Many selections' states: one workgroup each clears its histogram's first region and starts the state (unseeded).
__global__ void __launch_bounds__(kBlock) k_topn_init_batch(const TopnSelectItem* __restrict__ items) {
    const TopnSelectItem it = items[blockIdx.x];
    for (uint32_t i = threadIdx.x; i < kHistWords; i += kBlock) it.hist[i] = 0ull;
    if (threadIdx.x == 0) {
        TopnState* s = it.state;
        s->prefix = 0;
        s->mask = 0;
        s->k = it.n;
        s->above = 0;
        s->finite = 0;
        s->ties = 0;
        s->keep_all_finite = 0;
        s->gathered = 0;
        s->done = 0;
        s->seed = 0;
        s->seeded = 0;
    }
}

// The digit select of pass `pass` for many selections, one workgroup each; with `last`, each state is also copied
// to its item's slot of the batch's contiguous state array (one read-back for all of them).
__global__ void __launch_bounds__(kBlock) k_topn_select_batch(const TopnSelectItem* __restrict__ items, int pass,
                                                              int last) {
    const TopnSelectItem it = items[blockIdx.x];
    TopnState* s = it.state;
    if (s->done <= (unsigned long long)pass) {  // uniform: one load, the same for every thread
        select_digit(s, it.hist, pass, it.n);
        if (threadIdx.x == 0) s->done = (unsigned long long)pass + 1ull;
    }
    if (last) {
        __syncthreads();  // the holder's updates of the state
        if (threadIdx.x == 0) *it.out = *s;
    }
}

// The seeded first pass's histograms: region 0 of hist counts the first digit of every term, region 1 the second
// digit of the terms whose first digit is the seed's.  (A third level, over the terms whose first two digits are the
// seed's, measured slower: at a TopN cap the second digit of the boundary moves from layer to layer, and the third
// histogram's LDS cost the pass more than it saved.)  Walks its buckets as k_topn_hist does.
template <typename T>
__global__ void __launch_bounds__(kBlock) k_topn_hist_seeded(const TopnHistArgs<T> a) {
    __shared__ uint32_t h[2][kTopnBins];
    __shared__ RowList list;
    for (int i = threadIdx.x; i < 2 * kTopnBins; i += kBlock) (&h[0][0])[i] = 0;
    const TopnState st = *a.state;
    const uint32_t spec0 = (uint32_t)(st.seed >> topn_shift(0)) & (kTopnBins - 1);
    const uint32_t b_lo = blockIdx.x * a.buckets_per_block;
    const uint32_t nb = min(a.num_buckets, b_lo + a.buckets_per_block) - b_lo;  // <= kHistBucketsMax
    const uint32_t total = list_rows(a.start, a.len, b_lo, nb, list);
    uint32_t j = 0;
    for (uint32_t g0 = threadIdx.x; g0 < total; g0 += 4 * kBlock) {
        uint64_t pos[4];
        bool in[4];
        list_positions(list, total, g0, j, pos, in);
        uint64_t u[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (in[q]) u[q] = rank_bits<T>(a.c, a.score, pos[q]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (!in[q] || (!a.score && is_nan_bits(u[q]))) continue;
            const uint32_t d0 = (uint32_t)(u[q] >> topn_shift(0)) & (kTopnBins - 1);
            atomicAdd(&h[0][d0], 1u);
            if (d0 != spec0) continue;
            atomicAdd(&h[1][(uint32_t)(u[q] >> topn_shift(1)) & (kTopnBins - 1)], 1u);
        }
    }
    __syncthreads();
    const uint32_t copy = (blockIdx.x % kHistCopies) * kTopnBins;
    for (int i = threadIdx.x; i < 2 * kTopnBins; i += kBlock) {
        const uint32_t v = (&h[0][0])[i];
        if (v) atomicAdd(&a.hist[(i / kTopnBins) * kHistWords + copy + (i % kTopnBins)], (unsigned long long)v);
    }
}

// The first digit from region 0, the second from region 1 when the first is the seed's; region 1 is cleared for the
// next selection when unused.
__global__ void __launch_bounds__(kBlock) k_topn_select_seeded(TopnState* s, unsigned long long* hist, uint64_t n) {
    __shared__ int go;
    select_digit(s, hist, 0, n);
    int done = 1;
    for (int r = 1; r < 2; ++r) {
        __syncthreads();  // the holder's update of the state is visible
        if (threadIdx.x == 0) {
            const uint64_t d = (s->prefix >> topn_shift(r - 1)) & (kTopnBins - 1);
            go = done == r && !s->keep_all_finite && d == ((s->seed >> topn_shift(r - 1)) & (kTopnBins - 1));
        }
        __syncthreads();
        if (go) {
            select_digit(s, hist + (size_t)r * kHistWords, r, n);
            done = r + 1;
        } else {
            for (uint32_t i = threadIdx.x; i < kHistWords; i += kBlock) hist[(size_t)r * kHistWords + i] = 0;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) s->done = s->keep_all_finite ? 3ull : (unsigned long long)done;
}

// The terms of the boundary bin: rank key equal to the prefix on the decided bits (a NaN never matches a finite
// prefix: its exponent bits are all ones).  Buckets are walked as in k_topn_hist.
template <int W, typename T>
__device__ __forceinline__ void topn_gather_body(const TopnTieArgs<W, T>& a, uint32_t block) {
    __shared__ RowList list;
    const uint64_t t = a.state->prefix, mask = a.state->mask;
    const uint32_t b_lo = block * a.buckets_per_block;
    const uint32_t nb = min(a.num_buckets, b_lo + a.buckets_per_block) - b_lo;  // <= kHistBucketsMax
    const uint32_t total = list_rows(a.start, a.len, b_lo, nb, list);
    uint32_t j = 0;
    for (uint32_t g0 = threadIdx.x; g0 < total; g0 += 4 * kBlock) {
        uint64_t pos[4];
        bool in[4];
        list_positions(list, total, g0, j, pos, in);
        uint64_t u[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (in[q]) u[q] = rank_bits<T>(a.c, a.score, pos[q]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (!in[q] || (u[q] & mask) != t || (!a.score && is_nan_bits(u[q]))) continue;
            const uint64_t slot = atomicAdd(&a.state->gathered, 1ull);
            if (slot >= a.tie_cap) continue;
            const Key<W> k = load_key<W>(a.x, a.z, a.cap, pos[q]);
#pragma unroll
            for (int w = 0; w < W; ++w) {
                a.tie_x[slot * W + w] = k.x[w];
                a.tie_z[slot * W + w] = k.z[w];
            }
            a.tie_bucket[slot] = bucket_of<W>(k, a.rows, a.ref_bits);
            a.tie_pos[slot] = pos[q];
            a.tie_rank[slot] = u[q];
        }
    }
}

template <int W, typename T>
__global__ void __launch_bounds__(kBlock) k_topn_gather_ties(const TopnTieArgs<W, T> a) {
    topn_gather_body<W, T>(a, blockIdx.x);
}

// The boundary bins of many selections in one launch (each item's ties into its own range of the batch's arrays).
template <int W, typename T>
__global__ void __launch_bounds__(kBlock) k_topn_gather_batch(const TopnTieArgs<W, T>* __restrict__ items,
                                                              const uint32_t* __restrict__ block_start,
                                                              uint32_t num_items) {
    const uint32_t i = batch_item(block_start, num_items);
    const TopnTieArgs<W, T> a = items[i];
    topn_gather_body<W, T>(a, blockIdx.x - block_start[i]);
}

// Whether the term at column position i (coefficient c) survives the selection: above the boundary bin on the
// decided bits, or in it and flagged (without flags, every term in it).
template <int W, typename T>
__device__ __forceinline__ bool retain_keeps(const TopnRetainArgs<W, T>& a, const TopnState& st, T c, uint64_t i) {
    const uint64_t u = a.score ? score_bits(a.score[i]) : magnitude_bits<T>(c);
    return topn_keeps(st, u, !a.score && is_nan_bits(u), a.tie_keep, i);
}

// In-place retain, 2 kBlock rows per step: both rows' loads are issued before the step's one scan, and a dropped
// row's key is never read.  Every write lands at or before its row's own position, and every row of the step was
// read before the scan's barrier.
template <int W, typename T>
__global__ void __launch_bounds__(kBlock) k_topn_retain(const TopnRetainArgs<W, T> a) {
    __shared__ uint32_t scan_scratch[2 * kWaves];
    const uint32_t b = blockIdx.x;
    const uint32_t n = a.len[b];
    const uint64_t s = a.start[b];
    const TopnState st = *a.state;
    uint32_t cur = 0;
    for (uint32_t base = 0; base < n; base += 2 * kBlock) {
        const uint32_t r0 = base + threadIdx.x, r1 = r0 + kBlock;
        T c0 = T(0), c1 = T(0);
        if (r0 < n) c0 = a.c[s + r0];
        if (r1 < n) c1 = a.c[s + r1];
        const bool keep0 = r0 < n && retain_keeps<W, T>(a, st, c0, s + r0);
        const bool keep1 = r1 < n && retain_keeps<W, T>(a, st, c1, s + r1);
        Key<W> k0, k1;
        if (keep0) k0 = load_key<W>(a.x, a.z, a.cap, s + r0);
        if (keep1) k1 = load_key<W>(a.x, a.z, a.cap, s + r1);
        bool f[2] = {keep0, keep1};
        uint32_t off[2], tot[2];
        block_flag_scan<2>(f, off, tot, scan_scratch);
        if (keep0 && cur + off[0] != r0) {
            const uint64_t pos = s + cur + off[0];
            store_key<W>(a.x, a.z, a.cap, pos, k0);
            store_coeff<T>(a.c, pos, c0);
        }
        if (keep1 && cur + tot[0] + off[1] != r1) {
            const uint64_t pos = s + cur + tot[0] + off[1];
            store_key<W>(a.x, a.z, a.cap, pos, k1);
            store_coeff<T>(a.c, pos, c1);
        }
        cur += tot[0] + tot[1];
    }
    if (threadIdx.x == 0) a.len[b] = cur;
}

__global__ void k_mark_positions(const uint64_t* pos, uint64_t n, uint8_t* flags) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) flags[pos[i]] = 1;
}

// The boundary flags of one selection: pos holds its boundary bin's positions in rank order, the first `kept` kept.
__global__ void k_topn_flag_ties(const uint64_t* pos, uint64_t ties, uint64_t kept, uint8_t* flags) {
    const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < ties) flags[pos[j]] = j < kept ? 1 : 0;
}

// The boundary flags of many selections, one workgroup each: every position of the item's boundary bin, in rank
// order, is flagged kept (its first `kept`) or dropped.  Only positions in the boundary bin are ever read, so no
// other flag needs a value.
__global__ void __launch_bounds__(kBlock) k_topn_flags_batch(const TopnFlagItem* __restrict__ items) {
    const TopnFlagItem it = items[blockIdx.x];
    for (uint64_t j = threadIdx.x; j < it.ties; j += kBlock) it.flags[it.pos[j]] = j < it.kept ? 1 : 0;
}

// ---- the windowed selection ---------------------------------------------------------------------------------

// The keys of a workgroup's buckets against the window: those at or above it and those that are numbers are counted,
// those inside collected.  The coefficients' (or scores') bytes, and above 10^7 keys the merging of the bins' counts,
// bound it: 8 us at 2^20 f64 terms and 48 at 2^24 (72 with twice the bins, 164 with one line of counters).  With the
// narrowing and the finish a selection is 26 and 84 us of kernels and one wait of the host, where the radix passes, the
// gather of the boundary bin and their selects were 50-60 and 170 with two or three synchronizations.
template <int W, typename T>
__global__ void __launch_bounds__(kBlock) k_window_scan(const WindowArgs<W, T> a) {
    __shared__ RowList list;
    __shared__ uint64_t su[kWindowStage], sp[kWindowStage];
    __shared__ uint32_t bins[kWindowBins];
    __shared__ uint32_t collected, totals[2];
    __shared__ unsigned long long base;
    if (threadIdx.x < 2) totals[threadIdx.x] = 0u;
    if (threadIdx.x == 2) collected = 0u;
    if (threadIdx.x < kWindowBins) bins[threadIdx.x] = 0u;
    const uint32_t b_lo = blockIdx.x * a.buckets_per_block;
    const uint32_t nb = min(a.num_buckets, b_lo + a.buckets_per_block) - b_lo;  // <= kHistBucketsMax
    const uint32_t total = list_rows(a.start, a.len, b_lo, nb, list);
    uint32_t above = 0, finite = 0, j = 0;
    for (uint32_t g0 = threadIdx.x; g0 < total; g0 += 8 * kBlock) {
        uint64_t pos[8];
        bool in[8];
        list_positions(list, total, g0, j, pos, in);
        uint64_t u[8];
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (in[q]) u[q] = rank_bits<T>(a.c, a.score, pos[q]);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if (!in[q] || (!a.score && is_nan_bits(u[q]))) continue;
            ++finite;
            if (u[q] >= a.hi) {
                ++above;
            } else if (u[q] >= a.lo) {
                const uint32_t slot = atomicAdd(&collected, 1u);
                if (slot < kWindowStage) {
                    su[slot] = u[q];
                    sp[slot] = pos[q];
                }
                if (a.narrow) atomicAdd(&bins[(uint32_t)((u[q] - a.lo) >> a.bin_shift)], 1u);
            }
        }
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        above += (uint32_t)__shfl_xor((int)above, d, 64);
        finite += (uint32_t)__shfl_xor((int)finite, d, 64);
    }
    if (lane_id() == 0) {
        atomicAdd(&totals[0], above);
        atomicAdd(&totals[1], finite);
    }
    __syncthreads();
    const uint32_t part = blockIdx.x % kWindowParts;
    if (threadIdx.x == 0) {
        WindowCounts::Part& p = a.counts->part[part];
        base = collected ? atomicAdd(&p.count, (unsigned long long)collected) : 0ull;
        if (totals[1]) atomicAdd(&p.above_finite, (unsigned long long)totals[0] | ((unsigned long long)totals[1] << 32));
        if (collected > kWindowStage) atomicOr(&p.overflow, 1ull);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < min(collected, kWindowStage); i += kBlock)
        if (base + i < a.room) {
            a.key[part * a.room + base + i] = su[i];
            a.pos[part * a.room + base + i] = sp[i];
        }
    if (a.narrow && threadIdx.x < kWindowBins && bins[threadIdx.x])
        atomicAdd(&a.counts->bins[blockIdx.x % kWindowCopies][threadIdx.x], bins[threadIdx.x]);
}

// The scan's counters of all parts, and the collected keys as one list: entry i of it lies at at(i).  Every thread of
// the workgroup calls read (one barrier); nothing is kept from a part with more keys than room.
struct WindowTotals {
    uint64_t first[kWindowParts + 1];
    uint64_t above, finite, fullest;

    __device__ __forceinline__ void read(const WindowCounts& w) {  // into LDS
        if (threadIdx.x < 64) {
            const uint32_t l = threadIdx.x & (kWindowParts - 1);
            const WindowCounts::Part p = w.part[l];
            uint64_t n = p.count, up = p.above_finite & 0xFFFFFFFFull, f = p.above_finite >> 32;
            uint64_t most = p.overflow ? ~0ull : n;
#pragma unroll
            for (int d = 1; d < (int)kWindowParts; d <<= 1) {
                const uint64_t o = __shfl_up(n, d, kWindowParts);
                if (l >= (uint32_t)d) n += o;
                up += __shfl_xor(up, d, kWindowParts);
                f += __shfl_xor(f, d, kWindowParts);
                const uint64_t m = __shfl_xor(most, d, kWindowParts);
                most = m > most ? m : most;
            }
            if (threadIdx.x < kWindowParts) first[l + 1] = n;
            if (threadIdx.x == 0) {
                first[0] = 0;
                above = up;
                finite = f;
                fullest = most;
            }
        }
        __syncthreads();
    }
    // whether the n-th key is inside the window, and every key inside collected
    __device__ __forceinline__ bool inside(uint64_t n) const { return above < n && above + first[kWindowParts] >= n; }
    __device__ __forceinline__ bool holds(uint64_t n, uint64_t room) const { return fullest <= room && inside(n); }
    __device__ __forceinline__ uint64_t at(uint64_t i, uint64_t room) const {
        uint32_t p = 0;
#pragma unroll
        for (uint32_t half = kWindowParts / 2; half > 0; half >>= 1)
            if (first[p + half] <= i) p += half;
        return p * room + (i - first[p]);
    }
};

// The bin (of BINS in ascending order, hist[bin]) that holds the k-th key from the top, the keys above it and its own,
// by a workgroup of BLOCK threads; k is at least 1 and at most the bins' total.  Every thread gets the answer.
template <uint32_t BINS, uint32_t BLOCK>
__device__ __forceinline__ void window_bin(const uint32_t* hist, uint64_t k, uint64_t* part, uint64_t (&answer)[3]) {
    constexpr uint32_t PER = (BINS + BLOCK - 1) / BLOCK;  // the threads past the last bin hold none
    static_assert(PER * BLOCK == BINS || PER == 1, "bins split evenly over the workgroup");
    uint64_t mine = 0;
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q)
        if (threadIdx.x * PER + q < BINS) mine += hist[threadIdx.x * PER + q];
    uint64_t suffix = mine;  // this lane's bins and the higher lanes' of its wave
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t o = __shfl_down(suffix, d, 64);
        if (lane_id() + (uint32_t)d < 64u) suffix += o;
    }
    if (lane_id() == 0) part[wave_id()] = suffix;
    __syncthreads();
    uint64_t above = suffix - mine;
    for (uint32_t w = wave_id() + 1; w < BLOCK / 64; ++w) above += part[w];
    if (above < k && above + mine >= k) {
        for (uint32_t q = PER; q-- > 0;) {
            const uint64_t h = hist[threadIdx.x * PER + q];
            if (above + h >= k) {
                part[BLOCK / 64] = threadIdx.x * PER + q;
                part[BLOCK / 64 + 1] = above;
                part[BLOCK / 64 + 2] = h;
                break;
            }
            above += h;
        }
    }
    __syncthreads();
    for (int i = 0; i < 3; ++i) answer[i] = part[BLOCK / 64 + i];
    __syncthreads();
}

// The copies of the scan's bins summed into hist (zero before), by a workgroup of BLOCK threads.
template <uint32_t BLOCK>
__device__ __forceinline__ void window_bins_sum(const WindowCounts& w, uint32_t* hist) {
    static_assert(BLOCK % kWindowBins == 0, "a group of threads per bin");
    uint32_t sum = 0;
#pragma unroll 8
    for (uint32_t c = threadIdx.x / kWindowBins; c < kWindowCopies; c += BLOCK / kWindowBins)
        sum += w.bins[c][threadIdx.x % kWindowBins];
    atomicAdd(&hist[threadIdx.x % kWindowBins], sum);
    __syncthreads();
}

// The collected keys of the boundary's bin, for a sum whose window holds too many for one workgroup.
template <int W, typename T>
__global__ void __launch_bounds__(kBlock) k_window_narrow(const WindowArgs<W, T> a) {
    __shared__ uint64_t part[kWaves + 3];
    __shared__ uint32_t hist[kWindowBins];
    __shared__ uint64_t su[kWindowStage], sp[kWindowStage];
    __shared__ uint32_t collected;
    __shared__ unsigned long long base;
    __shared__ WindowTotals t;
    WindowCounts& w = *a.counts;
    if (threadIdx.x < kWindowBins) hist[threadIdx.x] = 0u;
    if (threadIdx.x == 0) collected = 0u;
    t.read(w);  // complete at this launch's start
    if (!t.holds(a.n, a.room)) return;  // uniform
    window_bins_sum<kBlock>(w, hist);
    uint64_t bin[3];
    window_bin<kWindowBins, kBlock>(hist, a.n - t.above, part, bin);
    if (blockIdx.x == 0 && threadIdx.x == 0) w.narrowed_above = t.above + bin[1];
    const uint64_t m = t.first[kWindowParts], stride = (uint64_t)gridDim.x * kBlock;
    for (uint64_t i0 = (uint64_t)blockIdx.x * kBlock; i0 < m; i0 += stride) {  // uniform
        const uint64_t i = i0 + threadIdx.x;
        if (i < m) {
            const uint64_t at = t.at(i, a.room), u = a.key[at];
            if (((u - a.lo) >> a.bin_shift) == bin[0]) {
                const uint32_t slot = atomicAdd(&collected, 1u);
                su[slot] = u;
                sp[slot] = a.pos[at];
            }
        }
        __syncthreads();
        const uint32_t held = collected;
        if (held > kWindowStage - kBlock || i0 + stride >= m) {  // uniform: the next step's keys may not fit, or the end
            if (threadIdx.x == 0) base = held ? atomicAdd(&w.narrowed, (unsigned long long)held) : 0ull;
            __syncthreads();
            for (uint32_t q = threadIdx.x; q < held; q += kBlock) {
                a.key2[base + q] = su[q];
                a.pos2[base + q] = sp[q];
            }
            __syncthreads();
            if (threadIdx.x == 0) collected = 0u;
        }
        __syncthreads();
    }
}

// The k-th largest of the n listed keys (su, with their positions sp), by a workgroup of kFinishBlock threads: the
// boundary, how many of the keys equal to it stay, and how many there are.  Only some staying, they are put into
// canonical order and flagged; false when they are more than the order holds.  Both counts take every thread the list
// leaves: a run of lanes per key, each over a part of the list.
constexpr uint32_t kFinishBlock = 1024;
template <int W>
struct RankScratch {
    uint64_t x[W][kWindowTies], z[W][kWindowTies], pos[kWindowTies];
    uint32_t bucket[kWindowTies];
    uint32_t ties;
    uint64_t found[3];  // the boundary key, the list's keys above it, the keys equal to it
};
__device__ __forceinline__ uint32_t lanes_per_key(uint32_t n) {
    uint32_t g = 1;
    while (2 * g * n <= kFinishBlock && g < 64) g *= 2;
    return g;
}
template <int W, typename Args>
__device__ __forceinline__ bool rank_ties(const Args& a, RankScratch<W>& r, const uint64_t* su, const uint64_t* sp,
                                          uint32_t n, uint64_t boundary, uint32_t equal, uint64_t stay) {
    if (equal > kWindowTies) return false;
    const uint32_t tid = threadIdx.x;
    for (uint32_t i = tid; i < n; i += kFinishBlock) {
        if (su[i] != boundary) continue;
        const uint32_t e = atomicAdd(&r.ties, 1u);
        const Key<W> kk = load_key<W>(a.x, a.z, a.cap, sp[i]);
#pragma unroll
        for (int v = 0; v < W; ++v) {
            r.x[v][e] = kk.x[v];
            r.z[v][e] = kk.z[v];
        }
        r.bucket[e] = bucket_of<W>(kk, a.rows, a.ref_bits);
        r.pos[e] = sp[i];
    }
    __syncthreads();
    const uint32_t g = lanes_per_key(equal), i = tid / g;
    uint32_t before = 0;
    if (i < equal)
        for (uint32_t q = tid % g; q < equal; q += g) {
            int order = r.bucket[q] < r.bucket[i] ? -1 : r.bucket[q] > r.bucket[i] ? 1 : 0;
#pragma unroll
            for (int v = 0; v < W; ++v)
                if (order == 0) order = r.x[v][q] < r.x[v][i] ? -1 : r.x[v][q] > r.x[v][i] ? 1 : 0;
#pragma unroll
            for (int v = 0; v < W; ++v)
                if (order == 0) order = r.z[v][q] < r.z[v][i] ? -1 : r.z[v][q] > r.z[v][i] ? 1 : 0;
            before += order < 0;
        }
    for (uint32_t d = 1; d < g; d *= 2) before += (uint32_t)__shfl_xor((int)before, (int)d, 64);
    if (i < equal && tid % g == 0) a.flags[r.pos[i]] = before < stay ? 1 : 0;
    return true;
}
template <int W, typename T, typename Args>
__device__ __forceinline__ bool rank_boundary(const Args& a, RankScratch<W>& r, const uint64_t* su, const uint64_t* sp,
                                              uint32_t n, uint64_t k, bool one, uint64_t& boundary, uint64_t& stay,
                                              uint32_t& equal) {
    const uint32_t tid = threadIdx.x;
    if (tid == 0) r.ties = 0u;
    if (one && tid == 0) {  // every digit decided: the listed keys are one key
        r.found[0] = su[0];
        r.found[1] = 0;
        r.found[2] = n;
    }
    const uint32_t g = lanes_per_key(n);
    for (uint32_t i0 = 0; !one && i0 < n; i0 += kFinishBlock / g) {  // uniform
        const uint32_t i = i0 + tid / g;
        const uint64_t u = i < n ? su[i] : 0;
        uint32_t greater = 0, same = 0;
        if (i < n)
            for (uint32_t q = tid % g; q < n; q += g) {
                greater += su[q] > u;
                same += su[q] == u;
            }
        for (uint32_t d = 1; d < g; d *= 2) {
            greater += (uint32_t)__shfl_xor((int)greater, (int)d, 64);
            same += (uint32_t)__shfl_xor((int)same, (int)d, 64);
        }
        if (i < n && greater < k && greater + same >= k) {  // every row equal to the boundary writes the same
            r.found[0] = u;
            r.found[1] = greater;
            r.found[2] = same;
        }
    }
    __syncthreads();
    boundary = r.found[0];
    stay = k - r.found[1];
    equal = (uint32_t)r.found[2];
    return stay == equal || rank_ties<W>(a, r, su, sp, n, boundary, equal, stay);
}

// A list of n keys (at most kWindowList, in [base, base + 2^shift)) cut by further digits until at most kWindowRank are left
// or they are equal: every pass in LDS, two keys a thread, where a pass over the collected keys is up to 40 us.  A run of
// more than kWindowRank equal keys takes five or six of them (60 000 f32 terms, 240 selections: 30.0 -> 26.5 us a finish).
__device__ __forceinline__ void narrow_list(uint64_t* su, uint64_t* sp, uint32_t& n, uint32_t* held, uint64_t& base,
                                            int& shift, uint64_t& k, uint32_t* hist, uint64_t* part) {
    constexpr uint32_t kDigits = 2048;
    static_assert(kWindowList == 2 * kFinishBlock, "two keys a thread");
    const uint32_t tid = threadIdx.x;
    while (n > kWindowRank && shift > 0) {  // uniform
        const int sh = max(shift - 11, 0);
        uint64_t u[2] = {0, 0}, p[2] = {0, 0};
#pragma unroll
        for (uint32_t q = 0; q < 2; ++q)
            if (tid + q * kFinishBlock < n) {
                u[q] = su[tid + q * kFinishBlock];
                p[q] = sp[tid + q * kFinishBlock];
            }
        for (uint32_t i = tid; i < kDigits; i += kFinishBlock) hist[i] = 0u;
        __syncthreads();
        if (tid == 0) *held = 0u;
#pragma unroll
        for (uint32_t q = 0; q < 2; ++q)
            if (tid + q * kFinishBlock < n) atomicAdd(&hist[(u[q] - base) >> sh], 1u);
        __syncthreads();
        uint64_t bin[3];
        window_bin<kDigits, kFinishBlock>(hist, k, part, bin);
        base += bin[0] << sh;
        k -= bin[1];
        shift = sh;
#pragma unroll
        for (uint32_t q = 0; q < 2; ++q)
            if (tid + q * kFinishBlock < n && ((u[q] - base) >> sh) == 0) {
                const uint32_t slot = atomicAdd(held, 1u);
                su[slot] = u[q];
                sp[slot] = p[q];
            }
        __syncthreads();
        n = (uint32_t)bin[2];  // = *held
    }
}

// The n-th key among the collected (or narrowed) ones, by one workgroup: 11-bit digits of the window until at most
// kWindowList keys are left, more of them on that list until at most kWindowRank are left or they are equal, those ranked
// by counting, and the keys equal to the boundary put into canonical order when
// only some of them stay.  Then the state the next layer reads, the answer to the host, and the counts cleared.
template <int W, typename T>
__global__ void __launch_bounds__(kFinishBlock) k_window_finish(const WindowArgs<W, T> a) {
    constexpr uint32_t kDigits = 2048;
    __shared__ uint32_t hist[kDigits];
    __shared__ uint64_t part[kFinishBlock / 64 + 3];
    __shared__ uint64_t su[kWindowList], sp[kWindowList];
    __shared__ RankScratch<W> ranked;
    __shared__ uint32_t held;
    __shared__ WindowTotals t;
    const uint32_t tid = threadIdx.x;
    WindowCounts& w = *a.counts;
    t.read(w);
    const bool keep_all = t.finite <= a.n;
    bool done = !keep_all && t.holds(a.n, a.room);  // uniform
    uint64_t boundary = 0, stay = 0;
    uint32_t equal = 0;
    if (done) {
        const uint64_t m = a.narrow ? w.narrowed : t.first[kWindowParts];
        const uint64_t* const key = a.narrow ? a.key2 : a.key;
        const uint64_t* const pos = a.narrow ? a.pos2 : a.pos;
        auto at = [&](uint64_t i) { return a.narrow ? i : t.at(i, a.room); };
        uint64_t k = a.n - (a.narrow ? w.narrowed_above : t.above);  // 1 <= k <= m
        uint64_t base = a.lo, left = m;
        int shift = 64;  // the keys sought lie in [base, base + 2^shift)
        if (m > kWindowRank) {
            shift = 64 - __builtin_clzll(a.hi - a.lo);
            while (left > kWindowList && shift > 0) {
                const int sh = max(shift - 11, 0);
                for (uint32_t i = tid; i < kDigits; i += kFinishBlock) hist[i] = 0u;
                __syncthreads();
                for (uint64_t i0 = tid; i0 < m; i0 += 4 * kFinishBlock) {  // four loads in flight per thread
                    uint64_t r[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        r[q] = i0 + q * kFinishBlock < m ? key[at(i0 + q * kFinishBlock)] - base : ~0ull;
#pragma unroll
                    for (int q = 0; q < 4; ++q)  // a smaller key wraps far past the range
                        if ((r[q] >> shift) == 0) atomicAdd(&hist[r[q] >> sh], 1u);
                }
                __syncthreads();
                uint64_t bin[3];
                window_bin<kDigits, kFinishBlock>(hist, k, part, bin);
                base += bin[0] << sh;
                k -= bin[1];
                left = bin[2];
                shift = sh;
            }
        }
        done = left <= kWindowList;  // else more equal keys than the list holds
        if (done) {
            if (tid == 0) held = 0u;
            __syncthreads();
            for (uint64_t i0 = tid; i0 < m; i0 += 4 * kFinishBlock) {
                uint64_t u[4];
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (i0 + q * kFinishBlock < m) u[q] = key[at(i0 + q * kFinishBlock)];
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (i0 + q * kFinishBlock < m && (shift == 64 || ((u[q] - base) >> shift) == 0)) {
                        const uint32_t slot = atomicAdd(&held, 1u);
                        su[slot] = u[q];
                        sp[slot] = pos[at(i0 + q * kFinishBlock)];
                    }
            }
            __syncthreads();
            uint32_t n = held;  // = left
            narrow_list(su, sp, n, &held, base, shift, k, hist, part);
            done = rank_boundary<W, T>(a, ranked, su, sp, n, k, shift == 0, boundary, stay, equal);
        }
    }
    const bool crowded = !done && !keep_all && a.narrow && t.fullest > a.room && t.inside(a.n);  // uniform
    uint64_t bin[3] = {0, 0, 0};
    if (crowded) {
        if (tid < kWindowBins) hist[tid] = 0u;
        __syncthreads();
        window_bins_sum<kFinishBlock>(w, hist);
        window_bin<kWindowBins, kFinishBlock>(hist, a.n - t.above, part, bin);
    }
    __syncthreads();  // the counts are no longer read
    if (a.narrow)
        for (uint32_t i = tid; i < kWindowCopies * kWindowBins / 4; i += kFinishBlock)
            reinterpret_cast<uint4*>(&w.bins[0][0])[i] = make_uint4(0u, 0u, 0u, 0u);
    if (tid < kWindowParts) {
        w.part[tid].above_finite = 0;
        w.part[tid].count = 0;
        w.part[tid].overflow = 0;
    }
    if (tid == 0) {
        w.narrowed = 0;
        w.narrowed_above = 0;
        if (done || keep_all) {
            TopnState& s = *a.state;
            s.prefix = boundary;
            s.mask = ~0ull;
            s.k = stay;
            s.above = a.n - stay;
            s.finite = t.finite;
            s.ties = equal;
            s.keep_all_finite = keep_all ? 1 : 0;
        }
        volatile unsigned long long* h = a.host;  // fine-grained host memory: the stores bypass the L2
        h[0] = done || keep_all ? kWindowDone : crowded ? kWindowCrowded : kWindowMissed;
        h[1] = keep_all ? 0ull : boundary;
        h[2] = t.fullest;
        h[3] = t.finite;
        h[5] = done && stay < equal ? 1 : 0;
        h[6] = bin[0];
        __builtin_amdgcn_s_waitcnt(0);  // the slot's words land before its sequence number
        h[4] = a.seq;
    }
}

// A whole selection by one workgroup, for many sums of up to kWholeTerms terms at once: the n-th key by 11-bit digits
// over every key of the sum, then as k_window_finish ranks.  It needs no boundary to start from.  Each wave reads four
// buckets at a time, sixteen loads in flight per lane: the latency of the one CU's reads bounds it, and the counts of keys
// that share a digit follow one another in the LDS.  64 sums keeping 2^15 of up to 2^16 terms: 37 us in one launch (48 with
// the octaves as the first digit), where the start, three radix passes and their selects were 46 in seven, with a second
// round trip for the boundary bins ordered on the host.  (The windowed selection batched the same way took 21, but with
// angles drawn from the whole circle some sum's boundary left its window in 788 of 823 steps.)
template <int W, typename T, typename F>
__device__ __forceinline__ void whole_keys(const WholeArgs<W, T>& a, const uint32_t* first, const uint16_t* len, F f) {
    constexpr uint32_t kWavesHere = kFinishBlock / 64;
    for (uint32_t b0 = wave_id(); b0 < a.num_buckets; b0 += 4 * kWavesHere) {
        uint32_t most = 0, from[4], n[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t b = b0 + q * kWavesHere;
            n[q] = b < a.num_buckets ? len[b] : 0u;
            from[q] = n[q] ? first[b] : 0u;
            most = max(most, n[q]);
        }
        for (uint32_t r0 = lane_id(); r0 - lane_id() < most; r0 += 256) {
            T c[4][4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (r0 + 64 * v < n[q]) c[q][v] = a.c[from[q] + r0 + 64 * v];
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (r0 + 64 * v < n[q]) {
                        const uint64_t u = magnitude_bits<T>(c[q][v]);
                        if (!is_nan_bits(u)) f(u, from[q] + r0 + 64 * v);
                    }
        }
    }
}

template <int W, typename T>
__global__ void __launch_bounds__(kFinishBlock) k_topn_whole(const WholeArgs<W, T>* __restrict__ items) {
    constexpr uint32_t kDigits = 2048;
    __shared__ uint32_t hist[kDigits];
    __shared__ uint64_t part[kFinishBlock / 64 + 3];
    __shared__ uint64_t su[kWindowList], sp[kWindowList];
    __shared__ RankScratch<W> ranked;
    __shared__ uint32_t first[kWholeBuckets];
    __shared__ uint16_t len[kWholeBuckets];
    __shared__ uint32_t held, finite_terms, above_terms;
    const WholeArgs<W, T> a = items[blockIdx.x];
    const uint32_t tid = threadIdx.x;
    for (uint32_t b = tid; b < a.num_buckets; b += kFinishBlock) {
        first[b] = (uint32_t)a.start[b];
        len[b] = (uint16_t)a.len[b];
    }
    for (uint32_t i = tid; i < kDigits; i += kFinishBlock) hist[i] = 0u;
    if (tid == 0) held = finite_terms = above_terms = 0u;
    __syncthreads();
    // The first digit: of eight octaves around the last boundary 256 parts each, which leaves a few keys to collect and
    // spreads the counts over the LDS; with no boundary, or one outside them, the octaves alone.
    const uint64_t low = a.seed ? max(a.seed >> 44, 1024ull) - 1024ull : 0ull;
    int shift = a.seed ? 44 : 52;
    uint32_t mine = 0, over = 0;
    whole_keys<W, T>(a, first, len, [&](uint64_t u, uint32_t) {
        ++mine;
        const uint64_t r = (u >> shift) - low;
        if (r < kDigits) atomicAdd(&hist[r], 1u);
        else over += (u >> shift) > low;
    });
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        mine += (uint32_t)__shfl_xor((int)mine, d, 64);
        over += (uint32_t)__shfl_xor((int)over, d, 64);
    }
    if (lane_id() == 0) {
        atomicAdd(&finite_terms, mine);
        if (over) atomicAdd(&above_terms, over);
    }
    __syncthreads();
    const uint32_t finite = finite_terms, above = above_terms;
    const bool keep_all = finite <= a.n;  // uniform
    bool done = keep_all;
    uint64_t boundary = 0, stay = 0;
    uint32_t equal = 0;
    if (!keep_all) {
        uint64_t k = a.n - above, base = 0, bin[3] = {0, 0, 0};
        bool outside = above >= a.n;  // uniform, as below
        if (!outside) {
            if (tid == 0) part[kFinishBlock / 64 + 2] = 0;  // window_bin leaves the answer as it is when there is none
            window_bin<kDigits, kFinishBlock>(hist, k, part, bin);
            outside = bin[2] == 0;
        }
        if (outside) {
            shift = 52;
            k = a.n;
            for (uint32_t i = tid; i < kDigits; i += kFinishBlock) hist[i] = 0u;
            __syncthreads();
            whole_keys<W, T>(a, first, len, [&](uint64_t u, uint32_t) { atomicAdd(&hist[u >> 52], 1u); });
            __syncthreads();
            window_bin<kDigits, kFinishBlock>(hist, k, part, bin);
        }
        base = (bin[0] + (outside ? 0 : low)) << shift;
        k -= bin[1];
        while (bin[2] > kWindowList && shift > 0) {
            const int sh = max(shift - 11, 0);
            for (uint32_t i = tid; i < kDigits; i += kFinishBlock) hist[i] = 0u;
            __syncthreads();
            whole_keys<W, T>(a, first, len, [&](uint64_t u, uint32_t) {
                const uint64_t r = u - base;  // a smaller key wraps far past the range
                if ((r >> shift) == 0) atomicAdd(&hist[r >> sh], 1u);
            });
            __syncthreads();
            window_bin<kDigits, kFinishBlock>(hist, k, part, bin);
            base += bin[0] << sh;
            k -= bin[1];
            shift = sh;
        }
        done = bin[2] <= kWindowList;  // else more equal keys than the list holds
        if (done) {
            whole_keys<W, T>(a, first, len, [&](uint64_t u, uint32_t at) {
                if (((u - base) >> shift) == 0) {
                    const uint32_t slot = atomicAdd(&held, 1u);
                    su[slot] = u;
                    sp[slot] = at;
                }
            });
            __syncthreads();
            uint32_t listed = held;
            narrow_list(su, sp, listed, &held, base, shift, k, hist, part);
            done = rank_boundary<W, T>(a, ranked, su, sp, listed, k, shift == 0, boundary, stay, equal);
        }
    }
    if (tid == 0) {
        if (done) {
            TopnState& s = *a.state;
            s.prefix = boundary;
            s.mask = ~0ull;
            s.k = stay;
            s.above = a.n - stay;
            s.finite = finite;
            s.ties = equal;
            s.keep_all_finite = keep_all ? 1 : 0;
        }
        volatile unsigned long long* h = a.host;  // fine-grained host memory: the stores bypass the L2
        h[0] = done ? kWindowDone : kWindowMissed;
        h[1] = boundary;
        h[3] = finite;
        h[5] = done && stay < equal ? 1 : 0;
        __builtin_amdgcn_s_waitcnt(0);  // the slot's words land before its sequence number
        h[4] = a.seq;
    }
}

template <int W, typename T>
hipError_t launch_topn_whole(hipStream_t st, const WholeArgs<W, T>* items, uint32_t num_items) {
    if (num_items == 0) return hipSuccess;
    hipLaunchKernelGGL((k_topn_whole<W, T>), dim3(num_items), dim3(kFinishBlock), 0, st, items);
    return hipGetLastError();
}

template <int W, typename T>
bool window_args_valid(const WindowArgs<W, T>& a) {
    return a.buckets_per_block != 0 && a.buckets_per_block <= kHistBucketsMax && a.hi > a.lo && a.n != 0 &&
           a.hi - a.lo < kWindowSpan && a.bin_shift >= 0 && a.bin_shift <= 63 &&
           ((a.hi - a.lo - 1) >> a.bin_shift) < kWindowBins;
}

template <int W, typename T>
hipError_t launch_topn_window(hipStream_t st, const WindowArgs<W, T>& a) {
    if (!window_args_valid<W, T>(a)) return hipErrorInvalidValue;
    const uint32_t blocks = (a.num_buckets + a.buckets_per_block - 1) / a.buckets_per_block;
    hipLaunchKernelGGL((k_window_scan<W, T>), dim3(blocks), dim3(kBlock), 0, st, a);
    if (a.narrow) hipLaunchKernelGGL((k_window_narrow<W, T>), dim3(256), dim3(kBlock), 0, st, a);
    hipLaunchKernelGGL((k_window_finish<W, T>), dim3(1), dim3(kFinishBlock), 0, st, a);
    return hipGetLastError();
}

// ---- ApproxTopN ---------------------------------------------------------------------------------------------

// octave(norm_sqr) = norm_sqr.to_bits() >> 52 (builtin.rs:276-279).  A NaN of either sign counts in octave 2047,
// as a positive NaN does in the reference; classify_octave (:281-288) puts it below every octave.
__device__ __forceinline__ uint32_t octave_of(uint64_t u) { return (uint32_t)((u >> 52) & 0x7FFu); }

template <typename T>
__global__ void __launch_bounds__(kBlock) k_octave_hist(const OctaveHistArgs<T> a) {
    __shared__ uint32_t h[kOctaveBins];
    for (int i = threadIdx.x; i < kOctaveBins; i += kBlock) h[i] = 0;
    __syncthreads();
    const uint32_t b_lo = blockIdx.x * a.buckets_per_block;
    const uint32_t b_hi = min(a.num_buckets, b_lo + a.buckets_per_block);
    for (uint32_t b = b_lo; b < b_hi; ++b) {
        const uint32_t n = a.len[b];
        const uint64_t s = a.start[b];
        for (uint32_t r = threadIdx.x; r < n; r += kBlock) atomicAdd(&h[octave_of(magnitude_bits<T>(a.c[s + r]))], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kOctaveBins; i += kBlock)
        if (h[i]) atomicAdd(&a.hist[i], (unsigned long long)h[i]);
}

// The boundary side of a term: 1 above the octave, 0 at it, -1 below (or NaN).
__device__ __forceinline__ int octave_side(uint64_t u, uint32_t bin) {
    if (is_nan_bits(u)) return -1;
    const uint32_t o = octave_of(u);
    return o > bin ? 1 : (o == bin ? 0 : -1);
}

// ---- the cut on the device: five launches and one wait of the host

// Octave counts, a copy of the LDS histogram per wave (a wave's keys share a few octaves).
template <int W, typename T>
__global__ void __launch_bounds__(kBlock) k_octave_scan(const OctaveSelectArgs<W, T> a) {
    __shared__ uint32_t h[kWaves][kOctaveBins];
    __shared__ RowList list;
    __shared__ uint32_t nan;
    for (uint32_t i = threadIdx.x; i < kWaves * kOctaveBins; i += kBlock) (&h[0][0])[i] = 0u;
    if (threadIdx.x == 0) nan = 0u;
    const uint32_t b_lo = blockIdx.x * a.buckets_per_block;
    const uint32_t nb = min(a.num_buckets, b_lo + a.buckets_per_block) - b_lo;  // <= kHistBucketsMax
    const uint32_t total = list_rows(a.start, a.len, b_lo, nb, list);
    uint32_t j = 0;
    for (uint32_t g0 = threadIdx.x; g0 < total; g0 += 8 * kBlock) {
        uint64_t pos[8];
        bool in[8];
        list_positions(list, total, g0, j, pos, in);
        T c[8];
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (in[q]) c[q] = a.c[pos[q]];
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (in[q]) {
                const uint64_t u = magnitude_bits<T>(c[q]);
                atomicAdd(&h[wave_id()][octave_of(u)], 1u);
                if (is_nan_bits(u)) atomicAdd(&nan, 1u);
            }
    }
    __syncthreads();
    const uint32_t copy = blockIdx.x % kOctaveCopies;
    for (uint32_t i = threadIdx.x; i < kOctaveBins; i += kBlock) {
        uint32_t v = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) v += h[w][i];
        if (v) atomicAdd(&a.counts->hist[copy][i], v);
    }
    if (threadIdx.x == 0 && nan) atomicAdd(&a.counts->nan[copy * 32], nan);
}

// octave_edge (builtin.rs:320-352): whole octaves from the top while they fit in n; the first that does not is the
// boundary.  One workgroup, two octaves a thread.
template <int W, typename T>
__global__ void __launch_bounds__(kFinishBlock) k_octave_edge(const OctaveSelectArgs<W, T> a) {
    constexpr uint32_t PER = kOctaveBins / kFinishBlock;
    __shared__ uint64_t part[kFinishBlock / 64];
    OctaveCounts& w = *a.counts;
    const uint32_t tid = threadIdx.x;
    uint64_t mine[PER], sum = 0;
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
        mine[q] = 0;
#pragma unroll
        for (uint32_t c = 0; c < kOctaveCopies; ++c) mine[q] += w.hist[c][tid * PER + q];
        sum += mine[q];
    }
    uint64_t suffix = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t o = __shfl_down(suffix, d, 64);
        if (lane_id() + (uint32_t)d < 64u) suffix += o;
    }
    if (lane_id() == 0) part[wave_id()] = suffix;
    __syncthreads();
    uint64_t above = suffix - sum;
    for (uint32_t v = wave_id() + 1; v < kFinishBlock / 64; ++v) above += part[v];
    if (above <= a.n && above + sum > a.n) {  // this thread's octaves hold the boundary
        for (uint32_t q = PER; q-- > 0;) {
            if (above + mine[q] > a.n) {
                uint64_t nan = 0;
                for (uint32_t c = 0; c < kOctaveCopies; ++c) nan += w.nan[c * 32];
                const uint32_t bin = tid * PER + q;
                w.bin = bin;
                w.quota = a.n - above;
                w.above = above - (bin < kOctaveBins - 1 ? nan : 0ull);  // NaNs count in the last octave, and go
                break;
            }
            above += mine[q];
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < kOctaveCopies * kOctaveBins; i += kFinishBlock) (&w.hist[0][0])[i] = 0u;
    if (tid < kOctaveCopies) w.nan[tid * 32] = 0u;
}

// A wave per device bucket: its terms of the boundary octave counted (FLAGS false), or flagged by whether the quota
// reaches their reference bucket (FLAGS true; the split bucket's are flagged already).
template <int W, typename T, bool FLAGS>
__global__ void __launch_bounds__(kBlock) k_octave_bucket(const OctaveSelectArgs<W, T> a) {
    const uint32_t b = blockIdx.x * kWaves + wave_id();
    if (b >= a.num_buckets) return;  // the whole wave
    const uint32_t bin = a.counts->bin;
    const uint32_t n = a.len[b];
    const uint64_t s = a.start[b];
    uint8_t flag = 0;
    if constexpr (FLAGS) {
        const uint32_t rb = b & (a.ref_buckets - 1u), split = a.split[0];
        if (rb == split) return;
        flag = rb < split ? 1 : 0;
    }
    uint32_t count = 0;
    for (uint32_t r0 = lane_id(); r0 < n; r0 += 4 * 64) {
        T c[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (r0 + q * 64 < n) c[q] = a.c[s + r0 + q * 64];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (r0 + q * 64 >= n || octave_side(magnitude_bits<T>(c[q]), bin) != 0) continue;
            if constexpr (FLAGS) a.flags[s + r0 + q * 64] = flag;
            else ++count;
        }
    }
    if constexpr (!FLAGS) {
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) count += (uint32_t)__shfl_xor((int)count, d, 64);
        if (lane_id() == 0) a.boundary[b] = count;
    }
}

// QuotaSplit::new (builtin.rs:160-197): the reference bucket where the quota runs out, and its first terms in
// lexicographic order ranked by counting.  One workgroup; each thread owns a run of reference buckets.
template <int W, typename T>
__global__ void __launch_bounds__(kFinishBlock) k_octave_split(const OctaveSelectArgs<W, T> a) {
    __shared__ uint64_t part[kFinishBlock / 64];
    __shared__ uint64_t kx[W][kCutRows], kz[W][kCutRows], kp[kCutRows];
    __shared__ uint32_t held, split;
    __shared__ uint64_t left;
    const OctaveCounts& w = *a.counts;
    const uint32_t tid = threadIdx.x, parts = a.num_buckets / a.ref_buckets;
    if (tid == 0) {
        held = 0u;
        split = a.ref_buckets;
        left = 0;
    }
    const uint32_t per = (a.ref_buckets + kFinishBlock - 1) / kFinishBlock;
    const uint32_t lo = min(tid * per, a.ref_buckets), hi = min(lo + per, a.ref_buckets);
    auto ref_count = [&](uint32_t rb) {
        uint32_t v = 0;
#pragma unroll 4
        for (uint32_t e = 0; e < parts; ++e) v += a.boundary[rb + e * a.ref_buckets];
        return v;
    };
    uint64_t mine = 0;
    for (uint32_t e = 0; e < parts; ++e) {
#pragma unroll 4
        for (uint32_t rb = lo; rb < hi; ++rb) mine += a.boundary[rb + e * a.ref_buckets];
    }
    uint64_t inc = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t o = __shfl_up(inc, d, 64);
        if (lane_id() >= (uint32_t)d) inc += o;
    }
    if (lane_id() == 63) part[wave_id()] = inc;
    __syncthreads();
    uint64_t seen = inc - mine, total = 0;
    for (uint32_t v = 0; v < kFinishBlock / 64; ++v) {
        seen += v < wave_id() ? part[v] : 0ull;
        total += part[v];
    }
    const uint64_t quota = w.quota;
    if (seen <= quota && seen + mine > quota)  // this thread's buckets hold the split
        for (uint32_t rb = lo; rb < hi; ++rb) {
            const uint32_t v = ref_count(rb);
            if (seen + v > quota) {
                split = rb;
                left = quota - seen;
                break;
            }
            seen += v;
        }
    __syncthreads();
    const uint32_t sb = split;
    const uint64_t remaining = left;
    if (sb < a.ref_buckets) {
        for (uint32_t e = 0; e < parts; ++e) {
            const uint32_t b = sb + e * a.ref_buckets;
            const uint32_t n = a.len[b];
            const uint64_t s = a.start[b];
            for (uint32_t r = tid; r < n; r += kFinishBlock) {
                if (octave_side(magnitude_bits<T>(a.c[s + r]), w.bin) != 0) continue;
                const uint32_t slot = atomicAdd(&held, 1u);
                if (slot >= kCutRows) continue;
                const Key<W> k = load_key<W>(a.x, a.z, a.cap, s + r);
#pragma unroll
                for (int v = 0; v < W; ++v) {
                    kx[v][slot] = k.x[v];
                    kz[v][slot] = k.z[v];
                }
                kp[slot] = s + r;
            }
        }
        __syncthreads();
        const uint32_t m = min(held, kCutRows);
        for (uint32_t i = tid; i < m; i += kFinishBlock) {
            uint32_t before = 0;
            for (uint32_t q = 0; q < m; ++q) {
                int order = 0;
#pragma unroll
                for (int v = 0; v < W; ++v)
                    if (order == 0) order = kx[v][q] < kx[v][i] ? -1 : kx[v][q] > kx[v][i] ? 1 : 0;
#pragma unroll
                for (int v = 0; v < W; ++v)
                    if (order == 0) order = kz[v][q] < kz[v][i] ? -1 : kz[v][q] > kz[v][i] ? 1 : 0;
                before += order < 0;
            }
            a.flags[kp[i]] = before < remaining ? 1 : 0;
        }
    }
    if (tid == 0) {
        a.split[0] = sb;
        TopnState& st = *a.state;
        st.prefix = (unsigned long long)w.bin << 52;
        st.mask = 0xFFF0000000000000ull;
        st.keep_all_finite = 0;
        volatile unsigned long long* h = a.host;  // fine-grained host memory: the stores bypass the L2
        h[0] = held > kCutRows ? 2 : 1;
        h[1] = w.above + (sb < a.ref_buckets ? quota : total);
        __builtin_amdgcn_s_waitcnt(0);  // the slot's words land before its sequence number
        h[4] = a.seq;
    }
}

template <int W, typename T>
hipError_t launch_octave_select(hipStream_t st, const OctaveSelectArgs<W, T>& a) {
    if (a.num_buckets == 0 || a.ref_buckets > a.num_buckets || a.buckets_per_block == 0 ||
        a.buckets_per_block > kHistBucketsMax)
        return hipErrorInvalidValue;
    const uint32_t blocks = (a.num_buckets + a.buckets_per_block - 1) / a.buckets_per_block;
    const uint32_t waves = (a.num_buckets + kWaves - 1) / kWaves;
    hipLaunchKernelGGL((k_octave_scan<W, T>), dim3(blocks), dim3(kBlock), 0, st, a);
    hipLaunchKernelGGL((k_octave_edge<W, T>), dim3(1), dim3(kFinishBlock), 0, st, a);
    hipLaunchKernelGGL((k_octave_bucket<W, T, false>), dim3(waves), dim3(kBlock), 0, st, a);
    hipLaunchKernelGGL((k_octave_split<W, T>), dim3(1), dim3(kFinishBlock), 0, st, a);
    hipLaunchKernelGGL((k_octave_bucket<W, T, true>), dim3(waves), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

template <int W, typename T>
__global__ void __launch_bounds__(kBlock) k_octave_counts(const OctaveCutArgs<W, T> a) {
    const uint32_t b = blockIdx.x;
    const uint32_t n = a.len[b];
    const uint64_t s = a.start[b];
    for (uint32_t r = threadIdx.x; r < n; r += kBlock) {
        if (octave_side(magnitude_bits<T>(a.c[s + r]), a.bin) != 0) continue;
        const Key<W> k = load_key<W>(a.x, a.z, a.cap, s + r);
        atomicAdd(&a.counts[bucket_of<W>(k, a.rows, a.ref_bits)], 1u);
    }
}

template <int W, typename T>
__global__ void __launch_bounds__(kBlock) k_octave_gather(const OctaveCutArgs<W, T> a) {
    const uint32_t b = blockIdx.x;
    const uint32_t n = a.len[b];
    const uint64_t s = a.start[b];
    for (uint32_t r = threadIdx.x; r < n; r += kBlock) {
        if (octave_side(magnitude_bits<T>(a.c[s + r]), a.bin) != 0) continue;
        const Key<W> k = load_key<W>(a.x, a.z, a.cap, s + r);
        if (bucket_of<W>(k, a.rows, a.ref_bits) != a.split_bucket) continue;
        const uint64_t slot = atomicAdd(a.gathered, 1ull);
        if (slot >= a.out_cap) continue;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            a.out_x[slot * W + w] = k.x[w];
            a.out_z[slot * W + w] = k.z[w];
        }
        a.out_pos[slot] = s + r;
    }
}

template <int W, typename T>
__global__ void __launch_bounds__(kBlock) k_octave_retain(const OctaveCutArgs<W, T> a) {
    __shared__ uint32_t scan_scratch[kWaves];
    const uint32_t b = blockIdx.x;
    const uint32_t n = a.len[b];
    const uint64_t s = a.start[b];
    uint32_t cur = 0;
    for (uint32_t base = 0; base < n; base += kBlock) {
        const uint32_t r = base + threadIdx.x;
        Key<W> k;
        T c = T(0);
        bool keep = false;
        if (r < n) {
            k = load_key<W>(a.x, a.z, a.cap, s + r);
            c = a.c[s + r];
            const int side = octave_side(magnitude_bits<T>(c), a.bin);
            if (side > 0) {
                keep = true;
            } else if (side == 0) {
                const uint32_t rb = bucket_of<W>(k, a.rows, a.ref_bits);
                keep = rb < a.split_bucket || (rb == a.split_bucket && a.keep != nullptr && a.keep[s + r] != 0);
            }
        }
        bool f[1] = {keep};
        uint32_t off[1], tot[1];
        block_flag_scan<1>(f, off, tot, scan_scratch);  // every read of the chunk precedes its writes
        if (keep && cur + off[0] != r) {
            const uint64_t pos = s + cur + off[0];
#pragma unroll
            for (int w = 0; w < W; ++w) {
                a.x[w * a.cap + pos] = k.x[w];
                a.z[w * a.cap + pos] = k.z[w];
            }
            a.c[pos] = c;
        }
        cur += tot[0];
    }
    if (threadIdx.x == 0) a.len[b] = cur;
}

template <typename T>
hipError_t launch_octave_hist(hipStream_t st, const OctaveHistArgs<T>& a, uint32_t blocks) {
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL((k_octave_hist<T>), dim3(blocks), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

template <int W, typename T>
hipError_t launch_octave_counts(hipStream_t st, const OctaveCutArgs<W, T>& a, uint32_t num_buckets) {
    if (num_buckets == 0) return hipSuccess;
    hipLaunchKernelGGL((k_octave_counts<W, T>), dim3(num_buckets), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

template <int W, typename T>
hipError_t launch_octave_gather(hipStream_t st, const OctaveCutArgs<W, T>& a, uint32_t num_buckets) {
    if (num_buckets == 0) return hipSuccess;
    hipLaunchKernelGGL((k_octave_gather<W, T>), dim3(num_buckets), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

template <int W, typename T>
hipError_t launch_octave_retain(hipStream_t st, const OctaveCutArgs<W, T>& a, uint32_t num_buckets) {
    if (num_buckets == 0) return hipSuccess;
    hipLaunchKernelGGL((k_octave_retain<W, T>), dim3(num_buckets), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_topn_init_batch(hipStream_t st, const TopnSelectItem* items, uint32_t num_items) {
    if (num_items == 0) return hipSuccess;
    hipLaunchKernelGGL(k_topn_init_batch, dim3(num_items), dim3(kBlock), 0, st, items);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_topn_hist_batch(hipStream_t st, const TopnHistArgs<T>* items, const uint32_t* block_start,
                                  uint32_t num_items, uint32_t blocks, int pass) {
    if (num_items == 0 || blocks == 0) return hipSuccess;
    hipLaunchKernelGGL((k_topn_hist_batch<T>), dim3(blocks), dim3(kBlock), 0, st, items, block_start, num_items,
                       (int32_t)pass);
    return hipGetLastError();
}

hipError_t launch_topn_select_batch(hipStream_t st, const TopnSelectItem* items, uint32_t num_items, int pass,
                                    bool last) {
    if (num_items == 0) return hipSuccess;
    hipLaunchKernelGGL(k_topn_select_batch, dim3(num_items), dim3(kBlock), 0, st, items, pass, last ? 1 : 0);
    return hipGetLastError();
}

template <int W, typename T>
hipError_t launch_topn_gather_batch(hipStream_t st, const TopnTieArgs<W, T>* items, const uint32_t* block_start,
                                    uint32_t num_items, uint32_t blocks) {
    if (num_items == 0 || blocks == 0) return hipSuccess;
    hipLaunchKernelGGL((k_topn_gather_batch<W, T>), dim3(blocks), dim3(kBlock), 0, st, items, block_start,
                       num_items);
    return hipGetLastError();
}

hipError_t launch_topn_flag_ties(hipStream_t st, const uint64_t* pos, uint64_t ties, uint64_t kept, uint8_t* flags) {
    if (ties == 0) return hipSuccess;
    hipLaunchKernelGGL(k_topn_flag_ties, dim3((uint32_t)((ties + 255) / 256)), dim3(256), 0, st, pos, ties, kept,
                       flags);
    return hipGetLastError();
}

hipError_t launch_topn_flags_batch(hipStream_t st, const TopnFlagItem* items, uint32_t num_items) {
    if (num_items == 0) return hipSuccess;
    hipLaunchKernelGGL(k_topn_flags_batch, dim3(num_items), dim3(kBlock), 0, st, items);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_topn_hist(hipStream_t st, const TopnHistArgs<T>& a, uint32_t blocks) {
    hipLaunchKernelGGL((k_topn_hist<T>), dim3(blocks), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_topn_select(hipStream_t st, TopnState* state, unsigned long long* hist, int pass, uint64_t n) {
    hipLaunchKernelGGL(k_topn_select, dim3(1), dim3(kBlock), 0, st, state, hist, pass, n);
    return hipGetLastError();
}

hipError_t launch_topn_init(hipStream_t st, TopnState* state, uint64_t n, unsigned long long* hist,
                            uint32_t hist_words, uint64_t seed, bool seeded) {
    hipLaunchKernelGGL(k_topn_init, dim3(1), dim3(kBlock), 0, st, state, n, seed, seeded ? 1u : 0u, hist,
                       hist_words);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_topn_hist_seeded(hipStream_t st, const TopnHistArgs<T>& a, uint32_t blocks) {
    hipLaunchKernelGGL((k_topn_hist_seeded<T>), dim3(blocks), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_topn_select_seeded(hipStream_t st, TopnState* state, unsigned long long* hist, uint64_t n) {
    hipLaunchKernelGGL(k_topn_select_seeded, dim3(1), dim3(kBlock), 0, st, state, hist, n);
    return hipGetLastError();
}

template <int W, typename T>
hipError_t launch_topn_gather_ties(hipStream_t st, const TopnTieArgs<W, T>& a, uint32_t num_buckets) {
    (void)num_buckets;
    if (a.buckets_per_block == 0 || a.buckets_per_block > kHistBucketsMax) return hipErrorInvalidValue;
    const uint32_t blocks = (a.num_buckets + a.buckets_per_block - 1) / a.buckets_per_block;
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL((k_topn_gather_ties<W, T>), dim3(blocks), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

template <int W, typename T>
hipError_t launch_topn_retain(hipStream_t st, const TopnRetainArgs<W, T>& a, uint32_t num_buckets) {
    hipLaunchKernelGGL((k_topn_retain<W, T>), dim3(num_buckets), dim3(kBlock), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_mark_positions(hipStream_t st, const uint64_t* pos, uint64_t n, uint8_t* flags) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_mark_positions, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, st, pos, n, flags);
    return hipGetLastError();
}

template hipError_t launch_topn_hist_batch<double>(hipStream_t, const TopnHistArgs<double>*, const uint32_t*, uint32_t,
                                                   uint32_t, int);
template hipError_t launch_topn_hist_batch<float>(hipStream_t, const TopnHistArgs<float>*, const uint32_t*, uint32_t,
                                                  uint32_t, int);
template hipError_t launch_topn_hist<double>(hipStream_t, const TopnHistArgs<double>&, uint32_t);
template hipError_t launch_topn_hist<float>(hipStream_t, const TopnHistArgs<float>&, uint32_t);
template hipError_t launch_topn_hist_seeded<double>(hipStream_t, const TopnHistArgs<double>&, uint32_t);
template hipError_t launch_topn_hist_seeded<float>(hipStream_t, const TopnHistArgs<float>&, uint32_t);
template hipError_t launch_octave_hist<double>(hipStream_t, const OctaveHistArgs<double>&, uint32_t);
template hipError_t launch_octave_hist<float>(hipStream_t, const OctaveHistArgs<float>&, uint32_t);
#define PP_TOPN_INSTANTIATE(W, T)                                                                       \
    template hipError_t launch_octave_select<W, T>(hipStream_t, const OctaveSelectArgs<W, T>&);         \
    template hipError_t launch_topn_window<W, T>(hipStream_t, const WindowArgs<W, T>&);                 \
    template hipError_t launch_topn_whole<W, T>(hipStream_t, const WholeArgs<W, T>*, uint32_t);         \
    template hipError_t launch_topn_gather_ties<W, T>(hipStream_t, const TopnTieArgs<W, T>&, uint32_t); \
    template hipError_t launch_topn_gather_batch<W, T>(hipStream_t, const TopnTieArgs<W, T>*, const uint32_t*, \
                                                       uint32_t, uint32_t);                               \
    template hipError_t launch_topn_retain<W, T>(hipStream_t, const TopnRetainArgs<W, T>&, uint32_t);   \
    template hipError_t launch_octave_counts<W, T>(hipStream_t, const OctaveCutArgs<W, T>&, uint32_t);  \
    template hipError_t launch_octave_gather<W, T>(hipStream_t, const OctaveCutArgs<W, T>&, uint32_t);  \
    template hipError_t launch_octave_retain<W, T>(hipStream_t, const OctaveCutArgs<W, T>&, uint32_t);
PP_TOPN_INSTANTIATE(1, double)
PP_TOPN_INSTANTIATE(1, float)
PP_TOPN_INSTANTIATE(2, double)
PP_TOPN_INSTANTIATE(2, float)

}  // namespace pp
