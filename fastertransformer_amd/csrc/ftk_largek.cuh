// The fused step for launches whose largest k is beyond what one read of a row can bound (k > 192), in one launch: a
// 1024-thread workgroup owns a row.
//
// The lean gather takes three launches for them (lean_gather_kernel in its SLOTS and PRESET modes, lean_select_kernel),
// bound by the latency of many small workgroups and by a selection on four waves. Here
//   1. every thread takes the exact maxima of three disjoint groups of its columns (3072 per row, in short rows
//      one per vector and edge column, each the final value of a column of its own, after temperature, history penalty and masks);
//   2. the row's bound: the largest P, to within its low sixteen bits, that at least k of those maxima reach (two
//      rounds of a 256-bin count over the keys' top bytes) - at least k columns lie at or above it;
//   3. the vectors that hold something at or above the bound are noted in LDS and evaluated exactly, one per lane, into
//      the row's list. Rows of at most LK_RING vectors per thread are still in registers, longer ones come from the caches;
//   4. all sixteen waves put the list in the reference's order (largek_order), then one thread draws.
// A list that outgrows LDS is gathered again under a bound that counts every column. Short lists (rows with a small k) end
// like those of ftk_rowwide.cuh; rows with more equal values than LDS holds, or whose values 2048 buckets cannot tell apart,
// like its rare rows.
// What bounds it, 256 x 51200 f16, k = 1024 (us inside a workgroup): set-up 1.9, first pass 2.4, bound 4.4, second pass 7.4
// with its barrier, order 5.6, draw 4.1; 31 a step, 65 with maxima, gather and selection in launches of their own. With 12
// instead of 9 vectors in registers the compiler spills 41 of them.
// Preconditions (checked by the host): no embedding bias, three vectors of a row for every two of k, the row's history bitmap
// fits the LDS window, logits on an element's boundary.
#pragma once
#include "ftk_rowwide.cuh"

namespace ftk {

constexpr int LK_THREADS    = 1024;
constexpr int LK_WAVES      = LK_THREADS / WAVE;
constexpr int LK_GROUPS     = 3;     // maxima per thread
constexpr int LK_RING       = 9;    // vectors a thread holds
constexpr int LK_HIST_U     = 4;     // history ids a thread requests at a time
constexpr int LK_BUCKETS    = 2048;  // of the final order: 256 for each of eight doublings of the distance to the bound
constexpr int LK_BUCKET_CAP = 512;   // entries of a bucket are compared with each other
constexpr int LK_BUCKET_FEW = 96;    // more, and a quarter of the list: the bucket is divided by buckets of its own
static_assert(LK_RING % LK_GROUPS == 0, "a slot of the ring always belongs to the same group");

struct LargekShared {
    int      noted[LK_WAVES][LK_RING * WAVE];  // vectors of a wave that may hold a candidate
    uint32_t count[LK_BUCKETS + 1];
    uint32_t hist[256];
    uint32_t chunk[32][8];  // entries of each stage-1 slice in 64 positions of the list
    uint32_t wave_sum[LK_WAVES];
    uint32_t pick[3];
    uint32_t key_max;
    int      slice_count[8];
    int      n_list;
    uint32_t fullest;         // not zero: a bucket is full; the second time its entries << 16 | its number
    uint32_t key_lo[2], key_hi[2];  // the range of its keys, twice
};

// The lane of wave 0 that holds bins 4 lane .. 4 lane + 3 of a 256-bin count finds the highest bin b with at least
// `want` entries in bins b .. 255. Returns true in the lane that found it, with the bin and the number of entries
// above it; false everywhere when there are fewer than `want` entries.
__device__ __forceinline__ bool largek_bin_of_rank(const uint32_t* hist, int lane, uint32_t want, uint32_t* bin,
                                                   uint32_t* above_out)
{
    const uint32_t c0 = hist[4 * lane], c1 = hist[4 * lane + 1], c2 = hist[4 * lane + 2], c3 = hist[4 * lane + 3];
    const uint32_t s    = c0 + c1 + c2 + c3;
    uint32_t       incl = s;  // entries in this lane's bins and in those of higher lanes
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        const uint32_t v = __shfl_down(incl, d, WAVE);
        if (lane + d < WAVE) {
            incl += v;
        }
    }
    const uint32_t above = incl - s;
    if (!(above < want && want <= incl)) {
        return false;
    }
    uint32_t run = above;
    if (run + c3 >= want) {
        *bin       = 4 * lane + 3;
        *above_out = run;
        return true;
    }
    run += c3;
    if (run + c2 >= want) {
        *bin       = 4 * lane + 2;
        *above_out = run;
        return true;
    }
    run += c2;
    if (run + c1 >= want) {
        *bin       = 4 * lane + 1;
        *above_out = run;
        return true;
    }
    run += c1;
    *bin       = 4 * lane;
    *above_out = run;
    return true;
}

// The list in ts.cand (256 < n <= TK_CCAP entries, all at or above thr_f, key_max the largest key) in the order of the
// reference, by all threads: stage 1 orders a slice by (value, thread, block), which gives every entry its rank in the
// slice, stage 2 the whole list by (value, what follows from slice and rank). Both need only neighbours of similar value:
// the entries are counted into 2048 buckets, put down bucket by bucket, and compared inside their bucket;
// what lies in higher buckets is a prefix sum (over all, and per slice). Weights and columns of the first min(k, n) go to
// ts.sel, padded with zeros to a multiple of 32. False, with ts.cand as it was, where a bucket stays crowded (many
// equal values) or a slice holds more than k entries.
// Bound by the latency of its barriers and by LDS: 5.6 us for 1400 entries, k = 1024, and 4.1 for the draw after it, two
// chains of 1024 dependent operations; selection and draw took 41 with the per-slice sorts and merges on four waves.
// AGAIN: a bucket holds a quarter of the list, or more than are compared, and all are counted once more, then in finer buckets. A
// function of its own, out of the way of other lists (inside the kernel it cost those 0.3 to 0.5 us). us a step of 64 x 50257, k =
// 1024, counted once / so: a column 3e4 ahead of the others f16 94.0 / 31.9, f32 94.1 / 32.4; 300 valid columns f16 53.4 / 28.6, f32
// 55.6 / 32.4; 800 f32 54.0 / 36.5; fp32 multiples of 0.25 78.4 / 80.1; ordinary rows f16 28.5 / 28.5, f32 29.2 / 29.2.
template<bool AGAIN>
__device__ __forceinline__ bool largek_order(TopkShared& ts, LargekShared& s, int n, int k, int max_top_k, float thr_f);
typedef __attribute__((address_space(3))) TopkShared*   TopkSharedPtr;  // (what is behind it is addressed as LDS in a call, too)
typedef __attribute__((address_space(3))) LargekShared* LargekSharedPtr;
__device__ __noinline__ bool largek_order_again(TopkSharedPtr ts, LargekSharedPtr s, int n, int k, int max_top_k, float thr_f)
{
    return largek_order<true>(*(TopkShared*)ts, *(LargekShared*)s, n, k, max_top_k, thr_f);
}

template<bool AGAIN>
__device__ __forceinline__ bool largek_order(TopkShared& ts, LargekShared& s, int n, int k, int max_top_k, float thr_f)
{
    const int   t       = threadIdx.x;
    const int   lane    = lane_id();
    const int   wv      = wave_id();
    const int   bs1_log = max_top_k <= 16 ? 7 : 8;
    const int   BS1     = 1 << bs1_log;
    const int   bs2_log = max_top_k <= 32 ? 7 : 8;
    const float x_max   = key_to_float(s.key_max);
    // 1 at the bound, 257 at the row's maximum: the bits of that number are close to its logarithm, which gives the dense
    // values near the bound most of the buckets, also where a single value lies ahead of all others
    float lo = thr_f, scale = 256.0f / (x_max - thr_f);
    if constexpr (AGAIN) {
        // (the bound may be the lowest value of the type: the limit keeps the quotient a normal number)
        scale = 256.0f / __builtin_fminf(x_max - thr_f, 1.0e30f);
        if (!(x_max < __builtin_inff() && scale < __builtin_inff())) {
            return false;
        }
        lds_barrier();
        s.count[2 * t]     = 0u;
        s.count[2 * t + 1] = 0u;
        if (t < 8) {
            s.slice_count[t] = 0;
        }
        if (t < 2) {
            s.key_lo[t] = 0xFFFFFFFFu;
            s.key_hi[t] = 0u;
        }
        if (t == 0) {
            s.fullest = 0u;
        }
        lds_barrier();
    }
    else if (!(scale > 0.0f && scale < __builtin_inff())) {
        return largek_order_again((TopkSharedPtr)&ts, (LargekSharedPtr)&s, n, k, max_top_k, thr_f);
    }
    auto bucket_of = [&](uint32_t key) -> int {  // (never falls as the value does)
        const float    x = (key_to_float(key) - lo) * scale + 1.0f;
        const uint32_t y = __float_as_uint(AGAIN ? __builtin_fmaxf(x, 1.0f) : x);
        return max(LK_BUCKETS - 1 - (int)((y - 0x3F800000u) >> 15), 0);
    };
    // lanes of the wave whose entry lies in the same slice
    auto same_slice = [&](bool have, int slice) -> unsigned long long {
        unsigned long long m = __ballot(have);
#pragma unroll
        for (int bit = 0; bit < 3; ++bit) {
            const unsigned long long b = __ballot((slice >> bit) & 1);
            m &= ((slice >> bit) & 1) ? b : ~b;
        }
        return m;
    };
    auto below_lane = [&](unsigned long long m) -> int {
        return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    };
    unsigned long long comp[2];  // slice(3) | ~key(32) | BS1-1-t (8) | j (21), column = (j*8 + slice)*BS1 + t
    int                bucket[2], slot[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int      i    = t + u * LK_THREADS;
        const bool     have = i < n;
        const uint32_t key = have ? ts.cand.key[i] : 0u, idx = have ? ts.cand.idx[i] : 0u;
        const int      blk = (int)(idx >> bs1_log), slice = blk & 7;
        comp[u] = ((unsigned long long)slice << 61) | ((unsigned long long)(~key) << 29)
                  | ((unsigned long long)(BS1 - 1 - (int)(idx & (uint32_t)(BS1 - 1))) << 21) | (unsigned long long)(blk >> 3);
        if constexpr (!AGAIN) {
            bucket[u] = have ? bucket_of(key) : 0;
            slot[u]   = have ? (int)atomicAdd(&s.count[bucket[u]], 1u) : 0;
        }
        const unsigned long long m = same_slice(have, slice);
        if (have && below_lane(m) == 0) {
            atomicAdd(&s.slice_count[slice], (int)__builtin_popcountll(m));
        }
    }
    auto key_of = [&](int u) -> uint32_t { return ~(uint32_t)(comp[u] >> 29); };
    const uint32_t full = (uint32_t)min(max(n >> 2, LK_BUCKET_FEW), LK_BUCKET_CAP);
    // the entries' buckets, and the entries in this thread's two buckets and all below them of the wave
    uint32_t c0, c1, incl;
    auto     count = [&]() {
        if constexpr (AGAIN) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const bool have = t + u * LK_THREADS < n;
                bucket[u]       = have ? bucket_of(key_of(u)) : 0;
                slot[u]         = have ? (int)atomicAdd(&s.count[bucket[u]], 1u) : 0;
            }
        }
        lds_barrier();
        c0   = s.count[2 * t];
        c1   = s.count[2 * t + 1];
        incl = c0 + c1;
#pragma unroll
        for (int d = 1; d < WAVE; d <<= 1) {
            const uint32_t v = __shfl_up(incl, d, WAVE);
            incl += lane >= d ? v : 0u;
        }
        if (lane == WAVE - 1) {
            s.wave_sum[wv] = incl;
        }
        const uint32_t most = max(c0, c1);
        if constexpr (AGAIN) {
            if (most > full) {
                atomicMax(&s.fullest, most << 16 | (uint32_t)(2 * t + (c0 == most ? 0 : 1)));
            }
        }
        else if (__ballot(most > full) != 0ull && lane == 0) {
            s.fullest = 1u;
        }
        lds_barrier();
    };
    count();
    if constexpr (AGAIN) {
#pragma unroll 1
        for (int round = 0; round < 2; ++round) {
            // The row's maximum is far ahead of the others, or the bound is the lowest value of the type (fewer than k valid
            // columns). Buckets for what the fullest one holds, with 1 to 17, about half of the buckets.
            const uint32_t fullest = s.fullest;
            if (fullest == 0u) {
                break;
            }
            uint32_t klo = 0xFFFFFFFFu, khi = 0u;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const bool in = t + u * LK_THREADS < n && bucket[u] == (int)(fullest & 0xFFFFu);
                klo           = min(klo, in ? key_of(u) : 0xFFFFFFFFu);
                khi           = max(khi, in ? key_of(u) : 0u);
            }
            klo = ~wave_max(~klo);
            khi = wave_max(khi);
            if (lane == 0 && khi != 0u) {
                atomicMin(&s.key_lo[round], klo);
                atomicMax(&s.key_hi[round], khi);
            }
            lds_barrier();
            const float from = key_to_float(s.key_lo[round]), to = key_to_float(s.key_hi[round]), finer = 16.0f / (to - from);
            // (not where its values are equal, or equal but for rounding: then finer buckets would crowd all others)
            if (!(finer > scale && to - from > __builtin_fabsf(to) * 0x1p-9f)) {
                break;
            }
            lo                 = from;
            scale              = finer;
            s.count[2 * t]     = 0u;
            s.count[2 * t + 1] = 0u;
            if (t == 0) {
                s.fullest = 0u;
            }
            lds_barrier();
            count();
        }
    }
    {  // bucket counts -> where each bucket starts
        const uint32_t sums  = s.wave_sum[lane & (LK_WAVES - 1)];
        uint32_t       start = incl - c0 - c1;
#pragma unroll
        for (int w = 0; w < LK_WAVES; ++w) {
            start += w < wv ? (uint32_t)__builtin_amdgcn_readlane((int)sums, w) : 0u;
        }
        s.count[2 * t]     = start;
        s.count[2 * t + 1] = start + c0;
        if (t == 0) {
            s.count[LK_BUCKETS] = (uint32_t)n;
        }
    }
    const uint32_t fullest    = s.fullest;
    bool           one_by_one = AGAIN && fullest >> 16 > (uint32_t)LK_BUCKET_CAP;
#pragma unroll
    for (int sl = 0; sl < 8; ++sl) {
        one_by_one = one_by_one || s.slice_count[sl] > k;
    }
    lds_barrier();
    if (one_by_one) {
        return false;
    }
    if (!AGAIN && fullest != 0u) {
        return largek_order_again((TopkSharedPtr)&ts, (LargekSharedPtr)&s, n, k, max_top_k, thr_f);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        if (t + u * LK_THREADS < n) {
            ts.keys[(int)s.count[bucket[u]] + slot[u]] = comp[u];  // (over ts.cand, which everybody has read)
        }
    }
    lds_barrier();
    // from here on a thread has positions t and t + 1024 of the list
    int first[2], last[2], rank[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int  at   = t + u * LK_THREADS;
        const bool have = at < n;
        comp[u]         = have ? ts.keys[at] : 0ull;
        const int b     = have ? bucket_of(~(uint32_t)(comp[u] >> 29)) : 0;
        first[u]        = have ? (int)s.count[b] : 0;
        last[u]         = have ? (int)s.count[b + 1] : 0;
        const int                slice = (int)(comp[u] >> 61);
        const unsigned long long m     = same_slice(have, slice);
        rank[u]                        = below_lane(m);
        if (have && rank[u] == 0) {
            s.chunk[u * LK_WAVES + wv][slice] = (uint32_t)__builtin_popcountll(m);
        }
    }
    lds_barrier();
    if (t < 256) {
        const uint32_t c    = s.chunk[t & 31][t >> 5];
        uint32_t       incl = c;
#pragma unroll
        for (int d = 1; d < 32; d <<= 1) {
            const uint32_t v = __shfl_up(incl, d, 32);
            incl += (t & 31) >= d ? v : 0u;
        }
        s.chunk[t & 31][t >> 5] = incl - c;
    }
    lds_barrier();
    unsigned long long c2[2];  // ~key(32) | BS2-1-pos%BS2 (8) | pos/BS2 (12) | 0 (12), pos = slice*k + rank in the slice
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int slice = (int)(comp[u] >> 61);
        int       r     = rank[u] + (int)s.chunk[u * LK_WAVES + wv][slice];  // entries of the slice in front of this one
        for (int j = first[u]; j < last[u]; ++j) {
            const unsigned long long o = ts.keys[j];
            if ((int)(o >> 61) == slice) {
                r += (o < comp[u] ? 1 : 0) - (j < t + u * LK_THREADS ? 1 : 0);
            }
        }
        const int pos = slice * k + r;
        c2[u]         = ((unsigned long long)(uint32_t)(comp[u] >> 29) << 32)
                | ((unsigned long long)((1 << bs2_log) - 1 - (pos & ((1 << bs2_log) - 1))) << 24)
                | ((unsigned long long)(pos >> bs2_log) << 12);
    }
    lds_barrier();
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        if (t + u * LK_THREADS < n) {
            ts.keys[t + u * LK_THREADS] = c2[u];
        }
    }
    lds_barrier();
    const int n_list = min(k, n);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        int q = first[u];
        for (int j = first[u]; j < last[u]; ++j) {
            q += ts.keys[j] < c2[u] ? 1 : 0;
        }
        if (t + u * LK_THREADS < n && q < n_list) {
            ts.sel.w[q]   = det_expf(key_to_float(~(uint32_t)(comp[u] >> 29)) - x_max);
            ts.sel.idx[q] = (((int)(comp[u] & 0x1FFFFFull) * 8 + (int)(comp[u] >> 61)) << bs1_log) + BS1 - 1
                            - (int)((comp[u] >> 21) & 0xFFull);
        }
    }
    if (n_list + t < ((n_list + 31) & ~31)) {
        ts.sel.w[n_list + t] = 0.0f;
    }
    lds_barrier();
    return true;
}

#ifdef FTK_LK_STAMPS  // development builds: wall-clock stamps of a row's phases
#define LK_STAMP(i) if (threadIdx.x == 0) { reinterpret_cast<unsigned long long*>(l.entries + (size_t)blockIdx.x * l.row_entries)[i] = wall_clock64(); }
#else
#define LK_STAMP(i)
#endif

template<int DT, int BMW>
__global__ void __launch_bounds__(LK_THREADS) largek_step_kernel(const RowwideArgs a)
{
    typedef Storage<DT>   S;
    typedef typename S::T T;
    constexpr int         EPV = (int)(16 / sizeof(T));
    static_assert(BMW > 0, "the history bitmap of the whole row lives in LDS");
    __shared__ LargekShared s;
    __shared__ TopkShared   ts;
    const FusedParams&      p    = a.p;
    const FusedLaunch&      l    = a.l;
    const int               t    = threadIdx.x;
    const int               lane = lane_id();
    const int               wv   = wave_id();
    const int               row  = blockIdx.x;
    const T*                rowp = (const T*)p.logits + (size_t)row * p.Vp;
    // the vectors start at the row's first 128-byte line; bit 0 of the history bitmap is `lead` columns in front of the
    // row, so that a vector's flags never straddle two words
    const int    head  = (int)((0ull - (unsigned long long)rowp) & 127ull) / (int)sizeof(T);
    const int    lead  = -head & 31;
    const uint4* base  = reinterpret_cast<const uint4*>(rowp + head);
    const int    nvec  = (p.V - head) / EPV;  // whole vectors inside columns [head, V)
    const int    turns = (nvec + LK_THREADS - 1) / LK_THREADS;
    const bool   skip  = row_flag_or(p.skip_decode, row, p.end_ids + row, false);
    const bool   fin   = row_flag_or(p.finished_in, row, p.end_ids + row, false);
    const int    k     = row_arg_or(p.top_ks, row, p.end_ids + row, p.max_top_k);
    const float  tp    = row_arg_or(p.top_ps, row, p.end_ids + row, 1.0f);
    const bool   hist  = p.bitmaps != nullptr && p.penalties != nullptr;
    int          ids[LK_HIST_U];
    auto         request_history = [&](int t0) {
#pragma unroll
        for (int u = 0; u < LK_HIST_U; ++u) {
            ids[u] = p.output_ids[(size_t)min(t0 + t + u * LK_THREADS, p.step - 1) * p.batch_size + row];
        }
    };
    if (hist) {
        request_history(0);
    }
    uint4 ring[LK_RING];
    // (every load is issued whatever the turn, one past the last fetches the last again, unused: with the same number
    // of loads on every path the waits can name the oldest load instead of everything in flight)
    auto vload = [&](int slot, int q) { ring[slot] = base[min(min(q, turns - 1) * LK_THREADS + t, nvec - 1)]; };
#pragma unroll
    for (int r = 0; r < LK_RING; ++r) {
        vload(r, r);
    }
    // the columns outside the vectors, one each: the first wave has those in front, the others those behind
    const int edge_v = t < WAVE ? (t < head ? t : p.V) : head + nvec * EPV + t - WAVE;
    T         edge   = (T)0;
    if (edge_v < p.V) {
        edge = rowp[edge_v];
    }
    FusedRow<DT, BMW> rowctx(p, row);
    TopkOutputs       out = topk_outputs(l.ids, l.sequence_length, l.finished, nullptr, nullptr, row, p.end_ids);
    LK_STAMP(0)
    if (skip || fin) {  // the row is skipped or has finished
        if (!skip && t == 0) {
            l.ids[row] = out.end_id_in;
        }
        return;
    }
    if (t == WAVE) {
        ts.misc[0] = __float_as_int(row_uniform(l.rng, l.uniforms, row));
    }
    for (int i = t; i < LK_BUCKETS; i += LK_THREADS) {
        s.count[i] = 0u;
    }
    if (t < 256) {
        s.hist[t]                   = 0u;
        (&s.chunk[0][0])[t] = 0u;
    }
    if (t < 8) {
        s.slice_count[t] = 0;
    }
    if (t == 0) {
        s.n_list  = 0;
        s.fullest = 0u;
        s.key_max = 0u;
    }
    uint32_t* window = fused_lds_bitmap<BMW>();
    if (hist) {
        const int words = min(BMW, (p.V + lead + 31) / 32 + 1);
        for (int i = t; i < words; i += LK_THREADS) {
            window[i] = 0u;
        }
        lds_barrier();
        for (int t0 = 0;;) {
#pragma unroll
            for (int u = 0; u < LK_HIST_U; ++u) {
                const int pos = t0 + t + u * LK_THREADS;
                if (pos < p.step && ids[u] >= 0 && ids[u] < p.V && rowctx.history_position_counts(pos)) {
                    atomicOr(&window[(ids[u] + lead) >> 5], 1u << ((ids[u] + lead) & 31));
                }
            }
            t0 += LK_HIST_U * LK_THREADS;
            if (t0 >= p.step) {
                break;
            }
            request_history(t0);
        }
        rowctx.bm_mode   = 1;
        rowctx.bm_origin = -lead;
    }
    lds_barrier();
    LK_STAMP(1)
    const float    mul     = rowctx.fast_mul;
    const bool     ordered = mul > 0.0f && mul < __builtin_inff();  // the plain transform keeps the order
    const float    NEG_INF = -__builtin_inff();
    const uint32_t KMIN    = min_valid_key<DT>();
    // history flags of the vector whose first column is `first`
    auto flags_of = [&](int first) -> uint32_t {
        const int bit = first + lead;  // (a multiple of EPV)
        return hist ? (window[bit >> 5] >> (bit & 31)) & ((1u << EPV) - 1u) : 0u;
    };
    // no column of the history, not the masked end id: one multiplication per column
    auto plain_vector = [&](int first) -> bool {
        return ordered && flags_of(first) == 0u && (uint32_t)(rowctx.masked_end_id - first) >= (uint32_t)EPV;
    };
    // the final values of a vector's columns; the masked end id counts as -MAX_T like in the reference
    auto values_of = [&](const uint4& v, int first, float* x) {
        const uint32_t bits = flags_of(first);
#pragma unroll
        for (int c = 0; c < EPV; ++c) {
            x[c] = rowctx.fast(vector_element<DT>(v, c));
        }
        if (bits != 0u) {
#pragma unroll
            for (int c = 0; c < EPV; ++c) {
                x[c] = (bits >> c) & 1u ? rowctx.flagged(x[c], first + c) : x[c];
            }
        }
#pragma unroll
        for (int c = 0; c < EPV; ++c) {
            x[c] = first + c == rowctx.masked_end_id ? -S::max_t() : x[c];
        }
    };
    const bool  has_edge = edge_v < p.V;
    const float edge_x   = has_edge ? rowctx.slow(edge_v, S::ld(edge), rowctx.vector_bits(edge_v, 1)) : NEG_INF;

    // ---- 1. three maxima per thread
    float g[LK_GROUPS];
#pragma unroll
    for (int i = 0; i < LK_GROUPS; ++i) {
        g[i] = NEG_INF;
    }
    g[LK_GROUPS - 1] = __builtin_fmaxf(NEG_INF, edge_x);
    auto first_pass  = [&](auto resident) {
        for (int q0 = 0; q0 < turns; q0 += LK_RING) {
            uint32_t again = 0u;
#pragma unroll
            for (int r = 0; r < LK_RING; ++r) {
                const int q = q0 + r;
                if (q < turns) {
                    const int   rel   = q * LK_THREADS + t;
                    const bool  plain = plain_vector(min(rel, nvec - 1) * EPV + head);
                    const float vm    = rowctx.fast(lean_raw_max<DT>(ring[r]));
                    g[r % LK_GROUPS]  = __builtin_fmaxf(g[r % LK_GROUPS], rel < nvec && plain ? vm : NEG_INF);
                    again |= rel < nvec && !plain ? 1u << r : 0u;
                }
                if constexpr (!decltype(resident)::value) {
                    vload(r, q + LK_RING);
                }
            }
            // few vectors: they are looked at again, column by column
            while (again != 0u) {
                const int r = __builtin_ctz(again);
                again &= again - 1u;
                const int rel = (q0 + r) * LK_THREADS + t;
                float     x[EPV];
                values_of(base[rel], rel * EPV + head, x);
                float vm = NEG_INF;
#pragma unroll
                for (int c = 0; c < EPV; ++c) {
                    vm = __builtin_fmaxf(vm, x[c]);
                }
#pragma unroll
                for (int i = 0; i < LK_GROUPS; ++i) {
                    g[i] = r % LK_GROUPS == i ? __builtin_fmaxf(g[i], vm) : g[i];
                }
            }
        }
    };
    const bool stays = turns <= LK_RING;
    if (stays) {
        first_pass(std::true_type());
    }
    else {
        first_pass(std::false_type());
        // (the second read's first vectors are requested now: they arrive while the bound is worked out)
#pragma unroll
        for (int r = 0; r < LK_RING; ++r) {
            vload(r, r);
        }
    }
    LK_STAMP(2)

    // ---- 2. the bound: the top byte of the k-th largest key, then its second byte among the keys that share the first
    uint32_t key[LK_GROUPS];
#pragma unroll
    for (int i = 0; i < LK_GROUPS; ++i) {
        key[i] = order_key(g[i]);
        // (nearly all top bytes of a wave are the same one or two: one atomic per value, not per lane)
        unsigned long long left = ~0ull;
        while (left != 0ull) {
            const int                leader = __builtin_ctzll(left);
            const uint32_t           byte   = (uint32_t)__builtin_amdgcn_readlane((int)(key[i] >> 24), leader);
            const unsigned long long m      = __ballot((key[i] >> 24) == byte);
            if (lane == leader) {
                atomicAdd(&s.hist[byte], (uint32_t)__builtin_popcountll(m));
            }
            left &= ~m;
        }
    }
    {
        const uint32_t top = wave_max(max(key[0], max(key[1], key[2])));
        if (lane == 0) {
            atomicMax(&s.key_max, top);
        }
    }
    lds_barrier();
    if (wv == 0) {
        uint32_t   bin = 0u, above = 0u;
        const bool mine = largek_bin_of_rank(s.hist, lane, (uint32_t)k, &bin, &above);
        if (__ballot(mine) == 0ull) {
            if (lane == 0) {
                s.pick[0] = 0xFFFFFFFFu;  // (fewer than k maxima at all: there are 3/2 k vectors)
            }
        }
        else if (mine) {
            s.pick[0] = bin;
            s.pick[1] = (uint32_t)k - above;  // rank inside the bin
        }
        // (the first wave alone has read the counts: it clears them for the second round)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s.hist[4 * lane + i] = 0u;
        }
    }
    lds_barrier();
    const uint32_t top_byte = s.pick[0];
    const uint32_t want     = s.pick[1];
#pragma unroll
    for (int i = 0; i < LK_GROUPS; ++i) {
        if ((key[i] >> 24) == top_byte) {
            atomicAdd(&s.hist[(key[i] >> 16) & 255u], 1u);
        }
    }
    lds_barrier();
    if (wv == 0) {
        uint32_t   bin = 0u, above = 0u;
        const bool mine = top_byte != 0xFFFFFFFFu && largek_bin_of_rank(s.hist, lane, want, &bin, &above);
        if (__ballot(mine) == 0ull) {
            if (lane == 0) {
                s.pick[2] = 0u;
            }
        }
        else if (mine) {
            s.pick[2] = (top_byte << 24) | (bin << 16);
        }
    }
    lds_barrier();
    LK_STAMP(3)
    const uint32_t P     = s.pick[2];
    uint32_t       thr   = P >= KMIN ? P : KMIN;  // (P >= KMIN: at least k columns with a valid value at or above it)
    float          thr_f = key_to_float(thr);     // x >= thr_f  <=>  order_key(x) >= thr (a NaN fails both)

    // ---- 3. what reaches the bound goes to the list
    auto second_pass = [&](auto resident) {
        for (int q0 = 0; q0 < turns; q0 += LK_RING) {
            int n_noted = 0;  // (the same in every lane)
#pragma unroll
            for (int r = 0; r < LK_RING; ++r) {
                const int q = q0 + r;
                if (q < turns) {
                    const int  rel   = q * LK_THREADS + t;
                    const bool plain = plain_vector(min(rel, nvec - 1) * EPV + head);
                    // (a plain vector whose largest element stays under the bound holds no candidate)
                    const bool hit = rel < nvec && (!plain || rowctx.fast(lean_raw_max<DT>(ring[r])) >= thr_f);
                    const unsigned long long m = __ballot(hit);
                    if (hit) {
                        s.noted[wv][n_noted + (int)__builtin_amdgcn_mbcnt_hi(
                                        (uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] = rel;
                    }
                    n_noted += (int)__builtin_popcountll(m);
                }
                if constexpr (!decltype(resident)::value) {
                    vload(r, q + LK_RING);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
            // one noted vector per lane, from the caches, the next round's requested ahead
            int   rel_next = lane < n_noted ? s.noted[wv][lane] : 0;
            uint4 v_next   = base[rel_next];
            for (int e0 = 0; e0 < n_noted; e0 += WAVE) {
                const int   rel   = rel_next;
                const uint4 v     = v_next;
                const bool  have  = e0 + lane < n_noted;
                const int   first = rel * EPV + head;
                rel_next          = e0 + WAVE + lane < n_noted ? s.noted[wv][e0 + WAVE + lane] : 0;
                v_next            = base[rel_next];
                float x[EPV];
                values_of(v, first, x);
                uint32_t hit = 0u;
#pragma unroll
                for (int c = 0; c < EPV; ++c) {
                    hit |= have && x[c] >= thr_f && first + c != rowctx.masked_end_id ? 1u << c : 0u;
                }
                const int cnt = __builtin_popcount(hit);
                int       pre = 0, total = 0;
#pragma unroll
                for (int bit = 0; (1 << bit) <= EPV; ++bit) {
                    const unsigned long long bm = __ballot((cnt >> bit) & 1);
                    pre += (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32),
                                                          __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u))
                           << bit;
                    total += (int)__builtin_popcountll(bm) << bit;
                }
                if (total > 0) {
                    int slot = 0;
                    if (lane == 0) {
                        slot = atomicAdd(&s.n_list, total);
                    }
                    slot = __builtin_amdgcn_readfirstlane(slot) + pre;
#pragma unroll
                    for (int c = 0; c < EPV; ++c) {
                        if ((hit >> c) & 1u) {
                            if (slot < TK_CCAP) {
                                ts.cand.key[slot] = order_key(x[c]);
                                ts.cand.idx[slot] = (uint32_t)(first + c);
                            }
                            ++slot;
                        }
                    }
                }
            }
            __builtin_amdgcn_wave_barrier();  // (the notes have been read before the next ones are written)
        }
    };
    if (stays) {
        second_pass(std::true_type());
    }
    else {
        second_pass(std::false_type());
    }
    if (has_edge && edge_x >= thr_f && edge_v != rowctx.masked_end_id) {
        const int slot = atomicAdd(&s.n_list, 1);
        if (slot < TK_CCAP) {
            ts.cand.key[slot] = order_key(edge_x);
            ts.cand.idx[slot] = (uint32_t)edge_v;
        }
    }
    LK_STAMP(4)
    lds_barrier();
    LK_STAMP(5)
    if (s.n_list > TK_CCAP) {
        // The maxima were no measure of the columns (most of the row masked, the best columns side by side): the k-th largest
        // key to within its low sixteen bits out of all columns, then the list again.
        uint32_t prefix = 0u, rank = (uint32_t)k;
        auto     count  = [&](float x, int round) {
            const uint32_t kx = order_key(x);
            if (x >= key_to_float(KMIN) && (round == 0 || kx >> 24 == prefix)) {
                atomicAdd(&s.hist[round == 0 ? kx >> 24 : (kx >> 16) & 255u], 1u);
            }
        };
        for (int round = 0; round < 2; ++round) {
            if (t < 256) {
                s.hist[t] = 0u;
            }
            lds_barrier();
            for (int rel = t; rel < nvec; rel += LK_THREADS) {
                float x[EPV];
                values_of(base[rel], rel * EPV + head, x);
#pragma unroll
                for (int c = 0; c < EPV; ++c) {
                    count(x[c], round);
                }
            }
            if (has_edge) {
                count(edge_x, round);
            }
            lds_barrier();
            if (wv == 0) {
                uint32_t   bin = 0u, above = 0u;
                const bool mine = largek_bin_of_rank(s.hist, lane, rank, &bin, &above);
                if (__ballot(mine) == 0ull) {
                    if (lane == 0) {
                        s.pick[0] = 0xFFFFFFFFu;  // fewer than k valid columns: all of them are candidates
                    }
                }
                else if (mine) {
                    s.pick[0] = bin;
                    s.pick[1] = rank - above;
                }
                s.n_list = 0;
            }
            lds_barrier();
            if (s.pick[0] == 0xFFFFFFFFu) {
                prefix = 0u;
                break;
            }
            prefix = round == 0 ? s.pick[0] : prefix << 24 | s.pick[0] << 16;
            rank   = s.pick[1];
        }
        thr        = prefix >= KMIN ? prefix : KMIN;
        thr_f      = key_to_float(thr);
        auto again = [&](float x, int v) {
            if (x >= thr_f && v != rowctx.masked_end_id) {
                const int slot = atomicAdd(&s.n_list, 1);
                if (slot < TK_CCAP) {
                    ts.cand.key[slot] = order_key(x);
                    ts.cand.idx[slot] = (uint32_t)v;
                }
            }
        };
        for (int rel = t; rel < nvec; rel += LK_THREADS) {
            float x[EPV];
            values_of(base[rel], rel * EPV + head, x);
#pragma unroll
            for (int c = 0; c < EPV; ++c) {
                again(x[c], rel * EPV + head + c);
            }
        }
        if (has_edge) {
            again(edge_x, edge_v);
        }
        lds_barrier();
    }

    // ---- 4. the selection
    const int   n       = s.n_list;
    const float u       = __int_as_float(ts.misc[0]);
    const bool  ordered_list = n > 256 && n <= TK_CCAP && largek_order<false>(ts, s, n, k, p.max_top_k, thr_f);
    if (ordered_list) {
        LK_STAMP(6)
        if (t == 0) {
            float     s_sum;
            const int pick = topk_sample_walk(ts.sel.w, min(k, n), u, tp, &s_sum);
            topk_emit(out, row, ts.sel.idx[pick], false, 0.0f, 0.0f, p.end_ids, true);
        }
        LK_STAMP(7)
        return;
    }
    if (wv >= TK_WAVES) {
        return;  // the first four waves, one per SIMD, do the rest
    }
    if (n <= 256) {
        const int n_list = topk_rank_few<DT>(ts, n, k, p.max_top_k);
        topk_finish_list<DT>(ts, n_list, row, p.Vp, tp, false, u, p.end_ids, out);
    }
    else {
        rowwide_rare<DT>(ts, (RowwideArgSegment)__builtin_amdgcn_kernarg_segment_ptr(), row, n, thr, k, tp, u, nullptr);
    }
}

// Launchers, one translation unit per element type (lean_kernels.hip). window: 1 = small LDS window, 2 = large.
int largek_launch_f32(int window, int rows, hipStream_t st, const FusedParams& p, const FusedLaunch& l, hipEvent_t start,
                      hipEvent_t stop);
int largek_launch_f16(int window, int rows, hipStream_t st, const FusedParams& p, const FusedLaunch& l, hipEvent_t start,
                      hipEvent_t stop);
int largek_launch_bf16(int window, int rows, hipStream_t st, const FusedParams& p, const FusedLaunch& l, hipEvent_t start,
                       hipEvent_t stop);

}  // namespace ftk
