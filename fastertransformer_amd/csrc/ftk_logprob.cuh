// Fused decode step for rows of the top-k layer when cum_log_probs / output_log_probs are requested.
//
// The reference then turns the penalised logits into probabilities over the whole row before it samples
// (src/fastertransformer/layers/sampling_layers/TopKSamplingLayer.cu:220-266: invokeAddBiasSoftMax, then the
// top-k kernels on probabilities, whose log-prob outputs are log p and log p - log S). Its kernel sequence
// moves the row nine times (temperature R+W, penalties, softmax 3R+3W, top-k k+2 R). Here the row is read
// twice and never written. Both reads apply temperature, history penalty and the min-length mask in registers:
//   1. the exact maximum of the row;
//   2. e_v = T(exp(y_v - max)) summed in the order of the reference's softmax
//      (sampling_topp_kernels.cu:1308-1344: thread t of 1024 adds columns t, t + 1024, ... one after the other;
//      reduce_kernel_utils.cuh:73-103: xor butterflies 16..1 inside 32-lane groups, then over the 32 group sums),
//      so the sum has the reference's bits. The candidates of the top-k selection are gathered by e_v,
//      with a bound lowered by what the division and rounding to T can merge, so that every column whose
//      probability ties with the k-th largest is among them. The candidates' e_v then become probabilities
//      T(e_v / (sum + 1e-6)), the reference's tie orders are replayed on them and the row is sampled
//      (topk_select_lds with probabilities in). Rows it cannot bound take the literal replay on probabilities
//      computed on the fly.
// Three forms:
//   lp_wide_kernel - the product's: one launch, one workgroup of 1024, 512 or 256 threads per row does both reads
//                    (the second one comes from the caches), a thread owning 1, 2 or 4 whole summation chains;
//   lp_short_kernel (ftk_logprob_short.cuh) - the product's for short rows: the same, column by column;
//   lp_rowmax_kernel + lp_row_kernel - two launches: the first streams the row in the launch shape of the lean
//                    gather and leaves the maximum of every workgroup's share in the workspace, the second gives
//                    a row to one 256-thread workgroup whose threads own four neighbouring chains each and walk
//                    them with 16-byte (fp32) or 8-byte (16-bit types) loads that are 1024 columns apart. The test
//                    build of the library can select it; the forms must agree bit for bit.
// Preconditions (checked by the host, which otherwise reports FTK_ERR_UNSUPPORTED and the layer runs the kernel
// sequence): no embedding bias, largest k <= 128, vocabulary >= 1024 (the reference's block is min(V, 1024)
// threads). Rows may have any pitch and start on any element boundary: vector loads are the aligned vectors of the
// memory, and the few columns of the first one that lie in front of the row are masked or looked at one by one.
#pragma once
#include <type_traits>

#include "ftk_exp16.cuh"
#include "ftk_lean.cuh"

namespace ftk {

constexpr int LP_THREADS = 256;
constexpr int LP_CHAINS  = 4;     // neighbouring summation chains per thread
constexpr int LP_BLOCK   = 1024;  // chains per row: the reference's block size
constexpr int LP_RING    = 8;     // loads in flight per thread
constexpr int LP_HEAD    = 4;     // rounds examined before the first bound exists
static_assert(LP_THREADS * LP_CHAINS == LP_BLOCK, "a workgroup owns all chains of its row");

struct LogProbLaunch {
    float* cum_log_probs;     // [rows] or null
    float* output_log_probs;  // [rows] or null
    float* partial_max;       // [rows][splits]
    int    splits;            // workgroups per row of lp_rowmax_kernel
};

// The exact value of the largest element of a 16-byte vector whose first element is column `first` (`a` columns of
// the row's first vector lie in front of the row): plain vectors through their raw maximum (rounding to T and a
// positive multiplier keep the order), the others element by element.
template<int DT, int BMW>
__device__ __forceinline__ float lp_vector_max(const FusedRow<DT, BMW>& rowctx, const uint4& v, int first, int a,
                                               bool bitsv, bool ordered)
{
    typedef Storage<DT> S;
    constexpr int       EPV  = (int)(16 / sizeof(typename S::T));
    uint32_t            bits = 0u;
    if (bitsv) {
        if (BMW > 0 && a == 0) {  // the flags of a vector never straddle a word of the bitmap
            const int rel = first - rowctx.bm_origin;
            bits          = (rowctx.bm_word(rel >> 5) >> (rel & 31)) & ((1u << EPV) - 1u);
        }
        else {
            bits = rowctx.vector_bits(first, EPV);
        }
    }
    const uint32_t rel_end = (uint32_t)(rowctx.masked_end_id - first);
    if (bits == 0u && rel_end >= (uint32_t)EPV && ordered) {
        return rowctx.fast(lean_raw_max<DT>(v));
    }
    float vm = -__builtin_inff();
#pragma unroll
    for (int c = 0; c < EPV; ++c) {
        float x = rowctx.fast(vector_element<DT>(v, c));
        if ((bits >> c) & 1u) {
            x = rowctx.flagged(x, first + c);
        }
        if ((uint32_t)c == rel_end) {
            x = -S::max_t();
        }
        vm = __builtin_fmaxf(vm, x);
    }
    return vm;
}

// ---- pass 1 --------------------------------------------------------------------------------------------
template<int DT, int BMW>
__global__ void __launch_bounds__(LG_THREADS, LG_OCCUPANCY) lp_rowmax_kernel(FusedParams p, FusedLaunch l, LogProbLaunch lp)
{
    typedef Storage<DT>   S;
    typedef typename S::T T;
    constexpr int         EPV = (int)(16 / sizeof(T));
    constexpr int         R   = LG_RING;
    __shared__ float      red[LG_WAVES];
    const int             t     = threadIdx.x;
    const int             row   = blockIdx.y;
    const int             chunk = blockIdx.x;
    // Rows may start anywhere: the 16-byte vectors are those of the memory, `a` columns of the first one lie in
    // front of the row. Vectors [vlo, vhi) lie inside columns [0, V); the first and the last workgroup of a row
    // look at the few columns in front of and behind them one by one.
    const T*              rowp  = (const T*)p.logits + (size_t)row * p.Vp;
    const int             a     = (int)(((uintptr_t)rowp & 15u) / sizeof(T));
    const uint4*          base  = reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(rowp) - a * sizeof(T));
    const int             vlo   = (a + EPV - 1) / EPV;
    const int             vhi   = max(vlo, (a + p.V) / EPV);
    const int             vb    = min(vhi, vlo + chunk * l.subs_per_wg * LG_SUB_VECS);
    const int             ve    = min(vhi, vb + l.subs_per_wg * LG_SUB_VECS);
    const int             nvec  = ve - vb;
    const int             nsub  = (nvec + LG_SUB_VECS - 1) / LG_SUB_VECS;

    const bool hist = BMW > 0 && p.bitmaps != nullptr && p.penalties != nullptr;
    int        hist_ids[LG_HIST_U];
    if (hist) {
#pragma unroll
        for (int u = 0; u < LG_HIST_U; ++u) {
            const int pos = t + u * LG_THREADS;
            hist_ids[u]   = pos < p.step ? p.output_ids[(size_t)pos * p.batch_size + row] : -1;
        }
    }
    uint4 raw[R][LG_NV];
    auto  load = [&](int slot, int q) {
#pragma unroll
        for (int j = 0; j < LG_NV; ++j) {
            const int vi = min(vb + q * LG_SUB_VECS + j * LG_THREADS + t, ve - 1);
            raw[slot][j] = stream_load(base + vi);
        }
    };
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (r < nsub) {
            load(r, r);
        }
    }
    const bool        skip = row_flag_or(p.skip_decode, row, p.end_ids + row, false);
    const bool        fin  = row_flag_or(p.finished_in, row, p.end_ids + row, false);
    FusedRow<DT, BMW> rowctx(p, row);
    if (skip || fin) {
        return;
    }
    const bool first_wg = chunk == 0;
    const bool last_wg  = chunk == (int)gridDim.x - 1;
    const int  lo_col   = first_wg ? 0 : vb * EPV - a;
    const int  hi_col   = last_wg ? p.V : ve * EPV - a;
    if (hist) {
        uint32_t* window = fused_lds_bitmap<FusedRow<DT, BMW>::LDS_WORDS>();
        const int origin = lo_col & ~31;
        const int words  = min(FusedRow<DT, BMW>::LDS_WORDS, (hi_col - origin + 31) / 32 + 1);
        for (int i = t; i < words; i += LG_THREADS) {
            window[i] = 0u;
        }
        lds_barrier();
        auto mark = [&](int pos, int id) {
            if (id >= lo_col && id < hi_col && rowctx.history_position_counts(pos)) {
                atomicOr(&window[(id - origin) >> 5], 1u << ((id - origin) & 31));
            }
        };
#pragma unroll
        for (int u = 0; u < LG_HIST_U; ++u) {
            mark(t + u * LG_THREADS, hist_ids[u]);
        }
        for (int pos = t + LG_HIST_U * LG_THREADS; pos < p.step; pos += LG_THREADS) {
            mark(pos, p.output_ids[(size_t)pos * p.batch_size + row]);
        }
        rowctx.bm_mode   = 1;
        rowctx.bm_origin = origin;
    }
    lds_barrier();
    const bool  bitsv   = rowctx.has_vector_bits();
    const float mul     = rowctx.fast_mul;
    const bool  ordered = mul > 0.0f && mul < __builtin_inff();  // the plain transform keeps the order
    const float NEG_INF = -__builtin_inff();
    float       m       = NEG_INF;
    auto vector_max = [&](const uint4& v, int first) -> float {
        return lp_vector_max<DT, BMW>(rowctx, v, first, a, bitsv, ordered);
    };
    for (int q0 = 0; q0 < nsub; q0 += R) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int q = q0 + r;
            if (q < nsub) {
#pragma unroll
                for (int j = 0; j < LG_NV; ++j) {
                    const int   rel = q * LG_SUB_VECS + j * LG_THREADS + t;
                    const float vm  = vector_max(raw[r][j], (vb + min(rel, nvec - 1)) * EPV - a);
                    m               = __builtin_fmaxf(m, rel < nvec ? vm : NEG_INF);
                }
                if (q + R < nsub) {
                    load(r, q + R);
                }
            }
        }
    }
    if (first_wg) {
        // the columns in front of the first whole vector
        for (int v = t; v < min(p.V, vlo * EPV - a); v += LG_THREADS) {
            m = __builtin_fmaxf(m, topk_value_at<DT>(rowctx, v));
        }
    }
    if (last_wg) {
        // the columns behind the last whole vector
        for (int v = vhi * EPV - a + t; v < p.V; v += LG_THREADS) {
            m = __builtin_fmaxf(m, topk_value_at<DT>(rowctx, v));
        }
    }
    m = wave_max(m);
    if (lane_id() == 0) {
        red[wave_id()] = m;
    }
    lds_barrier();
    if (t == 0) {
        float r = red[0];
#pragma unroll
        for (int w = 1; w < LG_WAVES; ++w) {
            r = __builtin_fmaxf(r, red[w]);
        }
        lp.partial_max[(size_t)row * lp.splits + chunk] = r;
    }
}

// ---- pass 2 --------------------------------------------------------------------------------------------
// Row accessor of the recovery paths: the key of column v is that of its probability.
template<int DT>
struct ProbRow {
    typedef Storage<DT>       S;
    typedef typename S::T     T;
    FusedRow<DT, 0>*          base;
    float                     row_max;
    float                     denom;  // sum + 1e-6
    static constexpr int      IN_FLIGHT = 1;
    __device__ __forceinline__ void prepare_whole_row()
    {
        base->prepare_whole_row();
    }
    __device__ __forceinline__ float prob_of(float y) const
    {
        const float e = round_t<DT>(det_expf(y - row_max));
        return round_t<DT>(e / denom);
    }
    __device__ __forceinline__ uint32_t key_at(int v) const
    {
        const uint32_t bit = base->bm_mode != 0 ? base->vector_bits(v, 1) : 0u;
        return order_key(prob_of(base->slow(v, S::ld(base->rowp[v]), bit)));
    }
};

// element c of a thread's chunk (four neighbouring columns) as fp32
template<int DT>
__device__ __forceinline__ float lp_chunk_element(const uint4& v, int c)
{
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    return __uint_as_float(w[c]);
}
template<int DT>
__device__ __forceinline__ float lp_chunk_element(const uint2& v, int c)
{
    const uint32_t w[2] = {v.x, v.y};
    return Storage<DT>::ld((uint16_t)(c & 1 ? w[c >> 1] >> 16 : w[c >> 1] & 0xFFFFu));
}

// Ties after the division: two e values give the same probability T(e / denom) only if they differ by less than
// a unit in the last place of that probability times denom. While the k-th largest probability is a normal
// number of T that is at most 2^-(mantissa bits - 1) of e (four half-units, to be safe): candidates are gathered
// down to e_bound * (1 - LP_TIE_REL). When it is subnormal the unit no longer shrinks with the value; binary16 rows
// with one likely token get there with ordinary k (a probability below 6e-5). The unit is then 2^-24, so candidates
// are gathered LP_TIE_DENOM units and a quarter below the bound, which is enough for denominators up to LP_TIE_DENOM
// (a row whose k-th probability is that small has most of its mass in a few columns, whose e are at most 1). Rows
// that neither rule covers are gathered again with the denominator at hand (topk_regather).
template<int DT>
__device__ __forceinline__ float lp_tie_rel()
{
    return DT == DT_F32 ? 2.384185791015625e-07f : (DT == DT_F16 ? 0.001953125f : 0.015625f);
}
template<int DT>
__device__ __forceinline__ bool lp_ties_bounded(float e_bound, float denom)
{
    const float smallest_normal = DT == DT_F16 ? 6.103515625e-05f : 1.17549435e-38f;
    return e_bound >= 2.0f * smallest_normal * denom;
}
constexpr float LP_TIE_DENOM = 8.0f;
constexpr float LP_TIE_UNIT  = 5.9604644775390625e-08f;  // 2^-24, binary16's smallest number
// where gathering stops, given a value of e that at least k columns reach
template<int DT>
__device__ __forceinline__ float lp_gather_floor(float e_bound)
{
    const float low = e_bound - e_bound * lp_tie_rel<DT>();
    if (DT == DT_F16 && !lp_ties_bounded<DT>(e_bound, LP_TIE_DENOM)) {
        return __builtin_fminf(low, __builtin_fmaxf(e_bound - 1.25f * LP_TIE_UNIT * LP_TIE_DENOM, LP_TIE_UNIT));
    }
    return low;
}
// whether everything that ties with the k-th largest probability was gathered
template<int DT>
__device__ __forceinline__ bool lp_gather_covers(float e_bound, float denom)
{
    return lp_ties_bounded<DT>(e_bound, denom)
           || (DT == DT_F16 && denom <= LP_TIE_DENOM && e_bound >= 2.5f * LP_TIE_UNIT * LP_TIE_DENOM);
}

// The end of a row, by TK_THREADS threads: the n candidates in s.cand carry e = T(exp(y - max)) as their keys (`probs`:
// T(e / denom) already); they become probabilities, the list is cut to little more than k entries and the reference's
// tie orders are replayed on probabilities (topk_select_lds), which also samples and writes the row's outputs. `slot` is
// scratch for TK_THREADS keys. n < 0: the literal replay. `equal`: see topk_rank_few.
template<int DT>
__device__ __forceinline__ void lp_finish(TopkShared& s, uint32_t* slot, int n, bool probs, float denom, float row_max,
                                          int k, float tp, float u, const FusedParams& p, const FusedLaunch& l, int row,
                                          const TopkOutputs& out, bool equal = false)
{
    const int      t    = threadIdx.x;
    const uint32_t KMIN = min_valid_key<DT>();
    if (n >= 0) {
        // ---- candidates: e -> probability
        if (!probs) {
            for (int i = t; i < n; i += TK_THREADS) {
                s.cand.key[i] = order_key(round_t<DT>(key_to_float(s.cand.key[i]) / denom));
            }
            lds_barrier();
        }
        if (n > k + k / 2 && n <= 4 * TK_THREADS) {
            // keep what reaches the k-th largest of 256 slot maxima (at least k candidates do, and everything
            // that ties with the k-th largest probability does)
            uint32_t mx = 0u;
            for (int i = t; i < n; i += TK_THREADS) {
                const uint32_t key = s.cand.key[i];
                mx                 = key > mx ? key : mx;
            }
            slot[t] = mx;
            lds_barrier();
            const uint32_t P = lean_kth_of_slots(slot, k);
            lds_barrier();
            if (P > KMIN) {
                n = topk_prune(s, n, P);
            }
        }
    }
    FusedRow<DT, 0> r0(p, row);
    r0.team = TK_THREADS;  // (the workgroup may have had more threads: those have left)
    ProbRow<DT>     prow{&r0, row_max, denom};
    topk_select_lds<DT, ProbRow<DT>, true>(prow, s, n, KMIN, row, p.Vp, k, tp, p.max_top_k,
                                           l.entries + (size_t)row * l.row_entries, true, u, p.end_ids, out, equal);
}

// Whether an fp32 row looks like values of a 16-bit type, which nearly always leave equal values among the candidates: the
// last thirteen bits of the first wave's first vectors are zero. Left in s.misc[3], which nothing else uses, for lp_finish.
// (us a step of bfloat16 values, without / with: 8 x 50257, k = 64, 23.5 / 22.5; 64 x 8000 17.5 / 16.1; 256 x 128256 51.0 / 49.6;
// of whole numbers 32.8 / 29.4, 22.4 / 19.6 and 59.2 / 56.0; other rows as before)
template<int DT>
__device__ __forceinline__ void lp_note_equal(TopkShared& s, const uint4& first)
{
    if constexpr (DT == DT_F32) {
        if (wave_id() == 0) {
            const unsigned long long fine = __ballot(((first.x | first.y | first.z | first.w) & 0x1FFFu) != 0u);
            if (lane_id() == 0) {
                s.misc[3] = fine == 0ull ? 1 : 0;
            }
        }
    }
}

template<int DT, int BMW>
__global__ void __launch_bounds__(LP_THREADS) lp_row_kernel(FusedParams p, FusedLaunch l, LogProbLaunch lp)
{
    typedef Storage<DT>   S;
    typedef typename S::T T;
    // a thread's load: LP_CHAINS neighbouring columns
    typedef typename std::conditional<sizeof(T) == 4, uint4, uint2>::type Chunk;
    // The row's history bitmap lives in LDS that nothing else uses while the row streams: the ordered-list area
    // of the select phase holds its first words, an array behind the select state the rest (four workgroups then
    // fit a compute unit even with the window of the largest vocabularies). Both are addressed as words of one
    // object, so that the choice between them is a choice between two uniform offsets.
    constexpr int LP_BM_OVERLAY = (int)(sizeof(TopkShared::sel) / sizeof(uint32_t));
    constexpr int LP_BM_TAIL    = BMW > LP_BM_OVERLAY ? BMW - LP_BM_OVERLAY : 1;
    struct LpShared {
        TopkShared s;
        uint32_t   bitmap_tail[LP_BM_TAIL];
    };
    static_assert(sizeof(TopkShared) % sizeof(uint32_t) == 0 && offsetof(LpShared, bitmap_tail) == sizeof(TopkShared),
                  "the tail follows the select state word for word");
    static_assert(LP_BM_OVERLAY % (LP_BLOCK / 32) == 0, "a round's bitmap words lie on one side of the seam");
    constexpr int LP_BM_HEAD_AT = (int)(offsetof(TopkShared, sel) / sizeof(uint32_t));
    constexpr int LP_BM_TAIL_AT = (int)(sizeof(TopkShared) / sizeof(uint32_t)) - LP_BM_OVERLAY;
    __shared__ LpShared   sh;
    TopkShared&           s = sh.s;
    __shared__ uint32_t   slot_key[2][LP_THREADS];
    __shared__ float      warp_sum[32];
    const int             t   = threadIdx.x;
    const int             row = blockIdx.x;
    // Rows may start anywhere: the chunks are those of the memory, `a` columns of the first one lie in front of
    // the row. Slot c of thread t then holds column n * LP_BLOCK + 4 t + c - a in round n, always of the same
    // summation chain (4 t + c - a modulo LP_BLOCK) and in ascending order; the chains are put back in their
    // places before they are added up.
    const T*              rowp = (const T*)p.logits + (size_t)row * p.Vp;
    const int             a    = (int)(((uintptr_t)rowp % sizeof(Chunk)) / sizeof(T));
    const Chunk*          base = reinterpret_cast<const Chunk*>(reinterpret_cast<const char*>(rowp) - a * sizeof(T));
    const int             rounds = (p.V + a + LP_BLOCK - 1) / LP_BLOCK;  // columns outside [0, V) are masked: e = 0 exactly

    // history first, then the first loads of the row, then the arguments
    const bool hist = BMW > 0 && p.bitmaps != nullptr && p.penalties != nullptr;
    int        hist_ids[LG_HIST_U];
    if (hist) {
#pragma unroll
        for (int u = 0; u < LG_HIST_U; ++u) {
            const int pos = t + u * LP_THREADS;
            hist_ids[u]   = pos < p.step ? p.output_ids[(size_t)pos * p.batch_size + row] : -1;
        }
    }
    Chunk        raw[LP_RING];
    const int    tcol  = t * LP_CHAINS;  // the thread's first column within a round
    const Chunk* tbase = base + t;
    // the last round may reach past the row: such a thread reads its chunk of the round before (never used).
    // A chunk of the memory that starts in front of the padded row's end holds at least one of its elements.
    const bool last_inside = (rounds - 1) * LP_BLOCK + tcol < a + p.Vp;
    // Every load is issued whatever the round (one past the row's end fetches the last round's chunk again, unused):
    // with the same number of loads on every path the waits can name the oldest load instead of all of them.
    auto load = [&](int slot, int n) {
        const int m = min(n, rounds - 1);
        raw[slot]   = tbase[(size_t)((m + 1 < rounds || last_inside) ? m : m - 1) * LP_THREADS];
    };
#pragma unroll
    for (int r = 0; r < LP_RING; ++r) {
        load(r, r);
    }
    const bool        skip = row_flag_or(p.skip_decode, row, p.end_ids + row, false);
    const bool        fin  = row_flag_or(l.finished, row, p.end_ids + row, false);
    const int         k    = row_arg_or(p.top_ks, row, p.end_ids + row, p.max_top_k);
    const float       tp   = row_arg_or(p.top_ps, row, p.end_ids + row, 1.0f);
    FusedRow<DT, BMW> rowctx(p, row);
    if (skip) {
        return;
    }
    if (fin) {
        if (t == 0) {
            l.ids[row] = p.end_ids[row];  // a finished row emits its end id: no draw, no log-prob, no length update
        }
        return;
    }
    int draw_bits = 0;
    if (t == 0) {
        draw_bits = __float_as_int(row_uniform(l.rng, l.uniforms, row));
    }
    const TopkOutputs out =
        topk_outputs(l.ids, l.sequence_length, l.finished, lp.cum_log_probs, lp.output_log_probs, row, p.end_ids);
    // the row's maximum: pass 1 left one per workgroup; pad columns count as -MAX_T
    float row_max = -3.402823466e+38f;
    for (int c = 0; c < lp.splits; ++c) {
        row_max = __builtin_fmaxf(row_max, lp.partial_max[(size_t)row * lp.splits + c]);
    }
    if (p.V < p.Vp) {
        row_max = __builtin_fmaxf(row_max, -S::max_t());
    }
    row_max = uniform_f(row_max);
    if (t == 0) {
        s.n_cand  = 0;
        s.misc[0] = draw_bits;
    }
    uint32_t* const lds_words = reinterpret_cast<uint32_t*>(&sh);
    auto            bitmap_at = [&](int w) { return (w < LP_BM_OVERLAY ? LP_BM_HEAD_AT : LP_BM_TAIL_AT) + w; };
    if (hist) {
        const int words = min(BMW, (p.V + 31) / 32 + 1);
        for (int i = t; i < words; i += LP_THREADS) {
            lds_words[bitmap_at(i)] = 0u;
        }
        lds_barrier();
        auto mark = [&](int pos, int id) {
            if (id >= 0 && id < p.V && rowctx.history_position_counts(pos)) {
                const int w = id >> 5;
                atomicOr(&lds_words[bitmap_at(w)], 1u << (id & 31));
            }
        };
#pragma unroll
        for (int u = 0; u < LG_HIST_U; ++u) {
            mark(t + u * LP_THREADS, hist_ids[u]);
        }
        for (int pos = t + LG_HIST_U * LP_THREADS; pos < p.step; pos += LP_THREADS) {
            mark(pos, p.output_ids[(size_t)pos * p.batch_size + row]);
        }
    }
    lds_barrier();
    const float u     = __int_as_float(s.misc[0]);
    const bool  bitsv = hist || rowctx.has_vector_bits();
    const uint32_t KMIN = min_valid_key<DT>();

    // e values of the LP_CHAINS columns of round n that a chunk holds; columns >= V give 0. What depends on the
    // round alone (the side of the bitmap seam, whether the round holds the masked end id or the end of the
    // vocabulary) is decided in scalar registers.
    auto e_values = [&](const Chunk& v, int n, float* e) {
        const int col  = n * LP_BLOCK + tcol - a;
        uint32_t  bits = 0u;
        if (bitsv) {
            if constexpr (BMW > 0) {
                if (a == 0) {
                    const int at = (n < LP_BM_OVERLAY / (LP_BLOCK / 32) ? LP_BM_HEAD_AT : LP_BM_TAIL_AT) + n * (LP_BLOCK / 32);
                    bits         = (lds_words[at + (tcol >> 5)] >> (tcol & 31)) & ((1u << LP_CHAINS) - 1u);
                }
                else if (col >= 0) {
                    // the four flags may straddle two words (the bitmap carries one word of slack)
                    const int sh = col & 31;
                    bits         = lds_words[bitmap_at(col >> 5)] >> sh;
                    if (sh + LP_CHAINS > 32) {
                        bits |= lds_words[bitmap_at((col >> 5) + 1)] << (32 - sh);
                    }
                    bits &= (1u << LP_CHAINS) - 1u;
                }
                else {
                    bits = (lds_words[bitmap_at(0)] << (-col)) & ((1u << LP_CHAINS) - 1u);  // columns 0 .. at slots -col ..
                }
            }
            else {
                bits = rowctx.vector_bits(col, LP_CHAINS);
            }
        }
        float y[LP_CHAINS];
#pragma unroll
        for (int c = 0; c < LP_CHAINS; ++c) {
            y[c] = rowctx.fast(lp_chunk_element<DT>(v, c));
        }
        // rare: a column of the history, the masked end id, the end of the vocabulary
        const bool     edge_round = (n + 1) * LP_BLOCK - a > p.V || (a != 0 && n == 0);
        const bool     end_round  = (uint32_t)(rowctx.masked_end_id - (n * LP_BLOCK - a)) < (uint32_t)LP_BLOCK;
        const uint32_t rel_end    = (uint32_t)(rowctx.masked_end_id - col);
        bool           rare       = bits != 0u;
        if (edge_round || end_round) {
            rare = rare || rel_end < (uint32_t)LP_CHAINS || col + LP_CHAINS > p.V || col < 0;
        }
        if (rare) {
#pragma unroll
            for (int c = 0; c < LP_CHAINS; ++c) {
                if ((bits >> c) & 1u) {
                    y[c] = rowctx.flagged(y[c], col + c);
                }
                if ((uint32_t)c == rel_end || (uint32_t)(col + c) >= (uint32_t)p.V) {
                    y[c] = -S::max_t();
                }
            }
        }
        float d[LP_CHAINS];
#pragma unroll
        for (int c = 0; c < LP_CHAINS; ++c) {
            d[c] = y[c] - row_max;
        }
        // one look for a NaN per chunk instead of one per column
        if (__builtin_isunordered(d[0], d[1]) || __builtin_isunordered(d[2], d[3])) {
#pragma unroll
            for (int c = 0; c < LP_CHAINS; ++c) {
                e[c] = round_t<DT>(det_expf_nonpos(d[c]));
            }
        }
        else {
#pragma unroll
            for (int c = 0; c < LP_CHAINS; ++c) {
                e[c] = round_t<DT>(det_expf_nonpos_number(d[c]));
            }
        }
        if (edge_round && (col + LP_CHAINS > p.V || col < 0)) {
#pragma unroll
            for (int c = 0; c < LP_CHAINS; ++c) {
                e[c] = (uint32_t)(col + c) < (uint32_t)p.V ? e[c] : 0.0f;  // (what lies outside the row adds nothing)
            }
        }
    };

    float    acc[LP_CHAINS] = {0.0f, 0.0f, 0.0f, 0.0f};  // the chains' running sums
    uint32_t thr            = KMIN;                      // candidates: e with key >= thr_low
    float    thr_low        = key_to_float(KMIN);
    uint32_t dmax           = 0u;  // largest key this thread has put on the list
    bool     valid          = false;
    int      par            = 0;
    auto     set_threshold  = [&](uint32_t key) {
        thr           = key;
        const float e = key_to_float(key);
        thr_low       = uniform_f(lp_gather_floor<DT>(e));
    };
    auto push = [&](float e, int col) {
        const uint32_t key  = order_key(e);
        const int      slot = atomicAdd(&s.n_cand, 1);
        if (slot < TK_CCAP) {
            s.cand.key[slot] = key;
            s.cand.idx[slot] = (uint32_t)col;
        }
        dmax = key > dmax ? key : dmax;
    };
    auto rebound = [&](uint32_t mine) {
        slot_key[par][t] = mine;
        lds_barrier();
        const uint32_t P = lean_kth_of_slots(slot_key[par], k);
        par ^= 1;
        if (P > thr && P > order_key(0.0f)) {  // at least k columns with e > 0 at or above it
            set_threshold(P);
            valid = true;
        }
    };

    // ---- head: the first rounds are summed and kept; their largest e per thread gives the first bound
    float head_e[LP_HEAD][LP_CHAINS];
    const int head = min(rounds, LP_HEAD);
    {
        float tmax = 0.0f;
#pragma unroll
        for (int n = 0; n < LP_HEAD; ++n) {
            if (n < head) {
                e_values(raw[n], n, head_e[n]);
#pragma unroll
                for (int c = 0; c < LP_CHAINS; ++c) {
                    acc[c] = acc[c] + head_e[n][c];
                    tmax   = __builtin_fmaxf(tmax, head_e[n][c]);
                }
            }
            load(n, n + LP_RING);
        }
        rebound(order_key(tmax));
#pragma unroll
        for (int n = 0; n < LP_HEAD; ++n) {
            if (n < head) {
#pragma unroll
                for (int c = 0; c < LP_CHAINS; ++c) {
                    const int col = n * LP_BLOCK + tcol + c - a;
                    if (head_e[n][c] >= thr_low && (uint32_t)col < (uint32_t)p.V) {
                        push(head_e[n][c], col);
                    }
                }
            }
        }
    }
    // ---- the rest of the row; the bound is raised again after 8, 16, 32, ... rounds
    static_assert(LP_RING % LP_HEAD == 0 && LP_RING > LP_HEAD, "the ring continues where the head stopped");
    int  next_tighten = 2 * LP_HEAD;
    auto one_round    = [&](int slot, int n) {
        float     e[LP_CHAINS];
        const int col0 = n * LP_BLOCK + tcol - a;
        e_values(raw[slot], n, e);
#pragma unroll
        for (int c = 0; c < LP_CHAINS; ++c) {
            acc[c] = acc[c] + e[c];
        }
        // one look per chunk for a candidate (a NaN is none, with or without the maximum)
        if (__builtin_fmaxf(__builtin_fmaxf(e[0], e[1]), __builtin_fmaxf(e[2], e[3])) >= thr_low) {
#pragma unroll
            for (int c = 0; c < LP_CHAINS; ++c) {
                if (e[c] >= thr_low && (uint32_t)(col0 + c) < (uint32_t)p.V) {
                    push(e[c], col0 + c);
                }
            }
        }
    };
    auto tighten = [&](int n) {
        if (n + 1 == next_tighten && n + 1 < rounds) {
            next_tighten *= 2;
            rebound(dmax);
        }
    };
    int n0 = LP_HEAD;
    // whole groups of LP_RING rounds: no guards, every slot is loaded again
    for (; n0 + LP_RING <= rounds; n0 += LP_RING) {
#pragma unroll
        for (int r = 0; r < LP_RING; ++r) {
            const int slot = (LP_HEAD + r) % LP_RING;
            one_round(slot, n0 + r);
            load(slot, n0 + r + LP_RING);
            tighten(n0 + r);
        }
    }
    // the last rounds (fewer than LP_RING): their chunks are on their way or here
#pragma unroll
    for (int r = 0; r < LP_RING - 1; ++r) {
        if (n0 + r < rounds) {
            one_round((LP_HEAD + r) % LP_RING, n0 + r);
            tighten(n0 + r);
        }
    }
    if (a != 0) {
        // chain 4 t + c - a (modulo LP_BLOCK) back to slot c of thread t; the bitmap's first words are done with
        float* chain = reinterpret_cast<float*>(lds_words + LP_BM_HEAD_AT);
        static_assert(sizeof(TopkShared::sel) >= LP_BLOCK * sizeof(float), "one float per chain");
        __syncthreads();
#pragma unroll
        for (int c = 0; c < LP_CHAINS; ++c) {
            chain[(tcol + c - a) & (LP_BLOCK - 1)] = acc[c];
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < LP_CHAINS; ++c) {
            acc[c] = chain[tcol + c];
        }
    }
    // ---- the sum, in the reference's order: chain t = 4 * thread + c; butterflies with masks 16, 8, 4 run
    // between the eight threads of a 32-chain group, masks 2 and 1 inside a thread
#pragma unroll
    for (int o = 4; o >= 1; o >>= 1) {
#pragma unroll
        for (int c = 0; c < LP_CHAINS; ++c) {
            acc[c] = acc[c] + __shfl_xor(acc[c], o, WAVE);
        }
    }
    acc[0] = acc[0] + acc[2];
    acc[1] = acc[1] + acc[3];
    acc[0] = acc[0] + acc[1];
    if ((t & 7) == 0) {
        warp_sum[t >> 3] = acc[0];
    }
    __syncthreads();
    float total = t < 32 ? warp_sum[t] : 0.0f;
    if (t < WAVE) {
#pragma unroll
        for (int o = 16; o >= 1; o >>= 1) {
            total = total + __shfl_xor(total, o, WAVE);
        }
        if (t == 0) {
            warp_sum[0] = total;
        }
    }
    __syncthreads();
    const float denom = uniform_f(warp_sum[0] + 1e-6f);
    const int   n     = s.n_cand;
    __syncthreads();
    const bool trusted = n <= TK_CCAP && valid && lp_gather_covers<DT>(key_to_float(thr), denom);
    lp_finish<DT>(s, slot_key[par], trusted ? n : -1, false, denom, row_max, k, tp, u, p, l, row, out);
}

// ---- one launch: a workgroup per row reads it twice ---------------------------------------------------------------
// With few rows lp_row_kernel's four waves per row are what bounds the step (about a microsecond per 1024 columns),
// and most compute units idle. Here THREADS threads share a row, thread t owning 1024 / THREADS neighbouring summation
// chains of the reference's 1024, so the sum has the reference's order without any regrouping. First pass: the row's
// maximum after temperature, penalties and masks, and every thread's own largest value, from which the bound of the
// candidates follows (the k-th largest of 256 joined thread maxima, each of them a column of its own). Second pass (the
// row comes from the caches this time): e = T(exp(y - max)) summed chain by chain, of fp32 rows with the candidates on the
// way; those of 16-bit rows are looked for afterwards, in the few groups of vectors whose largest raw value reaches the
// bound. Then all waves but four leave and those finish like lp_row_kernel (lp_finish).
// THREADS = 1024 for launches of at most one row per compute unit; with more rows, workgroups of fewer threads share a
// compute unit and one's first pass (memory) runs beside another's second (arithmetic).
constexpr int LPW_THREADS = 1024;

#ifdef FTK_LP_STAMPS  // development builds: wall-clock stamps of a row's phases in its candidate list area
#define LPW_STAMP(i) if (threadIdx.x == 0) { reinterpret_cast<unsigned long long*>(l.entries + (size_t)blockIdx.x * l.row_entries)[i] = wall_clock64(); }
#else
#define LPW_STAMP(i)
#endif

// Whether any lane of the wave has it, in a branch that the whole wave takes: what it leads to is out of the way of the
// straight line (a branch for some lanes would be jumped over by all others, at the cost of a fetch).
__device__ __forceinline__ bool lp_rare(bool mine)
{
    return __builtin_expect(__ballot(mine) != 0ull, 0);
}

// Bound by the arithmetic of the second pass (vector instructions, and its waits where only eight waves share a compute
// unit). 1024 x 152064 f16, k = 64: 166 us a step with every column through det_expf, columns one by one and candidates
// looked for in both passes; 141 us now. 16-bit types hold their values in pairs and take det_expf only where the
// hardware's exponential leaves the rounding open (ftk_exp16.cuh), the first pass looks at raw values alone, 16-bit candidates
// are looked for in some ninety groups of 64 columns, and flags of the history cost a bit test per sixteen columns. Other
// sizes, us before / now: 256 x 152064 f16 53.7 / 48.7, 512 x 50257 f16 51.9 / 45.2, 1024 x 32000 bf16 56.6 / 43.5, 256 x
// 128256 f16 with 2000 ids of history 70.8 / 58.1, 8 x 50257 f32 24.0 / 22.9, 400 x 152064 f32 89.2 / 85.8, 1024 x 152064
// f32 203 / 199.
template<int DT, int BMW, int THREADS>
__global__ void __launch_bounds__(THREADS) lp_wide_kernel(FusedParams p, FusedLaunch l, LogProbLaunch lp)
{
    typedef Storage<DT>   S;
    typedef typename S::T T;
    constexpr bool        WORD16 = DT != DT_F32;
    constexpr int         CH = LP_BLOCK / THREADS;     // neighbouring chains of a thread
    constexpr int         N  = WORD16 ? 16 : 8;        // columns of a thread's batch
    constexpr int         U  = N / CH;                 // ... in rounds of 1024 columns
    // Candidates are gathered on the way of the sum: two more operations per four columns. fp32 rows looked at again after the
    // sum are out of the second-level cache by then (us a step, again / on the way: 8 x 50257 23.1 / 22.9, 256 x 128256
    // 50.4 / 48.5, 400 x 152064 87.2 / 85.8, 512 x 152064 113.6 / 107.5, 2048 x 50257 150.5 / 140.2, 1024 x 152064 212 / 199).
    constexpr bool        IN_SUM = !WORD16;
    constexpr int         NR = WORD16 && CH > 1 ? N / 2 : N;  // registers a batch is loaded into
    constexpr int         NY = WORD16 ? N / 2 : N;            // ... and its values, 16-bit types in pairs
    static_assert(THREADS * CH == LP_BLOCK && U * CH == N && THREADS % 32 == 0 && THREADS >= TK_THREADS,
                  "a workgroup owns all chains of its row");
    typedef std::conditional_t<WORD16 && CH == 1, uint16_t, uint32_t> Raw;
    typedef std::conditional_t<WORD16, uint32_t, float>               Val;
    __shared__ TopkShared s;
    __shared__ uint32_t   wide_key[THREADS];
    __shared__ uint32_t   slot_key[TK_THREADS];
    __shared__ float      warp_sum[32];
    __shared__ float      redf[THREADS / WAVE];
    const int             t    = threadIdx.x;
    // The last rows first: whatever produced the logits wrote them shortly before this launch, and of a batch that is
    // larger than the last-level cache the rows written last are the ones still in it.
    const int             row  = (int)gridDim.x - 1 - (int)blockIdx.x;
    const T*              rowp = (const T*)p.logits + (size_t)row * p.Vp;
    // A workgroup that shares its compute unit with others is served first while it waits for memory more than it
    // computes (set-up, first pass, selection): its few instructions then do not queue behind the arithmetic of a
    // neighbour's second pass, and its loads stay in flight.
    if constexpr (THREADS < LPW_THREADS) {
        __builtin_amdgcn_s_setprio(3);
    }
    // slot j of a batch: round j / CH of the batch, chain CH * t + j % CH
    auto offset_of = [](int j) { return (j / CH) * LP_BLOCK + j % CH; };
    // First pass, for the maximum only: the order of the columns does not matter, so the row comes in as the 16-byte
    // vectors of the memory, thread t taking vectors vlo + t, vlo + t + THREADS, ... (`a` columns of the row's first
    // vector lie in front of the row; what lies in front of vector vlo and behind vector vhi is looked at column by
    // column). The first vectors are on their way before anything else is read.
    constexpr int EPV   = (int)(16 / sizeof(T));
    constexpr int R1    = 8;  // vectors a thread keeps in flight
    const int     a     = (int)(((uintptr_t)rowp & 15u) / sizeof(T));
    const uint4*  base  = reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(rowp) - a * sizeof(T));
    const int     vlo   = (a + EPV - 1) / EPV;
    const int     vhi   = max(vlo + 1, (a + p.V) / EPV);  // (a row has at least 1024 columns)
    const int     nvec  = vhi - vlo;
    const int     turns = (nvec + THREADS - 1) / THREADS;
    // (the history before them: its ids are scattered reads that nothing should queue behind)
    constexpr int HU   = 2048 / THREADS;
    const bool    hist = p.bitmaps != nullptr && p.penalties != nullptr;
    int           hist_ids[HU];
    T             hist_raw[HU];
    if (hist) {
#pragma unroll
        for (int i = 0; i < HU; ++i) {
            const int pos = t + i * THREADS;
            hist_ids[i]   = pos < p.step ? p.output_ids[(size_t)pos * p.batch_size + row] : -1;
        }
    }
    uint4         ring[R1];
    // (every load is issued whatever the turn, one past the last fetches the last again, unused: with the same number
    // of loads on every path the waits can name the oldest load instead of everything in flight)
    auto vload = [&](int slot, int q) { ring[slot] = base[vlo + min(min(q, turns - 1) * THREADS + t, nvec - 1)]; };
#pragma unroll
    for (int r = 0; r < R1; ++r) {
        vload(r, r);
    }
    // Second pass: thread t takes columns of its own chains, batches of N
    const int nfull = p.V / (U * LP_BLOCK);  // batches that every thread holds in full
    constexpr int R2 = WORD16 && CH > 1 ? 4 : 2;  // batches in registers, the one in use included
    Raw       buf[R2][NR];
    auto      load = [&](Raw* raw, int b) {
#pragma unroll
        for (int r = 0; r < U; ++r) {
            __builtin_memcpy(raw + r * (NR / U), rowp + (b * U + r) * LP_BLOCK + CH * t, CH * sizeof(T));
        }
    };
    const bool            skip = row_flag_or(p.skip_decode, row, p.end_ids + row, false);
    const bool            fin  = row_flag_or(l.finished, row, p.end_ids + row, false);
    const int             k    = row_arg_or(p.top_ks, row, p.end_ids + row, p.max_top_k);
    const float           tp   = row_arg_or(p.top_ps, row, p.end_ids + row, 1.0f);
    FusedRow<DT, BMW>     rowctx(p, row);
    LPW_STAMP(0)
    if (skip) {
        return;
    }
    if (fin) {
        if (t == 0) {
            l.ids[row] = p.end_ids[row];  // a finished row emits its end id: no draw, no log-prob, no length update
        }
        return;
    }
    if (t == 0) {
        s.n_cand  = 0;
        s.misc[1] = 0;  // groups of vectors kept in mind
    }
    const TopkOutputs out =
        topk_outputs(l.ids, l.sequence_length, l.finished, lp.cum_log_probs, lp.output_log_probs, row, p.end_ids);
    // (the first and last columns of a row, outside its whole vectors, are nobody's: at >= 0 && at < nvec fails)
    uint32_t own_flags = 0u;  // bit b % 32: a column of the thread's batch b has a value of its own
    auto     flag_of   = [&](int v) { return 1u << ((v / (U * LP_BLOCK)) & 31); };
    auto     owner_of  = [&](int v) { return (v & (LP_BLOCK - 1)) / CH; };
    if (hist) {
        // which columns of the row are in its history: a bitmap in LDS (launches with a window; others have one in
        // memory), and per thread which of its batches hold one
        wide_key[t] = 0u;
        if constexpr (BMW > 0) {
            uint32_t* window = fused_lds_bitmap<FusedRow<DT, BMW>::LDS_WORDS>();
            const int words  = min(FusedRow<DT, BMW>::LDS_WORDS, (p.V + 31) / 32 + 1);
            for (int i = t; i < words; i += THREADS) {
                window[i] = 0u;
            }
            rowctx.bm_mode   = 1;
            rowctx.bm_origin = 0;
        }
        __syncthreads();
        auto mark = [&](int pos, int id) {
            id -= p.col_offset;
            if (id >= 0 && id < p.V && rowctx.history_position_counts(pos)) {
                if constexpr (BMW > 0) {
                    atomicOr(&fused_lds_bitmap<FusedRow<DT, BMW>::LDS_WORDS>()[id >> 5], 1u << (id & 31));
                }
                atomicOr(&wide_key[owner_of(id)], flag_of(id));
            }
        };
#pragma unroll
        for (int i = 0; i < HU; ++i) {
            if (hist_ids[i] >= 0) {
                mark(t + i * THREADS, hist_ids[i]);
            }
        }
        for (int pos = t + HU * THREADS; pos < p.step; pos += THREADS) {
            mark(pos, p.output_ids[(size_t)pos * p.batch_size + row]);
        }
#pragma unroll
        for (int i = 0; i < HU; ++i) {  // what the columns of the history hold, for the maximum
            hist_raw[i] = rowp[min(max(hist_ids[i] - p.col_offset, 0), p.V - 1)];
        }
    }
    __syncthreads();
    if (hist) {
        own_flags = wide_key[t];
    }
    if (rowctx.masked_end_id >= 0 && rowctx.masked_end_id < p.V && owner_of(rowctx.masked_end_id) == t) {
        own_flags |= flag_of(rowctx.masked_end_id);
    }
    // visit(v, raw) for the columns of the history and the masked end id, by whichever thread
    auto for_special = [&](auto&& visit) {
        if (hist) {
#pragma unroll
            for (int i = 0; i < HU; ++i) {
                const int id = hist_ids[i] - p.col_offset;
                if (hist_ids[i] >= 0 && id >= 0 && id < p.V && rowctx.history_position_counts(t + i * THREADS)) {
                    visit(id, hist_raw[i]);
                }
            }
#pragma unroll 1
            for (int pos = t + HU * THREADS; pos < p.step; pos += THREADS) {
                const int id = p.output_ids[(size_t)pos * p.batch_size + row] - p.col_offset;
                if (id >= 0 && id < p.V && rowctx.history_position_counts(pos)) {
                    visit(id, rowp[id]);
                }
            }
        }
        if (t == 0 && rowctx.masked_end_id >= 0 && rowctx.masked_end_id < p.V) {
            visit(rowctx.masked_end_id, rowp[rowctx.masked_end_id]);
        }
    };
    LPW_STAMP(1)
    const uint32_t KMIN    = min_valid_key<DT>();
    const float    NEG_INF = -__builtin_inff();
    // The values of a batch's columns (v0 = the first one) after temperature, history penalty and the min-length mask.
    // Batches without a flag need no more than the multiplication. `whole`: all columns lie in the row.
    const bool bitsv = rowctx.has_vector_bits();
    auto values = [&](auto whole, int v0, const Raw* raw, Val* y) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NY; ++i) {
            if constexpr (!WORD16) {
                y[i] = rowctx.fast(u2f(raw[i]));
            }
            else {
                uint32_t pair;
                if constexpr (CH == 1) {
                    pair = (uint32_t)raw[2 * i] | ((uint32_t)raw[2 * i + 1] << 16);
                }
                else {
                    pair = raw[i];
                }
                y[i] = ExpPairs<DT>::times(pair, rowctx.fast_mul);
            }
        }
        if (lp_rare((own_flags & flag_of(v0)) != 0u)) {
            const uint32_t to_end = (uint32_t)(rowctx.masked_end_id - v0);  // offset_of(j) for the masked end id at slot j
            const int      bsh    = v0 & 31;  // (a thread's columns of a round are neighbouring bits of one word)
            uint32_t       special, flags = 0u;
            if (bitsv) {
#pragma unroll
                for (int r = 0; r < U; ++r) {
                    const int at = (v0 >> 5) + r * (LP_BLOCK / 32);
                    flags |= ((rowctx.bm_word(decltype(whole)::value ? at : min(at, p.V >> 5)) >> bsh) & ((1u << CH) - 1u))
                             << (r * CH);
                }
            }
            special = flags;
#pragma unroll
            for (int j = 0; j < N; ++j) {
                special |= to_end == (uint32_t)offset_of(j) ? 1u << j : 0u;
            }
            while (special != 0u) {  // (a slot per lane and turn: one or two turns as a rule)
                const int j = __builtin_ctz(special), v = v0 + offset_of(j);
                special &= special - 1u;
                if constexpr (!WORD16) {
                    float x = register_pick<N>(y, j);
                    x       = (flags >> j) & 1u ? rowctx.flagged(x, v) : x;
                    x       = to_end == (uint32_t)offset_of(j) ? -S::max_t() : x;
#pragma unroll
                    for (int i = 0; i < N; ++i) {
                        y[i] = i == j ? x : y[i];
                    }
                }
                else {
                    const uint32_t pair  = register_pick<NY>(y, j >> 1);
                    const int      shift = 16 * (j & 1);
                    float          x     = S::ld((T)(pair >> shift));
                    x                    = (flags >> j) & 1u ? rowctx.flagged(x, v) : x;
                    x                    = to_end == (uint32_t)offset_of(j) ? -S::max_t() : x;
                    const uint32_t other = (pair & (0xFFFF0000u >> shift)) | ((uint32_t)S::st(x) << shift);
#pragma unroll
                    for (int i = 0; i < NY; ++i) {
                        y[i] = i == j >> 1 ? other : y[i];
                    }
                }
            }
        }
    };
    // the same for one column
    auto value = [&](int v, T raw) -> float {
        float y = rowctx.fast(S::ld(raw));
        if (bitsv && ((rowctx.bm_word(v >> 5) >> (v & 31)) & 1u)) {
            y = rowctx.flagged(y, v);
        }
        return v == rowctx.masked_end_id ? -S::max_t() : y;
    };
    // The values of any batch of the row, -inf behind its end.
    auto some_values = [&](int v0, Val* y) __attribute__((always_inline)) {
        Raw raw[NR];
#pragma unroll
        for (int r = 0; r < U; ++r) {
            T         one[CH];
            const int v = v0 + r * LP_BLOCK;
            __builtin_memcpy(one, rowp + min(v, p.V - CH), CH * sizeof(T));
            if (CH > 1 && v < p.V && v + CH > p.V) {  // (one thread at most)
#pragma unroll
                for (int c = 0; c < CH; ++c) {
                    one[c] = rowp[min(v + c, p.V - 1)];
                }
            }
            __builtin_memcpy(raw + r * (NR / U), one, CH * sizeof(T));
        }
        values(std::false_type(), v0, raw, y);
#pragma unroll
        for (int j = 0; j < N; ++j) {
            if (v0 + offset_of(j) >= p.V) {
                if constexpr (!WORD16) {
                    y[j] = NEG_INF;
                }
                else {
                    const uint32_t none = S::st(NEG_INF);
                    y[j / 2] = j % 2 == 0 ? (y[j / 2] & 0xFFFF0000u) | none : (y[j / 2] & 0xFFFFu) | (none << 16);
                }
            }
        }
    };
    // The second pass over the row: whole batches with the next one's loads issued before the current one is used,
    // then the columns behind them in a batch that ends with -inf. use_batch(v0, y, rounds) takes a batch's values, as
    // many rounds of them as there are.
    auto stream = [&](auto&& use_batch) {
        if (nfull > 0) {
#pragma unroll
            for (int r = 0; r < R2 - 1; ++r) {
                load(buf[r], min(r, nfull - 1));
            }
        }
        // (every load is issued whatever the batch, one past the last fetches the last again, unused: with the same
        // number of loads on every path the waits can name the older batch instead of everything in flight)
        for (int b0 = 0; b0 < nfull; b0 += R2) {
#pragma unroll
            for (int r = 0; r < R2; ++r) {
                load(buf[(r + R2 - 1) % R2], min(b0 + r + R2 - 1, nfull - 1));
                if (b0 + r < nfull) {
                    Val       y[NY];
                    const int v0 = (b0 + r) * U * LP_BLOCK + CH * t;
                    values(std::true_type(), v0, buf[r], y);
                    use_batch(v0, y, U);
                }
            }
        }
        const int rest = p.V - nfull * U * LP_BLOCK;
        if (rest > 0) {
            Val       y[NY];
            const int v0 = nfull * U * LP_BLOCK + CH * t;
            some_values(v0, y);
            use_batch(v0, y, (rest + LP_BLOCK - 1) / LP_BLOCK);
        }
    };

    lp_note_equal<DT>(s, ring[0]);
    // ---- first pass: the maximum (pad columns count as -MAX_T), and the thread's own
    // The plain transform keeps the order, so a thread's maximum is that of its raw values - columns of the history and
    // the masked end id apart, which have values of their own. Looking for them vector by vector costs more than the
    // maximum itself; instead every history id looks whether its raw value is the largest of the thread that owns its
    // column. Such a thread says nothing about its columns (nothing follows for the candidates' bound), unless its raw
    // maximum lies above everything else: then a wave goes through its vectors with the flags at hand.
    // 16-bit types: the maxima of groups of a thread's vectors stay behind in the candidates' array: once the bound is there
    // they tell which groups to look into for candidates.
    constexpr int GROUPS = 2 * TK_CCAP / THREADS;  // per thread
    const float   mul     = rowctx.fast_mul;
    const bool    ordered = mul > 0.0f && mul < __builtin_inff();  // the plain transform keeps the order
    int           glog    = 3;                                     // log2 of the turns of a group
    while ((GROUPS << glog) < turns) {
        ++glog;
    }
    float* group_max = reinterpret_cast<float*>(&s.cand);  // [group][thread]
    static_assert(sizeof(s.cand) >= GROUPS * THREADS * sizeof(float) && R1 == 8, "a group is a whole number of rings");
    float m       = NEG_INF;
    float raw_own = NEG_INF;
    if (ordered) {
        typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
        float group = NEG_INF;
        auto  ring_of = [&](auto last, int q0) {  // `last`: not every thread has all of these vectors
            const _Float16 low  = -__builtin_inff16();
            f16x2          pair = {low, low};
            float          most = NEG_INF;
#pragma unroll
            for (int r = 0; r < R1; ++r) {
                if (!decltype(last)::value || (q0 + r) * THREADS + t < nvec) {
                    const uint4& v = ring[r];
                    if constexpr (DT == DT_F16) {
                        const f16x2 x = __builtin_bit_cast(f16x2, v.x), y = __builtin_bit_cast(f16x2, v.y);
                        const f16x2 z = __builtin_bit_cast(f16x2, v.z), w = __builtin_bit_cast(f16x2, v.w);
                        pair = __builtin_elementwise_max(
                            __builtin_elementwise_max(pair, __builtin_elementwise_max(x, y)),
                            __builtin_elementwise_max(z, w));
                    }
                    else {
                        most = __builtin_fmaxf(most, lean_raw_max<DT>(v));
                    }
                }
                vload(r, q0 + r + R1);
            }
            if constexpr (DT == DT_F16) {
                most = __builtin_fmaxf((float)pair.x, (float)pair.y);
            }
            group   = __builtin_fmaxf(group, most);
            raw_own = __builtin_fmaxf(raw_own, most);
            if (!IN_SUM && (((q0 + R1) & ((1 << glog) - 1)) == 0 || q0 + R1 >= turns)) {
                group_max[(q0 >> glog) * THREADS + t] = group;
                group                                 = NEG_INF;
            }
        };
        int q0 = 0;
        for (; (q0 + R1) * THREADS <= nvec; q0 += R1) {
            ring_of(std::false_type(), q0);
        }
        if (q0 < turns) {
            ring_of(std::true_type(), q0);
        }
    }
    else {
        for (int q0 = 0; q0 < turns; q0 += R1) {
#pragma unroll
            for (int r = 0; r < R1; ++r) {
                const int rel = (q0 + r) * THREADS + t;
                if (q0 + r < turns) {
                    const float vm = lp_vector_max<DT, BMW>(rowctx, ring[r], (vlo + min(rel, nvec - 1)) * EPV - a, a,
                                                            bitsv, ordered);
                    m              = __builtin_fmaxf(m, rel < nvec ? vm : NEG_INF);
                }
                vload(r, q0 + r + R1);
            }
        }
    }
    // the columns in front of the first whole vector and behind the last
    auto for_outer = [&](auto&& visit) {
        for (int v = t; v < min(p.V, vlo * EPV - a); v += THREADS) {
            visit(v);
        }
        for (int v = vhi * EPV - a + t; v < p.V; v += THREADS) {
            visit(v);
        }
    };
    for_outer([&](int v) { m = __builtin_fmaxf(m, value(v, rowp[v])); });
    float unsure = NEG_INF;  // an upper bound of this thread's columns where no more is known
    float seen   = m;        // what counts for the row's maximum
    // the vector of column v, counted from the row's first whole one
    auto vector_of = [&](int v) { return (v + a) / EPV - vlo; };
    if (ordered) {
        wide_key[t] = f2u(raw_own);
        if (t < THREADS / 32) {
            slot_key[t] = 0u;  // bit t % 32 of word t / 32: thread t's raw maximum is a column with a value of its own
        }
        __syncthreads();
        for_special([&](int v, T raw) {
            const int at = vector_of(v), owner = at & (THREADS - 1);
            if (at >= 0 && at < nvec && S::ld(raw) >= u2f(wide_key[owner])) {
                atomicOr(&slot_key[owner >> 5], 1u << (owner & 31));
            }
            seen = __builtin_fmaxf(seen, value(v, raw));
        });
        __syncthreads();
        const float top = rowctx.fast(raw_own);
        if ((slot_key[t >> 5] >> (t & 31)) & 1u) {
            unsure = top;
        }
        else {
            m    = __builtin_fmaxf(m, top);
            seen = __builtin_fmaxf(seen, top);
        }
    }
    LPW_STAMP(2)
    if (t == 0) {
        s.misc[0] = __float_as_int(row_uniform(l.rng, l.uniforms, row));  // (read behind the barriers of the sum)
    }
    seen                      = wave_max(seen);
    const float unsure_of_all = wave_max(unsure);
    if (lane_id() == 0) {
        redf[wave_id()]     = seen;
        warp_sum[wave_id()] = unsure_of_all;
    }
    __syncthreads();
    constexpr int NW      = THREADS / WAVE;
    float         row_max = wave_max(lane_id() < NW ? redf[lane_id()] : NEG_INF);
    if (wave_max(lane_id() < NW ? warp_sum[lane_id()] : NEG_INF) > row_max) {  // (the same for every wave)
        // the vectors of the threads in question again, past the columns that have values of their own: each wave those of its
        // lanes, two lanes' at a time
        float found = NEG_INF;
        for (unsigned long long again = __ballot(unsure > row_max); again != 0ull;) {
            const int one = __builtin_ctzll(again);
            again &= again - 1ull;
            const int other = again != 0ull ? __builtin_ctzll(again) : one;
            again &= again - 1ull;
            for (int q = 0; q < turns; q += WAVE) {
                uint4 v[2];
                int   rel[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    rel[i] = (q + lane_id()) * THREADS + (t & ~(WAVE - 1)) + (i == 0 ? one : other);
                    v[i]   = base[vlo + min(rel[i], nvec - 1)];
                }
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int      first = (vlo + rel[i]) * EPV - a;
                    const uint32_t end   = (uint32_t)(rowctx.masked_end_id - first);
                    uint32_t       bits  = end < (uint32_t)EPV ? 1u << end : 0u;
                    if (rel[i] >= nvec) {
                        bits = (1u << EPV) - 1u;
                    }
                    else if (bitsv) {
                        bits |= rowctx.vector_bits(first, EPV);
                    }
#pragma unroll
                    for (int j = 0; j < EPV; ++j) {
                        found = __builtin_fmaxf(found, (bits >> j) & 1u ? NEG_INF : vector_element<DT>(v[i], j));
                    }
                }
            }
        }
        found = rowctx.fast(found);
        __syncthreads();
        row_max = __builtin_fmaxf(row_max, block_max<float, NW>(found, redf, NEG_INF));
    }
    LPW_STAMP(3)
    row_max       = __builtin_fmaxf(-3.402823466e+38f, row_max);
    if (p.V < p.Vp) {
        row_max = __builtin_fmaxf(row_max, -S::max_t());
    }
    row_max = uniform_f(row_max);
    // the bound: every thread's largest e belongs to a column of its own
    wide_key[t] = order_key(round_t<DT>(det_expf_nonpos(m - row_max)));
    __syncthreads();
    if (t < TK_THREADS) {
        uint32_t key = wide_key[t];
#pragma unroll
        for (int g = 1; g < THREADS / TK_THREADS; ++g) {
            key = max(key, wide_key[t + g * TK_THREADS]);
        }
        slot_key[t] = key;
    }
    __syncthreads();
    uint32_t       thr     = KMIN;
    float          thr_low = key_to_float(KMIN);
    bool           valid   = false;
    const uint32_t P       = lean_kth_of_slots(slot_key, k);
    if (P > order_key(0.0f)) {  // at least k columns with e > 0 at or above it
        thr           = P;
        const float e = key_to_float(P);
        thr_low       = uniform_f(lp_gather_floor<DT>(e));
        valid         = true;
    }

    // ---- where the candidates of a 16-bit row are: groups of vectors with a raw value that the bound does not rule out
    // (the list lies where the selection keeps its own later on)
    int*      parked    = s.sel.idx;
    float     raw_floor = NEG_INF;
    bool      raises    = false;  // the history penalty raises values
    // (the mask of the end id raises a value of -inf to -MAX_T, which is the largest of rows that are masked throughout: the
    // end id is considered whatever its raw value)
    const int end_vector =
        rowctx.masked_end_id >= 0 && rowctx.masked_end_id < p.V ? vector_of(rowctx.masked_end_id) : -1;
    if (!IN_SUM && valid && ordered) {
        // an unflagged column with e >= thr_low has at least this raw value (e's rounding, the logarithm's, y's)
        const float rounding = DT == DT_F16 ? (thr_low < 2.44140625e-04f ? 0.4f : 0.998f) : 0.98f;
        float       y        = row_max + det_logf(thr_low * rounding);
        y                    = lean_below_rounding<DT>(y - __builtin_fabsf(row_max) * 1e-6f - 1e-5f) / mul;
        y                    = y - __builtin_fabsf(y) * 1e-6f;
        raw_floor            = uniform_f(y < 3.0e38f ? y : NEG_INF);
        uint32_t mine        = 0u;
        for (int g = 0; g << glog < turns; ++g) {
            mine |= (group_max[g * THREADS + t] >= raw_floor ? 1u : 0u) << g;
        }
        if (end_vector >= 0 && end_vector < nvec && (end_vector & (THREADS - 1)) == t) {
            mine |= 1u << ((end_vector / THREADS) >> glog);
        }
        // (a penalty that raises values: the columns of the history can reach the bound from any raw value)
        raises = hist && !(p.penalty_type == 0 ? rowctx.penalty >= 0.0f : rowctx.penalty >= 1.0f);
        if (raises) {
            __syncthreads();
            wide_key[t] = mine;
            __syncthreads();
            for_special([&](int v, T) {
                const int at = vector_of(v);
                if (at >= 0 && at < nvec) {
                    atomicOr(&wide_key[at & (THREADS - 1)], 1u << ((at / THREADS) >> glog));
                }
            });
            __syncthreads();
            mine = wide_key[t];
        }
        while (mine != 0u) {
            const int g    = __builtin_ctz(mine);
            const int slot = atomicAdd(&s.misc[1], 1);
            if (slot < TK_CCAP) {
                parked[slot] = (g << glog) * THREADS + t;  // the group's first vector
            }
            mine &= mine - 1u;
        }
    }
    LPW_STAMP(4)
    if constexpr (THREADS < LPW_THREADS) {
        __builtin_amdgcn_s_setprio(0);
    }
    // ---- second pass: the sum chain by chain, and the candidates of an fp32 row
    float acc[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        acc[c] = 0.0f;
    }
    auto push = [&](int v, float e) {
        const int slot = atomicAdd(&s.n_cand, 1);
        if (slot < TK_CCAP) {
            s.cand.key[slot] = order_key(e);
            s.cand.idx[slot] = (uint32_t)v;
        }
    };
    const auto  ex   = [&] {
        if constexpr (WORD16) {
            return ExpPairs<DT>(row_max);
        }
        else {
            return 0;
        }
    }();
    const float        sum_low = valid ? thr_low : __builtin_inff();  // of a column that the sum keeps as a candidate
    unsigned long long far = 0ull;  // bfloat16: lanes that have met columns far below the maximum
    // e of slots [j0, j0 + G) of a batch. 16-bit types: half a batch in a straight line (a wave waits for every branch).
    constexpr int G = WORD16 ? 8 : 4;
    auto numerators = [&](auto wide, const Val* y, Val* e, int j0) __attribute__((always_inline)) {
        if constexpr (!WORD16) {
            float d[G];
#pragma unroll
            for (int j = 0; j < G; ++j) {
                d[j] = y[j0 + j] - row_max;
            }
#pragma unroll
            for (int j = 0; j < G; ++j) {
                e[j0 + j] = det_expf_nonpos_number(d[j]);
            }
            if (lp_rare(__builtin_isunordered(d[0], d[1]) || __builtin_isunordered(d[2], d[3]))) {
#pragma unroll
                for (int j = 0; j < G; ++j) {
                    e[j0 + j] = d[j] != d[j] ? d[j] : e[j0 + j];
                }
            }
        }
        else if constexpr (decltype(wide)::value) {
            ex.template wide_numerators<G / 2>(y + j0 / 2, e + j0 / 2);
        }
        else {
            ex.template numerators<G / 2>(y + j0 / 2, e + j0 / 2, far);
        }
    };
    auto add_batch = [&](auto wide, int v0, const Val* y, int rounds) __attribute__((always_inline)) {
#pragma unroll
        for (int j0 = 0; j0 < N; j0 += G) {
            if (j0 / CH < rounds) {  // (whole batches: always)
                Val e[NY];
                numerators(wide, y, e, j0);
                if constexpr (IN_SUM) {
                    const float top = __builtin_fmaxf(__builtin_fmaxf(e[j0], e[j0 + 1]), __builtin_fmaxf(e[j0 + 2], e[j0 + 3]));
                    if (lp_rare(top >= sum_low)) {  // (a NaN is no candidate)
#pragma unroll
                        for (int j = j0; j < j0 + G; ++j) {
                            if (e[j] >= sum_low && v0 + offset_of(j) < p.V) {
                                push(v0 + offset_of(j), e[j]);
                            }
                        }
                    }
                }
                // (slots of a chain in ascending order of their columns)
#pragma unroll
                for (int j = j0; j < j0 + G; ++j) {
                    if constexpr (!WORD16) {
                        acc[j % CH] = acc[j % CH] + e[j];
                    }
                    else if (j % 2 == 0) {
                        acc[j % CH]       = ex.add_low(acc[j % CH], e[j / 2]);
                        acc[(j + 1) % CH] = ex.add_high(acc[(j + 1) % CH], e[j / 2]);
                    }
                }
            }
        }
    };
    stream([&](int v0, const Val* y, int rounds) __attribute__((always_inline)) {
        // (bfloat16: from the first far column on a wave takes the wide bounds for the rest of its columns)
        if (DT == DT_BF16 && __builtin_expect(far != 0ull, 0)) {
            add_batch(std::integral_constant<bool, DT == DT_BF16>(), v0, y, rounds);
        }
        else {
            add_batch(std::false_type(), v0, y, rounds);
        }
    });
    const float pad_e = p.V < p.Vp ? round_t<DT>(det_expf_nonpos(-S::max_t() - row_max)) : 0.0f;
    if (pad_e > 0.0f) {
        // pad columns count once nothing of the vocabulary is far above -MAX_T (rows that are masked throughout)
#pragma unroll 1
        for (int v0 = (p.V & ~(LP_BLOCK - 1)) + CH * t; v0 < p.Vp; v0 += LP_BLOCK) {
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                acc[c] = v0 + c >= p.V && v0 + c < p.Vp ? acc[c] + pad_e : acc[c];
            }
        }
    }
    LPW_STAMP(5)
    if constexpr (THREADS < LPW_THREADS) {
        __builtin_amdgcn_s_setprio(3);
    }
    // the reference's order: xor butterflies inside 32-chain groups, then over the 32 group sums
    // (chains that are CH or more apart belong to other lanes, nearer ones to the same thread)
#pragma unroll
    for (int o = 16; o >= 1; o >>= 1) {
        float other[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            other[c] = o >= CH ? __shfl_xor(acc[c], o >= CH ? o / CH : 0, 32) : acc[c ^ (o & (CH - 1))];
        }
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            acc[c] = acc[c] + other[c];
        }
    }
    if (((CH * t) & 31) == 0) {
        warp_sum[(CH * t) >> 5] = acc[0];
    }
    __syncthreads();
    float total = warp_sum[lane_id() & 31];
#pragma unroll
    for (int o = 16; o >= 1; o >>= 1) {
        total = total + __shfl_xor(total, o, 32);
    }
    const float denom = uniform_f(total + 1e-6f);
    const float u     = __int_as_float(s.misc[0]);
    // the candidates of a 16-bit row: the columns at or above the bound in the groups kept in mind (the whole row where raw
    // values say nothing), a vector per thread and turn, and those outside the whole vectors
    const int   n_parked = __builtin_amdgcn_readfirstlane(s.misc[1]);
    const float e_bound  = key_to_float(thr);
    const bool  covered  = valid && lp_gather_covers<DT>(e_bound, denom);
    if (covered && n_parked <= TK_CCAP) {
        auto consider = [&](int v) {
            const float e = round_t<DT>(det_expf_nonpos(value(v, rowp[v]) - row_max));
            if (e >= thr_low) {  // (a NaN is no candidate)
                push(v, e);
            }
        };
        const int vectors = IN_SUM ? 0 : ordered ? n_parked << glog : nvec;
#pragma unroll 1
        for (int i = t; i < vectors; i += THREADS) {
            const int rel = ordered ? parked[i >> glog] + (i & ((1 << glog) - 1)) * THREADS : i;
            if (rel < nvec) {
                const uint4 v    = base[vlo + rel];
                uint32_t    hits = 0u;
#pragma unroll
                for (int j = 0; j < EPV; ++j) {
                    hits |= (!(vector_element<DT>(v, j) < raw_floor) ? 1u : 0u) << j;
                }
                if (rel == end_vector) {
                    hits |= 1u << ((rowctx.masked_end_id + a) % EPV);
                }
                if (raises) {
                    hits = (1u << EPV) - 1u;
                }
                while (hits != 0u) {
                    consider((vlo + rel) * EPV - a + __builtin_ctz(hits));
                    hits &= hits - 1u;
                }
            }
        }
        if (!IN_SUM) {
            for_outer(consider);
        }
        if (pad_e > 0.0f && pad_e >= thr_low) {
            for (int v = p.V + t; v < p.Vp; v += THREADS) {
                push(v, pad_e);
            }
        }
    }
    __syncthreads();
    int  n     = __builtin_amdgcn_readfirstlane(s.n_cand);
    bool probs = false;
    __syncthreads();
    if (!covered || n_parked > TK_CCAP || n > TK_CCAP) {
        // (fewer than k columns with e > 0: columns of probability zero are picked too, by the reference's tie rules)
        probs = true;
        n     = topk_regather<DT, THREADS, true>(
            s, wide_key, p.Vp, k, p.max_top_k <= 16 ? 7 : 8, valid ? order_key(round_t<DT>(e_bound / denom)) : 0u,
            [&](int v) -> uint32_t {
                const float y = v < p.V ? value(v, rowp[v]) : -S::max_t();
                return order_key(round_t<DT>(round_t<DT>(det_expf_nonpos(y - row_max)) / denom));
            });
        n = __builtin_amdgcn_readfirstlane(n);
        __syncthreads();
    }
    if (wave_id() >= TK_WAVES) {
        return;  // the first four waves select
    }
    LPW_STAMP(6)
    lp_finish<DT>(s, slot_key, n, probs, denom, row_max, k, tp, u, p, l, row, out, DT == DT_F32 && s.misc[3] != 0);
    LPW_STAMP(7)
}

// Launchers, one translation unit per element type (logprob_kernels.hip built with FTK_LP_DT = 0, 1, 2).
// window: 0 = history bitmaps in global memory, 1 = small LDS window, 2 = large.
int lp_rowmax_launch_f32(int window, dim3 grid, hipStream_t st, const FusedParams& p, const FusedLaunch& l,
                         const LogProbLaunch& lp);
int lp_rowmax_launch_f16(int window, dim3 grid, hipStream_t st, const FusedParams& p, const FusedLaunch& l,
                         const LogProbLaunch& lp);
int lp_rowmax_launch_bf16(int window, dim3 grid, hipStream_t st, const FusedParams& p, const FusedLaunch& l,
                          const LogProbLaunch& lp);
int lp_row_launch_f32(int window, int rows, hipStream_t st, const FusedParams& p, const FusedLaunch& l,
                      const LogProbLaunch& lp);
int lp_row_launch_f16(int window, int rows, hipStream_t st, const FusedParams& p, const FusedLaunch& l,
                      const LogProbLaunch& lp);
int lp_row_launch_bf16(int window, int rows, hipStream_t st, const FusedParams& p, const FusedLaunch& l,
                       const LogProbLaunch& lp);
// threads: 1024, 512 or 256 per row
int lp_wide_launch_f32(int window, int threads, int rows, hipStream_t st, const FusedParams& p, const FusedLaunch& l,
                       const LogProbLaunch& lp);
int lp_wide_launch_f16(int window, int threads, int rows, hipStream_t st, const FusedParams& p, const FusedLaunch& l,
                       const LogProbLaunch& lp);
int lp_wide_launch_bf16(int window, int threads, int rows, hipStream_t st, const FusedParams& p, const FusedLaunch& l,
                        const LogProbLaunch& lp);

}  // namespace ftk
