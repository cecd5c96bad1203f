// One step of beam search over [batch * beam_width, vocab] logits: log-softmax, the 2K best tokens of every beam,
// the K best continuations of every batch entry, finished hypotheses moved to the BeamHypotheses arrays.
//
// Reference behaviour restated (src/fastertransformer/kernels/online_softmax_beamsearch_kernels.cu):
//   :366-514  beam_online_softmax_topk_stage1 / stage2 - per row (max, sum of exponentials) and the 2K best
//             elements under TopK<T, MAX_K>::insert (kernels/reduce_kernel_utils.cuh:275-322): value
//             descending, id ascending, which no merge order changes
//   :99-262   batch_topk_kernel - the 2 * MAX_K best of a batch entry's K * 2K candidates after length penalty
//             and diversity term, then one thread walks them: end tokens among the first K go to the
//             hypotheses (kernels/beam_search_topk_kernels.h:31-58), the others become the next beams
//   :549-701  launchers and the beam-width classes
//
// The reference finds the best elements by inserting into per-thread sorted arrays and merging them with cub. Here
// every selection is an exact radix select over 64-bit keys (order-preserving value bits, then the complement of
// the position, so that keys are distinct and ties need no rule of their own): byte by byte from the top, a
// 256-bin LDS histogram of the keys that match the bytes fixed so far; as soon as few enough match they are moved
// to LDS and the remaining bytes are settled there.
#include "ftk_columns.cuh"
#include "ftk_device.cuh"
#include "ftk_sampling.h"
#include "ftk_transform.cuh"
#ifdef FTK_TEST_HOOKS
#include "ftk_test_hooks.h"
#endif

namespace ftk {

constexpr int BM_THREADS = 256;
constexpr int BM_WAVES   = BM_THREADS / WAVE;
constexpr int BM_CAP     = 2048;  // keys settled in LDS
constexpr int BM_MAX_N   = 128;   // 2 * beam_width and 2 * MAX_K are at most this

struct BeamSelect {
    __attribute__((aligned(16))) unsigned long long list[BM_CAP];
    unsigned long long cand[BM_CAP];     // a section's elements at or above the bound from the thread maxima
    unsigned long long slots[BM_THREADS];
    unsigned long long out[BM_MAX_N];
    int                n_cand;
    uint32_t           hist[256];
    uint32_t           wave_total[BM_WAVES];
    int                n_list;
    int                n_out;
    int                found_bin;
    int                found_above;
};

// The `need`-th largest of `count` keys key(i), 1 <= need <= count, distinct at least down to that one (zero keys
// that pad a list may repeat below it): every thread of the workgroup gets it. key(i) is evaluated once per byte
// that is settled on the caller's data (until BM_CAP or fewer keys match).
template<class F>
__device__ __forceinline__ unsigned long long beam_nth_key(BeamSelect& s, F&& key, int count, int need)
{
    const int          t      = threadIdx.x;
    unsigned long long prefix = 0ull;
    bool               in_lds = false;
    int                n      = count;
    for (int shift = 56; shift >= 0; shift -= 8) {
        s.hist[t] = 0u;
        __syncthreads();
        for (int i = t; i < n; i += BM_THREADS) {
            const unsigned long long k = in_lds ? s.list[i] : key(i);
            if (shift == 56 || (k >> (shift + 8)) == prefix) {
                atomicAdd(&s.hist[(uint32_t)(k >> shift) & 255u], 1u);
            }
        }
        __syncthreads();
        // thread t looks at bin 255 - t: inclusive sums from the top bin down
        const uint32_t mine = s.hist[255 - t];
        uint32_t       inc  = mine;
#pragma unroll
        for (int o = 1; o < WAVE; o <<= 1) {
            const uint32_t up = __shfl_up(inc, o, WAVE);
            if (lane_id() >= o) {
                inc += up;
            }
        }
        if (lane_id() == WAVE - 1) {
            s.wave_total[wave_id()] = inc;
        }
        __syncthreads();
        for (int w = 0; w < wave_id(); ++w) {
            inc += s.wave_total[w];
        }
        if (inc >= (uint32_t)need && inc - mine < (uint32_t)need) {
            s.found_bin   = 255 - t;
            s.found_above = (int)(inc - mine);
        }
        __syncthreads();
        const int bin     = s.found_bin;
        const int matched = (int)s.hist[bin];
        need -= s.found_above;
        prefix = (prefix << 8) | (unsigned long long)bin;
        if (!in_lds && matched <= BM_CAP && shift > 0) {
            // few enough keys carry the bytes fixed so far: the rest is settled on a copy in LDS
            if (t == 0) {
                s.n_list = 0;
            }
            __syncthreads();
            for (int i = t; i < n; i += BM_THREADS) {
                const unsigned long long k = key(i);
                if ((k >> shift) == prefix) {
                    s.list[atomicAdd(&s.n_list, 1)] = k;
                }
            }
            __syncthreads();
            in_lds = true;
            n      = matched;
        }
        __syncthreads();
    }
    return prefix;
}

// Leaves the `need` largest of `count` distinct keys in s.out, largest first; need <= BM_MAX_N, need <= count.
template<class F>
__device__ __forceinline__ void beam_select(BeamSelect& s, F&& key, int count, int need)
{
    const int t = threadIdx.x;
    if (count <= BM_THREADS) {
        // one key per thread: its place is the number of larger keys
        const unsigned long long k = t < count ? key(t) : 0ull;
        __syncthreads();  // (the caller may still be reading what key() reads from, or s.list)
        s.list[t] = k;  // (zeros behind the last key: they are larger than nothing)
        __syncthreads();
        const ulonglong2* pairs = reinterpret_cast<const ulonglong2*>(s.list);
        int               r     = 0;
        for (int j = 0; j < (count + 3) / 4; ++j) {
            const ulonglong2 a = pairs[2 * j];
            const ulonglong2 b = pairs[2 * j + 1];
            r += (a.x > k ? 1 : 0) + (a.y > k ? 1 : 0) + (b.x > k ? 1 : 0) + (b.y > k ? 1 : 0);
        }
        if (t < count && r < need) {
            s.out[r] = k;
        }
        __syncthreads();
        return;
    }
    const unsigned long long bound = beam_nth_key(s, key, count, need);
    if (t == 0) {
        s.n_out = 0;
    }
    __syncthreads();
    for (int i = t; i < count; i += BM_THREADS) {
        const unsigned long long k = key(i);
        if (k >= bound) {
            s.list[atomicAdd(&s.n_out, 1)] = k;  // exactly `need` of them
        }
    }
    __syncthreads();
    if (t < need) {
        const unsigned long long k = s.list[t];
        int                      r = 0;
        for (int j = 0; j < need; ++j) {
            r += s.list[j] > k ? 1 : 0;
        }
        s.out[r] = k;
    }
    __syncthreads();
}

__device__ __forceinline__ unsigned long long beam_key(float value, uint32_t position)
{
    return ((unsigned long long)order_key(value) << 32) | (unsigned long long)(0xFFFFFFFFu - position);
}
__device__ __forceinline__ uint32_t beam_key_position(unsigned long long k)
{
    return 0xFFFFFFFFu - (uint32_t)k;
}
__device__ __forceinline__ float beam_key_value(unsigned long long k)
{
    return key_to_float((uint32_t)(k >> 32));
}

// element `v` of row `r` as the reference's kernels see it (:341-347, :410-416)
template<int DT>
__device__ __forceinline__ float beam_element(const typename Storage<DT>::T* __restrict__ x,
                                              const typename Storage<DT>::T* __restrict__ bias, size_t row_base, int v)
{
    typedef Storage<DT> S;
    const float         b = bias != nullptr ? S::ld(bias[v]) : 0.0f;
    return round_t<DT>(S::ld(x[row_base + v]) + b);
}

// the same from a value that is already loaded
template<int DT>
__device__ __forceinline__ float beam_element_of(float xv, const typename Storage<DT>::T* __restrict__ bias, int v)
{
    if (bias == nullptr) {
        return xv;  // adding T(0) changes -0 into +0 and nothing else: same key, same exponential
    }
    return round_t<DT>(xv + Storage<DT>::ld(bias[v]));
}

struct BeamPlan {
    int    parts;  // sections per row
    int    section;
    size_t off_pmax, off_psum, off_pkeys, off_cand_id, off_cand_val, off_before, bytes;
};

static inline size_t beam_align(size_t x)
{
    return (x + 255) & ~(size_t)255;
}

static BeamPlan beam_plan(int rows, int beam_width, int vocab)
{
    BeamPlan  p;
    const int N = 2 * beam_width;
    int       parts = (1024 + rows - 1) / (rows > 0 ? rows : 1);
    const int by_len = vocab / 4096 > 0 ? vocab / 4096 : 1;
    parts   = parts < by_len ? parts : by_len;
    parts   = parts < BM_CAP / N ? parts : BM_CAP / N;  // the lists of a row are merged in LDS
    parts   = parts < 1 ? 1 : parts;
    while (parts > 1 && (vocab + parts - 1) / parts < N) {
        parts--;  // every section holds at least 2K elements
    }
    p.parts   = parts;
    p.section = (vocab + parts - 1) / parts;
    const size_t r = (size_t)(rows > 0 ? rows : 1);
    size_t       off = 0;
    p.off_pmax = off;
    off += beam_align(r * parts * sizeof(float));
    p.off_psum = off;
    off += beam_align(r * parts * sizeof(double));
    p.off_pkeys = off;
    off += beam_align(r * parts * N * sizeof(unsigned long long));
    p.off_cand_id = off;
    off += beam_align(r * N * sizeof(int));
    p.off_cand_val = off;
    off += beam_align(r * N * sizeof(float));
    p.off_before = off;
    off += beam_align(r * sizeof(int2));
    p.bytes = off;
    return p;
}

// What a finished row offers (:328-336): MAX_T at its end id, -MAX_T elsewhere, so the end id first, then the lowest
// ids. Element t of that list.
struct BeamFinishedRow {
    bool  inside;  // the end id is a column
    float m, d;    // maximum and sum of exponentials: inside, every other exponential is 0
};
template<int DT>
__device__ __forceinline__ BeamFinishedRow beam_finished_row(int end_id, int vocab)
{
    const bool inside = end_id >= 0 && end_id < vocab;
    return BeamFinishedRow{inside, inside ? Storage<DT>::max_t() : -Storage<DT>::max_t(), inside ? 1.0f : (float)vocab};
}
template<int DT>
__device__ __forceinline__ unsigned long long beam_finished_key(const BeamFinishedRow& f, int end_id, int t)
{
    const int   id = f.inside ? (t == 0 ? end_id : (t - 1 < end_id ? t - 1 : t)) : t;
    const float u  = f.inside && t == 0 ? Storage<DT>::max_t() : -Storage<DT>::max_t();
    return beam_key(u, (uint32_t)id);
}

// A row's flag and length as they were before the step: the batch kernel of a step that updates them in the same
// launch reads those of other entries' rows.
__device__ __forceinline__ void beam_keep_before(int2* __restrict__ before, const bool* __restrict__ finished,
                                                 const int* __restrict__ sequence_lengths, int row)
{
    before[row] = make_int2(finished[row] ? 1 : 0, sequence_lengths != nullptr ? sequence_lengths[row] : 0);
}

// (parts x rows) workgroups: the maximum of a section
template<int DT>
__global__ void __launch_bounds__(BM_THREADS)
beam_section_max_kernel(const typename Storage<DT>::T* __restrict__ x, const typename Storage<DT>::T* __restrict__ bias,
                        const bool* __restrict__ finished, int vocab, int section, float* __restrict__ pmax)
{
    __shared__ float red[BM_WAVES];
    const int        row = blockIdx.y;
    const int        t   = threadIdx.x;
    if (finished[row]) {
        return;
    }
    const int    lo = min(vocab, (int)blockIdx.x * section);
    const int    hi = min(vocab, lo + section);
    const size_t rb = (size_t)row * vocab;
    float        m  = -Storage<DT>::max_t();
    stream_columns<DT, BM_THREADS>(x + rb, lo, hi, [&](int v, float xv) {
        const float e = beam_element_of<DT>(xv, bias, v);
        m             = e > m ? e : m;
    });
    m = block_max<float, BM_WAVES>(m, red, -Storage<DT>::max_t());
    if (t == 0) {
        pmax[(size_t)row * gridDim.x + blockIdx.x] = m;
    }
}

// (parts x rows) workgroups: the sum of exponentials of a section against the row's maximum and its 2K best
template<int DT>
__global__ void __launch_bounds__(BM_THREADS)
beam_section_kernel(const typename Storage<DT>::T* __restrict__ x, const typename Storage<DT>::T* __restrict__ bias,
                    const bool* __restrict__ finished, int vocab, int section, int N, const float* __restrict__ pmax,
                    double* __restrict__ psum, unsigned long long* __restrict__ pkeys)
{
    __shared__ BeamSelect s;
    __shared__ double     red[BM_WAVES];
    const int             row   = blockIdx.y;
    const int             part  = blockIdx.x;
    const int             parts = gridDim.x;
    const int             t     = threadIdx.x;
    if (finished[row]) {
        return;
    }
    const int    lo = min(vocab, part * section);
    const int    hi = min(vocab, lo + section);
    const size_t rb = (size_t)row * vocab;
    float        m  = -Storage<DT>::max_t();
    for (int p = 0; p < parts; ++p) {
        const float pm = pmax[(size_t)row * parts + p];
        m              = pm > m ? pm : m;
    }
    // first pass: the sum, and every thread's largest element
    double d    = 0.0;
    float  fmax = -__builtin_inff();
    stream_columns<DT, BM_THREADS>(x + rb, lo, hi, [&](int v, float xv) {
        const float e = beam_element_of<DT>(xv, bias, v);
        d += (double)det_expf_nonpos(e - m);  // m is the row's maximum: the argument is never positive
        fmax = __builtin_fmaxf(fmax, e);      // (a NaN is never the maximum, as under order_key)
    });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        d += __shfl_xor(d, o, WAVE);
    }
    if (lane_id() == 0) {
        red[wave_id()] = d;
    }
    // N <= 32 needs no more than 64 maxima to choose the N-th largest from, N <= 64 no more than 128: neighbouring
    // threads join theirs, and the ranking below is that much shorter
    const int group = N <= 32 ? 4 : N <= 64 ? 2 : 1;
    if (group >= 2) {
        fmax = __builtin_fmaxf(fmax, __shfl_xor(fmax, 1, WAVE));
    }
    if (group == 4) {
        fmax = __builtin_fmaxf(fmax, __shfl_xor(fmax, 2, WAVE));
    }
    const int n_slots = BM_THREADS / group;
    if (t % group == 0) {
        s.slots[t / group] = ((unsigned long long)order_key(fmax) << 32) | (unsigned long long)(BM_THREADS - 1 - t);
    }
    if (t == 0) {
        s.n_cand = 0;
    }
    __syncthreads();
    if (t == 0) {
        double tot = 0.0;
        for (int w = 0; w < BM_WAVES; ++w) {
            tot += red[w];
        }
        psum[(size_t)row * parts + part] = tot;
    }
    // a short last section gives fewer than N keys; the rest of its list is 0, below every key of an element
    const int take = min(N, hi - lo);
    // The N-th largest of the thread maxima is an element with at least N elements at or above it (N threads hold
    // one each): nothing below it can be among the N best. Usually a few times N elements pass.
    // (a group that saw no element reports -inf, which lowers the bound at most to "every number")
    beam_select(s, [&](int i) { return s.slots[i]; }, n_slots, N);
    const uint32_t floor_key = (uint32_t)(s.out[N - 1] >> 32);
    const float    floor_val = key_to_float(floor_key);
    const bool     all_pass  = floor_key <= order_key(-__builtin_inff());  // then NaN columns are wanted too
    stream_columns<DT, BM_THREADS>(x + rb, lo, hi, [&](int v, float xv) {
        const float e = beam_element_of<DT>(xv, bias, v);
        if (e >= floor_val || all_pass) {
            const int at = atomicAdd(&s.n_cand, 1);
            if (at < BM_CAP) {
                s.cand[at] = beam_key(e, (uint32_t)v);
            }
        }
    });
    __syncthreads();
    const int passed = s.n_cand;
    if (take > 0) {
        if (passed <= BM_CAP) {
            beam_select(s, [&](int i) { return s.cand[i]; }, passed, take);
        }
        else {
            // (rows of many equal values) the selection runs over the section itself
            beam_select(s, [&](int i) { return beam_key(beam_element<DT>(x, bias, rb, lo + i), (uint32_t)(lo + i)); },
                        hi - lo, take);
        }
    }
    if (t < N) {
        pkeys[((size_t)row * parts + part) * N + t] = t < take ? s.out[t] : 0ull;
    }
}

// one workgroup per row: the row's 2K best from its sections' lists, val = u - m - log(d) + cum_log_probs as T
template<int DT>
__global__ void __launch_bounds__(BM_THREADS)
beam_row_kernel(const bool* __restrict__ finished, const int* __restrict__ end_ids,
                const float* __restrict__ cum_log_probs, int vocab, int K, int parts, const float* __restrict__ pmax,
                const double* __restrict__ psum, const unsigned long long* __restrict__ pkeys,
                int* __restrict__ cand_id, float* __restrict__ cand_val, const int* __restrict__ sequence_lengths,
                int2* __restrict__ before)
{
    typedef Storage<DT>   S;
    __shared__ BeamSelect s;
    const int             row  = blockIdx.x;
    const int             t    = threadIdx.x;
    const int             N    = 2 * K;
    const float           MAXT = S::max_t();
    const float           cum  = cum_log_probs[row];
    if (t == 0) {
        beam_keep_before(before, finished, sequence_lengths, row);
    }
    if (finished[row]) {
        const int             end_id = end_ids[row / K];
        const BeamFinishedRow f      = beam_finished_row<DT>(end_id, vocab);
        if (t < N) {
            const unsigned long long k   = beam_finished_key<DT>(f, end_id, t);
            cand_id[(size_t)row * N + t] = (int)beam_key_position(k) + row * vocab;
            cand_val[(size_t)row * N + t] = round_t<DT>((beam_key_value(k) - f.m - det_logf(f.d)) + cum);
        }
        return;
    }
    float  m = -MAXT;
    double d = 0.0;
    for (int p = 0; p < parts; ++p) {
        const float pm = pmax[(size_t)row * parts + p];
        m              = pm > m ? pm : m;
        d += psum[(size_t)row * parts + p];
    }
    const float               logd = det_logf((float)d);
    const unsigned long long* keys = pkeys + (size_t)row * parts * N;
    if (parts == 1) {
        if (t < N) {
            s.out[t] = keys[t];
        }
        __syncthreads();
    }
    else {
        beam_select(s, [&](int i) { return keys[i]; }, parts * N, N);
    }
    if (t < N) {
        const unsigned long long k    = s.out[t];
        cand_id[(size_t)row * N + t]  = (int)beam_key_position(k) + row * vocab;
        cand_val[(size_t)row * N + t] = round_t<DT>((beam_key_value(k) - m - logd) + cum);
    }
}

// The three kernels above in one launch: one 1024-thread workgroup per row finds the row's maximum, the sum of exponentials and every thread's largest
// element, takes a bound from 256 (128, 64) joined thread maxima, collects what reaches it and leaves the row's 2K
// best with their values. The passes over the row are the section kernels' with the whole row as the one section
// (the second and third come from the caches); the bound is found by the first wave alone (a bisection with
// ballots over the top 24 key bits: a floor at or below the 2K-th largest maximum, which is all the argument
// needs) so that the other fifteen waves only wait at two barriers; after the last pass twelve waves leave and the
// first four select with the code of the 256-thread kernels (a barrier counts the waves that are left).
// With more rows than compute units the workgroups have 512 threads and two of them share a compute unit: one's reads
// run beside the other's exponentials (64 x 8 beams x 152064 fp16: 120 -> 116 us).
constexpr int BR_THREADS = 1024;

// A value at or below the row's 2K-th largest, from the threads' maxima: the maxima of neighbouring threads joined into
// slots, in LDS behind the next barrier, and, by one wave behind that barrier, the bound. Leaves the candidates' count at
// zero.
__device__ __forceinline__ int beam_n_slots(int N)
{
    // 2K <= 32 needs no more than 64 maxima to choose the 2K-th largest from, 2K <= 64 no more than 128
    return N <= 32 ? 64 : N <= 64 ? 128 : 256;
}
template<int THREADS>
__device__ __forceinline__ void beam_slots(BeamSelect& s, float fmax, int N)
{
    const int t       = threadIdx.x;
    const int n_slots = beam_n_slots(N);
    const int join    = THREADS / n_slots;  // neighbouring threads that join their maxima: 2 to 16
    fmax              = __builtin_fmaxf(fmax, __shfl_xor(fmax, 1, WAVE));
    if (join >= 4) {
        fmax = __builtin_fmaxf(fmax, __shfl_xor(fmax, 2, WAVE));
    }
    if (join >= 8) {
        fmax = __builtin_fmaxf(fmax, __shfl_xor(fmax, 4, WAVE));
    }
    if (join == 16) {
        fmax = __builtin_fmaxf(fmax, __shfl_xor(fmax, 8, WAVE));
    }
    uint32_t* slot_key = reinterpret_cast<uint32_t*>(s.slots);
    if (t % join == 0) {
        slot_key[t / join] = order_key(fmax);
    }
    if (t == 0) {
        s.n_cand = 0;
    }
}
__device__ __forceinline__ uint32_t beam_floor(const BeamSelect& s, int N)
{
    const int       n_slots  = beam_n_slots(N);
    const uint32_t* slot_key = reinterpret_cast<const uint32_t*>(s.slots);
    // The 2K-th largest of the maxima is an element with at least 2K elements at or above it: nothing below it
    // can be among the 2K best; so is any value below that one. (A group that saw no element reports -inf.)
    uint32_t P = 0u;
    if (n_slots == WAVE) {
        // every lane counts the maxima above its own and those at or above it: the 2K-th largest lies between
        const uint32_t mine  = slot_key[lane_id()];
        int            above = 0, reach = 0;
#pragma unroll
        for (int j = 0; j < WAVE; ++j) {
            const uint32_t other = __builtin_amdgcn_readlane(mine, j);
            above += other > mine ? 1 : 0;
            reach += other >= mine ? 1 : 0;
        }
        const unsigned long long at = __ballot(above < N && reach >= N);
        P = __builtin_amdgcn_readlane(mine, __builtin_ctzll(at));
    }
    else {
        uint32_t kk[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int i = lane_id() + g * WAVE;
            kk[g]       = i < n_slots ? slot_key[i] : 0u;
        }
        for (int bit = 31; bit >= 8; --bit) {
            const uint32_t cand = P | (1u << bit);
            int            c    = 0;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                c += (int)__builtin_popcountll(__ballot(kk[g] >= cand));
            }
            P = c >= N ? cand : P;
        }
    }
    return P;
}

// The same and the row's sum from the waves' sums, by the first wave alone while the others wait at two barriers.
template<int THREADS>
__device__ __forceinline__ void beam_bound(BeamSelect& s, const double* red, float fmax, int N, double& row_sum,
                                           uint32_t& floor)
{
    beam_slots<THREADS>(s, fmax, N);
    __syncthreads();
    if (wave_id() == 0) {
        const uint32_t P = beam_floor(s, N);
        if (lane_id() == 0) {
            double tot = 0.0;
            for (int w = 0; w < THREADS / WAVE; ++w) {
                tot += red[w];
            }
            row_sum = tot;
            floor   = P;
        }
    }
    __syncthreads();
}

template<int DT, int THREADS>
__global__ void __launch_bounds__(THREADS)
beam_rowwide_kernel(const typename Storage<DT>::T* __restrict__ x, const typename Storage<DT>::T* __restrict__ bias,
                    const bool* __restrict__ finished, const int* __restrict__ end_ids,
                    const float* __restrict__ cum_log_probs, int vocab, int K, int* __restrict__ cand_id,
                    float* __restrict__ cand_val, const int* __restrict__ sequence_lengths, int2* __restrict__ before)
{
    typedef Storage<DT>   S;
    constexpr int         BR_WAVES = THREADS / WAVE;
    static_assert(THREADS == 1024 || THREADS == 512, "256, 128 or 64 joined maxima");
    __shared__ BeamSelect s;
    __shared__ double     red[BR_WAVES];
    __shared__ float      redf[BR_WAVES];
    __shared__ double     row_sum;
    __shared__ uint32_t   row_floor;
    const int             row  = blockIdx.x;
    const int             t    = threadIdx.x;
    const int             N    = 2 * K;
    const float           MAXT = S::max_t();
    const float           cum  = cum_log_probs[row];
    if (t == 0) {
        beam_keep_before(before, finished, sequence_lengths, row);
    }
    if (finished[row]) {
        const int             end_id = end_ids[row / K];
        const BeamFinishedRow f      = beam_finished_row<DT>(end_id, vocab);
        if (t < N) {
            const unsigned long long k   = beam_finished_key<DT>(f, end_id, t);
            cand_id[(size_t)row * N + t] = (int)beam_key_position(k) + row * vocab;
            cand_val[(size_t)row * N + t] = round_t<DT>((beam_key_value(k) - f.m - det_logf(f.d)) + cum);
        }
        return;
    }
    const size_t rb = (size_t)row * vocab;
    // first pass: the row's maximum
    float m = -MAXT;
    stream_columns<DT, THREADS>(x + rb, 0, vocab, [&](int v, float xv) {
        const float e = beam_element_of<DT>(xv, bias, v);
        m             = e > m ? e : m;
    });
    m = block_max<float, BR_WAVES>(m, redf, -MAXT);
    // second pass: the sum, and every thread's largest element
    double d    = 0.0;
    float  fmax = -__builtin_inff();
    stream_columns<DT, THREADS>(x + rb, 0, vocab, [&](int v, float xv) {
        const float e = beam_element_of<DT>(xv, bias, v);
        d += (double)det_expf_nonpos(e - m);
        fmax = __builtin_fmaxf(fmax, e);
    });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        d += __shfl_xor(d, o, WAVE);
    }
    if (lane_id() == 0) {
        red[wave_id()] = d;
    }
    beam_bound<THREADS>(s, red, fmax, N, row_sum, row_floor);
    const uint32_t floor_key = row_floor;
    const float    floor_val = key_to_float(floor_key);
    const bool     all_pass  = floor_key <= order_key(-__builtin_inff());  // then NaN columns are wanted too
    stream_columns<DT, THREADS>(x + rb, 0, vocab, [&](int v, float xv) {
        const float e = beam_element_of<DT>(xv, bias, v);
        if (e >= floor_val || all_pass) {
            const int at = atomicAdd(&s.n_cand, 1);
            if (at < BM_CAP) {
                s.cand[at] = beam_key(e, (uint32_t)v);
            }
        }
    });
    __syncthreads();
    if (wave_id() >= BM_WAVES) {
        return;  // the first four waves select
    }
    const int passed = s.n_cand;
    const int take   = min(N, vocab);
    if (passed <= BM_CAP) {
        beam_select(s, [&](int i) { return s.cand[i]; }, passed, take);
    }
    else {
        // (rows of many equal values) the selection runs over the row itself
        beam_select(s, [&](int i) { return beam_key(beam_element<DT>(x, bias, rb, i), (uint32_t)i); }, vocab, take);
    }
    const float logd = det_logf((float)row_sum);
    if (t < N) {
        const unsigned long long k    = t < take ? s.out[t] : 0ull;
        cand_id[(size_t)row * N + t]  = (int)beam_key_position(k) + row * vocab;
        cand_val[(size_t)row * N + t] = round_t<DT>((beam_key_value(k) - m - logd) + cum);
    }
}

// Rows of up to 65536 columns, read once: a thread keeps its vectors in registers through the three passes, and with
// at most half as many rows as compute units 2, 4 or 8 workgroups share a row. Every workgroup of a row reads all of it
// for the maximum (100 KB of a row of 50257 fp16, from the XCD's L2 after the first), so they need nothing of each
// other; the exponentials, which bound the kernel (23 vector instructions and a double addition each), and the
// candidates are those of its own part. A part leaves its 2K best, largest first, and its sum; beam_batch_kernel merges.
// The bound of the candidates is worked out by the first wave while the others are at their exponentials, and the few
// threads that can hold a candidate look for it. 32 x 4 rows of 50257 fp16: 19.6 us with one workgroup per row that reads it
// three times, 14.4 us with the bound behind the exponentials and a comparison per column, 12.8 us here (traced).
constexpr int BT_COLUMNS   = 65536;
constexpr int BT_MAX_PARTS = 8;

template<int DT>
__global__ void __launch_bounds__(BR_THREADS)
beam_team_kernel(const typename Storage<DT>::T* __restrict__ x, const typename Storage<DT>::T* __restrict__ bias,
                 const bool* __restrict__ finished, const int* __restrict__ end_ids,
                 const int* __restrict__ sequence_lengths, int vocab, int K, float* __restrict__ pmax,
                 double* __restrict__ psum, unsigned long long* __restrict__ pkeys, int2* __restrict__ before)
{
    typedef Storage<DT>   S;
    typedef typename S::T T;
    constexpr int         EPV   = (int)(16 / sizeof(T));
    constexpr int         NV    = BT_COLUMNS / EPV / BR_THREADS;  // vectors of a thread: 8, or 16 of floats
    constexpr int         WAVES = BR_THREADS / WAVE;
    __shared__ BeamSelect s;
    __shared__ double     red[WAVES];
    __shared__ float      redf[WAVES];
    __shared__ uint32_t   part_floor;
    const int             row   = blockIdx.x;
    const int             part  = blockIdx.y;
    const int             parts = gridDim.y;
    const int             t     = threadIdx.x;
    const int             N     = 2 * K;
    const float           NEG   = -__builtin_inff();
    const bool            done  = finished[row];
    // the row: up to seven columns in front of the first 16-byte boundary, vectors, up to seven columns behind the last
    const T*     rowp  = x + (size_t)row * vocab;
    const int    head  = min((int)(((16u - ((uintptr_t)rowp & 15u)) & 15u) / sizeof(T)), vocab);
    const int    nvec  = (vocab - head) / EPV;
    const int    tail0 = head + nvec * EPV;
    const uint4* vec   = reinterpret_cast<const uint4*>(rowp + head);
    const int    lo    = nvec * part / parts;  // this part's vectors: at most NV * BR_THREADS
    const int    own   = nvec * (part + 1) / parts - lo;
    uint4        raw[NV];
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = t + u * BR_THREADS;
        raw[u]      = i < own ? vec[lo + i] : make_uint4(0, 0, 0, 0);
    }
    // threads 0..6 hold the columns in front, the second wave's first seven those behind
    const int  edge     = t < head ? t : (t >= WAVE && t - WAVE < vocab - tail0 ? tail0 + t - WAVE : -1);
    const bool edge_own = edge >= 0 && (edge < head ? part == 0 : part == parts - 1);
    const float edge_x  = edge >= 0 ? beam_element_of<DT>(S::ld(rowp[edge]), bias, edge) : NEG;
    if (t == 0 && part == 0) {
        beam_keep_before(before, finished, sequence_lengths, row);
    }
    unsigned long long* keys = pkeys + ((size_t)row * parts + part) * N;
    if (done) {
        const int             end_id = end_ids[row / K];
        const BeamFinishedRow f      = beam_finished_row<DT>(end_id, vocab);
        if (t < N) {
            keys[t] = part == 0 ? beam_finished_key<DT>(f, end_id, t) : 0ull;  // (0 is below every element's key)
        }
        if (t == 0) {
            psum[(size_t)row * parts + part] = part == 0 ? (double)f.d : 0.0;
            if (part == 0) {
                pmax[row] = f.m;
            }
        }
        return;
    }
    auto each_own = [&](auto&& visit) {
        if (edge_own) {
            visit(edge, edge_x);
        }
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int i = t + u * BR_THREADS;
            if (i < own) {
                const T*  e = reinterpret_cast<const T*>(&raw[u]);
                const int v = head + (lo + i) * EPV;
#pragma unroll
                for (int j = 0; j < EPV; ++j) {
                    visit(v + j, beam_element_of<DT>(S::ld(e[j]), bias, v + j));
                }
            }
        }
    };
    // the row's maximum, and the thread's own largest element
    float m    = -S::max_t();
    float fmax = NEG;
    // the other parts' vectors, seen only here
    constexpr int U      = 4;
    const int     others = nvec - own;
    for (int o0 = t; o0 < others; o0 += U * BR_THREADS) {
        uint4 ov[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int o = o0 + u * BR_THREADS;
            ov[u]       = o < others ? vec[o < lo ? o : o + own] : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int o = o0 + u * BR_THREADS;
            if (o < others && bias == nullptr) {
                m = __builtin_fmaxf(m, lean_raw_max<DT>(ov[u]));
            }
            else if (o < others) {
                const T*  e = reinterpret_cast<const T*>(&ov[u]);
                const int v = head + (o < lo ? o : o + own) * EPV;
#pragma unroll
                for (int j = 0; j < EPV; ++j) {
                    m = __builtin_fmaxf(m, beam_element_of<DT>(S::ld(e[j]), bias, v + j));
                }
            }
        }
    }
    m = __builtin_fmaxf(m, edge_x);
    // (a NaN is never the maximum)
    if (bias == nullptr) {
        fmax = __builtin_fmaxf(edge_own ? edge_x : NEG, NEG);
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            if (t + u * BR_THREADS < own) {
                fmax = __builtin_fmaxf(fmax, lean_raw_max<DT>(raw[u]));
            }
        }
    }
    else {
        each_own([&](int, float e) { fmax = __builtin_fmaxf(fmax, e); });
    }
    beam_slots<BR_THREADS>(s, fmax, N);
    m = block_max<float, WAVES>(__builtin_fmaxf(m, fmax), redf, -S::max_t());  // (barriers: the slots are there)
    if (wave_id() == 0) {
        const uint32_t P = beam_floor(s, N);  // while the other waves go on
        if (t == 0) {
            part_floor = P;
        }
    }
    double d = 0.0;
    each_own([&](int, float e) { d += (double)det_expf_nonpos(e - m); });
    d = wave_reduce_unordered(d, [](double p, double q) { return p + q; });
    if (lane_id() == 0) {
        red[wave_id()] = d;
    }
    __syncthreads();
    const uint32_t floor_key = part_floor;
    const float    floor_val = key_to_float(floor_key);
    const bool     all_pass  = floor_key <= order_key(NEG);  // then NaN columns are wanted too
    auto push = [&](int v, float e) {
        if (e >= floor_val || all_pass) {
            const int at = atomicAdd(&s.n_cand, 1);
            if (at < BM_CAP) {
                s.cand[at] = beam_key(e, (uint32_t)v);
            }
        }
    };
    if (bias != nullptr || all_pass) {
        each_own(push);
    }
    else if (fmax >= floor_val) {  // (few threads hold a candidate; short code, since it waits for its own fetch)
        if (edge_own) {
            push(edge, edge_x);
        }
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int i = t + u * BR_THREADS;
            if (u * BR_THREADS < own && i < own && lean_raw_max<DT>(raw[u]) >= floor_val) {
                const T* e    = reinterpret_cast<const T*>(&raw[u]);
                uint32_t hits = 0u;
#pragma unroll
                for (int j = 0; j < EPV; ++j) {
                    hits |= (S::ld(e[j]) >= floor_val ? 1u : 0u) << j;
                }
                const uint32_t w[4] = {raw[u].x, raw[u].y, raw[u].z, raw[u].w};
                while (hits != 0u) {
                    const int      j    = __builtin_ctz(hits);
                    const uint32_t word = register_pick<4>(w, j * (int)sizeof(T) / 4);
                    float          x;
                    if constexpr (sizeof(T) == 4) {
                        x = u2f(word);
                    }
                    else {
                        x = S::ld((T)(word >> (16 * (j & 1))));
                    }
                    push(head + (lo + i) * EPV + j, x);
                    hits &= hits - 1u;
                }
            }
        }
    }
    __syncthreads();
    if (wave_id() >= BM_WAVES) {
        return;  // the first four waves select
    }
    const int passed = s.n_cand;
    if (passed <= BM_CAP) {
        beam_select(s, [&](int i) { return s.cand[i]; }, passed, N);
    }
    else {
        // (rows of many equal values) the selection runs over the part itself
        const int from  = part == 0 ? 0 : head + lo * EPV;
        const int until = part == parts - 1 ? vocab : head + (lo + own) * EPV;
        beam_select(s, [&](int i) { return beam_key(beam_element<DT>(rowp, bias, 0, from + i), (uint32_t)(from + i)); },
                    until - from, N);
    }
    if (t < N) {
        keys[t] = s.out[t];
    }
    if (t == 0) {
        double sum = 0.0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            sum += red[w];
        }
        psum[(size_t)row * parts + part] = sum;
        if (part == 0) {
            pmax[row] = m;
        }
    }
}

struct BeamHypsDevice {
    int*         output_ids_tgt;
    int*         sequence_lengths_tgt;
    float*       cum_log_probs;
    float*       normed_scores;
    float*       log_probs;
    float*       min_normed_scores;
    int*         num_beams;
    bool*        is_done;
    const int*   output_ids_src;
    const int*   parent_ids_src;
    const int*   end_ids;
    const float* log_probs_src;
    int          step;
    int          ite;
    int          batch_size;
    int          local_batch_size;
    int          max_seq_len;
    int          early_stopping;
};

// Where the rows' candidates come from: a list per row, ranked and valued (parts == 0), or per part of a row (1 to 8)
// its best keys in order and its sum, with the row's maximum.
struct BeamCandidates {
    const int*                id;
    const float*              val;
    int                       parts;
    const float*              pmax;
    const double*             psum;
    const unsigned long long* pkeys;
    const int2*               before;  // per row: finished and length before the step
};

// What a whole step does after the beams are chosen (all of it, or nothing: parent_ids == nullptr)
struct BeamUpdate {
    bool*      finished;
    int*       sequence_length;
    int*       parent_ids;
    int*       cache_tgt;  // nullptr: the cache indirection is left to a launch of its own
    const int* cache_src;
    int        start_step, num_steps, max_seq_len, step;
};

constexpr int BB_HISTORY = 1024;  // (step, beam) pairs of the history kept in LDS
constexpr int BB_MERGED  = 1024;  // keys of an entry that are merged here
constexpr int BB_SHARED  = 512;   // the same where rows are shared: two per thread
constexpr int BB_CACHE   = 4096;  // cache positions of an entry that are copied here: 16 per thread

// One workgroup per batch entry (:99-262). Bound by latency: a few hundred candidates and one thread that walks the
// best of them. So everything the walk may read is requested before anything is computed - the hypotheses' state and
// the last BB_HISTORY (step, beam) pairs of tokens, parents and log-probs among it, through which a finished beam is
// traced in LDS instead of one dependent read per step - and the launches that followed it (token and parent split,
// flags, lengths, cache indirection: 4.4 and 3.6 us of mostly latency) are its last lines.
// 32 entries of 4 beams: 16.8 us in three launches, 9.7 us here (traced); the step 34 -> 25 us.
template<int DT>
__global__ void __launch_bounds__(BM_THREADS)
beam_batch_kernel(BeamCandidates cd, int* ids, float* cum_log_probs, float* __restrict__ output_log_probs,
                  const int* __restrict__ end_ids, BeamHypsDevice h, BeamUpdate up, int K, int max_k2, int vocab,
                  float length_penalty, float diversity_rate)
{
    __shared__ BeamSelect s;
    __shared__ float      old_cum[64];
    __shared__ float      normed[BM_MAX_N];
    __shared__ int        hist_id[BB_HISTORY], hist_parent[BB_HISTORY];
    __shared__ float      hist_lp[BB_HISTORY];
    __shared__ int        cand_x[BM_MAX_N], cand_beam[BM_MAX_N], cand_ends[BM_MAX_N];
    __shared__ float      cand_y[BM_MAX_N], score_of[BM_MAX_N];
    __shared__ int        chosen[WAVE], counted[WAVE], parent_of[WAVE], live[WAVE];
    __shared__ int        complete;  // the entry has its beam_width hypotheses
    __shared__ int        merged_id[BB_MERGED];
    __shared__ float      merged_val[BB_MERGED];
    __shared__ int        cached[BB_MERGED];
    __shared__ float      row_max[WAVE], row_logd[WAVE];
    const int             b         = blockIdx.x;
    const int             t         = threadIdx.x;
    const int             N         = 2 * K;
    const int             C         = K * N;
    const bool            with_hyps = h.num_beams != nullptr;
    const bool            updates   = up.parent_ids != nullptr;
    const int             g         = h.ite * h.local_batch_size + b;
    // ---- what is read, all of it requested before the first value is used (indices of idle threads are clamped: a
    // branch per thread would make every group of loads wait for the one before)
    const int   nb0     = with_hyps ? h.num_beams[g] : 0;
    const int   nb_here = with_hyps ? h.num_beams[b] : 0;
    const float mn0     = with_hyps ? h.min_normed_scores[g] : 0.0f;
    const int   end_h   = with_hyps ? h.end_ids[b] : -1;
    const int   end_u   = end_ids[b];
    const int2  before  = cd.before[b];
    const int   own     = b * K + min(t, K - 1);
    const float r_cum   = cum_log_probs[own];
    int         r_id = 0, r_len = 0;
    bool        r_fin = false;
    if (updates) {
        r_id  = ids[own];
        r_len = up.sequence_length[own];
        r_fin = up.finished[own];
    }
    constexpr int      TURNS   = BB_MERGED / BM_THREADS;
    const int          per_row = cd.parts * N;
    const int          n_keys  = K * per_row;
    unsigned long long r_key[TURNS];
    double             r_sum = 0.0;
    float              r_max = 0.0f;
    if (cd.parts > 0) {
#pragma unroll
        for (int u = 0; u < TURNS; ++u) {
            if (u * BM_THREADS < n_keys) {
                r_key[u] = cd.pkeys[(size_t)b * n_keys + min(t + u * BM_THREADS, n_keys - 1)];
            }
        }
        r_sum = cd.psum[(size_t)b * K * cd.parts + min(t, K * cd.parts - 1)];  // (2 K K parts <= BB_MERGED: one wave has all)
        r_max = cd.pmax[own];
    }
    const int  kept    = with_hyps ? min(h.step, BB_HISTORY / K) : 0;  // steps of the history in LDS: the last ones
    const bool with_lp = h.log_probs != nullptr && h.log_probs_src != nullptr;
    float      r_normed = 0.0f;
    int        r_hid[TURNS], r_hparent[TURNS];
    float      r_hlp[TURNS];
    if (with_hyps) {
        r_normed = h.normed_scores[(size_t)g * N + min(t, N - 1)];
#pragma unroll
        for (int u = 0; u < TURNS; ++u) {
            if (u * BM_THREADS < kept * K) {
                const int    i   = min(t + u * BM_THREADS, kept * K - 1);
                const size_t src = (size_t)(h.step - kept + i / K) * h.batch_size * K + (size_t)g * K + i % K;
                r_hid[u]         = h.output_ids_src[src];
                r_hparent[u]     = h.parent_ids_src[src];
                r_hlp[u]         = with_lp ? h.log_probs_src[src] : 0.0f;
            }
        }
    }
    const bool cache_here = up.cache_tgt != nullptr && K * up.num_steps <= BB_MERGED;  // its source goes to LDS, too
    int        r_cache[TURNS];
    if (cache_here) {
#pragma unroll
        for (int u = 0; u < TURNS; ++u) {
            if (u * BM_THREADS < K * up.num_steps) {
                const int i    = min(t + u * BM_THREADS, K * up.num_steps - 1);
                const int circ = (up.start_step + i % up.num_steps) % up.max_seq_len;
                r_cache[u]     = up.cache_src[((size_t)b * K + i / up.num_steps) * up.max_seq_len + circ];
            }
        }
    }
    // ---- and kept
    if (t < K) {
        old_cum[t] = r_cum;
        if (updates) {
            chosen[t]  = r_id;  // (kept where the walk chooses nothing)
            counted[t] = r_fin ? r_len : r_len + 1;
        }
        if (cd.parts > 0) {
            row_max[t] = r_max;
        }
    }
    if (with_hyps) {
        if (t < N) {
            normed[t] = r_normed;
        }
#pragma unroll
        for (int u = 0; u < TURNS; ++u) {
            const int i = t + u * BM_THREADS;
            if (i < kept * K) {
                hist_id[i]     = r_hid[u];
                hist_parent[i] = r_hparent[u];
                hist_lp[i]     = r_hlp[u];
            }
        }
    }
    if (cache_here) {
#pragma unroll
        for (int u = 0; u < TURNS; ++u) {
            const int i = t + u * BM_THREADS;
            if (i < K * up.num_steps) {
                cached[i] = r_cache[u];
            }
        }
    }
    const int*   x = cd.id + (size_t)b * C;
    const float* y = cd.val + (size_t)b * C;
    if (cd.parts > 0) {
        if (t < WAVE) {
            // a row's sums lie in neighbouring lanes; added and turned into a logarithm once per row
            double d = 0.0;
            for (int p = 0; p < cd.parts; ++p) {
                d += __shfl(r_sum, min(t * cd.parts + p, WAVE - 1), WAVE);
            }
            if (t < K) {
                row_logd[t] = det_logf((float)d);
            }
        }
#pragma unroll
        for (int u = 0; u < TURNS; ++u) {
            const int i = t + u * BM_THREADS;
            if (i < n_keys) {
                s.cand[i] = r_key[u];
            }
        }
        __syncthreads();
        for (int i = t; i < n_keys; i += BM_THREADS) {
            const unsigned long long k     = s.cand[i];
            const int                r     = i / per_row;
            int                      place = i - r * per_row;
            if (cd.parts > 1) {
                // its rank among the row's keys, four looked at at a time
                const ulonglong2* pairs = reinterpret_cast<const ulonglong2*>(s.cand + r * per_row);
                place                   = 0;
#pragma unroll 2
                for (int j = 0; j < per_row / 4; ++j) {
                    const ulonglong2 m = pairs[2 * j];
                    const ulonglong2 n = pairs[2 * j + 1];
                    place += (m.x > k ? 1 : 0) + (m.y > k ? 1 : 0) + (n.x > k ? 1 : 0) + (n.y > k ? 1 : 0);
                }
            }
            // (a finished row's other parts hold zeros, below the first part's 2K keys: they get no place)
            if (place < N && k != 0ull) {
                merged_id[r * N + place] = (int)beam_key_position(k) + (b * K + r) * vocab;
                merged_val[r * N + place] =
                    round_t<DT>((beam_key_value(k) - row_max[r] - row_logd[r]) + old_cum[r]);
            }
        }
        x = merged_id;
        y = merged_val;
    }
    __syncthreads();
    const bool  skip = with_hyps && nb0 == K;
    const float none = 3.402823466e+38f;
    if (!skip) {
        // (:146-156) the batch entry's own flag and length are used for all of its beams, as in the reference
        float denom = 1.0f;
        if (length_penalty != 0.0f) {
            const int length = before.x != 0 ? before.y : before.y + 1;
            if (length != 1) {
                denom = round_t<DT>(det_expf(length_penalty * det_logf((float)length)));
            }
            else {
                length_penalty = 0.0f;
            }
        }
        const float div_t = round_t<DT>(diversity_rate);
        auto        score = [&](int c) {
            float elem = y[c];
            if (length_penalty != 0.0f) {
                elem = round_t<DT>(elem / denom);
            }
            return round_t<DT>(elem + round_t<DT>(div_t * round_t<DT>((float)(c % K))));
        };
        const int take = max_k2 < C ? max_k2 : C;
        beam_select(s, [&](int c) { return beam_key(score(c), (uint32_t)c); }, C, take);
        // what the walk asks about its candidates, worked out by one thread each
        if (t < take) {
            const int p  = (int)beam_key_position(s.out[t]);
            score_of[t]  = score(p);
            cand_x[t]    = x[p];
            cand_y[t]    = y[p];
            cand_beam[t] = (cand_x[t] / vocab) % K;
            cand_ends[t] = with_hyps && cand_x[t] % vocab == end_h ? 1 : 0;
        }
        __syncthreads();
        if (t == 0) {
            float* v        = cum_log_probs + (size_t)b * K;
            int    selected = 0;
            int    nb       = nb0;
            float  mn       = nb0 == 0 ? none : mn0;
            bool   closed   = false;
            for (int i = 0; i < take; ++i) {
                const int   xp = cand_x[i];
                const float yp = cand_y[i];
                if (cand_ends[i] != 0) {
                    if (i < K) {
                        const float normed_score = score_of[i];
                        int         beam_idx     = nb;
                        if (nb == K) {
                            if (normed_score < mn) {
                                break;
                            }
                            for (int j = 0; j < K; ++j) {
                                if (normed[j] == mn) {
                                    beam_idx = j;
                                    nb--;
                                    mn        = none;
                                    normed[j] = normed_score;
                                    for (int l = 0; l < K; ++l) {
                                        mn = __builtin_fminf(mn, normed[l]);
                                    }
                                    break;
                                }
                            }
                        }
                        const int    tgt_beam = g * N + beam_idx;
                        const size_t tgt      = (size_t)tgt_beam * h.max_seq_len;
                        int          prev_id  = cand_beam[i];
                        h.output_ids_tgt[tgt + h.step] = end_h;
                        if (h.log_probs != nullptr) {
                            h.log_probs[tgt + h.step] = yp - old_cum[prev_id];
                        }
                        for (int j = h.step - 1; j >= 0; --j) {
                            const int back = j - (h.step - kept);
                            int       id, parent;
                            float     lp = 0.0f;
                            // (a parent outside the beams of an entry - the caller's arrays are not checked - is
                            // looked up in them like before)
                            if (back >= 0 && prev_id >= 0 && prev_id < K) {
                                id     = hist_id[back * K + prev_id];
                                parent = hist_parent[back * K + prev_id];
                                lp     = hist_lp[back * K + prev_id];
                            }
                            else {
                                const size_t src = (size_t)j * h.batch_size * K + (size_t)g * K + prev_id;
                                id               = h.output_ids_src[src];
                                parent           = h.parent_ids_src[src];
                                if (with_lp) {
                                    lp = h.log_probs_src[src];
                                }
                            }
                            h.output_ids_tgt[tgt + j] = id;
                            if (with_lp) {
                                h.log_probs[tgt + j] = lp;
                            }
                            prev_id = parent;
                        }
                        h.sequence_lengths_tgt[tgt_beam] = h.step;
                        h.normed_scores[tgt_beam]        = normed_score;
                        normed[beam_idx]                 = normed_score;
                        mn                               = __builtin_fminf(mn, normed_score);
                        nb++;
                        h.cum_log_probs[tgt_beam] = yp;
                    }
                }
                else if ((with_hyps && i < N) || (!with_hyps && i < K)) {
                    if (updates) {
                        chosen[selected] = xp;
                    }
                    else {
                        ids[(size_t)b * K + selected] = xp;
                    }
                    if (output_log_probs != nullptr) {
                        output_log_probs[b * K + selected] = yp - old_cum[cand_beam[i]];
                    }
                    v[selected] = yp;
                    selected++;
                }
                if (selected >= K) {
                    break;
                }
            }
            if (with_hyps) {
                if (nb0 == 0 || nb != nb0 || mn != mn0) {
                    h.min_normed_scores[g] = mn;
                }
                if (nb != nb0) {
                    h.num_beams[g] = nb;
                }
                closed         = (g == b ? nb : nb_here) >= K;
                if (!closed) {
                    h.is_done[b] = false;
                }
                else if (h.early_stopping) {
                    h.is_done[b] = true;
                }
            }
            complete = with_hyps && nb == K ? 1 : 0;
        }
    }
    else if (t == 0) {
        complete = 1;
    }
    if (!updates) {
        return;
    }
    __syncthreads();
    // layers/beam_search_layers/OnlineBeamSearchLayer.cu:24-61, as beam_update_kernel
    if (t < K) {
        const int  i       = b * K + t;
        const int  word    = chosen[t];
        const int  end_id  = end_u;
        const bool valid   = word >= 0;  // (as there: a slot left untouched holds whatever the buffer held)
        const int  beam_id = valid ? (word / vocab) % K : t;
        const int  word_id = valid ? word % vocab : end_id;
        const bool done    = complete != 0 || word_id == end_id;
        up.sequence_length[i] = counted[beam_id];
        up.finished[i]        = done;
        up.parent_ids[i]      = beam_id;
        ids[i]                = word_id;
        parent_of[t]          = beam_id;
        live[t]               = done ? 0 : 1;
    }
    if (up.cache_tgt == nullptr) {
        return;
    }
    __syncthreads();
    // layers/beam_search_layers/BaseBeamSearchLayer.cu:22-49, as beam_indir_cache_kernel
    for (int i = t; i < K * up.num_steps; i += BM_THREADS) {
        const int beam = i / up.num_steps;
        if (live[beam] != 0) {
            const int    time_step = up.start_step + i % up.num_steps;
            const int    circ      = time_step % up.max_seq_len;
            const size_t base      = (size_t)b * K * up.max_seq_len + circ;
            const int    from      = parent_of[beam];
            const int    value     = cache_here ? cached[from * up.num_steps + i % up.num_steps] :
                                                  up.cache_src[base + (size_t)from * up.max_seq_len];
            up.cache_tgt[base + (size_t)beam * up.max_seq_len] = time_step == up.step ? beam : value;
        }
    }
}

// ---- the kernels around the step -----------------------------------------------------------------------------
// kernels/beam_search_penalty_kernels.cu:24-86 (add_bias_temperature, generic and half2 forms): one workgroup per
// (chunk, row); pad columns are masked in both forms here (the sampling layers' half2 form leaves them alone).
template<int DT>
__global__ void __launch_bounds__(BM_THREADS)
beam_bias_temperature_kernel(typename Storage<DT>::T* __restrict__ logits,
                             const typename Storage<DT>::T* __restrict__ bias, int V, int Vp, int chunk,
                             float temperature)
{
    typedef Storage<DT>   S;
    const int             row   = blockIdx.y;
    const float           inv   = 1.0f / (temperature + 1e-6f);
    const float           inv_t = round_t<DT>(inv);
    const bool            pairs = DT == DT_F16 && V % 2 == 0 && Vp % 2 == 0;
    const int             lo    = min(Vp, (int)blockIdx.x * chunk);
    const int             hi    = min(Vp, lo + chunk);
    typename S::T*        rowp  = logits + (size_t)row * Vp;
    transform_columns<DT, BM_THREADS>(rowp, lo, hi, [&](int v, float x) {
        if (v >= V) {
            return -S::max_t();
        }
        if (pairs) {
            const float y = bias != nullptr ? round_t<DT>(x + S::ld(bias[v])) : x;
            return y * inv_t;
        }
        const float b = bias != nullptr ? S::ld(bias[v]) : 0.0f;
        return round_t<DT>(x + b) * (DT == DT_F32 ? inv : inv_t);
    });
}

// :88-154 (apply_repetition_penalty): one workgroup per beam; thread 0 follows the beam back through parent_ids and
// computes every penalised value from the row as it is, then all threads store. Dynamic LDS: step values and ids.
template<int DT>
__global__ void __launch_bounds__(BM_THREADS)
beam_repetition_kernel(typename Storage<DT>::T* __restrict__ logits, int batch_size, int K, int Vp, int step,
                       const int* __restrict__ current_ids, const int* __restrict__ previous_ids,
                       const int* __restrict__ parent_ids, const int* __restrict__ input_lengths,
                       int max_input_length, float repetition_penalty, int additive)
{
    typedef Storage<DT>   S;
    extern __shared__ int beam_hist[];  // [step] ids, then [step] values
    int*                  idx  = beam_hist;
    float*                val  = reinterpret_cast<float*>(beam_hist + step);
    const int             t    = threadIdx.x;
    const int             r    = blockIdx.x;
    const int             b    = r / K;
    typename S::T*        row  = logits + (size_t)r * Vp;
    const int             len  = input_lengths != nullptr ? input_lengths[r] : max_input_length;
    if (t == 0) {
        const int   bbsize = batch_size * K;
        const float pen    = round_t<DT>(repetition_penalty);
        auto        penalised = [&](float x) {
            if (additive) {
                return round_t<DT>(x - pen);
            }
            return x > 0.0f ? round_t<DT>(x / pen) : round_t<DT>(x * pen);
        };
        int prev_id   = current_ids[r];
        idx[step - 1] = prev_id;
        val[step - 1] = penalised(S::ld(row[prev_id]));
        int beam      = r % K;
        for (int i = step - 2; i >= 0; --i) {
            if (i >= len && i < max_input_length) {
                continue;
            }
            beam    = parent_ids[(size_t)i * bbsize + b * K + beam];
            prev_id = previous_ids[(size_t)i * bbsize + b * K + beam];
            idx[i]  = prev_id;
            val[i]  = penalised(S::ld(row[prev_id]));
        }
    }
    __syncthreads();
    for (int i = t; i < step; i += BM_THREADS) {
        if (i >= len && i < max_input_length) {
            continue;
        }
        row[idx[i]] = S::st(val[i]);
    }
}

// :156-173 (apply_min_length_penalty)
template<int DT>
__global__ void beam_min_length_kernel(typename Storage<DT>::T* __restrict__ logits, int min_length,
                                       const int* __restrict__ end_ids, const int* __restrict__ sequence_lengths,
                                       int max_input_length, int K, int Vp, int rows)
{
    const int r = threadIdx.x + blockIdx.x * blockDim.x;
    if (r < rows && sequence_lengths[r] + 1 - max_input_length < min_length) {
        logits[(size_t)r * Vp + end_ids[r / K]] = Storage<DT>::st(-Storage<DT>::max_t());
    }
}

// layers/beam_search_layers/OnlineBeamSearchLayer.cu:24-61 (update_kernel): one wave per batch entry, so that what
// the reference leaves to the order of its threads is fixed: every row counts its token, then takes the length of
// the beam it continues; an entry with beam_width hypotheses is finished.
__global__ void __launch_bounds__(WAVE)
beam_update_kernel(bool* __restrict__ finished, int* __restrict__ parent_ids, int* __restrict__ sequence_length,
                   int* word_ids, int* output_ids, const int* __restrict__ num_beams, int ite, int hyps_local_batch,
                   int K, int Vp, const int* __restrict__ end_ids)
{
    __shared__ int counted[WAVE];
    const int      b = blockIdx.x;
    const int      k = threadIdx.x;
    const int      i = b * K + k;
    int            word = 0;
    if (k < K) {
        counted[k] = finished[i] ? sequence_length[i] : sequence_length[i] + 1;
        word       = word_ids[i];
    }
    __syncthreads();
    if (k < K) {
        // A slot the step left untouched (an entry that is complete, or one with fewer than K continuations) holds
        // whatever the caller's buffer held: a negative value counts as "this beam, its end token", so that no index
        // below leaves its range (the reference reads other rows' memory there; ids are absolute over the batch,
        // (entry * K + beam) * Vp + token, and any non-negative one is brought into range by the modulo).
        const bool valid   = word >= 0;
        const int  beam_id = valid ? (word / Vp) % K : k;
        const int  word_id = valid ? word % Vp : end_ids[b];
        const bool done    = num_beams != nullptr && num_beams[ite * hyps_local_batch + b] == K;
        sequence_length[i] = counted[beam_id];
        finished[i]        = done || word_id == end_ids[b];
        parent_ids[i]      = beam_id;
        word_ids[i]        = word_id;
        output_ids[i]      = word_id;
    }
}

// layers/beam_search_layers/BaseBeamSearchLayer.cu:22-49 (update_indir_cache_kernel)
__global__ void beam_indir_cache_kernel(int* __restrict__ tgt, const int* __restrict__ src,
                                        const int* __restrict__ beam_ids, const bool* __restrict__ finished,
                                        int start_step, int local_batch_size, int K, int max_seq_len, int step)
{
    int       time_step = threadIdx.x + blockIdx.x * blockDim.x;
    const int bb        = blockIdx.y;
    const int b         = bb / K;
    const int beam      = bb % K;
    if (bb >= K * local_batch_size || time_step >= min(step + 1, max_seq_len) || finished[bb]) {
        return;
    }
    time_step += start_step;
    const int    circ     = time_step % max_seq_len;
    const int    src_beam = beam_ids[b * K + beam];
    const size_t t_off    = (size_t)b * K * max_seq_len + (size_t)beam * max_seq_len + circ;
    const size_t s_off    = (size_t)b * K * max_seq_len + (size_t)src_beam * max_seq_len + circ;
    tgt[t_off]            = time_step == step ? beam : src[s_off];
}

}  // namespace ftk

using namespace ftk;

constexpr int BR_SHORT_ROW = 65536;
constexpr int BR_MANY_ROWS = 192;
#ifdef FTK_TEST_HOOKS
// Test hook (hooks build of the library only): 1 = sections of rows and three launches everywhere, 2 = one
// 1024-thread workgroup per row everywhere, 3 = one 512-thread workgroup per row everywhere, 0 = by the shape.
static int g_beam_path = 0;
extern "C" void ftk_test_set_beam_path(int v)
{
    g_beam_path = v;
}
#endif

// How many workgroups share a row of beam_team_kernel: as many as the compute units allow, as long as every part has at
// least 4096 columns to itself and an entry's keys fit the merge. Rows too long for the registers, and more rows than
// compute units, take the other forms (0). Requests of four steps through the layer, fp16, us, other forms / this one:
//   32 x 4 x 50257, two parts        124 / 106    (8192 columns, one part: 86 / 87)
//    8 x 4 x 50257, eight parts      117 / 94     (32000 columns, four parts: 102 / 89)
//   64 x 4 x 50257, one part         132 / 126    (fp32: 160 / 139)
//    1 x 8 x 50257, four parts       127 / 106    (8192 columns, two parts: 91 / 91)
//    8 x 16 x 50257, one part        186 / 180    (8192 columns: 146 / 146)
// Where rows are shared a merge takes two keys per thread at most: with four, ranked one by one, the last two took 186 and
// 211 us.
static int beam_team_parts(int rows, int beam_width, int vocab, const BeamPlan& plan)
{
    if (vocab > BT_COLUMNS || rows > 256) {
        return 0;
    }
    int parts = 1;
    while (parts < BT_MAX_PARTS && 2 * parts * rows <= 256 && vocab / (2 * parts) >= 4096 && 2 * parts <= plan.parts) {
        parts *= 2;
    }
    while (parts > 0 && 2 * beam_width * beam_width * parts > (parts > 1 ? BB_SHARED : BB_MERGED)) {
        parts /= 2;
    }
    return parts;
}

static int beam_step(int dtype, const void* log_probs, const void* bias, const bool* finished,
                     const int* sequence_lengths, float* cum_log_probs, float* output_log_probs, int* ids,
                     void* temp_storage, size_t* temp_storage_size, const ftk_beam_hypotheses* beam_hyps,
                     int batch_size, int beam_width, int vocab_size, const int* end_ids, float diversity_rate,
                     float length_penalty, BeamUpdate up, ftk_stream_t stream)
{
    if (dtype < 0 || dtype > 2) {
        return FTK_ERR_DTYPE;
    }
    if (beam_width < 2 || beam_width > 64) {
        return FTK_ERR_ARGUMENT;  // the reference's launcher covers 1..64 (:650-688) and rejects 1 (:625)
    }
    if (batch_size < 0 || vocab_size < 2 * beam_width || (long long)batch_size * beam_width > 65535
        || (long long)batch_size * beam_width * vocab_size > 0x7FFFFFFFll) {
        return FTK_ERR_ARGUMENT;  // candidate ids are row * vocab + token in an int, as in the reference
    }
    const int      rows = batch_size * beam_width;
    const BeamPlan plan = beam_plan(rows, beam_width, vocab_size);
    if (temp_storage == nullptr) {
        if (temp_storage_size == nullptr) {
            return FTK_ERR_ARGUMENT;
        }
        *temp_storage_size = plan.bytes;
        return 0;
    }
    if (temp_storage_size != nullptr && *temp_storage_size < plan.bytes) {
        return FTK_ERR_WORKSPACE;
    }
    if (batch_size == 0) {
        return 0;
    }
    if (length_penalty != 0.0f && sequence_lengths == nullptr) {
        return FTK_ERR_ARGUMENT;  // (:572)
    }
    if (log_probs == nullptr || finished == nullptr || cum_log_probs == nullptr || ids == nullptr
        || end_ids == nullptr) {
        return FTK_ERR_ARGUMENT;  // the reference's kernels read and write all of these
    }
    if (beam_hyps != nullptr && beam_hyps->num_beams != nullptr
        && (beam_hyps->output_ids_tgt == nullptr || beam_hyps->sequence_lengths_tgt == nullptr
            || beam_hyps->cum_log_probs == nullptr || beam_hyps->normed_scores == nullptr
            || beam_hyps->min_normed_scores == nullptr || beam_hyps->is_done == nullptr
            || beam_hyps->end_ids == nullptr
            || (beam_hyps->step > 0 && (beam_hyps->output_ids_src == nullptr || beam_hyps->parent_ids_src == nullptr))
            || beam_hyps->step < 0 || beam_hyps->step >= beam_hyps->max_seq_len)) {
        return FTK_ERR_ARGUMENT;  // a hypothesis is written at position `step` of a max_seq_len-long row
    }
    char*               ws       = (char*)temp_storage;
    float*              pmax     = (float*)(ws + plan.off_pmax);
    double*             psum     = (double*)(ws + plan.off_psum);
    unsigned long long* pkeys    = (unsigned long long*)(ws + plan.off_pkeys);
    int*                cand_id  = (int*)(ws + plan.off_cand_id);
    float*              cand_val = (float*)(ws + plan.off_cand_val);
    hipStream_t         st       = (hipStream_t)stream;
    const int           N        = 2 * beam_width;
    const int           max_k    = beam_width <= 4 ? 4 : beam_width <= 8 ? 8 : beam_width <= 16 ? 16 : beam_width <= 32 ? 32 : 64;
    BeamHypsDevice      h        = {};
    if (beam_hyps != nullptr) {
        h.output_ids_tgt       = beam_hyps->output_ids_tgt;
        h.sequence_lengths_tgt = beam_hyps->sequence_lengths_tgt;
        h.cum_log_probs        = beam_hyps->cum_log_probs;
        h.normed_scores        = beam_hyps->normed_scores;
        h.log_probs            = beam_hyps->log_probs;
        h.min_normed_scores    = beam_hyps->min_normed_scores;
        h.num_beams            = beam_hyps->num_beams;
        h.is_done              = beam_hyps->is_done;
        h.output_ids_src       = beam_hyps->output_ids_src;
        h.parent_ids_src       = beam_hyps->parent_ids_src;
        h.end_ids              = beam_hyps->end_ids;
        h.log_probs_src        = beam_hyps->log_probs_src;
        h.step                 = beam_hyps->step;
        h.ite                  = beam_hyps->ite;
        h.batch_size           = beam_hyps->batch_size;
        h.local_batch_size     = beam_hyps->local_batch_size;
        h.max_seq_len          = beam_hyps->max_seq_len;
        h.early_stopping       = beam_hyps->early_stopping ? 1 : 0;
    }
    int2*      before = (int2*)(ws + plan.off_before);
    const dim3 sections(plan.parts, rows);
    // A few long rows would leave most compute units idle with one workgroup each: they go in sections (measured on
    // MI355X, f16: 32 rows of 128256 take 40 us in one launch and 34 us in sections; 512 rows of 152064 112 against
    // 115 us).
    int  team        = beam_team_parts(rows, beam_width, vocab_size, plan);
    bool one_per_row = vocab_size <= BR_SHORT_ROW || rows >= BR_MANY_ROWS;
    bool half_size   = rows > 256;  // two 512-thread workgroups per compute unit
#ifdef FTK_TEST_HOOKS
    team        = g_beam_path == 0 ? team : 0;
    one_per_row = g_beam_path == 0 ? one_per_row : g_beam_path >= 2;
    half_size   = g_beam_path <= 1 ? half_size : g_beam_path == 3;
#endif
    const BeamCandidates cd{cand_id, cand_val, team, pmax, psum, pkeys, before};
    FTK_DISPATCH_DTYPE(dtype, {
        typedef Storage<DT>::T T;
        if (team > 0) {
            beam_team_kernel<DT><<<dim3(rows, team), BR_THREADS, 0, st>>>((const T*)log_probs, (const T*)bias, finished,
                                                                          end_ids, sequence_lengths, vocab_size,
                                                                          beam_width, pmax, psum, pkeys, before);
            FTK_LAUNCH_CHECK();
        }
        else if (one_per_row && half_size) {
            beam_rowwide_kernel<DT, BR_THREADS / 2><<<rows, BR_THREADS / 2, 0, st>>>(
                (const T*)log_probs, (const T*)bias, finished, end_ids, cum_log_probs, vocab_size, beam_width, cand_id,
                cand_val, sequence_lengths, before);
            FTK_LAUNCH_CHECK();
        }
        else if (one_per_row) {
            beam_rowwide_kernel<DT, BR_THREADS><<<rows, BR_THREADS, 0, st>>>(
                (const T*)log_probs, (const T*)bias, finished, end_ids, cum_log_probs, vocab_size, beam_width, cand_id,
                cand_val, sequence_lengths, before);
            FTK_LAUNCH_CHECK();
        }
        else {
            beam_section_max_kernel<DT><<<sections, BM_THREADS, 0, st>>>((const T*)log_probs, (const T*)bias, finished,
                                                                         vocab_size, plan.section, pmax);
            FTK_LAUNCH_CHECK();
            beam_section_kernel<DT><<<sections, BM_THREADS, 0, st>>>((const T*)log_probs, (const T*)bias, finished,
                                                                     vocab_size, plan.section, N, pmax, psum, pkeys);
            FTK_LAUNCH_CHECK();
            beam_row_kernel<DT><<<rows, BM_THREADS, 0, st>>>(finished, end_ids, cum_log_probs, vocab_size, beam_width,
                                                             plan.parts, pmax, psum, pkeys, cand_id, cand_val,
                                                             sequence_lengths, before);
            FTK_LAUNCH_CHECK();
        }
        beam_batch_kernel<DT><<<batch_size, BM_THREADS, 0, st>>>(cd, ids, cum_log_probs, output_log_probs, end_ids, h,
                                                                 up, beam_width, 2 * max_k, vocab_size, length_penalty,
                                                                 diversity_rate);
        FTK_LAUNCH_CHECK();
    });
    return 0;
}

extern "C" {

int ftk_invoke_topk_softmax(int dtype, const void* log_probs, const void* bias, const bool* finished,
                            const int* sequence_lengths, float* cum_log_probs, float* output_log_probs, int* ids,
                            void* temp_storage, size_t* temp_storage_size, const ftk_beam_hypotheses* beam_hyps,
                            int batch_size, int beam_width, int vocab_size, const int* end_ids, float diversity_rate,
                            float length_penalty, ftk_stream_t stream)
{
    return beam_step(dtype, log_probs, bias, finished, sequence_lengths, cum_log_probs, output_log_probs, ids,
                     temp_storage, temp_storage_size, beam_hyps, batch_size, beam_width, vocab_size, end_ids,
                     diversity_rate, length_penalty, BeamUpdate{}, stream);
}

int ftk_fused_beam_step(int dtype, const void* log_probs, bool* finished, int* sequence_lengths, float* cum_log_probs,
                        float* output_log_probs, int* ids, int* parent_ids, int* tgt_indir_cache,
                        const int* src_indir_cache, void* temp_storage, size_t temp_storage_size,
                        const ftk_beam_hypotheses* beam_hyps, int batch_size, int beam_width, int vocab_size,
                        int max_seq_len, int step, const int* end_ids, float diversity_rate, float length_penalty,
                        ftk_stream_t stream)
{
    if (temp_storage == nullptr) {
        return FTK_ERR_WORKSPACE;
    }
    if (max_seq_len < 1 || step < 0
        || (batch_size > 0
            && (sequence_lengths == nullptr || parent_ids == nullptr || tgt_indir_cache == nullptr
                || src_indir_cache == nullptr))) {
        return FTK_ERR_ARGUMENT;
    }
    BeamUpdate up{};
    up.finished        = finished;
    up.sequence_length = sequence_lengths;
    up.parent_ids      = parent_ids;
    up.max_seq_len     = max_seq_len;
    up.step            = step;
    up.start_step      = step + 1 - max_seq_len > 0 ? step + 1 - max_seq_len : 0;
    up.num_steps       = step + 1 < max_seq_len ? step + 1 : max_seq_len;
    // a long cache is copied by as many workgroups as it needs, in a launch of its own
    const bool copies = (long long)beam_width * up.num_steps <= BB_CACHE;
    if (copies) {
        up.cache_tgt = tgt_indir_cache;
        up.cache_src = src_indir_cache;
    }
    const int rc = beam_step(dtype, log_probs, nullptr, finished, sequence_lengths, cum_log_probs, output_log_probs, ids,
                             temp_storage, &temp_storage_size, beam_hyps, batch_size, beam_width, vocab_size, end_ids,
                             diversity_rate, length_penalty, up, stream);
    if (rc != 0 || copies) {
        return rc;
    }
    return ftk_invoke_update_indir_cache(tgt_indir_cache, src_indir_cache, parent_ids, finished, batch_size, batch_size,
                                         beam_width, max_seq_len, step, stream);
}

int ftk_invoke_add_bias_apply_penalties(int dtype, int step, void* logits, const int* current_ids,
                                        const int* previous_ids, const int* parent_ids, const int* input_lengths,
                                        const int* sequence_lengths, const void* bias, int ite, int max_input_length,
                                        int local_batch_size, int batch_size, int beam_width, int vocab_size,
                                        int vocab_size_padded, const int* end_ids, float temperature,
                                        float repetition_penalty, int repetition_penalty_type, int min_length,
                                        ftk_stream_t stream)
{
    if (dtype < 0 || dtype > 2) {
        return FTK_ERR_DTYPE;
    }
    if (local_batch_size < 0 || beam_width < 1 || vocab_size < 1 || vocab_size_padded < vocab_size || step < 0
        || (long long)local_batch_size * beam_width > 65535) {
        return FTK_ERR_ARGUMENT;
    }
    const int rows = local_batch_size * beam_width;
    if (rows == 0) {
        return 0;
    }
    if (logits == nullptr) {
        return FTK_ERR_ARGUMENT;
    }
    hipStream_t st = (hipStream_t)stream;
    if (bias != nullptr || temperature != 1.0f || vocab_size != vocab_size_padded) {
        int chunks = (1024 + rows - 1) / rows;
        chunks     = chunks < (vocab_size_padded + 8191) / 8192 ? chunks : (vocab_size_padded + 8191) / 8192;
        const int  chunk = ((vocab_size_padded + chunks - 1) / chunks + 7) / 8 * 8;
        const dim3 grid((vocab_size_padded + chunk - 1) / chunk, rows);
        FTK_DISPATCH_DTYPE(dtype, beam_bias_temperature_kernel<DT><<<grid, BM_THREADS, 0, st>>>(
                                      (Storage<DT>::T*)logits, (const Storage<DT>::T*)bias, vocab_size,
                                      vocab_size_padded, chunk, temperature));
        FTK_LAUNCH_CHECK();
    }
    const bool  additive = repetition_penalty_type == FTK_PENALTY_ADDITIVE;
    const float neutral  = repetition_penalty_type == FTK_PENALTY_MULTIPLICATIVE ? 1.0f : 0.0f;
    if (repetition_penalty_type != FTK_PENALTY_NONE && step > 0 && repetition_penalty != neutral) {
        if (current_ids == nullptr || (step > 1 && (previous_ids == nullptr || parent_ids == nullptr))) {
            return FTK_ERR_ARGUMENT;
        }
        const size_t smem = (size_t)step * 2 * sizeof(int);
        if (smem > 64 * 1024) {
            return FTK_ERR_ARGUMENT;  // a history of more than 8192 steps does not fit the kernel's table
        }
        FTK_DISPATCH_DTYPE(dtype, beam_repetition_kernel<DT><<<rows, BM_THREADS, smem, st>>>(
                                      (Storage<DT>::T*)logits, batch_size, beam_width, vocab_size_padded, step,
                                      current_ids, previous_ids,
                                      parent_ids != nullptr ? parent_ids + (size_t)ite * beam_width * local_batch_size :
                                                              nullptr,
                                      input_lengths, max_input_length, repetition_penalty, additive ? 1 : 0));
        FTK_LAUNCH_CHECK();
    }
    if (step - max_input_length < min_length) {
        if (sequence_lengths == nullptr || end_ids == nullptr) {
            return FTK_ERR_ARGUMENT;  // the reference checks the same two
        }
        FTK_DISPATCH_DTYPE(dtype, beam_min_length_kernel<DT><<<(rows + 255) / 256, 256, 0, st>>>(
                                      (Storage<DT>::T*)logits, min_length, end_ids, sequence_lengths, max_input_length,
                                      beam_width, vocab_size_padded, rows));
        FTK_LAUNCH_CHECK();
    }
    return 0;
}

int ftk_invoke_beam_update(bool* finished, int* parent_ids, int* sequence_length, int* word_ids, int* output_ids,
                           const ftk_beam_hypotheses* beam_hyps, int local_batch_size, int beam_width,
                           int vocab_size_padded, const int* end_ids, ftk_stream_t stream)
{
    if (local_batch_size < 0 || beam_width < 1 || beam_width > WAVE || vocab_size_padded < 1) {
        return FTK_ERR_ARGUMENT;
    }
    if (local_batch_size == 0) {
        return 0;
    }
    if (finished == nullptr || parent_ids == nullptr || sequence_length == nullptr || word_ids == nullptr
        || output_ids == nullptr || end_ids == nullptr) {
        return FTK_ERR_ARGUMENT;
    }
    const int* num_beams = beam_hyps != nullptr ? beam_hyps->num_beams : nullptr;
    beam_update_kernel<<<local_batch_size, WAVE, 0, (hipStream_t)stream>>>(
        finished, parent_ids, sequence_length, word_ids, output_ids, num_beams, beam_hyps != nullptr ? beam_hyps->ite : 0,
        beam_hyps != nullptr ? beam_hyps->local_batch_size : 0, beam_width, vocab_size_padded, end_ids);
    FTK_LAUNCH_CHECK();
    return 0;
}

int ftk_invoke_update_indir_cache(int* tgt_indir_cache, const int* src_indir_cache, const int* beam_ids,
                                  const bool* finished, int batch_dim, int local_batch_size, int beam_width,
                                  int max_seq_len, int step, ftk_stream_t stream)
{
    (void)batch_dim;
    if (local_batch_size < 0 || beam_width < 1 || max_seq_len < 1 || step < 0
        || (long long)local_batch_size * beam_width > 65535) {
        return FTK_ERR_ARGUMENT;
    }
    if (local_batch_size == 0) {
        return 0;
    }
    if (tgt_indir_cache == nullptr || src_indir_cache == nullptr || beam_ids == nullptr || finished == nullptr) {
        return FTK_ERR_ARGUMENT;
    }
    const int  start_step = step + 1 - max_seq_len > 0 ? step + 1 - max_seq_len : 0;
    const int  num_steps  = step + 1 < max_seq_len ? step + 1 : max_seq_len;
    const dim3 grid((num_steps + 63) / 64, local_batch_size * beam_width);
    beam_indir_cache_kernel<<<grid, 64, 0, (hipStream_t)stream>>>(tgt_indir_cache, src_indir_cache, beam_ids, finished,
                                                                  start_step, local_batch_size, beam_width, max_seq_len,
                                                                  step);
    FTK_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
