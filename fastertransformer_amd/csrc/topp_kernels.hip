// Masked softmax and top-p (nucleus) sampling.
//
// Reference behaviour restated (src/fastertransformer/kernels/sampling_topp_kernels.cu):
//   :1294-1345 addBiasSoftMax          - in-place masked softmax, result rounded to T
//   :801-860   topp_beam_topk_kernel   - arg-max shortcut when max prob >= top_p
//   :1106-1119 cub segmented sort      - stable descending sort of every row
//   :877-1004  topp_sampling           - inclusive prefix sum over 256-wide tiles, first crossing
//   :1381-1412 computeToppDecay
//
// The replacement orders only the part of a row in front of the draw (see the top-p section).
#include <algorithm>

#include "ftk_device.cuh"
#include "ftk_sampling.h"
#ifdef FTK_TEST_HOOKS
#include "ftk_test_hooks.h"
#endif
#include "ftk_topp.cuh"
#include "ftk_topp_sample.h"

namespace ftk {

// =============================================================================================
// softmax
// =============================================================================================
constexpr int SM_THREADS = 1024;

// The reference block has BLK = min(n, 1024) threads and thread t owns columns t, t+BLK, ...;
// summation order (reduce_kernel_utils.cuh:73-103) = sequential per thread, xor butterfly
// (16,8,4,2,1) inside each 32-lane group, lane-0 partials through shared memory, butterfly again.
// STATS_ONLY: stops after the sum and leaves (maximum, denominator) of the row in `stats`; the row itself is
// not written (softmax_finish_histogram_kernel divides).
template<int DT, bool STATS_ONLY>
__global__ void __launch_bounds__(SM_THREADS)
softmax_kernel(typename Storage<DT>::T* __restrict__ logits, const typename Storage<DT>::T* __restrict__ bias,
               const int* __restrict__ end_ids, const bool* __restrict__ finished, int n_padded, int n,
               float2* __restrict__ stats)
{
    typedef Storage<DT> S;
    __shared__ float    sh[32];
    __shared__ float    sh_bcast;
    const int           row    = blockIdx.x;
    const int           t      = threadIdx.x;
    const int           BLK    = min(n, SM_THREADS);
    const bool          active = t < BLK;
    const bool          fin    = finished != nullptr ? finished[row] : false;
    const int           end_id = fin ? end_ids[row] : -1;
    typename S::T*      rowp   = logits + (size_t)row * n_padded;
    const float         MAXT   = S::max_t();

    auto masked = [&](int v) -> float {
        if (v >= n) {
            return -MAXT;
        }
        if (fin) {
            return v == end_id ? MAXT : -MAXT;
        }
        const float b = bias != nullptr ? S::ld(bias[v]) : 0.0f;
        return round_t<DT>(S::ld(rowp[v]) + b);
    };

    if (!fin && bias == nullptr) {
        // Ordinary rows. The maximum and the final division do not depend on the order of the columns
        // and go through 16-byte accesses; the sum keeps the reference's order (thread t adds its
        // columns t, t + BLK, ... one after the other), eight or sixteen loads in flight.
        float mx = -3.402823466e+38f;
        stream_columns<DT, SM_THREADS>(rowp, 0, n, [&](int, float x) { mx = __builtin_fmaxf(mx, x + 0.0f); });
        if (n_padded > n) {
            mx = __builtin_fmaxf(mx, -MAXT);
        }
        mx = block_max<float, SM_THREADS / WAVE>(mx, sh, -3.402823466e+38f);
        if (BLK < 1024) {
            mx = __builtin_fmaxf(mx, -1e20f);
        }
        const float pad_e = round_t<DT>(det_expf_nonpos(-MAXT - mx));
        float       sum   = 0.0f;
        if (active) {
            constexpr int U = DT == DT_F32 ? 8 : 16;  // 2-byte loads move half as much per instruction
            int           v = t;
            for (; v + (U - 1) * BLK < n; v += U * BLK) {
                float x[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    x[u] = S::ld(rowp[v + u * BLK]);
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    sum += round_t<DT>(det_expf_nonpos((x[u] + 0.0f) - mx));
                }
            }
            for (; v < n; v += BLK) {
                sum += round_t<DT>(det_expf_nonpos((S::ld(rowp[v]) + 0.0f) - mx));
            }
            for (; v < n_padded; v += BLK) {
                sum += pad_e;
            }
        }
#pragma unroll
        for (int m = 16; m > 0; m >>= 1) {
            sum += __shfl_xor(sum, m, 32);
        }
        if ((t & 31) == 0) {
            sh[t >> 5] = sum;
        }
        __syncthreads();
        if (t < 32) {
            float v = ((float)t < (float)BLK / 32.0f) ? sh[t] : 0.0f;
#pragma unroll
            for (int m = 16; m > 0; m >>= 1) {
                v += __shfl_xor(v, m, 32);
            }
            if (t == 0) {
                sh_bcast = v;
            }
        }
        __syncthreads();
        const float denom = sh_bcast + 1e-6f;
        if constexpr (STATS_ONLY) {
            if (t == 0) {
                stats[row] = make_float2(mx, denom);
            }
            return;
        }
        const RowDivisor div(denom);
        if (div.ok) {
            transform_columns<DT, SM_THREADS>(rowp, 0, n, [&](int, float x) {
                return div.divide(round_t<DT>(det_expf_nonpos((x + 0.0f) - mx)));
            });
        }
        else {
            transform_columns<DT, SM_THREADS>(rowp, 0, n, [&](int, float x) {
                return round_t<DT>(det_expf_nonpos((x + 0.0f) - mx)) / denom;
            });
        }
        transform_columns<DT, SM_THREADS>(rowp, n, n_padded, [&](int, float) { return pad_e / denom; });
        return;
    }

    float mx = -3.402823466e+38f;
    if (active) {
        for (int v = t; v < n_padded; v += BLK) {
            mx = __builtin_fmaxf(mx, masked(v));
        }
    }
    mx = block_max<float, SM_THREADS / WAVE>(mx, sh, -3.402823466e+38f);
    if (BLK < 1024) {
        mx = __builtin_fmaxf(mx, -1e20f);  // blockReduceMax pads its second stage with -1e20f
    }

    float sum = 0.0f;
    if (active) {
        for (int v = t; v < n_padded; v += BLK) {
            sum += round_t<DT>(det_expf_nonpos(masked(v) - mx));
        }
    }
#pragma unroll
    for (int m = 16; m > 0; m >>= 1) {
        sum += __shfl_xor(sum, m, 32);
    }
    if ((t & 31) == 0) {
        sh[t >> 5] = sum;
    }
    __syncthreads();
    if (t < 32) {
        float v = ((float)t < (float)BLK / 32.0f) ? sh[t] : 0.0f;
#pragma unroll
        for (int m = 16; m > 0; m >>= 1) {
            v += __shfl_xor(v, m, 32);
        }
        if (t == 0) {
            sh_bcast = v;
        }
    }
    __syncthreads();
    const float denom = sh_bcast + 1e-6f;
    if constexpr (STATS_ONLY) {
        if (t == 0) {
            stats[row] = make_float2(mx, denom);
        }
        return;
    }
    if (active) {
        for (int v = t; v < n_padded; v += BLK) {
            const float e = round_t<DT>(det_expf_nonpos(masked(v) - mx));
            rowp[v]       = S::st(e / denom);
        }
    }
}

// =============================================================================================
// top-p
// =============================================================================================
//
// The reference sorts every row completely and then scans it. Only the part of the sorted order in
// front of the draw matters, so the rows are cut first and only the part above the cut is ordered:
//   histogram  - (chunks x rows) workgroups stream the probabilities once: entries per bucket (six
//                mantissa bits under the exponent, 32 octaves below 1.0), a fixed-point lower bound
//                of the mass per bucket, and the arg-max;
//   cut        - one workgroup per row: the lowest bucket whose suffix of mass certainly covers the
//                draw, where every bucket and every chunk writes inside the ordered prefix, and the
//                prefix divided into segments of whole buckets;
//   gather     - second stream: entries at or above the cut go to their bucket's range as
//                (~key, id) pairs;
//   sort       - segments are sorted independently, dealt out over the workgroups of one launch: the
//                keys of a segment are spread over bins, neighbouring bins joined into groups of a few
//                dozen entries, and every group sorted by one wave in registers (a long group of equal
//                keys by the whole workgroup in LDS, a segment that one bucket alone makes too long
//                by a radix sort in memory);
//   pick       - one workgroup per row replays the reference's scan on the ordered prefix with its
//                exact rounding order (32 raking lanes x 8 items, Kogge-Stone over the 32 partials,
//                sequential carry over tiles) and emits the token.
// A row whose draw is not crossed inside its prefix (it cannot be unless the bound above fails)
// falls back to a stable radix sort of all its positive entries.
// Callers that do not need the probabilities afterwards take a second form of the step, which only reads the logits
// (topp_sample_kernels.hip).

// Workspace sections (all offsets multiples of 256 bytes). `sorted` keeps the reference's shape of
// two 64-bit arrays per row; the second one is only touched by the radix sorts.
struct ToppPlan {
    int    splits;  // chunks per row of the two streaming kernels
    int    chunk;   // columns per chunk
    int    sorters; // workgroups of the sort kernel
    size_t off_pcnt, off_pmass, off_pbest, off_start, off_boff, off_seg, off_meta, bytes;
};

static inline size_t align256(size_t x)
{
    return (x + 255) & ~(size_t)255;
}

static ToppPlan topp_plan(int batch, size_t vocab)
{
    ToppPlan p;
    const int rows = batch > 0 ? batch : 1;
    int       s    = (1024 + rows - 1) / rows;
    const int cap  = (int)(vocab / 8192) > 0 ? (int)(vocab / 8192) : 1;
    s              = s < cap ? s : cap;
    s              = s < 64 ? s : 64;
    p.splits       = s;
    p.chunk        = (int)(((vocab + s - 1) / s + 7) / 8 * 8);
    p.sorters      = 512;
    size_t off     = align256((size_t)rows * vocab * 2 * sizeof(unsigned long long));
    p.off_pcnt     = off;
    off += align256((size_t)rows * s * TPB_NB * sizeof(uint32_t));
    p.off_pmass = off;
    off += align256((size_t)rows * s * TPB_NB * sizeof(uint32_t));
    p.off_pbest = off;
    off += align256((size_t)rows * s * sizeof(unsigned long long));
    p.off_start = off;
    off += align256((size_t)rows * s * TPB_NB * sizeof(uint32_t));
    p.off_boff = off;
    off += align256((size_t)rows * TPB_NB * sizeof(uint32_t));
    p.off_seg = off;
    off += align256((size_t)rows * TPB_NB * sizeof(uint32_t));
    p.off_meta = off;
    off += align256((size_t)rows * sizeof(ToppRowMeta));
    p.bytes = off;
    return p;
}

template<int DT>
__global__ void __launch_bounds__(TPH_THREADS)
topp_histogram_kernel(const typename Storage<DT>::T* __restrict__ probs, int vocab, int chunk,
                      const bool* __restrict__ skip_decode, uint32_t* __restrict__ part_cnt,
                      uint32_t* __restrict__ part_mass, unsigned long long* __restrict__ part_best)
{
    __shared__ uint32_t           cnt[TPB_NB];
    __shared__ uint32_t           mass[TPB_NB];
    __shared__ unsigned long long red[16];
    const int                     row = blockIdx.y;
    const int                     j   = blockIdx.x;
    const int                     S   = gridDim.x;
    const int                     t   = threadIdx.x;
    if (skip_decode != nullptr && skip_decode[row]) {
        return;
    }
    for (int b = t; b < TPB_NB; b += TPH_THREADS) {
        cnt[b]  = 0u;
        mass[b] = 0u;
    }
    __syncthreads();
    const int lo   = (int)min((long long)vocab, (long long)j * chunk);
    const int hi   = (int)min((long long)vocab, (long long)lo + chunk);
    uint32_t  tmax = 0;
    int       tidx = 0x7FFFFFFF;
    stream_columns<DT, TPH_THREADS>(probs + (size_t)row * vocab, lo, hi, [&](int v, float x) {
        const uint32_t k = order_key(x);
        if (k > tmax) {
            tmax = k;
            tidx = v;
        }
        if (k > ZERO_KEY) {
            const int b = topp_bucket(k);
            atomicAdd(&cnt[b], 1u);
            // truncation keeps the sum a lower bound of the mass
            atomicAdd(&mass[b], (uint32_t)(__builtin_fminf(x, 1.0f) * 2147483648.0f));
        }
    });
    __syncthreads();
    const size_t base = ((size_t)row * S + j) * TPB_NB;
    for (int b = t; b < TPB_NB; b += TPH_THREADS) {
        part_cnt[base + b]  = cnt[b];
        part_mass[base + b] = mass[b];
    }
    unsigned long long best = ((unsigned long long)tmax << 32) | (uint32_t)(~(uint32_t)tidx);
    best                    = block_max<unsigned long long, TPH_THREADS / WAVE>(best, red, 0ull);
    if (t == 0) {
        part_best[(size_t)row * S + j] = best;
    }
}

// Second half of the softmax for the fused step, (chunks x rows) workgroups: divides every column by the
// row's denominator (same expression as softmax_kernel, so the stored probabilities are the same bits) and
// tallies what topp_histogram_kernel would read back from the row, in the same pass.
template<int DT>
__global__ void __launch_bounds__(TPH_THREADS)
softmax_finish_histogram_kernel(typename Storage<DT>::T* __restrict__ logits,
                                const typename Storage<DT>::T* __restrict__ bias, const int* __restrict__ end_ids,
                                const bool* __restrict__ finished, const float2* __restrict__ stats, int n_padded,
                                int n, int chunk, const bool* __restrict__ skip_decode,
                                uint32_t* __restrict__ part_cnt, uint32_t* __restrict__ part_mass,
                                unsigned long long* __restrict__ part_best)
{
    typedef Storage<DT>           S;
    __shared__ uint32_t           cnt[TPB_NB];
    __shared__ uint32_t           mass[TPB_NB];
    __shared__ unsigned long long red[16];
    const int                     row    = blockIdx.y;
    const int                     j      = blockIdx.x;
    const int                     NS     = gridDim.x;
    const int                     t      = threadIdx.x;
    const bool                    tally  = !(skip_decode != nullptr && skip_decode[row]);
    const bool                    fin    = finished != nullptr ? finished[row] : false;
    const int                     end_id = fin ? end_ids[row] : -1;
    const float                   MAXT   = S::max_t();
    const float2                  st     = stats[row];
    const float                   mx     = st.x;
    const float                   denom  = st.y;
    for (int b = t; b < TPB_NB; b += TPH_THREADS) {
        cnt[b]  = 0u;
        mass[b] = 0u;
    }
    __syncthreads();
    const int lo   = (int)min((long long)n_padded, (long long)j * chunk);
    const int hi   = (int)min((long long)n_padded, (long long)lo + chunk);
    uint32_t  tmax = 0;
    int       tidx = 0x7FFFFFFF;
    auto finish = [&](int v, float y) {
        // y <= mx (or NaN): the argument of the exponential is never positive
        const float p = round_t<DT>(det_expf_nonpos(y - mx)) / denom;
        if (tally) {
            const float    pr = round_t<DT>(p);
            const uint32_t k  = order_key(pr);
            if (k > tmax) {
                tmax = k;
                tidx = v;
            }
            if (k > ZERO_KEY) {
                const int b = topp_bucket(k);
                atomicAdd(&cnt[b], 1u);
                atomicAdd(&mass[b], (uint32_t)(__builtin_fminf(pr, 1.0f) * 2147483648.0f));
            }
        }
        return p;
    };
    typename S::T*   rowp = logits + (size_t)row * n_padded;
    const RowDivisor div(denom);
    if (!fin && bias == nullptr && div.ok) {
        // Ordinary rows: no per-column cases in front of the arithmetic, the division with the row's reciprocal,
        // and keys of values that cannot be negative (the exponential is in [0, 1] or NaN, the denominator at
        // least 1: probabilities in [0, 1]). `x + 0.0f` is left out: it only turns -0 into +0, and the
        // exponential of both differences is the same.
        auto quick = [&](int v, float y) {
            const float p = div.divide(round_t<DT>(det_expf_nonpos(y - mx)));
            if (tally) {
                const float    pr = round_t<DT>(p);
                const uint32_t k  = order_key_nonneg(pr);
                if (k > tmax) {
                    tmax = k;
                    tidx = v;
                }
                if (k > ZERO_KEY) {
                    const int b = topp_bucket(k);
                    atomicAdd(&cnt[b], 1u);
                    atomicAdd(&mass[b], (uint32_t)(pr * 2147483648.0f));
                }
            }
            return p;
        };
        const int mid = min(hi, max(lo, n));
        transform_columns<DT, TPH_THREADS>(rowp, lo, mid, [&](int v, float x) { return quick(v, x); });
        transform_columns<DT, TPH_THREADS>(rowp, mid, hi, [&](int v, float) { return quick(v, -MAXT); });
    }
    else {
        transform_columns<DT, TPH_THREADS>(rowp, lo, hi, [&](int v, float x) {
            float y;
            if (v >= n) {
                y = -MAXT;
            }
            else if (fin) {
                y = v == end_id ? MAXT : -MAXT;
            }
            else {
                // (rows without a bias come here, too, when their denominator is no ordinary number)
                y = round_t<DT>(x + (bias != nullptr ? S::ld(bias[v]) : 0.0f));
            }
            return finish(v, y);
        });
    }
    if (!tally) {
        return;
    }
    __syncthreads();
    const size_t base = ((size_t)row * NS + j) * TPB_NB;
    for (int b = t; b < TPB_NB; b += TPH_THREADS) {
        part_cnt[base + b]  = cnt[b];
        part_mass[base + b] = mass[b];
    }
    unsigned long long best = ((unsigned long long)tmax << 32) | (uint32_t)(~(uint32_t)tidx);
    best                    = block_max<unsigned long long, TPH_THREADS / WAVE>(best, red, 0ull);
    if (t == 0) {
        part_best[(size_t)row * NS + j] = best;
    }
}

__global__ void __launch_bounds__(TPC_THREADS)
topp_cut_kernel(int S, const uint32_t* __restrict__ part_cnt, const uint32_t* __restrict__ part_mass,
                const unsigned long long* __restrict__ part_best, uint32_t* __restrict__ start,
                uint32_t* __restrict__ bucket_off, uint32_t* __restrict__ seg_ends, ToppRowMeta* __restrict__ meta,
                const RngState* rng,
                const float* __restrict__ uniforms, float top_p, const float* __restrict__ top_ps,
                const bool* __restrict__ skip_decode)
{
    __shared__ uint32_t           cnt[TPB_NB];
    __shared__ uint32_t           off[TPB_NB];
    __shared__ unsigned long long mass[TPB_NB];
    __shared__ unsigned long long red64[16];
    __shared__ uint32_t           wcnt[TPC_THREADS / WAVE];
    __shared__ unsigned long long wmass[TPC_THREADS / WAVE];
    __shared__ uint32_t           red32[16];
    const int                     row = blockIdx.x;
    const int                     t   = threadIdx.x;
    ToppRowMeta                   m;
    m.best = 0ull;
    m.cut = TPB_NB;
    m.n = m.n_pos = m.nseg = 0;
    m.flags = 0;
    m.safe  = 0.0f;
    if (skip_decode != nullptr && skip_decode[row]) {
        if (t == 0) {
            m.flags   = TOPP_SKIP;
            meta[row] = m;
        }
        return;
    }
    // sums over the chunks; what the chunks before chunk j hold of a bucket goes to `start` on the way.
    // All loads of one chunk are issued together: the chunks follow each other, not the buckets.
    constexpr int      K    = (TPB_NB + TPC_THREADS - 1) / TPC_THREADS;
    const size_t       base = (size_t)row * S * TPB_NB;
    uint32_t           c[K];
    unsigned long long ms[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        c[i]  = 0u;
        ms[i] = 0ull;
    }
    constexpr int J = 8;  // chunks whose loads are in flight together
    for (int j0 = 0; j0 < S; j0 += J) {
        uint32_t pc[J][K], pm[J][K];
#pragma unroll
        for (int jj = 0; jj < J; ++jj) {
#pragma unroll
            for (int i = 0; i < K; ++i) {
                const int  b  = t + i * TPC_THREADS;
                const bool ok = j0 + jj < S && b < TPB_NB;
                pc[jj][i]     = ok ? part_cnt[base + (size_t)(j0 + jj) * TPB_NB + b] : 0u;
                pm[jj][i]     = ok ? part_mass[base + (size_t)(j0 + jj) * TPB_NB + b] : 0u;
            }
        }
#pragma unroll
        for (int jj = 0; jj < J; ++jj) {
#pragma unroll
            for (int i = 0; i < K; ++i) {
                const int b = t + i * TPC_THREADS;
                if (j0 + jj < S && b < TPB_NB) {
                    start[base + (size_t)(j0 + jj) * TPB_NB + b] = c[i];
                }
                c[i] += pc[jj][i];
                ms[i] += pm[jj][i];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const int b = t + i * TPC_THREADS;
        if (b < TPB_NB) {
            cnt[b]  = c[i];
            mass[b] = ms[i];
        }
    }
    unsigned long long best = 0ull;
    for (int j = t; j < S; j += TPC_THREADS) {
        const unsigned long long v = part_best[(size_t)row * S + j];
        best                       = v > best ? v : best;
    }
    best = block_max<unsigned long long, TPC_THREADS / WAVE>(best, red64, 0ull);  // (also orders the LDS writes above)
    m.best = best;

    const float p         = top_ps != nullptr ? top_ps[row] : top_p;
    const float best_prob = (uint32_t)(best >> 32) == 0u ? __builtin_nanf("") : key_to_float((uint32_t)(best >> 32));
    if (best_prob >= p) {
        // arg-max shortcut of the reference (:842-849): nothing else of the row is needed
        if (t == 0) {
            m.flags   = TOPP_SHORTCUT;
            meta[row] = m;
        }
        return;
    }
    const float              rand_num = row_uniform_peek(rng, uniforms, row) * p;
    // smallest fixed-point mass that certainly covers the draw under the scan's own rounding
    const unsigned long long target = (unsigned long long)((double)rand_num * (1.0 + 1.0 / 1024.0) * 2147483648.0) + 64ull;

    // descending scan over buckets: thread t owns the descending positions [K*t, K*t + K)
    uint32_t           lc = 0;
    unsigned long long lm = 0;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const int d = K * t + i;
        if (d < TPB_NB) {
            lc += cnt[TPB_NB - 1 - d];
            lm += mass[TPB_NB - 1 - d];
        }
    }
    uint32_t           ic = lc;
    unsigned long long im = lm;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        const uint32_t           uc = __shfl_up(ic, o, WAVE);
        const unsigned long long um = __shfl_up(im, o, WAVE);
        if (lane_id() >= o) {
            ic += uc;
            im += um;
        }
    }
    if (lane_id() == WAVE - 1) {
        wcnt[wave_id()]  = ic;
        wmass[wave_id()] = im;
    }
    __syncthreads();
    uint32_t           ec = ic - lc;
    unsigned long long em = im - lm;
    uint32_t           total = 0;
    for (int w = 0; w < TPC_THREADS / WAVE; ++w) {
        if (w < wave_id()) {
            ec += wcnt[w];
            em += wmass[w];
        }
        total += wcnt[w];
    }
    uint32_t first = 0xFFFFFFFFu;  // first descending position where the suffix covers the target
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const int d = K * t + i;
        if (d < TPB_NB) {
            const int b = TPB_NB - 1 - d;
            off[b]      = ec;
            ec += cnt[b];
            em += mass[b];
            if (em >= target && first == 0xFFFFFFFFu) {
                first = (uint32_t)d;
            }
        }
    }
    first = block_min<uint32_t, TPC_THREADS / WAVE>(first, red32, 0xFFFFFFFFu);
    const int cut = first == 0xFFFFFFFFu ? 0 : TPB_NB - 1 - (int)first;
    m.cut         = cut;
    m.n_pos       = (int)total;
    m.n           = (int)(off[cut] + cnt[cut]);

    // where the bucket starts in the ordered prefix (the gather adds what earlier chunks hold)
    for (int b = cut + t; b < TPB_NB; b += TPC_THREADS) {
        bucket_off[(size_t)row * TPB_NB + b] = off[b];
    }
    // Segments of whole buckets, in descending order: a bucket closes a segment when a multiple of
    // TPS_SEG lies inside it or at its end, and the last gathered bucket closes the last one. A segment
    // is therefore shorter than TPS_SEG plus its closing bucket. Segment i is [ends[i-1], ends[i]).
    const uint32_t n_gathered = (uint32_t)m.n;
    uint32_t       closes[K];
    uint32_t       lclose = 0;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const int d = K * t + i;
        closes[i]   = 0u;
        if (d < TPB_NB && TPB_NB - 1 - d >= cut) {
            const int      b = TPB_NB - 1 - d;
            const uint32_t o = off[b];
            const uint32_t e = o + cnt[b];
            if (cnt[b] != 0u && (e / TPS_SEG != o / TPS_SEG || e == n_gathered)) {
                closes[i] = e;
                lclose++;
            }
        }
    }
    uint32_t iclose = lclose;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        const uint32_t up = __shfl_up(iclose, o, WAVE);
        if (lane_id() >= o) {
            iclose += up;
        }
    }
    __syncthreads();
    if (lane_id() == WAVE - 1) {
        wcnt[wave_id()] = iclose;
    }
    __syncthreads();
    uint32_t at   = iclose - lclose;
    uint32_t nseg = 0;
    for (int w = 0; w < TPC_THREADS / WAVE; ++w) {
        at += w < wave_id() ? wcnt[w] : 0u;
        nseg += wcnt[w];
    }
    uint32_t* ends = seg_ends + (size_t)row * TPB_NB;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        if (closes[i] != 0u) {
            ends[at++] = closes[i];
        }
    }
    if (t == 0) {
        m.nseg    = (int)nseg;
        meta[row] = m;
    }
}

template<int DT>
__global__ void __launch_bounds__(TPH_THREADS)
topp_gather_kernel(const typename Storage<DT>::T* __restrict__ probs, int vocab, int chunk,
                   const ToppRowMeta* __restrict__ meta, const uint32_t* __restrict__ start,
                   const uint32_t* __restrict__ bucket_off, unsigned long long* __restrict__ sorted)
{
    __shared__ uint32_t cur[TPB_NB];
    const int           row = blockIdx.y;
    const int           j   = blockIdx.x;
    const int           S   = gridDim.x;
    const int           t   = threadIdx.x;
    const ToppRowMeta   m   = meta[row];
    if (m.flags != 0 || m.n == 0) {
        return;
    }
    const size_t base = ((size_t)row * S + j) * TPB_NB;
    for (int b = m.cut + t; b < TPB_NB; b += TPH_THREADS) {
        cur[b] = bucket_off[(size_t)row * TPB_NB + b] + start[base + b];
    }
    __syncthreads();
    const int           lo  = (int)min((long long)vocab, (long long)j * chunk);
    const int           hi  = (int)min((long long)vocab, (long long)lo + chunk);
    const int           cut = m.cut;
    unsigned long long* A   = sorted + (size_t)row * 2 * vocab;
    stream_columns<DT, TPH_THREADS>(probs + (size_t)row * vocab, lo, hi, [&](int v, float x) {
        const uint32_t k = order_key(x);
        if (k > ZERO_KEY) {
            const int b = topp_bucket(k);
            if (b >= cut) {
                const uint32_t slot = atomicAdd(&cur[b], 1u);
                A[slot]             = ((unsigned long long)(~k) << 32) | (uint32_t)v;
            }
        }
    });
}
// Every workgroup takes the segments whose running number over all rows is its own modulo the grid.
__global__ void __launch_bounds__(TP_THREADS)
topp_sort_kernel(unsigned long long* __restrict__ sorted, const uint32_t* __restrict__ seg_ends,
                 const ToppRowMeta* __restrict__ meta, int vocab, int rows)
{
    __shared__ ToppSortShared s;
    const int                 t     = threadIdx.x;
    const uint32_t            G     = gridDim.x;
    uint32_t                  first = 0;  // running number of the first segment of the tile
    for (int rb = 0; rb < rows; rb += TP_THREADS) {
        const int row = rb + t;
        uint32_t  my  = 0;
        if (row < rows && meta[row].flags == 0) {
            my = (uint32_t)meta[row].nseg;
        }
        uint32_t       tile_total;
        const uint32_t incl = block_scan_incl(my, s.wtot, tile_total);
        s.psum[t]           = incl;
        __syncthreads();
        uint32_t w = first + (blockIdx.x + G - first % G) % G;
        for (; w < first + tile_total; w += G) {
            const uint32_t local = w - first;
            int            lo = 0, hi = TP_THREADS - 1;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (s.psum[mid] > local) {
                    hi = mid;
                }
                else {
                    lo = mid + 1;
                }
            }
            const int       r    = rb + lo;
            const int       i    = (int)(local - (lo > 0 ? s.psum[lo - 1] : 0u));
            const uint32_t* ends = seg_ends + (size_t)r * TPB_NB;
            const uint32_t  s0   = i > 0 ? ends[i - 1] : 0u;
            const int       n    = (int)(ends[i] - s0);
            unsigned long long* A   = sorted + (size_t)r * 2 * vocab;
            unsigned long long* seg = A + s0;
            topp_sort_one(s, seg, A + vocab + s0, n);
        }
        first += tile_total;
        __syncthreads();
    }
}
template<int DT>
__global__ void __launch_bounds__(TP_THREADS)
topp_pick_kernel(const typename Storage<DT>::T* __restrict__ probs, int* ids, int* __restrict__ sequence_length,
                 bool* __restrict__ finished, float* __restrict__ cum_log_probs, float* __restrict__ output_log_probs,
                 RngState* rng, const float* __restrict__ uniforms, int vocab, const int* __restrict__ end_ids,
                 float top_p, const float* top_ps, const bool* __restrict__ skip_decode,
                 unsigned long long* __restrict__ sorted, const ToppRowMeta* __restrict__ meta, int force_deep,
                 ToppDecayArgs dec)
{
    typedef Storage<DT>           S;
    __shared__ TopPScan           s;
    __shared__ unsigned long long digits[TP_DIGITS];
    const int                     row = blockIdx.x;
    const int                     t   = threadIdx.x;
    // thread 0 writes the row's id itself (a skipped row keeps what an earlier kernel left there) and every
    // thread reads the row's top_p before the first barrier
    auto decay = [&]() {
        if (dec.runtime_top_p != nullptr && t == 0) {
            topp_decay_row(dec, row, ids[row]);
        }
    };
    if (skip_decode != nullptr && skip_decode[row]) {
        decay();
        return;
    }
    const typename S::T* rowp = probs + (size_t)row * vocab;
    const float          p    = top_ps != nullptr ? top_ps[row] : top_p;
    const ToppRowMeta    m    = meta[row];
    int                  best_id = (int)(~(uint32_t)m.best);
    if ((uint32_t)(m.best >> 32) == 0u) {
        best_id = 0;  // nothing comparable in the row (all NaN): the reference keeps index 0
    }
    auto           prob_at   = [&](int v) -> float { return S::ld(rowp[v]); };
    const float    best_prob = prob_at(best_id);
    const TopPEmit emit{ids, sequence_length, finished, cum_log_probs, output_log_probs, end_ids, row};
    if (t == 0) {
        const float u = row_uniform(rng, uniforms, row);  // drawn for every non-skipped row
        s.fmisc[0]    = u * p;
    }
    __syncthreads();
    const float rand_num = s.fmisc[0];

    // ---- shortcut: sum_prob = T(0) + max prob, compared in fp32 (:842-849)
    if (round_t<DT>(0.0f + best_prob) >= p) {
        if (t == 0) {
            emit(best_id, best_prob);
        }
        decay();
        return;
    }
    if (t == 0) {
        ids[row] = best_id;  // kept when no prefix sum ever reaches the draw (:954)
    }

    unsigned long long* A = sorted + (size_t)row * 2 * vocab;
    auto scan = [&](const unsigned long long* src, int n) -> int {
        return n > 0 ? scan_tiles<8>(s, (n + TP_TILE - 1) / TP_TILE, rand_num,
                                     [&](int tile, int l, float* x) { tile_load(src, n, tile, l, x); }) :
                       -1;
    };
    auto emit_at = [&](const unsigned long long* src, int n, int found) {
        found = min(found, vocab - 1);  // (the zeros that fill the last tile can hold the crossing)
        if (found < n) {
            const unsigned long long e = src[found];
            emit((int)(uint32_t)e, key64_prob(e));
        }
        else {
            const int id = nth_zero_entry(prob_at, vocab, found - n);
            emit(id, prob_at(id));
        }
    };
    if (!force_deep && m.flags == 0) {
        const bool all   = m.n == m.n_pos;
        const int  found = scan(A, m.n);
        if (found >= 0 && (found < m.n || all)) {
            if (t == 0) {
                emit_at(A, m.n, found);
            }
            decay();
            return;
        }
        if (all) {
            decay();
            return;  // every positive entry scanned, never crossed: ids keeps the arg-max
        }
    }
    const unsigned long long* src   = sort_whole_row(s, digits, prob_at, vocab, A, A + vocab);
    const int                 n_all = s.misc[2];
    const int                 found = scan(src, n_all);
    if (found >= 0 && t == 0) {
        emit_at(src, n_all, found);
    }
    decay();
}

__global__ void topp_decay_kernel(float* __restrict__ runtime_top_p, const float* __restrict__ initial_top_p,
                                  const int* __restrict__ output_ids, const float* __restrict__ decay,
                                  const float* __restrict__ top_p_min, const int32_t* __restrict__ reset_ids, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) {
        return;
    }
    if (output_ids[i] == reset_ids[i]) {
        runtime_top_p[i] = initial_top_p[i];
    }
    else {
        runtime_top_p[i] = __builtin_fmaxf(runtime_top_p[i] * decay[i], top_p_min[i]);
    }
}

__global__ void topp_initialize_kernel(int* id_vals, int* offsets, int* begin_offsets, int batch, int n)
{
    const size_t tid = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && offsets != nullptr) {
        for (int i = threadIdx.x; i < batch + 1; i += blockDim.x) {
            offsets[i] = i * n;
            if (begin_offsets != nullptr) {
                begin_offsets[i] = i * n;
            }
        }
    }
    if (id_vals != nullptr) {
        for (size_t i = tid; i < (size_t)batch * n; i += (size_t)gridDim.x * blockDim.x) {
            id_vals[i] = (int)(i % n);
        }
    }
}

}  // namespace ftk

using namespace ftk;

extern "C" {

int ftk_invoke_add_bias_softmax(int dtype, void* logits, const void* bias, const int* end_ids, const bool* finished,
                                int m, int n_padded, int n, ftk_stream_t stream)
{
    if (m <= 0 || n <= 0) {
        return 0;
    }
    FTK_DISPATCH_DTYPE(dtype, (softmax_kernel<DT, false><<<m, SM_THREADS, 0, (hipStream_t)stream>>>(
                                  (Storage<DT>::T*)logits, (const Storage<DT>::T*)bias, end_ids, finished, n_padded, n,
                                  nullptr)));
    FTK_LAUNCH_CHECK();
    return 0;
}

int ftk_invoke_topp_initialize(int* topp_id_val_buf, int* topp_offset_buf, int* begin_topp_offset_buf,
                               size_t batch_size, int n, ftk_stream_t stream)
{
    if (batch_size == 0 || (topp_id_val_buf == nullptr && topp_offset_buf == nullptr)) {
        return 0;
    }
    topp_initialize_kernel<<<32, 512, 0, (hipStream_t)stream>>>(topp_id_val_buf, topp_offset_buf,
                                                                begin_topp_offset_buf, (int)batch_size, n);
    FTK_LAUNCH_CHECK();
    return 0;
}

#ifdef FTK_TEST_HOOKS
// Test hook (hooks build of the library only): a non-zero value routes every row through the radix-sort
// fallback, so that it can be exercised on small inputs.
static int g_topp_force_deep = 0;
void       ftk_test_set_topp_force_deep(int v)
{
    g_topp_force_deep = v;
}
#else
static constexpr int g_topp_force_deep = 0;
#endif

}  // extern "C"

int ftk::topp_force_deep()
{
    return g_topp_force_deep;
}

extern "C" {

// Shared by the two entry points below. `softmax_first`: `log_probs` holds logits on entry; the softmax runs as
// two kernels, the second of which also tallies the histogram, and the decay runs at the end of the pick.
static int topp_sampling_launch(int dtype, void* workspace, size_t* workspace_size, size_t* cub_temp_storage_size,
                                int* output_ids, int* sequence_length, bool* finished, float* cum_log_probs,
                                float* output_log_probs, void* log_probs, ftk_rng_state* rng_state,
                                const float* uniform_draws, int batch_size, size_t vocab_size_padded,
                                const int* end_ids, float max_top_p, const float* top_ps, hipStream_t st,
                                const bool* skip_decode, bool softmax_first, const void* bias, int vocab_size,
                                ToppDecayArgs dec)
{
    if (dtype < 0 || dtype > 2) {
        return FTK_ERR_DTYPE;
    }
    if (batch_size < 0 || batch_size > 65535) {
        return FTK_ERR_ARGUMENT;
    }
    const ToppPlan plan      = topp_plan(batch_size, vocab_size_padded);
    const size_t   off_stats = plan.bytes;
    // (the sizes of both forms of the step are one, so that a caller may take either with one workspace)
    const size_t   need      = softmax_first ?
                                   std::max(plan.bytes + align256((size_t)(batch_size > 0 ? batch_size : 1) * sizeof(float2)),
                                            topp_sample_bytes(dtype, batch_size, vocab_size, vocab_size_padded, false)) :
                                   plan.bytes;
    if (workspace == nullptr) {
        if (workspace_size == nullptr) {
            return FTK_ERR_ARGUMENT;
        }
        *workspace_size = need;
        if (cub_temp_storage_size != nullptr) {
            *cub_temp_storage_size = 0;
        }
        return 0;
    }
    if (workspace_size != nullptr && *workspace_size < need) {
        return FTK_ERR_WORKSPACE;
    }
    if (batch_size <= 0) {
        return 0;
    }
    if (rng_state == nullptr && uniform_draws == nullptr) {
        return FTK_ERR_ARGUMENT;
    }
    if (log_probs == nullptr || output_ids == nullptr
        || (end_ids == nullptr && finished != nullptr && (sequence_length != nullptr || softmax_first))) {
        return FTK_ERR_ARGUMENT;  // (the kernels read and write these unconditionally)
    }
    if (vocab_size_padded > (size_t)65535 * TP_THREADS) {
        return FTK_ERR_ARGUMENT;
    }
    if (softmax_first && (vocab_size <= 0 || (size_t)vocab_size > vocab_size_padded)) {
        return FTK_ERR_ARGUMENT;
    }
    char*               ws      = (char*)workspace;
    unsigned long long* sorted  = (unsigned long long*)ws;
    uint32_t*           pcnt    = (uint32_t*)(ws + plan.off_pcnt);
    uint32_t*           pmass   = (uint32_t*)(ws + plan.off_pmass);
    unsigned long long* pbest   = (unsigned long long*)(ws + plan.off_pbest);
    uint32_t*           start   = (uint32_t*)(ws + plan.off_start);
    uint32_t*           boff    = (uint32_t*)(ws + plan.off_boff);
    uint32_t*           segs    = (uint32_t*)(ws + plan.off_seg);
    ToppRowMeta*        meta    = (ToppRowMeta*)(ws + plan.off_meta);
    const int           vocab   = (int)vocab_size_padded;
    const dim3          chunks(plan.splits, batch_size);
    if (softmax_first) {
        float2* stats = (float2*)(ws + off_stats);
        FTK_DISPATCH_DTYPE(dtype, (softmax_kernel<DT, true><<<batch_size, SM_THREADS, 0, st>>>(
                                      (Storage<DT>::T*)log_probs, (const Storage<DT>::T*)bias, end_ids, finished, vocab,
                                      vocab_size, stats)));
        FTK_LAUNCH_CHECK();
        FTK_DISPATCH_DTYPE(dtype, softmax_finish_histogram_kernel<DT><<<chunks, TPH_THREADS, 0, st>>>(
                                      (Storage<DT>::T*)log_probs, (const Storage<DT>::T*)bias, end_ids, finished, stats,
                                      vocab, vocab_size, plan.chunk, skip_decode, pcnt, pmass, pbest));
        FTK_LAUNCH_CHECK();
    }
    else {
        FTK_DISPATCH_DTYPE(dtype, topp_histogram_kernel<DT><<<chunks, TPH_THREADS, 0, st>>>(
                                      (const Storage<DT>::T*)log_probs, vocab, plan.chunk, skip_decode, pcnt, pmass,
                                      pbest));
        FTK_LAUNCH_CHECK();
    }
    topp_cut_kernel<<<batch_size, TPC_THREADS, 0, st>>>(plan.splits, pcnt, pmass, pbest, start, boff, segs, meta,
                                                        (const RngState*)rng_state, uniform_draws, max_top_p, top_ps,
                                                        skip_decode);
    FTK_LAUNCH_CHECK();
    if (!g_topp_force_deep) {
        FTK_DISPATCH_DTYPE(dtype, topp_gather_kernel<DT><<<chunks, TPH_THREADS, 0, st>>>(
                                      (const Storage<DT>::T*)log_probs, vocab, plan.chunk, meta, start, boff, sorted));
        FTK_LAUNCH_CHECK();
        topp_sort_kernel<<<plan.sorters, TP_THREADS, 0, st>>>(sorted, segs, meta, vocab, batch_size);
        FTK_LAUNCH_CHECK();
    }
    FTK_DISPATCH_DTYPE(dtype, topp_pick_kernel<DT><<<batch_size, TP_THREADS, 0, st>>>(
                                  (const Storage<DT>::T*)log_probs, output_ids, sequence_length, finished,
                                  cum_log_probs, output_log_probs, (RngState*)rng_state, uniform_draws, vocab,
                                  end_ids, max_top_p, top_ps, skip_decode, sorted, meta, g_topp_force_deep, dec));
    FTK_LAUNCH_CHECK();
    return 0;
}

int ftk_invoke_batch_topp_sampling(int dtype, void* workspace, size_t* workspace_size, size_t* cub_temp_storage_size,
                                   int* output_ids, int* sequence_length, bool* finished, float* cum_log_probs,
                                   float* output_log_probs, const void* log_probs, const int* id_vals,
                                   int* offset_buf, int* begin_offset_buf, ftk_rng_state* rng_state,
                                   const float* uniform_draws, int batch_size, size_t vocab_size_padded,
                                   const int* end_ids, float max_top_p, const float* top_ps, ftk_stream_t stream,
                                   const bool* skip_decode)
{
    (void)id_vals;
    (void)offset_buf;
    (void)begin_offset_buf;
    const ToppDecayArgs none = {nullptr, nullptr, nullptr, nullptr, nullptr};
    return topp_sampling_launch(dtype, workspace, workspace_size, cub_temp_storage_size, output_ids, sequence_length,
                                finished, cum_log_probs, output_log_probs, const_cast<void*>(log_probs), rng_state,
                                uniform_draws, batch_size, vocab_size_padded, end_ids, max_top_p, top_ps,
                                (hipStream_t)stream, skip_decode, false, nullptr, 0, none);
}

int ftk_fused_topp_step(int dtype, void* workspace, size_t* workspace_size, void* logits, const void* bias,
                        int vocab_size, size_t vocab_size_padded, int batch_size, const int* end_ids, bool* finished,
                        int* sequence_length, int* output_ids, float* cum_log_probs, float* output_log_probs,
                        ftk_rng_state* rng_state, const float* uniform_draws, float max_top_p, float* runtime_top_p,
                        const float* initial_top_p, const float* top_p_decay, const float* top_p_min,
                        const int32_t* top_p_reset_ids, const bool* skip_decode, ftk_stream_t stream)
{
    ToppDecayArgs dec = {nullptr, nullptr, nullptr, nullptr, nullptr};
    if (top_p_decay != nullptr) {
        if (runtime_top_p == nullptr || initial_top_p == nullptr || top_p_min == nullptr || top_p_reset_ids == nullptr) {
            return FTK_ERR_ARGUMENT;
        }
        dec = ToppDecayArgs{runtime_top_p, initial_top_p, top_p_decay, top_p_min, top_p_reset_ids};
    }
    return topp_sampling_launch(dtype, workspace, workspace_size, nullptr, output_ids, sequence_length, finished,
                                cum_log_probs, output_log_probs, logits, rng_state, uniform_draws, batch_size,
                                vocab_size_padded, end_ids, max_top_p, runtime_top_p, (hipStream_t)stream,
                                skip_decode, true, bias, vocab_size, dec);
}

// Checks and size query shared by the two entry points that sample straight from logits.
static int topp_sample_entry(ToppSampleCall& c, size_t* workspace_size, hipStream_t st)
{
    if (c.dtype < 0 || c.dtype > 2) {
        return FTK_ERR_DTYPE;
    }
    const bool history = c.penalties != nullptr && c.penalty_type != FTK_PENALTY_NONE;
    if (!topp_sample_covers(c.dtype, c.rows, c.vocab_size, history)) {
        return FTK_ERR_UNSUPPORTED;
    }
    if (c.rows < 0 || c.rows > 65535 || (size_t)c.vocab_size > c.vocab_size_padded
        || c.vocab_size_padded > (size_t)65535 * TP_THREADS) {
        return FTK_ERR_ARGUMENT;
    }
    if (c.top_p_decay != nullptr
        && (c.runtime_top_p == nullptr || c.initial_top_p == nullptr || c.top_p_min == nullptr
            || c.top_p_reset_ids == nullptr)) {
        return FTK_ERR_ARGUMENT;
    }
    const bool   keeps_y = c.temperatures != nullptr || history || c.min_lengths != nullptr;
    const size_t vp      = c.vocab_size_padded;
    size_t       need    = topp_sample_bytes(c.dtype, c.rows, c.vocab_size, vp, keeps_y);
    if (!keeps_y) {
        need = std::max(need, topp_plan(c.rows, vp).bytes + align256((size_t)(c.rows > 0 ? c.rows : 1) * sizeof(float2)));
    }
    if (c.workspace == nullptr) {
        if (workspace_size == nullptr) {
            return FTK_ERR_ARGUMENT;
        }
        *workspace_size = need;
        return 0;
    }
    if (workspace_size != nullptr && *workspace_size < need) {
        return FTK_ERR_WORKSPACE;
    }
    c.workspace_size = workspace_size != nullptr ? *workspace_size : need;
    if (c.rows <= 0) {
        return 0;
    }
    if ((c.rng_state == nullptr && c.uniform_draws == nullptr) || c.logits == nullptr || c.output_ids == nullptr
        || (c.end_ids == nullptr && (c.finished != nullptr || c.min_lengths != nullptr))
        || (c.bias != nullptr && c.temperatures == nullptr) || (history && c.history == nullptr)
        || (history && c.penalty_type != FTK_PENALTY_ADDITIVE && c.penalty_type != FTK_PENALTY_MULTIPLICATIVE)
        || (c.min_lengths != nullptr && c.sequence_length == nullptr)) {
        return FTK_ERR_ARGUMENT;
    }
    return topp_sample_launch(c, st);
}

int ftk_fused_topp_sample_step(int dtype, void* workspace, size_t* workspace_size, const void* logits,
                               int vocab_size, size_t vocab_size_padded, int batch_size, const int* end_ids,
                               bool* finished, int* sequence_length, int* output_ids, float* cum_log_probs,
                               float* output_log_probs, ftk_rng_state* rng_state, const float* uniform_draws,
                               float max_top_p, float* runtime_top_p, const float* initial_top_p,
                               const float* top_p_decay, const float* top_p_min, const int32_t* top_p_reset_ids,
                               const bool* skip_decode, ftk_stream_t stream)
{
    ToppSampleCall c{};
    c.dtype             = dtype;
    c.workspace         = workspace;
    c.logits            = logits;
    c.vocab_size        = vocab_size;
    c.vocab_size_padded = vocab_size_padded;
    c.rows              = batch_size;
    c.penalty_type      = FTK_PENALTY_NONE;
    c.batch_size        = batch_size;
    c.end_ids           = end_ids;
    c.finished          = finished;
    c.sequence_length   = sequence_length;
    c.output_ids        = output_ids;
    c.cum_log_probs     = cum_log_probs;
    c.output_log_probs  = output_log_probs;
    c.rng_state         = rng_state;
    c.uniform_draws     = uniform_draws;
    c.max_top_p         = max_top_p;
    c.runtime_top_p     = runtime_top_p;
    c.initial_top_p     = initial_top_p;
    c.top_p_decay       = top_p_decay;
    c.top_p_min         = top_p_min;
    c.top_p_reset_ids   = top_p_reset_ids;
    c.skip_decode       = skip_decode;
    return topp_sample_entry(c, workspace_size, (hipStream_t)stream);
}

int ftk_fused_topp_penalty_step(ftk_fused_topp_args* args, ftk_stream_t stream)
{
    if (args == nullptr) {
        return FTK_ERR_ARGUMENT;
    }
    const ftk_fused_topk_args& a = args->row;
    if (a.frequency_penalties != nullptr) {
        return FTK_ERR_UNSUPPORTED;
    }
    ToppSampleCall c{};
    c.dtype             = a.dtype;
    c.workspace         = a.workspace;
    c.logits            = a.logits;
    c.bias              = a.embedding_bias;
    c.vocab_size        = a.vocab_size;
    c.vocab_size_padded = (size_t)a.vocab_size_padded;
    c.rows              = a.local_batch_size;
    c.temperatures      = a.temperatures;
    c.penalties         = a.penalties;
    c.penalty_type      = a.penalties != nullptr ? a.penalty_type : FTK_PENALTY_NONE;
    c.min_lengths       = a.min_lengths;
    c.input_lengths     = a.input_lengths;
    c.history           = a.output_ids;
    c.batch_size        = a.batch_size;
    c.step              = a.step;
    c.max_input_length  = a.max_input_length;
    c.end_ids           = a.end_ids;
    c.finished          = a.finished;
    c.sequence_length   = a.sequence_length;
    c.output_ids        = a.ids;
    c.cum_log_probs     = a.cum_log_probs;
    c.output_log_probs  = a.output_log_probs;
    c.rng_state         = a.rng_state;
    c.uniform_draws     = a.uniform_draws;
    c.max_top_p         = args->max_top_p;
    c.runtime_top_p     = args->runtime_top_p;
    c.initial_top_p     = args->initial_top_p;
    c.top_p_decay       = args->top_p_decay;
    c.top_p_min         = args->top_p_min;
    c.top_p_reset_ids   = args->top_p_reset_ids;
    c.skip_decode       = a.skip_decode;
    return topp_sample_entry(c, &args->row.workspace_size, (hipStream_t)stream);
}

int ftk_invoke_compute_topp_decay(float* runtime_top_p, const float* runtime_initial_top_p, const int* output_ids,
                                  const float* top_p_decay, const float* top_p_min, const int32_t* top_p_reset_ids,
                                  int local_batch_size, ftk_stream_t stream)
{
    if (local_batch_size <= 0) {
        return 0;
    }
    topp_decay_kernel<<<(local_batch_size + 255) / 256, 256, 0, (hipStream_t)stream>>>(
        runtime_top_p, runtime_initial_top_p, output_ids, top_p_decay, top_p_min, top_p_reset_ids, local_batch_size);
    FTK_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
