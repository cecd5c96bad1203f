// The log-prob step (ftk_logprob.cuh) for short rows: the same two passes over a row by one workgroup, column by column and
// with every column through det_expf.
//
// Bound by latency: rounds of memory, barriers and the fetch of instructions that a short row executes once. What
// lp_wide_kernel does to save arithmetic on long rows costs more than it saves here: raw maxima need a second look where the
// largest column is one of the history (2 to 3 us), pairs of columns a batch of 16384 for a whole workgroup, of which any part
// takes as long as all of it, and candidates that are looked for behind the sum another round of memory (2.7 us). us a step,
// lp_wide_kernel / here: 256 x 1100 f16 25.7 / 14.5, 256 x 9000 f16 20.9 / 17.2, bf16 21.9 / 17.2, f32 17.3 / 16.2, 300 x 8193 bf16
// 23.4 / 19.7; where batches are nearly full it loses: 256 x 32000 f16 22.3 / 23.5, 300 x 16384 f16 21.1 / 23.9 (the rule is
// beside the launch). Sums and candidates are the same bit for bit.
#pragma once
#include "ftk_logprob.cuh"

namespace ftk {

template<int DT, int BMW, int THREADS>
__global__ void __launch_bounds__(THREADS) lp_short_kernel(FusedParams p, FusedLaunch l, LogProbLaunch lp)
{
    typedef Storage<DT>   S;
    typedef typename S::T T;
    constexpr int         CH = LP_BLOCK / THREADS;  // chains of a thread
    constexpr int         U  = 8 / CH;              // rounds (1024 columns each) of a thread's batch: 8 columns
    constexpr int         N  = U * CH;
    static_assert(THREADS * CH == LP_BLOCK && U * CH == 8 && THREADS % 32 == 0 && THREADS >= TK_THREADS,
                  "a workgroup owns all chains of its row");
    __shared__ TopkShared s;
    __shared__ uint32_t   wide_key[THREADS];
    __shared__ uint32_t   slot_key[TK_THREADS];
    __shared__ float      warp_sum[32];
    __shared__ float      redf[THREADS / WAVE];
    const int             t    = threadIdx.x;
    const int             row  = blockIdx.x;
    const T*              rowp = (const T*)p.logits + (size_t)row * p.Vp;
    // (as in lp_wide_kernel: served first while it waits for memory more than it computes)
    if constexpr (THREADS < LPW_THREADS) {
        __builtin_amdgcn_s_setprio(3);
    }
    // slot j of a batch: round j / CH of the batch, chain (j % CH) * THREADS + t
    auto offset_of = [](int j) { return (j / CH) * LP_BLOCK + (j % CH) * THREADS; };
    // First pass, for the maximum only: the 16-byte vectors of the memory, thread t taking vectors vlo + t, vlo + t +
    // THREADS, ... (`a` columns of the row's first vector lie in front of the row; what lies in front of vector vlo and
    // behind vector vhi is looked at column by column). The first ones are on their way before anything else is read.
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
    const bool    hist = BMW > 0 && p.bitmaps != nullptr && p.penalties != nullptr;
    int           hist_ids[HU];
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
    T         buf[2][N];
    auto      load = [&](T* raw, int b) {
#pragma unroll
        for (int j = 0; j < N; ++j) {
            raw[j] = rowp[b * U * LP_BLOCK + offset_of(j) + t];
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
        s.n_cand = 0;
    }
    const TopkOutputs out =
        topk_outputs(l.ids, l.sequence_length, l.finished, lp.cum_log_probs, lp.output_log_probs, row, p.end_ids);
    if (hist) {
        // the row's history bitmap in LDS (launches with a window and a history penalty)
        uint32_t* window = fused_lds_bitmap<FusedRow<DT, BMW>::LDS_WORDS>();
        const int words  = min(FusedRow<DT, BMW>::LDS_WORDS, (p.V + 31) / 32 + 1);
        for (int i = t; i < words; i += THREADS) {
            window[i] = 0u;
        }
        __syncthreads();
        auto mark = [&](int pos, int id) {
            id -= p.col_offset;
            if (id >= 0 && id < p.V && rowctx.history_position_counts(pos)) {
                atomicOr(&window[id >> 5], 1u << (id & 31));
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
        rowctx.bm_mode   = 1;
        rowctx.bm_origin = 0;
    }
    __syncthreads();
    LPW_STAMP(1)
    const uint32_t KMIN    = min_valid_key<DT>();
    const float    NEG_INF = -__builtin_inff();
    // The values of a batch's columns (v0 = the first one's, t included) after temperature, history penalty and the
    // min-length mask. A column's history flag is bit t % 32 of word v / 32 of the bitmap. The words of a batch are
    // read together, and one look tells whether any of its columns needs more than the multiplication.
    const bool bitsv = rowctx.has_vector_bits();
    const int  bsh   = t & 31;
    auto values = [&](int v0, const T* raw, float* y) {
        uint32_t w[N];
        uint32_t any = 0u;
        if (bitsv) {
#pragma unroll
            for (int j = 0; j < N; ++j) {
                w[j] = rowctx.bm_word((v0 + offset_of(j)) >> 5);
            }
#pragma unroll
            for (int j = 0; j < N; ++j) {
                any |= w[j];
            }
            any = (any >> bsh) & 1u;
        }
#pragma unroll
        for (int j = 0; j < N; ++j) {
            y[j] = rowctx.fast(S::ld(raw[j]));
        }
        const uint32_t to_end = (uint32_t)(rowctx.masked_end_id - v0);  // offset_of(j) for the masked end id at slot j
        if (any != 0u || (to_end < (uint32_t)(U * LP_BLOCK) && (to_end & (THREADS - 1)) == 0u)) {  // rare
#pragma unroll
            for (int j = 0; j < N; ++j) {
                if (bitsv && ((w[j] >> bsh) & 1u)) {
                    y[j] = rowctx.flagged(y[j], v0 + offset_of(j));
                }
                if (to_end == (uint32_t)offset_of(j)) {
                    y[j] = -S::max_t();
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
    // The second pass over the row: whole batches with the next one's loads issued before the current one is used,
    // then the columns behind them one by one, loaded together.
    // use_batch(v0, y) takes a batch's values, use_one(j, v, y) the value of column v at slot j.
    auto stream = [&](auto&& use_batch, auto&& use_one) {
        if (nfull > 0) {
            load(buf[0], 0);
        }
        auto batch = [&](const T* raw, int b) {
            float     y[N];
            const int v0 = b * U * LP_BLOCK + t;
            values(v0, raw, y);
            use_batch(v0, y);
        };
        // (every load is issued whatever the batch, one past the last fetches the last again, unused: with the same
        // number of loads on every path the waits can name the older batch instead of everything in flight)
        for (int b = 0; b < nfull; b += 2) {
            load(buf[1], min(b + 1, nfull - 1));
            batch(buf[0], b);
            load(buf[0], min(b + 2, nfull - 1));
            if (b + 1 < nfull) {
                batch(buf[1], b + 1);
            }
        }
        const int v0 = nfull * U * LP_BLOCK + t;
        if (v0 < p.V) {
            T raw[N];
#pragma unroll
            for (int j = 0; j < N; ++j) {
                raw[j] = rowp[min(v0 + offset_of(j), p.V - 1)];
            }
#pragma unroll
            for (int j = 0; j < N; ++j) {
                if (v0 + offset_of(j) < p.V) {
                    use_one(j, v0 + offset_of(j), value(v0 + offset_of(j), raw[j]));
                }
            }
        }
    };

    lp_note_equal<DT>(s, ring[0]);
    // ---- first pass: the maximum (pad columns count as -MAX_T), and the thread's own
    float m = NEG_INF;
    {
        const float mul     = rowctx.fast_mul;
        const bool  ordered = mul > 0.0f && mul < __builtin_inff();  // the plain transform keeps the order
        for (int q0 = 0; q0 < turns; q0 += R1) {
#pragma unroll
            for (int r = 0; r < R1; ++r) {
                const int q = q0 + r;
                if (q < turns) {
                    const int   rel = q * THREADS + t;
                    const float vm  = lp_vector_max<DT, BMW>(rowctx, ring[r], (vlo + min(rel, nvec - 1)) * EPV - a, a,
                                                            bitsv, ordered);
                    m               = __builtin_fmaxf(m, rel < nvec ? vm : NEG_INF);
                }
                vload(r, q + R1);
            }
        }
        // the columns in front of the first whole vector and behind the last
        for (int v = t; v < min(p.V, vlo * EPV - a); v += THREADS) {
            m = __builtin_fmaxf(m, value(v, rowp[v]));
        }
        for (int v = vhi * EPV - a + t; v < p.V; v += THREADS) {
            m = __builtin_fmaxf(m, value(v, rowp[v]));
        }
    }
    LPW_STAMP(2)
    if (t == 0) {
        s.misc[0] = __float_as_int(row_uniform(l.rng, l.uniforms, row));  // (read behind the barriers of the sum)
    }
    float row_max = block_max<float, THREADS / WAVE>(m, redf, NEG_INF);
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

    LPW_STAMP(4)
    if constexpr (THREADS < LPW_THREADS) {
        __builtin_amdgcn_s_setprio(0);
    }
    // ---- second pass: the sum chain by chain, candidates on the way
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
    stream(
        [&](int v0, const float* y) {
            float d[N], e[N];
            bool  number = true;  // one look for a NaN per pair of columns instead of one per column
#pragma unroll
            for (int j = 0; j < N; ++j) {
                d[j] = y[j] - row_max;
            }
#pragma unroll
            for (int j = 0; j < N; j += 2) {
                number = number && !__builtin_isunordered(d[j], d[j + 1]);
            }
            if (number) {
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    e[j] = round_t<DT>(det_expf_nonpos_number(d[j]));
                }
            }
            else {
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    e[j] = round_t<DT>(det_expf_nonpos(d[j]));
                }
            }
            float top = e[0];
#pragma unroll
            for (int j = 0; j < N; ++j) {
                acc[j % CH] = acc[j % CH] + e[j];  // (slots of a chain in ascending order of their columns)
                top         = __builtin_fmaxf(top, e[j]);
            }
            if (top >= thr_low) {  // (a NaN is no candidate, with or without the maximum)
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    if (e[j] >= thr_low) {
                        push(v0 + offset_of(j), e[j]);
                    }
                }
            }
        },
        [&](int j, int v, float y) {
            const float e = round_t<DT>(det_expf_nonpos(y - row_max));
            acc[j % CH]   = acc[j % CH] + e;
            if (e >= thr_low) {
                push(v, e);
            }
        });
    if (p.V < p.Vp) {
        // pad columns count once nothing of the vocabulary is far above -MAX_T (rows that are masked throughout)
        const float pad_e = round_t<DT>(det_expf_nonpos(-S::max_t() - row_max));
        if (pad_e > 0.0f) {
#pragma unroll 1
            for (int v = p.V + ((t - p.V) & (THREADS - 1)); v < p.Vp; v += THREADS) {
                const int chain = (v & (LP_BLOCK - 1)) / THREADS;
#pragma unroll
                for (int c = 0; c < CH; ++c) {
                    acc[c] = c == chain ? acc[c] + pad_e : acc[c];
                }
                if (pad_e >= thr_low) {
                    push(v, pad_e);
                }
            }
        }
    }
    LPW_STAMP(5)
    if constexpr (THREADS < LPW_THREADS) {
        __builtin_amdgcn_s_setprio(3);
    }
    // the reference's order: xor butterflies inside 32-chain groups, then over the 32 group sums
#pragma unroll
    for (int c = 0; c < CH; ++c) {
#pragma unroll
        for (int o = 16; o >= 1; o >>= 1) {
            acc[c] = acc[c] + __shfl_xor(acc[c], o, 32);
        }
        if ((t & 31) == 0) {
            warp_sum[(c * THREADS + t) >> 5] = acc[c];
        }
    }
    __syncthreads();
    if (t < 32) {
        float total = warp_sum[t];
#pragma unroll
        for (int o = 16; o >= 1; o >>= 1) {
            total = total + __shfl_xor(total, o, 32);
        }
        if (t == 0) {
            warp_sum[0] = total;
        }
    }
    __syncthreads();
    const float denom = uniform_f(warp_sum[0] + 1e-6f);
    const float u     = __int_as_float(s.misc[0]);
    int         n     = __builtin_amdgcn_readfirstlane(s.n_cand);
    bool        probs = false;
    __syncthreads();
    const float e_bound = key_to_float(thr);
    if (n > TK_CCAP || !valid || !lp_gather_covers<DT>(e_bound, denom)) {
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

// threads: 1024, 512 or 256 per row; window: 0 or 1 (history bitmaps in global memory, small LDS window)
int lp_short_launch_f32(int window, int threads, int rows, hipStream_t st, const FusedParams& p, const FusedLaunch& l,
                        const LogProbLaunch& lp);
int lp_short_launch_f16(int window, int threads, int rows, hipStream_t st, const FusedParams& p, const FusedLaunch& l,
                        const LogProbLaunch& lp);
int lp_short_launch_bf16(int window, int threads, int rows, hipStream_t st, const FusedParams& p, const FusedLaunch& l,
                         const LogProbLaunch& lp);

}  // namespace ftk
