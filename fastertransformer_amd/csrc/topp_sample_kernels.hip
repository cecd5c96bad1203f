// The top-p step that samples straight from logits (ftk_fused_topp_sample_step, ftk_fused_topp_penalty_step).
//
// What TopPSamplingLayer runs per step - temperature, repetition / presence penalty and minimum length
// (src/fastertransformer/layers/sampling_layers/BaseSamplingLayer.cc:302-352), softmax, nucleus sampling and decay
// (layers/sampling_layers/TopPSamplingLayer.cu:256-343) - without writing penalised logits or probabilities to the
// caller's buffer. Results are bit for bit those of the kernel sequence. Three launches (four for fp32):
//
//   stage  reads the logits once: the values y after temperature, penalties and masks (kept in the workspace when there
//          are any), the row's maximum, whether there is a NaN, and, 16-bit types: the maximum of every block of 512
//          columns, fp32: a histogram of y;
//   sum    reads y: e = T(exp(y - max)) summed in the order of the reference's softmax
//          (sampling_topp_kernels.cu:1308-1344: thread t of 1024 adds columns t, t + 1024, ... one after the other, then
//          xor butterflies). A workgroup owns whole summation chains, so that a row can spread over several workgroups
//          and the sum keeps the reference's bits. On the way
//            16-bit types: counts how often every value of e occurs (there are few: at most 3970 / 15361);
//            fp32: the histogram of the stage says where the draw must lie; what is at or above that cut goes to
//            its bucket's place in the ordered prefix;
//   sort   (fp32) long prefixes, in segments dealt out over the launch;
//   pick   one workgroup per row replays the reference's scan and emits the token.
//
// 16-bit types need no sort: the counts are the sorted row in run-length form, the scan reads its values from the
// runs, and the one id that is emitted is looked up in the row: the n-th column, in order of ids, whose value is the
// picked one. Long runs of equal values, which 16-bit logits have everywhere, cost nothing.
#include <algorithm>
#include <type_traits>

#include "ftk_topp.cuh"
#include "ftk_sampling.h"
#include "ftk_topp_sample.h"

namespace ftk {

constexpr int   TSP_STAGE   = 256;        // threads of a stage workgroup, fp32
// 16-bit types: of a workgroup with and without penalties
constexpr int   topp_stage16_threads(bool penalties) { return penalties ? 512 : 256; }
constexpr int   TSP_SUM16   = 1024;       // threads of a sum workgroup, 16-bit types
constexpr int   TSP_SUM32   = 256;        // fp32
constexpr int   TSP_CHAINS  = 1024;       // summation chains of a row (the reference's block)
// Where the code of the large fp32 kernels starts. The same instructions at another multiple of 256 bytes take longer or
// shorter with every change to the file: 256 x 128256, at 1.5 KB behind a multiple of 2 KB / at one, stage 27.7 / 27.3 and sum 28.7 / 28.25
// us, a step 71.0 / 70.4.
constexpr int   TSP_CODE_ALIGN = 2048;
constexpr int   TSP_STAGE_WAVES = 4096;   // waves of a stage launch, 16-bit types
constexpr int   TSP_SPLITS  = 64;         // most workgroups per row of the 16-bit stage
constexpr int   TSP_BLOCK   = 512;        // columns whose maximum the 16-bit stage keeps: one 16-byte vector per lane
constexpr int   TSP_WINDOW  = 5120 + 4;   // words of the history bitmap of a workgroup
constexpr int   TSP_BUCKETS = 2048;       // fp32: buckets of y, 1/64 wide, downwards from TSP_ABOVE over the reference
constexpr float TSP_SCALE   = 64.0f;
constexpr float TSP_ABOVE   = 8.0f;
constexpr float TSP_LOWEST  = -3.402823466e+38f;

struct ToppStep {
    const void*  logits;
    const void*  bias;
    int          n, Vp, rows;  // columns of the vocabulary, pitch of a row
    void*        y;            // [rows][y_pitch], or null: y is the logits themselves
    int          y_pitch;
    const float* temperatures;
    const float* penalties;
    int          penalty_type;  // 2: none
    const int*   min_lengths;
    const int*   end_ids;
    const int*   input_lengths;
    const int*   history;  // element (t, row) at history[t * batch_size + row]
    const int*   sequence_length;
    int          batch_size, step, max_input_length;
    const bool*  finished;
    const bool*  skip;
    const RngState* rng;
    const float* uniforms;
    float        top_p;
    const float* top_ps;
    int          splits, chunk;  // 16-bit stage: workgroups per row and columns of one
    int          parts;          // sum (and the fp32 stage): workgroups per row
    int          blocks;         // blocks of TSP_BLOCK columns per row
    float2*      pmax;           // [rows][TSP_SPLITS]: maximum of a stage workgroup, and 1 when it saw a NaN
    float*       block_max;      // [rows][blocks]
    float*       ref;            // [rows]
    float*       gsum;           // [rows][32]
    uint32_t*    counts;         // 16-bit: [rows][counters]; fp32: [rows][parts][TSP_BUCKETS]
    ToppRowMeta* meta;
    uint32_t*    segs;           // [rows][TPB_NB] ends of segments
    uint32_t*    queue;          // [0]: segments left to the sort's workgroups, then the segments (row * TPB_NB + number)
    unsigned long long* sorted;
};

// Counters of the 16-bit types. binary16: one per value of e up to 1. bfloat16: one per value from 2^-31 to 1; a draw
// that falls among smaller ones takes the exact fallback.
template<int DT>
struct ToppCode;
template<>
struct ToppCode<DT_F16> {
    static constexpr int COUNTERS = 16384, USED = 15361, BASE = 0;
};
template<>
struct ToppCode<DT_BF16> {
    static constexpr int COUNTERS = 4096, BASE = ((127 - 31) << 7) - 1, USED = 127 * 128 - BASE + 1;
};
static_assert(ToppCode<DT_BF16>::USED <= ToppCode<DT_BF16>::COUNTERS, "bfloat16 counters");

// The value a column has after temperature, penalties and the minimum length, as the kernel sequence leaves it.
template<int DT>
struct ToppTransform {
    TemperatureCtx<DT> temperature;
    bool               temperature_active;
    float              penalty;
    int                penalty_type, masked_end;
    const typename Storage<DT>::T* bias;
    // (every load is requested before the first value is used)
    __device__ __forceinline__ ToppTransform(const ToppStep& s, int row): ToppTransform(s, Args(s, row), row) {}

private:
    struct Args {
        float temperature, penalty;
        int   min_length, length, end_id;
        __device__ __forceinline__ Args(const ToppStep& s, int row)
        {
            const void* safe = s.gsum;
            temperature      = row_arg_or(s.temperatures, row, safe, 1.0f);
            penalty          = row_arg_or(s.penalties, row, safe, 0.0f);
            min_length       = row_arg_or(s.min_lengths, row, safe, 0);
            length           = row_arg_or(s.min_lengths != nullptr ? s.sequence_length : nullptr, row, safe, 0);
            end_id           = row_arg_or(s.min_lengths != nullptr ? s.end_ids : nullptr, row, safe, -1);
        }
    };
    __device__ __forceinline__ ToppTransform(const ToppStep& s, const Args& a, int):
        temperature(a.temperature, s.n, s.Vp, false)
    {
        temperature_active = s.temperatures != nullptr;
        bias               = (const typename Storage<DT>::T*)s.bias;
        penalty_type       = s.penalties != nullptr ? s.penalty_type : 2;
        penalty            = a.penalty;
        masked_end = s.min_lengths != nullptr && min_length_masks(a.length, s.max_input_length, a.min_length) ? a.end_id : -1;
    }

public:
    __device__ __forceinline__ float operator()(int v, float x, bool in_history) const
    {
        if (temperature_active) {
            x = temperature.value(x, bias != nullptr, bias != nullptr ? Storage<DT>::ld(bias[v]) : 0.0f);
        }
        if (in_history) {
            x = round_t<DT>(repetition_value(x, penalty, penalty_type));
        }
        return v == masked_end ? -Storage<DT>::max_t() : x;
    }
};

// The tokens of a row's history that the penalty counts. Every id is a cache line of its own: eight in flight per thread.
// The first eight are requested ahead of everything else that a workgroup reads: vector loads complete in order, and what
// the history marks is needed first.
template<int THREADS>
struct ToppHistory {
    static constexpr int H = 8;
    int                  ids[H];
    __device__ __forceinline__ void request(const ToppStep& s, int row, int first)
    {
#pragma unroll
        for (int u = 0; u < H; ++u) {
            if (first + u * THREADS < s.step) {  // (the same for the workgroup)
                ids[u] = s.history[(size_t)min(first + u * THREADS + (int)threadIdx.x, s.step - 1) * s.batch_size + row];
            }
        }
    }
    // Calls mark(id) for all of them; `request(s, row, 0)` came before.
    template<class Mark>
    __device__ __forceinline__ void walk(const ToppStep& s, int row, Mark&& mark)
    {
        const int len = s.input_lengths != nullptr ? s.input_lengths[row] : s.max_input_length;
        for (int first = 0; first < s.step; first += H * THREADS) {
            if (first > 0) {
                request(s, row, first);
            }
#pragma unroll
            for (int u = 0; u < H; ++u) {
                const int at = first + u * THREADS + (int)threadIdx.x;
                // (the padding between a short prompt and max_input_length does not count)
                if (at < s.step && !(at >= len && at < s.max_input_length)) {
                    mark(ids[u]);
                }
            }
        }
    }
};

__device__ __forceinline__ bool topp_row_idle(const ToppStep& s, int row)
{
    const void* safe = s.pmax;
    const bool  skip = row_flag_or(s.skip, row, safe, false);
    const bool  fin  = row_flag_or(s.finished, row, safe, false);
    return skip || fin;
}

// Eight neighbouring 16-bit columns from any column on: one access where the memory allows.
__device__ __forceinline__ uint4 topp_load8(const uint16_t* from)
{
    uint4 raw;
    __builtin_memcpy(&raw, from, 16);
    return raw;
}

// ---- stage, 16-bit types ------------------------------------------------------------------------------------------
// (rows x splits) workgroups, each over a run of blocks of 512 columns, a block per wave at a time. The counters that
// several workgroups of the sum add to are cleared on the way. Bound by latency where there are few rows: flags and
// history (2 us), then a few blocks per wave. Requesting the history first and a short loop instead of 25 KB of
// straight-line code, which every wave fetched to run it once: 64 x 128256 bfloat16 with temperature and penalty
// 15.1 -> 12.8 us (16 MB read, 16 MB written; 0.2 of the copy rate), 128 x 152064 with 51 rows of its own 17.9 -> 14.6.
// An embedding bias has an instantiation of its own and is read like the row, sixteen bytes from any column on. us a step with
// a bias, its columns through the loop of the row's end / one two-byte load each / so: 256 x 128256 bfloat16 128.5 / 108.6 /
// 75.5, binary16 143.2 / 124.4 / 91.3; 64 x 128256 52.4 / 53.3 / 40.2; 1 x 32000 with penalties 27.0 / 29.4 / 26.1.
template<int DT, bool TRANSFORM, bool BIASED>
__global__ void __launch_bounds__(topp_stage16_threads(TRANSFORM)) topp_stage_kernel(ToppStep s)
{
    typedef Storage<DT>   S;
    typedef typename S::T T;
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    constexpr int         EPV = 8, THREADS = topp_stage16_threads(TRANSFORM), NW = THREADS / WAVE;
    constexpr uint32_t    INF16 = DT == DT_F16 ? 0x7C00u : 0x7F80u;
    __shared__ uint32_t   window[TRANSFORM ? TSP_WINDOW : 1];
    __shared__ float      red[16];
    __shared__ uint32_t   any_nan;
    const int             row = blockIdx.x, j = blockIdx.y, t = threadIdx.x;
    const int lo   = min(s.n, j * s.chunk);
    const int hi   = min(s.n, lo + s.chunk);
    const int nblk = (hi - lo + TSP_BLOCK - 1) / TSP_BLOCK;
    const T*  rowp = (const T*)s.logits + (size_t)row * s.Vp;
    // the history, the first blocks and everything about the row are requested together
    const bool  hist = TRANSFORM && s.penalties != nullptr && s.penalty_type != 2;
    ToppHistory<THREADS> history;
    if (hist) {
        history.request(s, row, 0);
    }
    auto load = [&](int b) {
        // (a vector that runs over the end is put right when it is used)
        return topp_load8(rowp + max(0, min(lo + b * TSP_BLOCK + lane_id() * EPV, s.n - EPV)));
    };
    uint4 r0 = load(wave_id()), r1 = load(wave_id() + NW), r2 = load(wave_id() + 2 * NW), r3 = load(wave_id() + 3 * NW);
    const bool              idle = topp_row_idle(s, row);
    const ToppTransform<DT> f(s, row);
    if (idle) {
        return;
    }
    T*        y    = (T*)s.y + (size_t)row * s.y_pitch;
    float*    bmax = s.block_max + (size_t)row * s.blocks;
    const float mul = f.temperature_active ? f.temperature.inv : 1.0f;
    if (s.parts > 1) {
        uint4* counters = reinterpret_cast<uint4*>(s.counts + (size_t)row * ToppCode<DT>::COUNTERS);
        for (int i = j * THREADS + t; i < ToppCode<DT>::COUNTERS / 4; i += s.splits * THREADS) {
            counters[i] = make_uint4(0u, 0u, 0u, 0u);
        }
    }
    if (t == 0) {
        any_nan = 0u;
    }
    if (hist) {
        const int words = (hi - lo + 31) / 32 + 1;
        for (int i = t; i < words; i += THREADS) {
            window[i] = 0u;
        }
        lds_barrier();
        history.walk(s, row, [&](int id) {
            if (id >= lo && id < hi) {
                atomicOr(&window[(id - lo) >> 5], 1u << ((id - lo) & 31));
            }
        });
    }
    lds_barrier();
    float mx   = TSP_LOWEST;
    u16x2 seen = {0, 0};  // largest magnitude bits (a NaN has the largest)
    // Four vectors of the lane are in flight. The loop stays a loop, and what few columns need are loops in it: a wave goes
    // through it a few times only, so that straight-line code waits for its own fetch.
#pragma unroll 1
    for (int b = wave_id(); b < nblk; b += NW) {
        uint4 raw = r0, add = {};
        if constexpr (BIASED) {  // (in front of the next block's load: what is waited for first)
            add = topp_load8(f.bias + max(0, min(lo + b * TSP_BLOCK + lane_id() * EPV, s.n - EPV)));
        }
        r0        = r1;
        r1        = r2;
        r2        = r3;
        r3        = load(b + 4 * NW);
        {   // One vector from here on. Left to itself the compiler takes it apart: loads of 12 and 8 bytes in binary16 (the kernel
            // at 160 x 50257 14.2 -> 15.3 us), a conversion per column instead of one per two in bfloat16 (64 x 128256 12.6 -> 13.2).
            typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
            u32x4 whole = __builtin_bit_cast(u32x4, raw);
            asm("" : "+v"(whole));
            raw = __builtin_bit_cast(uint4, whole);
        }
        const int      v    = lo + b * TSP_BLOCK + lane_id() * EPV;
        const int      rel  = v - lo;
        const uint32_t bits = TRANSFORM && hist && v < hi ? (window[rel >> 5] >> (rel & 31)) & 0xFFu : 0u;
        float          vm   = TSP_LOWEST;
        if (v + EPV > s.n) {
            // two columns at a time; the words of the vector take turns in `raw.x`
#pragma unroll 1
            for (int k = 0; k < EPV / 2; ++k) {
                uint32_t word = 0u;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const int col = v + 2 * k + c;
                    if (col < s.n) {
                        T e = rowp[col];
                        if constexpr (TRANSFORM) {
                            e = S::st(f(col, S::ld(e), ((bits >> (2 * k + c)) & 1u) != 0u));
                        }
                        vm = __builtin_fmaxf(vm, S::ld(e));
                        word |= (uint32_t)e << (16 * c);
                    }
                }
                raw = make_uint4(raw.y, raw.z, raw.w, word);
            }
        }
        else {
            if constexpr (TRANSFORM) {
                T* e = reinterpret_cast<T*>(&raw);
                if constexpr (BIASED) {
                    const T* a = reinterpret_cast<const T*>(&add);
#pragma unroll
                    for (int c = 0; c < EPV; ++c) {
                        e[c] = S::st(S::ld(e[c]) + S::ld(a[c]));
                    }
                }
#pragma unroll
                for (int c = 0; c < EPV; ++c) {
                    e[c] = S::st(S::ld(e[c]) * mul);
                }
                // columns of the history and a masked end id: few lanes, a column of each at a time
                const uint32_t end  = (uint32_t)(f.masked_end - v);
                uint32_t       todo = bits | (end < (uint32_t)EPV ? 1u << end : 0u);
                while (todo != 0u) {
                    const uint32_t c = (uint32_t)__builtin_ctz(todo);
                    todo &= todo - 1u;
                    const uint32_t word = c < 4u ? (c < 2u ? raw.x : raw.y) : (c < 6u ? raw.z : raw.w);
                    const uint32_t sh   = (c & 1u) * 16u;
                    T              x    = (T)(word >> sh);
                    if ((bits >> c) & 1u) {
                        x = S::st(repetition_value(S::ld(x), f.penalty, f.penalty_type));
                    }
                    if (c == end) {
                        x = S::st(-S::max_t());
                    }
                    const uint32_t put = (word & ~(0xFFFFu << sh)) | ((uint32_t)x << sh);
                    raw.x              = c >> 1 == 0u ? put : raw.x;
                    raw.y              = c >> 1 == 1u ? put : raw.y;
                    raw.z              = c >> 1 == 2u ? put : raw.z;
                    raw.w              = c >> 1 == 3u ? put : raw.w;
                }
            }
            const T* e = reinterpret_cast<const T*>(&raw);
#pragma unroll
            for (int c = 0; c < EPV; ++c) {
                vm = __builtin_fmaxf(vm, S::ld(e[c]));
            }
        }
        if constexpr (TRANSFORM) {
            // (rows of y are padded to whole vectors; y that does not stay in the L2s, which the stage writes back at its end,
            // makes the stage faster and the sum slower: 64 x 128256 12.6 -> 11.8 and 11.4 -> 12.0 us, a step of 128 x 152064 with
            // 51 rows of its own 74 -> 75)
            if (v < hi) {
                *reinterpret_cast<uint4*>(y + v) = raw;
            }
        }
        const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int c = 0; c < EPV / 2; ++c) {
            seen = __builtin_elementwise_max(seen, __builtin_bit_cast(u16x2, w[c] & 0x7FFF7FFFu));
        }
        mx = __builtin_fmaxf(mx, vm);
        vm = wave_reduce_unordered(vm, [](float a, float c) { return __builtin_fmaxf(a, c); });
        if (lane_id() == 0) {
            bmax[lo / TSP_BLOCK + b] = vm;
        }
    }
    if (max((uint32_t)seen.x, (uint32_t)seen.y) > INF16) {
        any_nan = 1u;
    }
    mx = block_max<float, NW>(mx, red, TSP_LOWEST);  // (barriers)
    if (t == 0) {
        s.pmax[(size_t)row * TSP_SPLITS + j] = make_float2(mx, any_nan != 0u ? 1.0f : 0.0f);
    }
}

// ---- stage, fp32 --------------------------------------------------------------------------------------------------
__device__ __forceinline__ int topp_y_bucket(float y, float top, float last = (float)(TSP_BUCKETS - 1))
{
    return (int)__builtin_amdgcn_fmed3f((top - y) * TSP_SCALE, 0.0f, last);
}

// (rows x parts) workgroups; a workgroup reads the columns of its summation chains, 1024 / parts neighbouring columns
// out of every 1024, so that its histogram says how many entries of every bucket the sum's workgroup of the same part
// will place. Rows are the fast index of the grid, and their number is rounded up to a multiple of eight: the parts of a
// row then run on one XCD, of the stage and of the sum, and its L2 keeps the row's histograms from the one to the other
// (us a step, as they come / rounded up: 1 x 8192 25.2 / 23.7, 33 x 8192 42 / 36, 95 x 8192 68 / 45; 255 x 128256
// 113 / 117). With the parts as the fast index every XCD would see the same quarter of every 4 KB and use a quarter of its
// L2's channels.
template<bool TRANSFORM>
__attribute__((aligned(TSP_CODE_ALIGN))) __global__ void __launch_bounds__(TSP_STAGE) topp_stage_f32_kernel(ToppStep s)
{
    // The last bucket is open below: masked columns, half of a row perhaps, lie there and would queue for its counter. It
    // is spread over a counter per lane (256 x 128256, every second column -inf: 153 -> 114 us a step).
    __shared__ uint32_t hist[TSP_BUCKETS - 1 + WAVE];
    __shared__ uint32_t window[TRANSFORM ? TSP_WINDOW : 1];
    __shared__ float    red[16];
    __shared__ uint32_t any_nan;
    const int           row = blockIdx.x, j = blockIdx.y, t = threadIdx.x;
    const float         last = (float)(TSP_BUCKETS - 1 + lane_id());
    if (row == 0 && j == 0 && t == 0) {
        s.queue[0] = 0u;
    }
    if (row >= s.rows || topp_row_idle(s, row)) {
        return;
    }
    const float* rowp  = (const float*)s.logits + (size_t)row * s.Vp;
    float*       y     = (float*)s.y + (size_t)row * s.y_pitch;
    const int    C     = TSP_CHAINS / s.parts;
    const int    shift = __builtin_ctz((unsigned)C);
    const int    c0    = j * C;
    const int    nit   = (s.n + TSP_CHAINS - 1) / TSP_CHAINS;
    // the origin of the buckets: the largest value among 1024 columns, 32 lines of 32 spread over the row (ids of one script
    // or of special tokens are neighbours), without the history; the same for every part. Everything 8 or more above it
    // lies in the first bucket (256 x 128256 with the first 1024 columns masked: 22 ms a step with those as the sample,
    // 0.12 ms). More and shorter stretches cost time on every row: 64 of 16, 0.7 us.
    constexpr int U0 = TSP_CHAINS / TSP_STAGE;
    auto  sample = [&](int u) { return (u * (TSP_STAGE / 32) + (t >> 5)) * ((s.n / 32) & ~31) + (t & 31); };
    const bool  marks = TRANSFORM && s.penalties != nullptr && s.penalty_type != 2;
    ToppHistory<TSP_STAGE> history;
    if (marks) {
        history.request(s, row, 0);
    }
    float plain[U0];
#pragma unroll
    for (int u = 0; u < U0; ++u) {
        plain[u] = rowp[sample(u)];
    }
    // (and the first vectors of the row, so that they do not wait for the sample's maximum)
    constexpr int U     = 8;
    const int     quads = C / 4, qshift = shift - 2;  // 16-byte vectors of a workgroup in one stretch of 1024 columns
    const int     nfull = s.n / TSP_CHAINS;           // stretches that lie inside the vocabulary
    const int     total = nfull * quads;              // vectors
    const bool    vec   = (s.Vp & 3) == 0 && ((uintptr_t)s.logits & 15u) == 0u;
    float4        raw[U];
    auto          load = [&](int i0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = min(i0 + u * TSP_STAGE, total - 1);
            raw[u]      = *reinterpret_cast<const float4*>(rowp + (size_t)(i >> qshift) * TSP_CHAINS + c0 + (i & (quads - 1)) * 4);
        }
    };
    if (vec) {
        load(t);
    }
    for (int i = t; i < TSP_BUCKETS - 1 + WAVE; i += TSP_STAGE) {
        hist[i] = 0u;
    }
    if (t == 0) {
        any_nan = 0u;
    }
    const ToppTransform<DT_F32> f(s, row);
    if (TRANSFORM && marks) {
        const int words = (nit * C + 31) / 32 + 1;
        for (int i = t; i < words; i += TSP_STAGE) {
            window[i] = 0u;
        }
    }
    float first = TSP_LOWEST;
#pragma unroll
    for (int u = 0; u < U0; ++u) {
        first = __builtin_fmaxf(first, TRANSFORM ? f(sample(u), plain[u], false) : plain[u]);
    }
    first = block_max<float, TSP_STAGE / WAVE>(first, red, TSP_LOWEST);  // (two barriers: both tables are clear)
    if (!(__builtin_fabsf(first) < 1e30f)) {
        first = 0.0f;
    }
    const float top = first + TSP_ABOVE;
    if (TRANSFORM && marks) {
        history.walk(s, row, [&](int id) {
            const int c = (id & (TSP_CHAINS - 1)) - c0;
            if (id >= 0 && id < s.n && c >= 0 && c < C) {
                const int at = ((id / TSP_CHAINS) << shift) + c;
                atomicOr(&window[at >> 5], 1u << (at & 31));
            }
        });
        __syncthreads();
    }
    float mx  = TSP_LOWEST;
    bool  nan = false;
    auto  one = [&](int it, int c, float x) -> float {  // column it * 1024 + c0 + c
        if constexpr (TRANSFORM) {
            const int  at     = (it << shift) + c;
            const bool marked = marks && ((window[at >> 5] >> (at & 31)) & 1u) != 0u;
            x                 = f(it * TSP_CHAINS + c0 + c, x, marked);
        }
        mx  = __builtin_fmaxf(mx, x);
        nan = nan || x != x;
        atomicAdd(&hist[topp_y_bucket(x, top, last)], 1u);
        return x;
    };
    int it0 = 0;
    if (vec) {
        for (int i0 = t; i0 < total; i0 += U * TSP_STAGE) {
            if (i0 != t) {
                load(i0);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = i0 + u * TSP_STAGE;
                if (i < total) {
                    const int it = i >> qshift;
                    const int c  = (i & (quads - 1)) * 4;
                    float4    r  = raw[u];
                    r.x          = one(it, c, r.x);
                    r.y          = one(it, c + 1, r.y);
                    r.z          = one(it, c + 2, r.z);
                    r.w          = one(it, c + 3, r.w);
                    if constexpr (TRANSFORM) {
                        *reinterpret_cast<float4*>(y + (size_t)it * TSP_CHAINS + c0 + c) = r;
                    }
                }
            }
        }
        it0 = nfull;
    }
    {
        constexpr int U     = 8;
        const int     total = (nit - it0) << shift;
        for (int i0 = t; i0 < total; i0 += U * TSP_STAGE) {
            float raw[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = i0 + u * TSP_STAGE;
                const int v = (it0 + (i >> shift)) * TSP_CHAINS + c0 + (i & (C - 1));
                raw[u]      = i < total && v < s.n ? rowp[v] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i  = i0 + u * TSP_STAGE;
                const int it = it0 + (i >> shift), c = i & (C - 1);
                const int v  = it * TSP_CHAINS + c0 + c;
                if (i < total && v < s.n) {
                    const float x = one(it, c, raw[u]);
                    if constexpr (TRANSFORM) {
                        y[v] = x;
                    }
                }
            }
        }
    }
    for (int v = s.n + t; v < s.Vp; v += TSP_STAGE) {  // pads lie in the last bucket
        const int c = (v & (TSP_CHAINS - 1)) - c0;
        if (c >= 0 && c < C) {
            atomicAdd(&hist[TSP_BUCKETS - 1 + lane_id()], 1u);
        }
    }
    if (nan) {
        any_nan = 1u;
    }
    mx = block_max<float, TSP_STAGE / WAVE>(mx, red, TSP_LOWEST);
    uint32_t* out = s.counts + ((size_t)row * s.parts + j) * TSP_BUCKETS;
    const int low = wave_sum_i((int)hist[TSP_BUCKETS - 1 + lane_id()]);
#pragma unroll
    for (int u = 0; u < TSP_BUCKETS / 4 / TSP_STAGE; ++u) {
        const int i = t + u * TSP_STAGE;
        uint4     c = reinterpret_cast<const uint4*>(hist)[i];
        c.w         = i == TSP_BUCKETS / 4 - 1 ? (uint32_t)low : c.w;
        reinterpret_cast<uint4*>(out)[i] = c;
    }
    if (t == 0) {
        s.pmax[(size_t)row * TSP_SPLITS + j] = make_float2(mx, any_nan != 0u ? 1.0f : 0.0f);
        if (j == 0) {
            s.ref[row] = first;
        }
    }
}

// The maximum of a row from what the stage's workgroups left (every lane of the wave gets it); a NaN when a sum over
// the row would be one: there is a NaN among the values, or the maximum is infinite.
struct ToppRowMax {
    float2 mine;
    __device__ __forceinline__ ToppRowMax(const ToppStep& s, int row, int n_partial)
    {
        const int l = min(lane_id(), n_partial - 1);
        mine        = s.pmax[(size_t)row * TSP_SPLITS + l];  // (requested here, used in the call below)
    }
    template<int DT>
    __device__ __forceinline__ float get(const ToppStep& s) const
    {
        float mx = mine.x;
        if (s.Vp > s.n) {
            mx = __builtin_fmaxf(mx, -Storage<DT>::max_t());
        }
        mx             = wave_reduce_unordered(mx, [](float a, float b) { return __builtin_fmaxf(a, b); });
        const bool nan = __ballot(mine.y != 0.0f) != 0ull || mx == __builtin_inff();
        return nan ? __builtin_nanf("") : mx;
    }
};

// exp of d <= 0 as det_expf_nonpos gives it, for numbers; below -86 something between 0 and 1e-37 instead of the exact
// value, which no sum over a row that holds a 1 can tell apart (its terms are far below half a unit of any such sum,
// and the group sums without the 1 vanish against it the same way). The integer part of the argument stays in the low
// bits of the sum with 3 * 2^22, from where it goes straight into the exponent.
__device__ __forceinline__ float topp_exp(float d)
{
    d               = __builtin_fmaxf(d, -86.0f);
    const float t   = d * 1.44269502162933349609375f + 12582912.0f;
    const float n   = t - 12582912.0f;
    float       r   = fma_rn(n, -0.693145751953125f, d);
    r               = fma_rn(n, -1.428606765330187045e-06f, r);
    float p         = 1.9875691500e-4f;
    p               = fma_rn(p, r, 1.3981999507e-3f);
    p               = fma_rn(p, r, 8.3334519073e-3f);
    p               = fma_rn(p, r, 4.1665795894e-2f);
    p               = fma_rn(p, r, 1.6666665459e-1f);
    p               = fma_rn(p, r, 5.0000001201e-1f);
    const float z   = r * r;
    const float y   = fma_rn(p, z, r) + 1.0f;
    return u2f(f2u(y) + (f2u(t) << 23));
}

// Four neighbouring lanes hold consecutive terms of one summation chain: added in their order, in every lane.
__device__ __forceinline__ float topp_chain_add(float sum, float e)
{
    sum += dpp_from<0x00>(e);
    sum += dpp_from<0x55>(e);
    sum += dpp_from<0xAA>(e);
    sum += dpp_from<0xFF>(e);
    return sum;
}

// Walks the columns of a workgroup's summation chains: LPC lanes share a chain and take its columns in turn.
// visit(v, raw) returns e; the chain's sum comes back. Batches of U columns per thread, the next batch requested before
// the current one is used (a uniform base and a 32-bit offset per lane: one load instruction per column and no address
// arithmetic in vector registers), the first one by topp_chains_load at the kernel's start. `pad` is what the columns
// behind the vocabulary hold.
template<class T, int LPC, int U>
__device__ __forceinline__ void topp_chains_load(T (&raw)[U], const T* __restrict__ y, int b, int chain, int q)
{
    constexpr int  STRIDE = LPC * TSP_CHAINS;
    const uint32_t lane   = (uint32_t)(chain + q * TSP_CHAINS);
    const T*       base   = y + (size_t)b * (U * STRIDE);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        raw[u] = (base + u * STRIDE)[lane];
    }
}

template<class T, int LPC, int U, class Visit>
__device__ __forceinline__ float topp_walk_chains(const T (&first)[U], const T* __restrict__ y, int n, int Vp, int chain, int q, T pad,
                                                  Visit&& visit)
{
    constexpr int  STRIDE = LPC * TSP_CHAINS;
    float          sum    = 0.0f;
    const uint32_t lane   = (uint32_t)(chain + q * TSP_CHAINS);
    const int      nb     = n / (U * STRIDE);  // batches that every lane of the workgroup holds in full
    T              buf[2][U];
    auto           load = [&](T (&raw)[U], int b) { topp_chains_load<T, LPC, U>(raw, y, b, chain, q); };
    auto add = [&](float e) {
        if constexpr (LPC == 1) {
            sum += e;
        }
        else {
            sum = topp_chain_add(sum, e);
        }
    };
    auto use = [&](const T* raw, int b) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            add(visit((int)lane + (b * U + u) * STRIDE, raw[u]));
        }
    };
#pragma unroll
    for (int u = 0; u < U; ++u) {
        buf[0][u] = first[u];
    }
    for (int b = 0; b < nb; b += 2) {
        load(buf[1], min(b + 1, nb - 1));
        use(buf[0], b);
        load(buf[0], min(b + 2, nb - 1));
        if (b + 1 < nb) {
            use(buf[1], b + 1);
        }
    }
    // what does not fill a batch (columns beyond the row count as nothing)
    for (int v0 = nb * U * STRIDE; v0 < Vp; v0 += U * STRIDE) {
        T raw[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int v = v0 + u * STRIDE + (int)lane;
            raw[u]      = y[min(v, n - 1)];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int v = v0 + u * STRIDE + (int)lane;
            if (v0 + u * STRIDE < Vp) {  // (the same for every lane)
                add(v < Vp ? visit(v, v < n ? raw[u] : pad) : 0.0f);
            }
        }
    }
    return sum;
}

// The xor butterflies inside 32-lane groups over the chain sums of the workgroup; the sums of the groups go to memory.
template<int THREADS, int LPC>
__device__ __forceinline__ void topp_group_sums(const ToppStep& s, int row, int part, float sum, float* chain_sum)
{
    constexpr int C = THREADS / LPC;
    const int     t = threadIdx.x;
    if (LPC == 1 || (t % LPC) == 0) {
        chain_sum[t / LPC] = sum;
    }
    __syncthreads();
    if (t < C) {
        float v = chain_sum[t];
#pragma unroll
        for (int m = 16; m > 0; m >>= 1) {
            v += __shfl_xor(v, m, 32);
        }
        if ((t & 31) == 0) {
            s.gsum[(size_t)row * 32 + part * (C / 32) + (t >> 5)] = v;
        }
    }
}

// ---- sum, 16-bit types ----------------------------------------------------------------------------------------------
// A workgroup owns C summation chains: C neighbouring columns out of every 1024 (a "stretch"). Its waves share the
// stretches out, read eight bytes - four chains - per lane and leave the e of a chunk of stretches in LDS, from where
// one thread per chain adds them up in the reference's order. (One chain per thread straight from memory would mean
// two-byte loads and a dependent addition per load.) Where a quarter of the threads adds, the others go on with the next
// chunk in a second buffer: 64 x 128256 bfloat16 13.0 -> 12.0 us, vector instructions in 0.6 of it; 51 rows of 152064 18.3 ->
// 17.7. Where all of them add, two buffers of half the size only cost barriers (a step of 256 x 128256 bfloat16 93.8 -> 95.4).
// e is a function of the 16 bits of y once the maximum is known, but a table of it in LDS, made by every workgroup, does
// not pay: gathers from it cost as much as the exponential (256 x 128256, us a step with a table / so: binary16 95 / 92,
// bfloat16 76 / 76; every second column masked 98 / 84 and 85 / 72).
template<int DT, int C>
__global__ void __launch_bounds__(TSP_SUM16) topp_sum_count_kernel(ToppStep s)
{
    typedef Storage<DT>   S;
    typedef typename S::T T;
    typedef ToppCode<DT>  Code;
    constexpr int         HALVES = C < TSP_SUM16 ? 2 : 1;  // buffers of e, 32 KB in all
    constexpr int         KI  = 16384 / HALVES / C;        // stretches of a chunk
    constexpr int         WS  = C / 4 / WAVE;              // waves side by side in a stretch
    constexpr int         PAR = TSP_SUM16 / WAVE / WS;     // stretches taken at a time
    constexpr int         U   = KI / PAR;                  // vectors per lane and chunk
    __shared__ uint32_t   cnt[Code::USED + WAVE];
    __shared__ uint2      e_of[HALVES][KI * C / 4];
    const int             row = blockIdx.x, part = blockIdx.y, t = threadIdx.x;
    const T* y = s.y != nullptr ? (const T*)s.y + (size_t)row * s.y_pitch : (const T*)s.logits + (size_t)row * s.Vp;
    const int q    = (t & (C / 4 - 1)) * 4 + part * C;  // first of this lane's four chains
    const int mine = t / (C / 4);                       // its first stretch
    const int nst  = (s.Vp + TSP_CHAINS - 1) / TSP_CHAINS;
    // Four vectors of the lane are in flight; the loop that uses them stays a loop (straight-line code of this length
    // runs once and waits for its own fetch).
    const int total = (nst + PAR - 1 - mine) / PAR;  // vectors of this lane
    auto      load  = [&](int k) -> uint2 {          // its k-th one
        const int v = (mine + min(k, total - 1) * PAR) * TSP_CHAINS + q;
        uint2     x;
        // (columns behind the vocabulary are put right where they are used: any four columns of the row will do here)
        __builtin_memcpy(&x, y + max(0, min(v, s.n - 4)), 8);
        return x;
    };
    const ToppRowMax rm(s, row, s.splits);
    uint2            r0 = load(0), r1 = load(1), r2 = load(2), r3 = load(3);
    if (topp_row_idle(s, row)) {
        return;
    }
    for (int i = t; i < Code::USED; i += TSP_SUM16) {
        cnt[i] = 0u;
    }
    const float mx = rm.get<DT>(s);
    if (!(mx == mx)) {
        return;  // (the pick sees the same and needs no sum)
    }
    __syncthreads();
    // The e of N values, counted; what has no counter goes to a word of the lane's own.
    auto e_bits = [&](const auto& x, auto& b) {
        constexpr int N = (int)(sizeof(x) / sizeof(x[0]));
#pragma unroll
        for (int c = 0; c < N; ++c) {
            b[c] = S::st(topp_exp(S::ld((T)x[c]) - mx));
        }
#pragma unroll
        for (int c = 0; c < N; ++c) {
            const int code = (int)b[c] - Code::BASE;
            atomicAdd(&cnt[code > 0 ? code : Code::USED + lane_id()], 1u);
        }
    };
    const uint32_t pad = S::st(-S::max_t());
    float          sum = 0.0f;
    int            at  = 0;
    int            half = 0;
    for (int i0 = 0; i0 < nst; i0 += KI, half ^= HALVES - 1) {
#pragma unroll 1
        for (int u = 0; u < U; ++u, ++at) {
            const int i = mine + u * PAR;
            const int v = (i0 + i) * TSP_CHAINS + q;
            if (i0 + i >= nst) {
                break;
            }
            const uint2 raw = r0;
            r0 = r1;
            r1 = r2;
            r2 = r3;
            r3 = load(at + 4);
            uint32_t b[4];
            if (v + 4 <= s.n) {
                const uint32_t x[4] = {raw.x & 0xFFFFu, raw.x >> 16, raw.y & 0xFFFFu, raw.y >> 16};
                e_bits(x, b);
            }
            else {
#pragma unroll 1
                for (int c = 0; c < 4; ++c) {
                    uint32_t e = 0u;
                    if (v + c < s.Vp) {
                        const uint32_t x[1] = {v + c < s.n ? (uint32_t)y[v + c] : pad};
                        uint32_t       one[1];
                        e_bits(x, one);
                        e = one[0];
                    }
                    b[0] = c == 0 ? e : b[0];
                    b[1] = c == 1 ? e : b[1];
                    b[2] = c == 2 ? e : b[2];
                    b[3] = c == 3 ? e : b[3];
                }
            }
            e_of[half][i * (C / 4) + (t & (C / 4 - 1))] = make_uint2(b[0] | (b[1] << 16), b[2] | (b[3] << 16));
        }
        lds_barrier();
        if (t < C) {
            const T*  e = reinterpret_cast<const T*>(e_of[half]) + t;
            const int k = min(KI, nst - i0);
#pragma unroll 8
            for (int i = 0; i < k; ++i) {
                sum += S::ld(e[i * C]);
            }
        }
        // (with two buffers the waves that add nothing go on with the other one; what is added here is overwritten behind the
        // next barrier only)
        if constexpr (HALVES == 1) {
            lds_barrier();
        }
    }
    if (t < C) {
#pragma unroll
        for (int m = 16; m > 0; m >>= 1) {
            sum += __shfl_xor(sum, m, 32);
        }
        if ((t & 31) == 0) {
            s.gsum[(size_t)row * 32 + part * (C / 32) + (t >> 5)] = sum;
        }
    }
    uint32_t* counters = s.counts + (size_t)row * Code::COUNTERS;
    if (gridDim.y == 1) {
        for (int i = t; i < Code::COUNTERS; i += TSP_SUM16) {
            counters[i] = i < Code::USED ? cnt[i] : 0u;
        }
    }
    else {
        for (int i = t; i < Code::USED; i += TSP_SUM16) {
            const uint32_t c = cnt[i];
            if (c != 0u) {
                atomicAdd(&counters[i], c);
            }
        }
    }
}

// ---- sum, fp32 --------------------------------------------------------------------------------------------------------
// Where the draw must lie comes from the stage's histogram: a bucket's mass is at least its count times the exponential
// of its lower edge and at most the same with its upper edge. Everything down to the bucket that certainly covers the
// draw - and two more, so that all entries which share a probability with the last one that can be drawn are
// there - goes to its bucket's place in the prefix, keyed by e (the division by the denominator keeps the order).
template<int LPC>
__attribute__((aligned(TSP_CODE_ALIGN))) __global__ void __launch_bounds__(TSP_SUM32) topp_sum_gather_kernel(ToppStep s)
{
    constexpr int       C  = TSP_SUM32 / LPC;
    constexpr int       K  = TSP_BUCKETS / TSP_SUM32;
    constexpr int       NW = TSP_SUM32 / WAVE;
    constexpr int       U  = 16;  // columns per batch
    __shared__ uint32_t cur[TSP_BUCKETS];
    __shared__ float    chain_sum[C];
    __shared__ float    wmass[NW], wupper[NW];
    __shared__ uint32_t wcnt[NW], wseg[NW];
    __shared__ uint32_t queue_at;  // where the row's segments go in the queue, plus one (0: the pick orders them)
    __shared__ uint32_t red32[16];
    const int           row = blockIdx.x, part = blockIdx.y, t = threadIdx.x;
    if (row >= s.rows || topp_row_idle(s, row)) {
        return;
    }
    const void*         safe = s.pmax;
    const RowDrawSource ds   = row_draw_source(s.rng, s.uniforms, row, safe);
    const float         p    = row_arg_or(s.top_ps, row, safe, s.top_p);
    const ToppRowMax    rm(s, row, s.parts);
    const float         ref = s.ref[row];
    const float* y    = s.y != nullptr ? (const float*)s.y + (size_t)row * s.y_pitch : (const float*)s.logits + (size_t)row * s.Vp;
    // thread t owns buckets [K t, K t + K), in descending order of y
    uint32_t tot[K], before[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        tot[i] = before[i] = 0u;
    }
    const uint4* counts = reinterpret_cast<const uint4*>(s.counts + (size_t)row * s.parts * TSP_BUCKETS);
#pragma unroll 4
    for (int q = 0; q < 4 * LPC; ++q) {
#pragma unroll
        for (int i = 0; i < K / 4; ++i) {
            const uint4    c    = counts[(q * TSP_BUCKETS + t * K) / 4 + i];
            const uint32_t w[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                before[i * 4 + k] += q < part ? w[k] : 0u;
                tot[i * 4 + k] += w[k];
            }
        }
    }
    // (behind the histograms in the queue, and there when the cut is known: 256 x 128256 29.9 -> 29.0 us, a step 65.5 -> 64.1
    // once p has decayed; with sixteen parts a row, 1 to 71 rows of 32000 to 128256 columns, steps take as long either way)
    float first_batch[U] = {};
    if (s.n >= U * LPC * TSP_CHAINS) {
        topp_chains_load<float, LPC, U>(first_batch, y, 0, part * C + t / LPC, t % LPC);
    }
    const float mx = rm.get<DT_F32>(s);
    if (!(mx == mx)) {
        return;  // (the pick sees the same and needs no sum)
    }
    uint64_t    next;
    const float draw = (s.uniforms != nullptr ? ds.injected : row_draw_generate(ds, &next)) * p;
    const float top  = ref + TSP_ABOVE;
    const float lead = top - mx;  // y of the first bucket's upper edge, relative to the maximum
    const int   mx_bucket = topp_y_bucket(mx, top);
    float       lower[K], upper[K], lm = 0.0f, lu = 0.0f;
    uint32_t    lc = 0u;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const int   b     = t * K + i;
        const float up    = b == 0 ? 1.0f : __builtin_amdgcn_exp2f(__builtin_fminf(lead - (float)b / TSP_SCALE, 0.0f) * 1.44269504f);
        const float below = b == TSP_BUCKETS - 1 ? 0.0f :
                                                   __builtin_amdgcn_exp2f(__builtin_fminf(lead - (float)(b + 1) / TSP_SCALE, 0.0f) * 1.44269504f);
        const float n     = (float)tot[i];
        lower[i]          = tot[i] == 0u ? 0.0f : n * below;
        upper[i]          = tot[i] == 0u ? 0.0f : n * up;
        if (b == mx_bucket) {
            lower[i] += 1.0f - below;  // the maximum itself lies here
        }
        lm += lower[i];
        lu += upper[i];
        lc += tot[i];
    }
    float    im = lm, iu = lu;  // running sums: im, ic from the first bucket on, iu from the last one back
    uint32_t ic = lc;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        const float    um = __shfl_up(im, o, WAVE), uu = __shfl_down(iu, o, WAVE);
        const uint32_t uc = __shfl_up(ic, o, WAVE);
        if (lane_id() >= o) {
            im += um;
            ic += uc;
        }
        if (lane_id() + o < WAVE) {
            iu += uu;
        }
    }
    if (lane_id() == WAVE - 1) {
        wmass[wave_id()] = im;
        wcnt[wave_id()]  = ic;
    }
    if (lane_id() == 0) {
        wupper[wave_id()] = iu;
    }
    __syncthreads();
    float em = im - lm, rest = __shfl_down(iu, 1, WAVE);
    rest     = lane_id() == WAVE - 1 ? 0.0f : rest;
    uint32_t ec = ic - lc;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        em += w < wave_id() ? wmass[w] : 0.0f;
        ec += w < wave_id() ? wcnt[w] : 0u;
        rest += w > wave_id() ? wupper[w] : 0.0f;
    }
    // The prefix holds the draw when (mass of the prefix) >= draw * (mass of the row), that is
    // mass * (1 - draw) >= draw * (mass behind it): with the mass from below on the left and from above on the right this
    // is sharp where little lies behind the prefix, however wide its buckets are. (Bounds on the whole row's mass differ
    // by a bucket's width, 1/64, so that draws above 0.98 would always take the whole row. 256 x 128256 N(0, 2.5), p = 0.9,
    // us a step: 406 with such bounds, 117; with two columns far ahead 601, 66.) The margin is the rounding of the
    // reference's scan.
    const float q     = draw * (1.0f + 1.0f / 1024.0f);
    uint32_t    first = 0xFFFFFFFFu;
    {
        float behind[K];
        behind[K - 1] = rest;
#pragma unroll
        for (int i = K - 1; i > 0; --i) {
            behind[i - 1] = behind[i] + upper[i];
        }
        float m = em;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            m += lower[i];
            if (m > 0.0f && m * (1.0f - q) >= q * (behind[i] + 1e-6f) && first == 0xFFFFFFFFu) {
                first = (uint32_t)(t * K + i);
            }
        }
    }
    first         = block_min<uint32_t, NW>(first, red32, 0xFFFFFFFFu);
    const int cut = (int)min(first == 0xFFFFFFFFu ? first : first + 2u, (uint32_t)(TSP_BUCKETS - 1));
    // (a row whose values are all -inf takes the exact fallback)
    const bool usable = mx > TSP_LOWEST;
    uint32_t   off[K + 1];
    off[0] = ec;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        off[i + 1]     = off[i] + tot[i];
        cur[t * K + i] = off[i] + before[i];
    }
    if (part == 0) {
        // the prefix in segments of whole buckets for the sort: a bucket closes a segment when a multiple of TPS_SEG
        // lies inside it or at its end, and the last gathered bucket closes the last one
        uint32_t n_mine = 0u;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            n_mine += t * K + i <= cut ? tot[i] : 0u;
        }
        n_mine = (uint32_t)wave_sum_i((int)n_mine);
        if (lane_id() == 0) {
            wseg[wave_id()] = n_mine;
        }
        __syncthreads();
        uint32_t n = 0u;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            n += wseg[w];
        }
        uint32_t closes[K], lclose = 0u;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            const bool in = t * K + i <= cut && tot[i] != 0u;
            closes[i]     = in && (off[i + 1] / TPS_SEG != off[i] / TPS_SEG || off[i + 1] == n) ? off[i + 1] : 0u;
            lclose += closes[i] != 0u ? 1u : 0u;
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
            wseg[wave_id()] = iclose;
        }
        __syncthreads();
        uint32_t at = iclose - lclose, nseg = 0u;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            at += w < wave_id() ? wseg[w] : 0u;
            nseg += wseg[w];
        }
        uint32_t* ends = s.segs + (size_t)row * TPB_NB;
#pragma unroll
        for (int i = 0; i < K; ++i) {
            if (closes[i] != 0u) {
                ends[at++] = closes[i];
            }
        }
        if (t == 0) {
            ToppRowMeta m;
            m.best  = 0ull;
            m.cut   = cut;
            m.n     = usable ? (int)n : 0;
            m.n_pos = (int)s.Vp;  // the prefix is the whole row exactly when it holds this many entries
            m.nseg  = (int)nseg;
            m.flags = 0;
            // (half a bucket under the one that covers the draw: a bucket and a half above what is not gathered)
            m.safe      = __builtin_amdgcn_exp2f((lead - ((float)cut - 0.5f) / TSP_SCALE) * 1.44269504f);
            s.meta[row] = m;
            // prefixes that fit its LDS are ordered by the pick kernel itself, longer ones by the sort's workgroups
            // (a word of its own: the other waves may still be reading wseg)
            queue_at = usable && n > (uint32_t)TPS_CAP ? atomicAdd(s.queue, nseg) + 1u : 0u;
        }
        __syncthreads();
        const uint32_t to = queue_at;
        if (to != 0u) {
            for (uint32_t i = (uint32_t)t; i < nseg; i += TSP_SUM32) {
                s.queue[to + i] = (uint32_t)row * TPB_NB + i;
            }
        }
    }
    __syncthreads();
    unsigned long long* A     = s.sorted + (size_t)row * 2 * s.Vp;
    // nothing under this lies in the gathered buckets (one bucket of margin)
    const float         y_low = cut >= TSP_BUCKETS - 1 ? -__builtin_inff() : top - (float)(cut + 2) / TSP_SCALE;
    const float sum = topp_walk_chains<float, LPC, U>(first_batch, y, s.n, s.Vp, part * C + t / LPC, t % LPC, -Storage<DT_F32>::max_t(), [&](int v, float x) -> float {
        const float e = topp_exp(x - mx);
        if (x >= y_low && usable) {
            const int b = topp_y_bucket(x, top);
            if (b <= cut) {
                const uint32_t slot = atomicAdd(&cur[b], 1u);
                const float    ex   = x - mx < -86.0f ? det_expf_nonpos(x - mx) : e;
                A[slot]             = ((unsigned long long)(~order_key_nonneg(ex)) << 32) | (uint32_t)v;
            }
        }
        return e;
    });
    topp_group_sums<TSP_SUM32, LPC>(s, row, part, sum, chain_sum);
}

// ---- sort, fp32: the segments of long prefixes, dealt out over the launch
__global__ void __launch_bounds__(TP_THREADS) topp_sort_queue_kernel(ToppStep s)
{
    __shared__ ToppSortShared ss;
    const uint32_t            n = s.queue[0];
    for (uint32_t w = blockIdx.x; w < n; w += gridDim.x) {
        const uint32_t      at   = s.queue[1 + w];
        const int           row  = (int)(at / TPB_NB), i = (int)(at % TPB_NB);
        const uint32_t*     ends = s.segs + (size_t)row * TPB_NB;
        const int           s0   = i > 0 ? (int)ends[i - 1] : 0;
        unsigned long long* A    = s.sorted + (size_t)row * 2 * s.Vp;
        topp_sort_one(ss, A + s0, A + s.Vp + s0, (int)ends[i] - s0);
        __syncthreads();
    }
}

// ---- pick -------------------------------------------------------------------------------------------------------------
// A pick is a chain of short steps on one row, bound by latency: everything it reads from memory that does not depend on
// an earlier step is requested at its start, without control flow (256 fp32 rows with short prefixes: 9 us, 31 us with
// loads where they are used and a sort of every prefix through memory).
struct ToppPickOut {
    int*          ids;
    int*          sequence_length;
    bool*         finished;
    float*        cum_log_probs;
    float*        output_log_probs;
    RngState*     rng;
    ToppDecayArgs dec;
    int           force_deep;
};

struct ToppPicked {
    int   id;
    float prob;
    bool  sampled;  // false: the draw was never reached; the id is kept, nothing else is updated (:954)
};

template<int DT>
struct ToppPickRow {
    typedef Storage<DT>  S;
    typedef typename S::T T;
    int           row;
    bool          skip, fin;
    float         p;
    RowDrawSource draw;
    ToppRowMax    rm;
    float         group;  // one group sum of the row
    int           end_id, length;
    float         cum, decay_p, decay_initial, decay_factor, decay_min;
    int           decay_reset;
    const T*      y;
    // worked out later
    float    mx, denom, rand_num;
    uint64_t next_draw;  // what the row's generator goes on with

    __device__ __forceinline__ ToppPickRow(const ToppStep& s, const ToppPickOut& o, int row_, int n_partial):
        row(row_), rm(s, row_, n_partial)
    {
        const void* safe = s.gsum;
        group         = s.gsum[(size_t)row * 32 + (lane_id() & 31)];
        skip          = row_flag_or(s.skip, row, safe, false);
        fin           = row_flag_or(s.finished, row, safe, false);
        p             = row_arg_or(s.top_ps, row, safe, s.top_p);
        draw          = row_draw_source(s.rng, s.uniforms, row, safe);
        end_id        = row_arg_or(s.end_ids, row, safe, -1);
        length        = row_arg_or(o.sequence_length, row, safe, 0);
        cum           = row_arg_or(o.cum_log_probs, row, safe, 0.0f);
        decay_p       = row_arg_or(o.dec.runtime_top_p, row, safe, 0.0f);
        decay_initial = row_arg_or(o.dec.runtime_top_p != nullptr ? o.dec.initial_top_p : nullptr, row, safe, 0.0f);
        decay_factor  = row_arg_or(o.dec.runtime_top_p != nullptr ? o.dec.decay : nullptr, row, safe, 0.0f);
        decay_min     = row_arg_or(o.dec.runtime_top_p != nullptr ? o.dec.top_p_min : nullptr, row, safe, 0.0f);
        decay_reset   = row_arg_or(o.dec.runtime_top_p != nullptr ? o.dec.reset_ids : nullptr, row, safe, 0);
        y             = s.y != nullptr ? (const T*)s.y + (size_t)row * s.y_pitch : (const T*)s.logits + (size_t)row * s.Vp;
    }
    // One wave or more: the draw, the maximum, the denominator: the reference's second butterfly.
    __device__ __forceinline__ void derive(const ToppStep& s)
    {
        next_draw     = 0;
        const float u = s.uniforms != nullptr ? draw.injected : row_draw_generate(draw, &next_draw);
        rand_num      = u * p;
        if (fin) {
            // a finished row: its end id alone has e = 1, or, when that lies outside the vocabulary, every column has
            const bool inside = end_id >= 0 && end_id < s.n;
            mx                = inside ? S::max_t() : -S::max_t();
            denom             = (inside ? 1.0f : (float)s.Vp) + 1e-6f;
        }
        else {
            mx      = rm.template get<DT>(s);
            float v = group;
#pragma unroll
            for (int m = 16; m > 0; m >>= 1) {
                v += __shfl_xor(v, m, 32);
            }
            denom = v + 1e-6f;  // (both halves of the wave hold the same group sums)
        }
    }
    // The generator's state goes on, for every row that is not skipped. Every wave has read the state for its own
    // derive(): unless only this thread's draw counts, a barrier lies between that and this.
    __device__ __forceinline__ void keep_draw(const ToppStep& s, const ToppPickOut& o) const
    {
        if (s.uniforms == nullptr && threadIdx.x == 0) {
            o.rng[row].offset = next_draw;
        }
    }
    // A single thread, once: what the row leaves behind, the decay of its p included.
    __device__ __forceinline__ void finish(const ToppPickOut& o, ToppPicked r) const
    {
        o.ids[row] = r.id;
        if (r.sampled) {
            if (o.cum_log_probs != nullptr || o.output_log_probs != nullptr) {
                const float lp = det_logf(r.prob);
                if (o.cum_log_probs != nullptr) {
                    o.cum_log_probs[row] = cum + lp;
                }
                if (o.output_log_probs != nullptr) {
                    o.output_log_probs[row] = lp;
                }
            }
            if (o.sequence_length != nullptr && o.finished != nullptr) {
                o.sequence_length[row] = fin ? length : length + 1;
                o.finished[row]        = r.id == end_id;
            }
        }
        decay(o, r.id);
    }
    __device__ __forceinline__ void decay(const ToppPickOut& o, int id) const
    {
        if (o.dec.runtime_top_p != nullptr) {
            o.dec.runtime_top_p[row] = id == decay_reset ? decay_initial : __builtin_fmaxf(decay_p * decay_factor, decay_min);
        }
    }
    // Rows that need no look at their columns (every thread gets the same answer): a NaN somewhere, so that no
    // probability is comparable and the reference keeps id 0, or finished with an ordinary end id.
    __device__ __forceinline__ bool trivial(const ToppStep& s, ToppPicked& r) const
    {
        if (!fin && !(mx == mx)) {
            r = ToppPicked{0, 0.0f, false};
            return true;
        }
        if (fin && end_id >= 0 && end_id < s.n) {
            const float one = topp_prob_of<DT>(1.0f, RowDivisor(denom), denom);
            r               = ToppPicked{end_id, one, round_t<DT>(0.0f + one) >= p || rand_num <= one};
            return true;
        }
        return false;
    }
};

// What the exact fallback needs of a row (the whole row, ordered): a draw that is not crossed inside what the step has
// ordered, or a row without anything ordered.
template<int DT>
struct ToppWholeRow {
    const typename Storage<DT>::T* y;
    int                            n, Vp, end_id;
    float                          mx, denom, p, rand_num;
    bool                           fin;
    unsigned long long*            sorted;
};

template<int DT>
__device__ __attribute__((noinline)) ToppPicked topp_pick_whole_row(TopPScan& sc, unsigned long long* digits, ToppWholeRow<DT> r)
{
    typedef Storage<DT> S;
    const RowDivisor    div(r.denom);
    const ToppRowValues vals{S::max_t(), r.fin, r.end_id, r.n};
    auto                prob_at = [&](int v) -> float {
        const float x = vals.masked(v, v < r.n ? S::ld(r.y[v]) : 0.0f);
        return topp_prob_of<DT>(round_t<DT>(det_expf_nonpos(x - r.mx)), div, r.denom);
    };
    const unsigned long long* src  = sort_whole_row(sc, digits, prob_at, r.Vp, r.sorted, r.sorted + r.Vp);
    const int                 n    = sc.misc[2];
    const int                 id   = n > 0 ? (int)(uint32_t)src[0] : 0;
    const float               best = n > 0 ? key64_prob(src[0]) : prob_at(0);
    if (round_t<DT>(0.0f + best) >= r.p) {
        return ToppPicked{id, best, true};
    }
    int found = n > 0 ? scan_tiles<1>(sc, (n + TP_TILE - 1) / TP_TILE, r.rand_num,
                                      [&](int tile, int l, float* x) { tile_load(src, n, tile, l, x); }) :
                        -1;
    if (found < 0) {
        return ToppPicked{id, best, false};
    }
    found = min(found, r.Vp - 1);  // (the zeros that fill the last tile can hold the crossing)
    if (found < n) {
        return ToppPicked{(int)(uint32_t)src[found], key64_prob(src[found]), true};
    }
    if (threadIdx.x == 0) {
        sc.misc[3] = nth_zero_entry(prob_at, r.Vp, found - n);
    }
    __syncthreads();
    const int z = sc.misc[3];
    return ToppPicked{z, prob_at(z), true};
}

// The scan of at most as many tiles as the workgroup's first THREADS threads have 32-lane groups, every group with its
// tile in registers: load(tile, l, x) as for scan_tiles. `agg` holds one float per group, `*found` (set to INT_MAX in
// front of the call, a barrier in between) gets the position the reference would pick. Two barriers; every thread of the
// workgroup calls.
template<int THREADS, class LoadTile>
__device__ __forceinline__ int scan_few_tiles(float* agg, int* found, int nt, float rand_num, LoadTile&& load)
{
    const int t = threadIdx.x, group = t >> 5, l = t & 31;
    float     x[8], incl = 0.0f;
    const bool mine = t < THREADS && group < nt;
    if (mine) {
        load(group, l, x);
        incl = tile_scan(x, l);
        if (l == 31) {
            agg[group] = incl;
        }
    }
    __syncthreads();
    if (mine) {
        float prefix = 0.0f;
        for (int g = 0; g < group; ++g) {
            prefix = prefix + agg[g];
        }
        const float excl = __shfl_up(incl, 1, 32);
        float       a    = l == 0 ? prefix : prefix + excl;
        uint32_t    m8   = 0u;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            a = a + x[j];
            if (rand_num <= a) {
                m8 |= 1u << j;
            }
        }
        // the reference looks at words of 32 positions, four lanes here: the first that holds a crossing counts
        // from its end
        int c = __popc(m8);
        c += dpp_from<DPP_QUAD_XOR1>(c);
        c += dpp_from<DPP_QUAD_XOR2>(c);
        const unsigned long long b     = __ballot(m8 != 0u);
        const uint32_t           lanes = (uint32_t)(b >> (lane_id() & 32));
        if (lanes != 0u) {
            const int first = __builtin_ctz(lanes) >> 2;
            if (l == first * 4) {
                atomicMin(found, group * TP_TILE + first * 32 + (32 - c));
            }
        }
    }
    __syncthreads();
    return *found == 0x7FFFFFFF ? -1 : *found;
}

// ---- pick, fp32
// The prefix is ordered by (e, id). Entries whose e differ can share a probability; the scan's sums do not depend on
// the order of equal values, only the emitted id does: the reference emits, of the entries that share the probability
// at position `found`, the one with as many smaller ids as there are entries of the run in front of `found`. Every
// thread calls and gets the entry.
template<class Prob>
__device__ __forceinline__ unsigned long long topp_settle_run(TopPScan& s, const unsigned long long* A, int n, int found,
                                                              int vocab, Prob&& prob)
{
    const int t = threadIdx.x;
    if (t == 0) {
        // both ends of the run are looked for outwards from `found` in doubling steps, then by bisection
        const float here = prob(A[found]);
        auto        same = [&](int i) { return prob(A[i]) == here; };
        int         hi = found, lo = 0;  // first position of the run: in [lo, hi], A[hi] belongs to it
        for (int step = 1;; step <<= 1) {
            const int probe = hi - step;
            if (probe < 0) {
                lo = 0;
                break;
            }
            if (!same(probe)) {
                lo = probe + 1;
                break;
            }
            hi = probe;
        }
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (same(mid)) {
                hi = mid;
            }
            else {
                lo = mid + 1;
            }
        }
        const int a = lo;
        lo          = found;
        hi          = n - 1;  // last position of the run: in [lo, hi], A[lo] belongs to it
        for (int step = 1;; step <<= 1) {
            const int probe = lo + step;
            if (probe > n - 1) {
                hi = n - 1;
                break;
            }
            if (!same(probe)) {
                hi = probe - 1;
                break;
            }
            lo = probe;
        }
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (same(mid)) {
                lo = mid;
            }
            else {
                hi = mid - 1;
            }
        }
        s.misc[4] = a;
        s.misc[5] = lo;
        s.misc[6] = (uint32_t)(A[a] >> 32) != (uint32_t)(A[lo] >> 32) ? 1 : 0;
    }
    __syncthreads();
    if (s.misc[6] == 0) {
        return A[found];  // one numerator: already in order of ids
    }
    // the id with exactly (found - a) smaller ids in the run: bisection over the ids, counting with all threads
    const int a = s.misc[4], b = s.misc[5];
    const int want = found - a;
    int       lo = 0, hi = vocab;
    while (hi - lo > 1) {
        const int mid = lo + (hi - lo) / 2;
        if (t == 0) {
            s.misc[7] = 0;
        }
        __syncthreads();
        int mine = 0;
        for (int i = a + t; i <= b; i += TP_THREADS) {
            mine += (int)(uint32_t)A[i] < mid ? 1 : 0;
        }
        mine = wave_sum_i(mine);
        if (lane_id() == 0 && mine != 0) {
            atomicAdd(&s.misc[7], mine);
        }
        __syncthreads();
        const int below_mid = s.misc[7];
        __syncthreads();
        if (below_mid > want) {
            hi = mid;
        }
        else {
            lo = mid;
        }
    }
    return (A[found] & 0xFFFFFFFF00000000ull) | (uint32_t)lo;
}

constexpr int TPF_SMALL = 512;  // prefixes up to this many entries are ordered by counting ranks in LDS

__global__ void __launch_bounds__(TP_THREADS) topp_pick_f32_kernel(ToppStep s, ToppPickOut o)
{
    __shared__ TopPScan       sc;
    __shared__ ToppSortShared ss;
    __shared__ int            sh_found;
    static_assert(sizeof(ss.buf) >= TP_DIGITS * sizeof(unsigned long long), "digit counters");
    static_assert(sizeof(ss.buf) >= 2 * TPF_SMALL * sizeof(unsigned long long), "ranks");
    const int           row = blockIdx.x;
    const int           t   = threadIdx.x;
    unsigned long long* A   = s.sorted + (size_t)row * 2 * s.Vp;
    ToppPickRow<DT_F32> r(s, o, row, s.parts);
    const ToppRowMeta   m    = s.meta[row];  // (a row without a record: what an earlier launch left, not looked at)
    unsigned long long  mine = A[min(t, s.Vp - 1)];
    if (t == 0) {
        sh_found = 0x7FFFFFFF;
    }
    if (r.skip) {
        if (t == 0) {
            r.decay(o, o.dec.runtime_top_p != nullptr ? o.ids[row] : 0);
        }
        return;
    }
    r.derive(s);
    ToppPicked res;
    if (r.trivial(s, res)) {
        r.keep_draw(s, o);
        if (t == 0) {
            r.finish(o, res);
        }
        return;
    }
    __syncthreads();
    r.keep_draw(s, o);
    const RowDivisor div(r.denom);
    auto prob = [&](unsigned long long entry) { return topp_prob_of<DT_F32>(key64_prob(entry), div, r.denom); };
    if (!r.fin && !o.force_deep && m.n > 0) {
        const int                 n   = m.n;
        const bool                all = n == m.n_pos;
        const unsigned long long* src = A;
        if (n <= TPF_SMALL) {
            // every entry's rank is the number of smaller ones (entries are distinct: ids are)
            unsigned long long* in  = ss.buf;
            unsigned long long* out = ss.buf + TPF_SMALL;
            if (t < n) {
                in[t] = mine;
            }
            __syncthreads();
            // (a whole number of waves per copy of the list: 1024 / copies threads look at n / copies entries each)
            const int per    = n <= 64 ? 64 : n <= 128 ? 128 : n <= 256 ? 256 : 512;
            const int copies = TP_THREADS / per;
            const int who = t & (per - 1), copy = t / per;
            uint32_t* rank = ss.hist;
            if (t < TPF_SMALL) {
                rank[t] = 0u;
            }
            __syncthreads();
            if (who < n) {
                const unsigned long long key  = in[who];
                const int                step = (n + copies - 1) / copies;
                const int                j0 = copy * step, j1 = min(n, j0 + step);
                uint32_t                 below = 0u;
                for (int j = j0; j < j1; ++j) {
                    below += in[j] < key ? 1u : 0u;
                }
                if (below != 0u) {
                    atomicAdd(&rank[who], below);
                }
            }
            __syncthreads();
            if (t < n) {
                out[rank[t]] = mine;
            }
            __syncthreads();
            src = out;
        }
        else if (n <= TPS_CAP) {
            topp_sort_one(ss, A, A, n);
            __threadfence_block();
            __syncthreads();
        }
        const unsigned long long best   = topp_settle_run(sc, src, n, 0, s.Vp, prob);
        const float              p_best = prob(best);
        // whether all entries that share the probability of the one at position i are in the prefix
        auto whole_run = [&](int i) { return all || key64_prob(src[i]) >= m.safe; };
        if (p_best > 0.0f && whole_run(0)) {
            if (0.0f + p_best >= r.p) {
                // arg-max shortcut of the reference (:842-849)
                if (t == 0) {
                    r.finish(o, ToppPicked{(int)(uint32_t)best, p_best, true});
                }
                return;
            }
            auto load = [&](int tile, int l, float* x) {
                const int i0 = tile * TP_TILE + l * 8;
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    x[k] = i0 + k < n ? prob(src[i0 + k]) : 0.0f;
                }
            };
            const int nt = (n + TP_TILE - 1) / TP_TILE;
            __syncthreads();
            const int found = nt <= TP_THREADS / 32 ? scan_few_tiles<TP_THREADS>(sc.agg, &sh_found, nt, r.rand_num, load) :
                                                      scan_tiles<2>(sc, nt, r.rand_num, load);
            if (found >= 0 && found < n && whole_run(found)) {
                __syncthreads();
                const unsigned long long e = topp_settle_run(sc, src, n, found, s.Vp, prob);
                if (t == 0) {
                    r.finish(o, ToppPicked{(int)(uint32_t)e, prob(e), true});
                }
                return;
            }
            if (found < 0 && all) {
                if (t == 0) {
                    r.finish(o, ToppPicked{(int)(uint32_t)best, p_best, false});  // never crossed: the arg-max stays
                }
                return;
            }
        }
        __syncthreads();
    }
    const ToppWholeRow<DT_F32> w{r.y, s.n, s.Vp, r.end_id, r.mx, r.denom, r.p, r.rand_num, r.fin, A};
    res = topp_pick_whole_row<DT_F32>(sc, ss.buf, w);
    if (t == 0) {
        r.finish(o, res);
    }
}

// ---- pick, 16-bit types
// 16-bit order-preserving image of a value's bits
__device__ __forceinline__ uint32_t topp_key16(uint32_t bits)
{
    return (bits & 0x8000u) ? (~bits & 0xFFFFu) : (bits | 0x8000u);
}

template<int DT>
union ToppRunsShared {
    struct {
        uint32_t start[ToppCode<DT>::USED + 1];  // entries in front of a run, in descending order of e
        uint16_t code[ToppCode<DT>::USED + 1];   // a run's value of e
        uint16_t prob[ToppCode<DT>::USED + 1];   // and its probability, both as stored values of the type
    };
    unsigned long long digits[TP_DIGITS];                          // the fallback's radix sort
    uint8_t            masks[TP_DIGITS * sizeof(unsigned long long)];  // the look-up's matches: a byte per eight columns
};

template<int DT>
__global__ void __launch_bounds__(TP_THREADS) topp_pick_runs_kernel(ToppStep s, ToppPickOut o)
{
    typedef Storage<DT>           S;
    typedef typename S::T         T;
    typedef ToppCode<DT>          Code;
    constexpr int                 CPT  = 16;                    // counters per thread
    constexpr int                 TEAM = Code::COUNTERS / CPT;  // threads that look at counters
    constexpr int                 TW   = TEAM / WAVE;
    constexpr int                 NW   = TP_THREADS / WAVE;
    constexpr int                 FEW  = 256;                   // threads of the short scan: eight tiles
    __shared__ TopPScan           sc;
    __shared__ ToppRunsShared<DT> rs;
    // the values of the row's first positions one by one: what the scan reads there
    constexpr int                 FLAT = DT == DT_F16 ? 8192 : 16384;
    __shared__ __align__(16) uint16_t flat[FLAT];
    __shared__ uint32_t           wcnt[TW], wrun[TW], wpick[NW];
    __shared__ float              wmass[TW];
    __shared__ uint32_t           sh_enough, key_lo, key_hi;
    __shared__ int                sh_found, code_lo, code_hi, sh_nth, sh_mixed;
    const int       row = blockIdx.x;
    const int       t   = threadIdx.x;
    ToppPickRow<DT> r(s, o, row, s.splits);
    // counters of this thread, descending: position d counts entries of code COUNTERS - 1 - d
    uint32_t c[CPT];
    {
        const uint4* from = reinterpret_cast<const uint4*>(s.counts + (size_t)row * Code::COUNTERS + (Code::COUNTERS - (min(t, TEAM - 1) + 1) * CPT));
#pragma unroll
        for (int i = 0; i < CPT / 4; ++i) {
            const uint4 w      = from[i];
            c[CPT - 1 - 4 * i] = w.x;
            c[CPT - 2 - 4 * i] = w.y;
            c[CPT - 3 - 4 * i] = w.z;
            c[CPT - 4 - 4 * i] = w.w;
        }
    }
    // the maxima of this wave's blocks of columns: a wave takes a contiguous run of them
    const int    bpw  = (s.blocks + NW - 1) / NW;
    const int    b0   = min(s.blocks, wave_id() * bpw), b1 = min(s.blocks, b0 + bpw);
    const float* bmax = s.block_max + (size_t)row * s.blocks;
    const float  bm   = bmax[min(b0 + lane_id(), s.blocks - 1)];
    if (t == 0) {
        sh_enough = 0xFFFFFFFFu;
        sh_found  = 0x7FFFFFFF;
    }
    if (r.skip) {
        if (t == 0) {
            r.decay(o, o.dec.runtime_top_p != nullptr ? o.ids[row] : 0);
        }
        return;
    }
    r.derive(s);
    ToppPicked res;
    if (r.trivial(s, res)) {
        r.keep_draw(s, o);
        if (t == 0) {
            r.finish(o, res);
        }
        return;
    }
    const ToppWholeRow<DT> whole{r.y, s.n, s.Vp, r.end_id, r.mx, r.denom, r.p, r.rand_num, r.fin, s.sorted + (size_t)row * 2 * s.Vp};
    if (r.fin || o.force_deep) {
        __syncthreads();
        r.keep_draw(s, o);
        res = topp_pick_whole_row<DT>(sc, rs.digits, whole);
        if (t == 0) {
            r.finish(o, res);
        }
        return;
    }
    const RowDivisor div(r.denom);
    const bool       quick = __builtin_amdgcn_readfirstlane((int)div.ok) != 0;
    auto             prob_of_code = [&](int code) -> float {
        const float e = S::ld((T)(code + Code::BASE));  // (at least 2^-31)
        return round_t<DT>(quick ? div.divide_normal(e) : e / r.denom);
    };
    // ---- the runs: counts, probabilities and places of the values that occur and whose probability is not zero
    float    pv[CPT];
    uint32_t lc = 0u, lr = 0u;
    float    lm = 0.0f;
    if (t < TEAM) {
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            pv[i] = 0.0f;
            if (c[i] != 0u) {
                pv[i] = prob_of_code(Code::COUNTERS - 1 - (t * CPT + i));
                if (pv[i] > 0.0f) {
                    lc += c[i];
                    lr += 1u;
                    lm += (float)c[i] * pv[i];
                }
            }
        }
    }
    uint32_t ic = lc, ir = lr;
    float    im = lm;
    if (t < TEAM) {
#pragma unroll
        for (int k = 1; k < WAVE; k <<= 1) {
            const uint32_t uc = __shfl_up(ic, k, WAVE), ur = __shfl_up(ir, k, WAVE);
            const float    um = __shfl_up(im, k, WAVE);
            if (lane_id() >= k) {
                ic += uc;
                ir += ur;
                im += um;
            }
        }
        if (lane_id() == WAVE - 1) {
            wcnt[wave_id()]  = ic;
            wrun[wave_id()]  = ir;
            wmass[wave_id()] = im;
        }
    }
    __syncthreads();
    r.keep_draw(s, o);
    uint32_t n = 0u, nruns = 0u;
    uint32_t at = ic - lc, run = ir - lr;
    float    mass = im - lm;
#pragma unroll
    for (int w = 0; w < TW; ++w) {
        const uint32_t wc = wcnt[w], wr = wrun[w];
        at += w < wave_id() ? wc : 0u;
        run += w < wave_id() ? wr : 0u;
        mass += w < wave_id() ? wmass[w] : 0.0f;
        n += wc;
        nruns += wr;
    }
    const uint32_t at0 = at, run0 = run;
    const float    mass0 = mass;
    // the place behind the run with which the mass certainly covers the draw: the scan need not look further
    const float want = r.rand_num * (1.0f + 1.0f / 256.0f) + 1e-5f;
    if (t < TEAM) {
        uint32_t enough = 0xFFFFFFFFu;
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            if (pv[i] > 0.0f) {
                rs.start[run] = at;
                rs.code[run]  = (uint16_t)(Code::COUNTERS - 1 - (t * CPT + i));
                rs.prob[run]  = S::st(pv[i]);
                at += c[i];
                mass += (float)c[i] * pv[i];
                run++;
                if (mass >= want && enough == 0xFFFFFFFFu) {
                    enough = at;
                }
            }
        }
        if (enough != 0xFFFFFFFFu && mass0 < want) {  // (one thread as a rule, a few next to it by rounding)
            atomicMin(&sh_enough, enough);
        }
        if (t == 0) {
            rs.start[nruns] = n;
        }
    }
    __syncthreads();
    const int enough = (int)min(n, sh_enough);
    // Whether the runs hold every positive probability: binary16's counters resolve all values of e, bfloat16's leave out
    // what lies below 2^-31.
    const bool complete = DT == DT_F16 || n == (uint32_t)s.Vp;
    int        found    = -1;
    bool       sampled  = true;
    float      prob     = 0.0f;
    bool       fallback = n == 0u;
    if (!fallback) {
        const float best = S::ld(rs.prob[0]);
        if (round_t<DT>(0.0f + best) >= r.p) {
            found = 0;  // arg-max shortcut of the reference (:842-849)
        }
        else {
            // the run of position i: the last one that starts at or before it
            auto run_at = [&](int i) -> int {
                int lo = 0, hi = (int)nruns;
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if ((int)rs.start[mid] <= i) {
                        lo = mid;
                    }
                    else {
                        hi = mid;
                    }
                }
                return lo;
            };
            // a lane's eight values from position i0 on, which lies in run `lo`; lo goes along
            auto values_from = [&](int i0, int& lo, float* x) {
                float v    = S::ld(rs.prob[lo]);
                int   next = (int)rs.start[lo + 1];
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    x[k] = 0.0f;
                    if (i0 + k < (int)n) {
                        if (i0 + k >= next) {
                            do {
                                ++lo;
                                next = (int)rs.start[lo + 1];
                            } while (i0 + k >= next);
                            v = S::ld(rs.prob[lo]);
                        }
                        x[k] = v;
                    }
                }
            };
            // Near the head of a row runs are short, and a tile taken out of them is a chain of look-ups (1.6 us per 32 tiles).
            // Sixteen threads write a run's value to its positions, and a lane's eight values are one read (128 x 152064
            // bf16: the scan for a draw behind 15000 entries 8.8 -> 5.2 us, behind 77000, with what follows, 20 -> 10). A row of
            // few distinct values has long runs at its head: sixteen bytes per store beyond SHORT positions. us a step of 64 x
            // 128256, two bytes per store throughout / so: bf16 of four values 72.5 / 46.1 (binary16 61.4 / 48.4), 16000 equal ones
            // at the head 63.0 / 37.3 (57.6 / 44.6), Zipf 37.0 / 36.0 (44.7 / 44.8); 8 x 32000 bf16 of four values 45.3 / 28.4. The
            // next run is requested ahead of the stores: without that binary16 lost 0.4 on rows of short runs.
            constexpr int SHORT  = 128;
            const int     flat_n = min(FLAT, (enough + TP_TILE - 1) / TP_TILE * TP_TILE);
            {
                const int lane = t & 15, last = (int)nruns;
                int       k = t >> 4, begin = (int)rs.start[min(k, last)], end = (int)rs.start[min(k + 1, last)];
                uint32_t  v = rs.prob[min(k, last)];
                while (k < last && begin < flat_n) {
                    k += TP_THREADS / 16;
                    const int      begin_next = (int)rs.start[min(k, last)], end_next = (int)rs.start[min(k + 1, last)];
                    const uint32_t v_next     = rs.prob[min(k, last)];
                    end                       = min(end, flat_n);
                    if (end - begin <= SHORT) {
#pragma unroll 1
                        for (int i = begin + lane; i < end; i += 16) {
                            flat[i] = (uint16_t)v;
                        }
                    }
                    else {
                        const int      lo = (begin + 7) & ~7, hi = end & ~7;
                        const uint32_t vv = v * 0x00010001u;
                        if (begin + lane < lo) {
                            flat[begin + lane] = (uint16_t)v;
                        }
                        if (hi + lane < end) {
                            flat[hi + lane] = (uint16_t)v;
                        }
#pragma unroll 4
                        for (int i = lo + lane * 8; i < hi; i += 128) {
                            *reinterpret_cast<uint4*>(flat + i) = make_uint4(vv, vv, vv, vv);
                        }
                    }
                    begin = begin_next;
                    end   = end_next;
                    v     = v_next;
                }
            }
            if ((int)n + t < flat_n) {  // (fewer than a tile's)
                flat[n + t] = 0;
            }
            __syncthreads();
            auto flat_load = [&](int i0, float* x) {
                const uint4    q    = *reinterpret_cast<const uint4*>(flat + i0);
                const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    x[2 * k]     = S::ld((T)w[k]);
                    x[2 * k + 1] = S::ld((T)(w[k] >> 16));
                }
            };
            auto load = [&](int tile, int l, float* x) {
                const int i0 = tile * TP_TILE + l * 8;
                if (i0 < flat_n) {
                    flat_load(i0, x);
                }
                else {
                    int lo = run_at(min(i0, (int)n - 1));
                    values_from(i0, lo, x);
                }
            };
            // Behind them: tiles of a few runs first, a thread each. All values of a tile are multiples of the last place of
            // its smallest one; where the largest is so near that 256 of it stay below 2^24 such places, no addition inside
            // the tile rounds, and its total is the sum of counts times values in any order. Other tiles go to 32-lane groups.
            auto totals = [&](int base, int count) {
                constexpr int RUNS = 8, SPREAD = 15 - (DT == DT_F16 ? 10 : 7);  // (of exponents)
                const int l  = t & 31;
                const int nf = max(0, min(count, flat_n / TP_TILE - base));
                if (t == 0) {
                    sh_mixed = 0;
                }
                for (int g = t >> 5; g < nf; g += TP_THREADS / 32) {
                    float x[8];
                    flat_load((base + g) * TP_TILE + l * 8, x);
                    const float total = tile_scan(x, l);
                    if (l == 31) {
                        sc.agg[g] = total;
                    }
                }
                if (nf == count) {
                    return;
                }
                __syncthreads();
                if (t >= nf && t < count) {
                    const int i0    = (base + t) * TP_TILE;
                    const int end   = min(i0 + TP_TILE, (int)n);
                    const int first = run_at(i0);
                    float     v     = S::ld(rs.prob[first]), sum = 0.0f;
                    const int top   = __float_as_int(v) >> 23;
                    int       from = i0, q = first;
                    bool      exact = true;
#pragma unroll 1
                    for (int k = 0; k < RUNS && from < end; ++k) {
                        const int to = min(end, (int)rs.start[++q]);
                        exact        = exact && top - (__float_as_int(v) >> 23) <= SPREAD;
                        sum          = sum + (float)(to - from) * v;
                        from         = to;
                        v            = S::ld(rs.prob[min(q, (int)nruns - 1)]);
                    }
                    if (exact && from == end) {
                        sc.agg[t] = sum;
                    }
                    else {
                        sc.carry[atomicAdd(&sh_mixed, 1)] = __int_as_float((t << 16) | first);
                    }
                }
                __syncthreads();
                const int mixed = sh_mixed;
                for (int m = t >> 5; m < mixed; m += TP_THREADS / 32) {
                    const int what = __float_as_int(sc.carry[m]);
                    const int tile = what >> 16, i = (base + tile) * TP_TILE + l * 8;
                    // (a lane's first entry: of the runs that begin inside the tile)
                    int lo = what & 0xFFFF, hi = min((int)nruns, lo + TP_TILE);
                    while (hi - lo > 1) {
                        const int mid = (lo + hi) >> 1;
                        if ((int)rs.start[mid] <= i) {
                            lo = mid;
                        }
                        else {
                            hi = mid;
                        }
                    }
                    float x[8];
                    values_from(i, lo, x);
                    const float total = tile_scan(x, l);
                    if (l == 31) {
                        sc.agg[tile] = total;
                    }
                }
            };
            const int nt_all = ((int)n + TP_TILE - 1) / TP_TILE;
            const int nt     = (enough + TP_TILE - 1) / TP_TILE;
            bool      over   = false;  // the scan has seen every tile
            if (nt <= FEW / 32) {
                found = scan_few_tiles<FEW>(sc.agg, &sh_found, nt, r.rand_num, load);
                over  = nt == nt_all;
            }
            else {
                found = scan_tiles(sc, nt, r.rand_num, load, totals);
                over  = nt == nt_all;
            }
            if (found < 0 && !over) {
                __syncthreads();
                found = scan_tiles(sc, nt_all, r.rand_num, load, totals);
            }
            __syncthreads();
            if (found < 0 || found >= (int)n) {
                if (complete && found < 0) {
                    found   = 0;  // never crossed: the arg-max stays (:954)
                    sampled = false;
                }
                else {
                    fallback = true;
                }
            }
        }
    }
    if (fallback) {
        // (a row without a value that the counters resolve, or a draw behind all of them)
        __syncthreads();
        res = topp_pick_whole_row<DT>(sc, rs.digits, whole);
        if (t == 0) {
            r.finish(o, res);
        }
        return;
    }
    // ---- the run of position `found`, together with neighbours whose numerators round to the same quotient
    if (t < TEAM && lc != 0u && found >= (int)at0 && found < (int)(at0 + lc)) {
        int q = (int)run0;
        while (found >= (int)rs.start[q + 1]) {
            ++q;
        }
        const uint16_t here = rs.prob[q];
        int            a = q, b = q;
        while (a > 0 && rs.prob[a - 1] == here) {
            --a;
        }
        while (b + 1 < (int)nruns && rs.prob[b + 1] == here) {
            ++b;
        }
        code_hi      = (int)rs.code[a];
        code_lo      = (int)rs.code[b];
        sh_nth       = found - (int)rs.start[a];
        sc.fmisc[1]  = S::ld(here);
    }
    __syncthreads();
    // ---- the values of y with these numerators: a range of the order-preserving image, found by two waves in three
    // rounds of 64 probes (e does not fall as y rises)
    if (wave_id() < 2) {
        const uint32_t key_mx  = topp_key16((uint32_t)S::st(r.mx));
        const uint32_t key_inf = topp_key16((uint32_t)S::st(-__builtin_inff()));
        auto           code_of = [&](uint32_t key) -> int {
            if (key >= key_mx) {
                return Code::USED - 1;
            }
            if (key < key_inf) {
                return 0;
            }
            const T bits = (T)((key & 0x8000u) ? (key & 0x7FFFu) : (~key & 0xFFFFu));
            return max((int)S::st(topp_exp(S::ld(bits) - r.mx)) - Code::BASE, 0);
        };
        const bool upper = wave_id() == 1;  // wave 0: the first key with code >= code_lo; wave 1: with code > code_hi
        const int  level = upper ? code_hi + 1 : code_lo;
        uint32_t   base  = 0u;  // keys below base have smaller codes
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int      width  = k == 0 ? 1024 : k == 1 ? 16 : 1;
            const int      probes = k == 2 ? 16 : 64;
            const uint32_t key    = base + (uint32_t)(lane_id() + 1) * (uint32_t)width - 1u;
            const bool     less   = lane_id() < probes && key < 65536u && code_of(key) < level;
            base += (uint32_t)__popcll(__ballot(less)) * (uint32_t)width;
        }
        if (lane_id() == 0) {
            if (upper) {
                key_hi = base;  // one past the last
            }
            else {
                key_lo = base;
            }
        }
    }
    __syncthreads();
    prob = sc.fmisc[1];
    // ---- the column: the sh_nth one in order of ids whose value lies in that range. Blocks whose maximum lies below it
    // cannot hold one: a draw near the head of the distribution reads a few blocks only.
    // (no value lies above the maximum; of zeros the positive one counts as the larger here, whichever the maximum is)
    const uint32_t klo = key_lo, khi = min(key_hi, topp_key16((uint32_t)S::st(r.mx + 0.0f)) + 1u);
    const int      nth = sh_nth;
    auto match = [&](uint32_t bits) -> bool {
        const uint32_t k = topp_key16(bits);
        return k >= klo && k < khi;
    };
    // Matches among a lane's eight columns of a block: bit k is column 2 k, bit 4 + k column 2 k + 1. Two columns at a
    // time: with a range of one sign the distance of the bits from its first value, otherwise of their images (with a
    // column at a time a deep draw, whose blocks are nearly all of the row, spent 10 us here at 128256 columns).
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    typedef short          i16x2 __attribute__((ext_vector_type(2)));
    const bool           positive = klo >= 0x8000u, one_sign = positive || khi <= 0x8000u;
    const unsigned short origin   = (unsigned short)(!one_sign ? klo : positive ? klo - 0x8000u : 0x10000u - khi);
    const unsigned short length   = (unsigned short)min(khi - klo, 0xFFFFu);  // (all 65536: a row of one value ends above)
    const u16x2          from = {origin, origin}, size = {length, length};
    const int whole_blocks = s.n / TSP_BLOCK;
    auto vector_of = [&](int blk) -> uint4 {
        return topp_load8(r.y + __builtin_amdgcn_readfirstlane(blk) * TSP_BLOCK + lane_id() * 8);
    };
    auto mask_whole = [&](const uint4& raw, auto same_sign) -> uint32_t {
        const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
        uint32_t       m    = 0u;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            u16x2 x = __builtin_bit_cast(u16x2, w[k]);
            if constexpr (!decltype(same_sign)::value) {
                const i16x2 sign = __builtin_bit_cast(i16x2, w[k]) >> 15;
                x = __builtin_bit_cast(u16x2, w[k] ^ (__builtin_bit_cast(uint32_t, sign) | 0x80008000u));
            }
            // (left to itself the compiler makes two comparisons and two selects of this minimum)
            uint32_t in = __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(size, (u16x2)(x - from)));
            asm("v_pk_min_u16 %0, %0, %1" : "+v"(in) : "v"(0x00010001u));
            m |= in << k;
        }
        return (m | (m >> 12)) & 0xFFu;
    };
    auto mask_part = [&]() -> uint32_t {  // of the block that runs over the end
        const int v0 = whole_blocks * TSP_BLOCK + lane_id() * 8;
        T         x[8];
        uint32_t  m = 0u;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            x[k] = r.y[min(v0 + k, s.n - 1)];  // (all of them requested before the first is looked at)
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (v0 + k < s.n && match((uint32_t)x[k])) {
                m |= 1u << ((k >> 1) + 4 * (k & 1));
            }
        }
        return m;
    };
    auto mask_of = [&](int blk) -> uint32_t {
        if (blk == whole_blocks) {
            return mask_part();
        }
        const uint4 raw = vector_of(blk);
        return one_sign ? mask_whole(raw, std::true_type()) : mask_whole(raw, std::false_type());
    };
    const bool kept = s.blocks <= (int)sizeof(rs.masks) / WAVE;  // the matches of every block fit LDS
    int        mine = 0;
    for (int g = b0; g < b1; g += WAVE) {  // (one turn unless the vocabulary has half a million columns)
        const float gm   = g == b0 ? bm : bmax[min(g + lane_id(), s.blocks - 1)];
        const bool  may  = g + lane_id() < b1 && topp_key16((uint32_t)S::st(gm)) >= klo;
        if (kept && g + lane_id() < b1 && !may) {
            uint4* z = reinterpret_cast<uint4*>(rs.masks + (g + lane_id()) * WAVE);
            z[0] = z[1] = z[2] = z[3] = make_uint4(0u, 0u, 0u, 0u);
        }
        unsigned long long todo = __ballot(may);
        auto count = [&](int blk, uint32_t m) {
            mine += __popc(m);
            if (kept) {
                rs.masks[blk * WAVE + lane_id()] = (uint8_t)m;
            }
        };
        if (whole_blocks >= g && whole_blocks < g + WAVE && ((todo >> (whole_blocks - g)) & 1ull) != 0ull) {
            todo &= ~(1ull << (whole_blocks - g));
            count(whole_blocks, mask_part());
        }
        // U blocks in flight, the next one requested as soon as one has been looked at (requested where they were looked at,
        // which kept one in flight, and with two comparisons per pair of columns: 10.1 us for the 297 blocks of 152064
        // columns; so: 6.1, the 43 KB/us that a compute unit gets from the last-level cache)
        auto look = [&](auto same_sign) {
            constexpr int U = 4;
            int           blk[U];
            uint4         raw[U];
            auto          next = [&]() -> int {
                const int b = todo != 0ull ? g + (int)__builtin_ctzll(todo) : -1;
                todo &= todo - 1ull;
                return __builtin_amdgcn_readfirstlane(b);
            };
#pragma unroll
            for (int u = 0; u < U; ++u) {
                blk[u] = next();
                raw[u] = vector_of(max(blk[u], 0));
            }
#pragma unroll 1
            while (blk[0] >= 0) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int      now = blk[u];
                    const uint32_t m   = mask_whole(raw[u], same_sign);
                    blk[u]             = next();
                    raw[u]             = vector_of(max(blk[u], 0));
                    if (now >= 0) {
                        count(now, m);
                    }
                }
            }
        };
        if (one_sign) {
            look(std::true_type());
        }
        else {
            look(std::false_type());
        }
    }
    mine = wave_sum_i(mine);
    if (lane_id() == 0) {
        wpick[wave_id()] = (uint32_t)mine;
    }
    __syncthreads();
    int before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const int x = (int)wpick[w];
        before += w < wave_id() ? x : 0;
        total += x;
    }
    if (nth >= before && nth < before + mine) {  // (one wave)
        int left = nth - before;
        for (int g = b0; g < b1; g += WAVE) {
            // lane i counts the matches of block g + i
            const int blk = g + lane_id();
            int       own = 0;
            if (kept && blk < b1) {
                const uint4* q = reinterpret_cast<const uint4*>(rs.masks + blk * WAVE);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint4 w = q[k];
                    own += __popc(w.x) + __popc(w.y) + __popc(w.z) + __popc(w.w);
                }
            }
            else if (!kept) {
                for (int i = g; i < min(b1, g + WAVE); ++i) {
                    const int x = wave_sum_i(__popc(mask_of(i)));
                    own         = lane_id() == i - g ? x : own;
                }
            }
            int inc = own;
#pragma unroll
            for (int k = 1; k < WAVE; k <<= 1) {
                const int up = __shfl_up(inc, k, WAVE);
                if (lane_id() >= k) {
                    inc += up;
                }
            }
            const unsigned long long hit = __ballot(inc > left);
            if (hit == 0ull) {
                left -= __shfl(inc, WAVE - 1, WAVE);
                continue;
            }
            const int which = __builtin_ctzll(hit);
            left -= __shfl(inc - own, which, WAVE);
            const uint32_t m = kept ? (uint32_t)rs.masks[(g + which) * WAVE + lane_id()] : mask_of(g + which);
            int            in = __popc(m);
            const int      c1 = in;
#pragma unroll
            for (int k = 1; k < WAVE; k <<= 1) {
                const int up = __shfl_up(in, k, WAVE);
                if (lane_id() >= k) {
                    in += up;
                }
            }
            int k = left - (in - c1);
            if (k >= 0 && k < c1) {
                uint32_t rest = 0u;  // in the order of the columns
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    rest |= (((m >> q) & 1u) | (((m >> (4 + q)) & 1u) << 1)) << (2 * q);
                }
                while (k-- > 0) {
                    rest &= rest - 1u;
                }
                r.finish(o, ToppPicked{(g + which) * TSP_BLOCK + lane_id() * 8 + (int)__builtin_ctz(rest), prob, sampled});
            }
            break;
        }
    }
    else if (nth >= total && t == 0) {
        // the pad columns follow the vocabulary; they match when their value does
        r.finish(o, ToppPicked{min(s.n + (nth - total), s.Vp - 1), prob, sampled});
    }
}

// ---- host -------------------------------------------------------------------------------------------------------------
static inline size_t up256(size_t x)
{
    return (x + 255) & ~(size_t)255;
}

struct ToppSamplePlan {
    int    parts, splits, chunk, blocks, y_pitch, sorters;
    size_t off_y, off_counts, off_pmax, off_blocks, off_ref, off_gsum, off_segs, off_queue, off_meta, bytes;
};

constexpr int TSP_MANY_ROWS   = 72;                     // fp32: from here on four workgroups per row, sixteen below
constexpr int TSP_WINDOW_BITS = (TSP_WINDOW - 4) * 32;  // most columns that the bitmap of the history covers
// the columns of a workgroup of the fp32 stage
static int topp_part_columns(int vocab, int parts)
{
    return (vocab + TSP_CHAINS - 1) / TSP_CHAINS * (TSP_CHAINS / parts);
}

static ToppSamplePlan topp_sample_plan(int dtype, int rows, int vocab, size_t vocab_padded, bool keeps_y)
{
    ToppSamplePlan p;
    rows = rows > 0 ? rows : 1;
    // The sum. fp32: 256-thread workgroups, one chain per thread and four workgroups per row from 72 rows on, sixteen with
    // four lanes to a chain below. Sixteen share a short batch out better, but each of them reads the histograms of all
    // sixteen (128 KB). us a step, zipf rows, p = 0.9, sixteen / four:
    //   rows      7         47        65        79        95        129       255
    //   8192      30 / 30   37 / 34   42 / 36   44 / 36   45 / 36   53 / 37   73 / 39
    //   32000     33 / 36   49 / 50   57 / 52   60 / 53   63 / 54   72 / 57  101 / 68
    //   128256    43 / 55   68 / 76   80 / 82   86 / 84   93 / 86  103 / 91  158 / 117
    // 16-bit types: 1024-thread workgroups, one per row from 192 rows on, four below; one / four:
    //   rows                64        96        128       160       224
    //   binary16  32000     38 / 37   38 / 43   39 / 45   40 / 51   40 / 59
    //             128256    75 / 61   79 / 76   81 / 79   85 / 93   90 / 110
    //   bfloat16  32000     33 / 31   33 / 32   33 / 33   34 / 36   35 / 38
    //             128256    63 / 49   66 / 55   67 / 56   70 / 65   74 / 74
    // (binary16, whose counters take four times the time to merge, would change over at some 130 rows)
    p.parts = dtype == DT_F32 ? (rows >= TSP_MANY_ROWS ? 4 : 16) : (rows >= 192 ? 1 : 4);
    // (a quarter of more than 655360 columns does not fit the bitmap of the history, a sixteenth does: whether a
    // vocabulary is covered must not depend on the rows of the call)
    if (dtype == DT_F32 && keeps_y && topp_part_columns(vocab, p.parts) > TSP_WINDOW_BITS) {
        p.parts = 16;
    }
    // 16-bit stage: about sixteen waves per compute unit, workgroups of at least four blocks of columns, no more columns than
    // a bitmap of the history covers. Workgroups of 512 threads where each walks the row's whole history (us of the stage
    // with 256 / 512 / 1024: 64 x 128256 12.9 / 12.8 / 13.2, 128 x 152064 with 51 rows of its own 15.1 / 14.6 / 15.5; twice
    // the waves, when that was 13.7 and 15.6, 14.1 and 15.7), of 256 where there are no penalties (a step of 8 x 50257 29.5, with 512 30.2). Eight blocks
    // per workgroup, one for each wave, instead of four: a step of 1 x 32000 with penalties 25.8 / 26.4.
    p.blocks = (vocab + TSP_BLOCK - 1) / TSP_BLOCK;
    int s    = (TSP_STAGE_WAVES / (topp_stage16_threads(keeps_y) / WAVE) + rows - 1) / rows;
    s        = std::min(s, std::max(1, p.blocks / 4));
    s        = std::max(s, (p.blocks + TSP_WINDOW_BITS / TSP_BLOCK - 1) / (TSP_WINDOW_BITS / TSP_BLOCK));
    p.splits = std::min(s, TSP_SPLITS);
    p.chunk  = (p.blocks + p.splits - 1) / p.splits * TSP_BLOCK;
    p.sorters       = (int)std::min<size_t>(512, (size_t)rows * (vocab_padded / TPS_SEG + 1));
    p.y_pitch       = (int)((vocab_padded + 7) / 8 * 8);
    const size_t el = dtype == DT_F32 ? 4 : 2;
    // (fp32: also as many as a call of fewer rows and more parts takes, so that a window of a batch never needs more)
    const size_t counters =
        dtype == DT_F32 ? (size_t)std::max(rows * p.parts, std::min(rows, TSP_MANY_ROWS - 1) * 16) * TSP_BUCKETS :
                          (size_t)rows * (dtype == DT_F16 ? ToppCode<DT_F16>::COUNTERS : ToppCode<DT_BF16>::COUNTERS);
    size_t off = up256((size_t)rows * vocab_padded * 2 * sizeof(unsigned long long));
    auto   take = [&](size_t bytes) {
        const size_t at = off;
        off += up256(bytes);
        return at;
    };
    p.off_counts = take(counters * sizeof(uint32_t));
    p.off_pmax   = take((size_t)rows * TSP_SPLITS * sizeof(float2));
    p.off_blocks = take(dtype == DT_F32 ? 0 : (size_t)rows * p.blocks * sizeof(float));
    p.off_ref    = take((size_t)rows * sizeof(float));
    p.off_gsum   = take((size_t)rows * 32 * sizeof(float));
    p.off_segs   = take((size_t)rows * TPB_NB * sizeof(uint32_t));
    p.off_queue  = take(((size_t)rows * TPB_NB + 1) * sizeof(uint32_t));
    p.off_meta   = take((size_t)rows * sizeof(ToppRowMeta));
    p.off_y      = keeps_y ? take((size_t)rows * p.y_pitch * el) : 0;
    p.bytes      = off;
    return p;
}

size_t topp_sample_bytes(int dtype, int rows, int vocab, size_t vocab_padded, bool keeps_y)
{
    return topp_sample_plan(dtype, rows, vocab, vocab_padded, keeps_y).bytes;
}

bool topp_sample_covers(int dtype, int rows, int vocab, bool history_penalty)
{
    if (vocab < TSP_CHAINS) {
        return false;  // the sum's order follows the softmax's block of min(n, 1024) threads
    }
    if (!history_penalty) {
        return true;
    }
    // the bitmap of the history that a stage's workgroup keeps
    const ToppSamplePlan p = topp_sample_plan(dtype, rows, vocab, (size_t)vocab, true);
    return (dtype == DT_F32 ? topp_part_columns(vocab, p.parts) : p.chunk) <= TSP_WINDOW_BITS;
}

int topp_sample_launch(const ToppSampleCall& c, hipStream_t st)
{
    const bool           keeps_y = c.temperatures != nullptr || (c.penalties != nullptr && c.penalty_type != 2) || c.min_lengths != nullptr;
    const ToppSamplePlan p       = topp_sample_plan(c.dtype, c.rows, c.vocab_size, c.vocab_size_padded, keeps_y);
    if (c.workspace_size < p.bytes) {
        return FTK_ERR_WORKSPACE;
    }
    char*    ws = (char*)c.workspace;
    ToppStep s{};
    s.logits = c.logits;
    s.bias   = c.bias;
    s.n      = c.vocab_size;
    s.Vp     = (int)c.vocab_size_padded;
    s.rows   = c.rows;
    s.y      = keeps_y ? ws + p.off_y : nullptr;
    s.y_pitch          = p.y_pitch;
    s.temperatures     = c.temperatures;
    s.penalties        = c.penalties;
    s.penalty_type     = c.penalty_type;
    s.min_lengths      = c.min_lengths;
    s.end_ids          = c.end_ids;
    s.input_lengths    = c.input_lengths;
    s.history          = c.history;
    s.sequence_length  = c.sequence_length;
    s.batch_size       = c.batch_size;
    s.step             = c.step;
    s.max_input_length = c.max_input_length;
    s.finished         = c.finished;
    s.skip             = c.skip_decode;
    s.rng              = (const RngState*)c.rng_state;
    s.uniforms         = c.uniform_draws;
    s.top_p            = c.max_top_p;
    s.top_ps           = c.runtime_top_p;
    s.splits           = p.splits;
    s.chunk            = p.chunk;
    s.parts            = p.parts;
    s.blocks           = p.blocks;
    s.pmax             = (float2*)(ws + p.off_pmax);
    s.block_max        = (float*)(ws + p.off_blocks);
    s.ref              = (float*)(ws + p.off_ref);
    s.gsum             = (float*)(ws + p.off_gsum);
    s.counts           = (uint32_t*)(ws + p.off_counts);
    s.meta             = (ToppRowMeta*)(ws + p.off_meta);
    s.segs             = (uint32_t*)(ws + p.off_segs);
    s.queue            = (uint32_t*)(ws + p.off_queue);
    s.sorted           = (unsigned long long*)ws;
    ToppPickOut o{};
    o.ids              = c.output_ids;
    o.sequence_length  = c.sequence_length;
    o.finished         = c.finished;
    o.cum_log_probs    = c.cum_log_probs;
    o.output_log_probs = c.output_log_probs;
    o.rng        = (RngState*)c.rng_state;
    o.dec        = ToppDecayArgs{c.top_p_decay != nullptr ? c.runtime_top_p : nullptr, c.initial_top_p, c.top_p_decay,
                                 c.top_p_min, c.top_p_reset_ids};
    o.force_deep = topp_force_deep();

    const dim3 parts(c.rows, p.parts), splits(c.rows, p.splits);
    if (c.dtype == DT_F32) {
        const dim3 grid((c.rows + 7) / 8 * 8, p.parts);
        if (keeps_y) {
            topp_stage_f32_kernel<true><<<grid, TSP_STAGE, 0, st>>>(s);
        }
        else {
            topp_stage_f32_kernel<false><<<grid, TSP_STAGE, 0, st>>>(s);
        }
        FTK_LAUNCH_CHECK();
        if (p.parts == 4) {
            topp_sum_gather_kernel<1><<<grid, TSP_SUM32, 0, st>>>(s);
        }
        else {
            topp_sum_gather_kernel<4><<<grid, TSP_SUM32, 0, st>>>(s);
        }
        FTK_LAUNCH_CHECK();
        topp_sort_queue_kernel<<<p.sorters, TP_THREADS, 0, st>>>(s);
        FTK_LAUNCH_CHECK();
        topp_pick_f32_kernel<<<c.rows, TP_THREADS, 0, st>>>(s, o);
        FTK_LAUNCH_CHECK();
        return 0;
    }
    auto run = [&](auto type) -> int {
        constexpr int DT = decltype(type)::value;
        if (keeps_y && s.temperatures != nullptr && s.bias != nullptr) {  // (the bias comes with the temperature)
            topp_stage_kernel<DT, true, true><<<splits, topp_stage16_threads(true), 0, st>>>(s);
        }
        else if (keeps_y) {
            topp_stage_kernel<DT, true, false><<<splits, topp_stage16_threads(true), 0, st>>>(s);
        }
        else {
            topp_stage_kernel<DT, false, false><<<splits, topp_stage16_threads(false), 0, st>>>(s);
        }
        FTK_LAUNCH_CHECK();
        if (p.parts == 1) {
            topp_sum_count_kernel<DT, 1024><<<parts, TSP_SUM16, 0, st>>>(s);
        }
        else {
            topp_sum_count_kernel<DT, 256><<<parts, TSP_SUM16, 0, st>>>(s);
        }
        FTK_LAUNCH_CHECK();
        topp_pick_runs_kernel<DT><<<c.rows, TP_THREADS, 0, st>>>(s, o);
        FTK_LAUNCH_CHECK();
        return 0;
    };
    if (c.dtype == DT_F16) {
        return run(std::integral_constant<int, DT_F16>());
    }
    return run(std::integral_constant<int, DT_BF16>());
}

}  // namespace ftk

#ifdef FTK_TEST_HOOKS
// Test hook (hooks build of the library only): what the last fp32 step in this workspace gathered of every row.
extern "C" int ftk_test_topp_prefix_lengths(const void* workspace, int rows, int vocab, size_t pitch, int keeps_y,
                                            int* lengths)
{
    const ftk::ToppSamplePlan p = ftk::topp_sample_plan(ftk::DT_F32, rows, vocab, pitch, keeps_y != 0);
    return (int)hipMemcpy2D(lengths, sizeof(int), (const char*)workspace + p.off_meta + offsetof(ftk::ToppRowMeta, n),
                            sizeof(ftk::ToppRowMeta), sizeof(int), rows, hipMemcpyDeviceToHost);
}
#endif
