// Top-p building blocks shared by the sampler on probabilities (topp_kernels.hip) and the step that samples straight
// from logits (topp_sample_kernels.hip): workspace records, the sorts, the replay of the reference's scan, the exact
// whole-row fallback and what a row's sample leaves behind.
#pragma once
#include "ftk_columns.cuh"
#include "ftk_device.cuh"
#include "ftk_transform.cuh"

namespace ftk {

constexpr int      TP_THREADS = 1024;
constexpr int      TP_TILE    = 256;          // the reference's scan tile
constexpr int      TP_ROUND   = 1024;         // tiles whose totals are held in LDS at a time
constexpr uint32_t ZERO_KEY   = 0x80000000u;  // order_key(+0.0f); entries at or below never join the scan

constexpr int TPH_THREADS = 256;
constexpr int TPC_THREADS = 1024;  // the cut kernel
constexpr int TPB_SHIFT   = 17;                        // key bits below a bucket (6 mantissa bits stay)
constexpr int TPB_ONE     = 0x3F800000 >> TPB_SHIFT;   // bucket of 1.0 before the shift of origin
constexpr int TPB_SPAN    = 32 * 64;                   // 32 octaves below 1.0 are resolved
constexpr int TPB_NB      = TPB_SPAN + 2;              // [0]: everything smaller, [NB-1]: above 1 + 1/64
constexpr int TPS_SEG     = 2048;                      // segment boundaries follow multiples of this
constexpr int TPS_CAP     = 5632;                      // longest segment sorted in LDS

constexpr int TOPP_SKIP     = 1;
constexpr int TOPP_SHORTCUT = 2;

struct ToppRowMeta {
    unsigned long long best;   // (key << 32) | ~id of the arg-max (lowest id among equals)
    int                cut;    // lowest gathered bucket
    int                n;      // entries at or above the cut
    int                n_pos;  // positive entries of the row (0x7FFFFFFF: not known, some may lie below the cut)
    int                nseg;
    int                flags;
    float              safe;   // (from logits) entries with e from here on share no probability with what is not gathered
};
__device__ __forceinline__ int topp_bucket(uint32_t key)
{
    const int raw = (int)((key & 0x7FFFFFFFu) >> TPB_SHIFT) - (TPB_ONE - TPB_SPAN);
    return min(max(raw, 0), TPB_NB - 1);
}

__device__ __forceinline__ float key64_prob(unsigned long long k)
{
    return key_to_float(~(uint32_t)(k >> 32));
}
struct ToppRowValues {
    // what the softmax sees of a row: y(v) as softmax_kernel's `masked`, rows without a bias
    float MAXT;
    bool  fin;
    int   end_id, n;
    __device__ __forceinline__ float masked(int v, float x) const
    {
        if (v >= n) {
            return -MAXT;
        }
        if (fin) {
            return v == end_id ? MAXT : -MAXT;
        }
        return x + 0.0f;
    }
};

// the probability the softmax would store for an element with e = T(exp(y - max)), as a float
template<int DT>
__device__ __forceinline__ float topp_prob_of(float e, const RowDivisor& div, float denom)
{
    return round_t<DT>(div.ok ? div.divide(e) : e / denom);
}
// Scratch of the radix sort below.
struct RadixScratch {
    unsigned short*     cnt16;  // [16][TP_THREADS]
    int*                wtot;   // [256]
    unsigned long long* red64;  // [16]
};

// Stable LSD radix sort (4-bit digits over bits [lowbit, 64)) of n 64-bit entries in memory by a
// TP_THREADS workgroup; digits that are constant over the range are skipped. Thread t owns the
// contiguous slice [t*chunk, (t+1)*chunk), n <= 65535 * TP_THREADS. Returns where the result is
// (a or b).
__device__ unsigned long long* radix_sort_range(unsigned long long* a, unsigned long long* b, int n, int lowbit,
                                                RadixScratch rs)
{
    const int t     = threadIdx.x;
    const int chunk = (n + TP_THREADS - 1) / TP_THREADS;
    const int lo    = min(n, t * chunk);
    const int hi    = min(n, lo + chunk);
    unsigned long long vor = 0ull, vand = ~0ull;
    for (int i = lo; i < hi; ++i) {
        vor |= a[i];
        vand &= a[i];
    }
    for (int o = 32; o > 0; o >>= 1) {
        vor |= __shfl_xor(vor, o, WAVE);
        vand &= __shfl_xor(vand, o, WAVE);
    }
    __syncthreads();
    if (lane_id() == 0) {
        rs.red64[wave_id()] = vor;
    }
    __syncthreads();
    unsigned long long all_or = 0ull;
    for (int w = 0; w < TP_THREADS / WAVE; ++w) {
        all_or |= rs.red64[w];
    }
    __syncthreads();
    if (lane_id() == 0) {
        rs.red64[wave_id()] = vand;
    }
    __syncthreads();
    unsigned long long all_and = ~0ull;
    for (int w = 0; w < TP_THREADS / WAVE; ++w) {
        all_and &= rs.red64[w];
    }
    __syncthreads();
    const unsigned long long diff = all_or ^ all_and;

    unsigned long long* src = a;
    unsigned long long* dst = b;
    for (int shift = lowbit; shift < 64; shift += 4) {
        if (((diff >> shift) & 0xFull) == 0ull) {
            continue;
        }
        // 1. private digit counts
        for (int d = 0; d < 16; ++d) {
            rs.cnt16[d * TP_THREADS + t] = 0;
        }
        for (int i = lo; i < hi; ++i) {
            const int d = (int)((src[i] >> shift) & 0xFull);
            rs.cnt16[d * TP_THREADS + t]++;
        }
        // 2. exclusive prefix over (digit major, thread minor)
        int base_off[16];
#pragma unroll
        for (int d = 0; d < 16; ++d) {
            const int val = rs.cnt16[d * TP_THREADS + t];
            int       inc = val;
#pragma unroll
            for (int o = 1; o < WAVE; o <<= 1) {
                const int up = __shfl_up(inc, o, WAVE);
                if (lane_id() >= o) {
                    inc += up;
                }
            }
            base_off[d] = inc - val;
            if (lane_id() == WAVE - 1) {
                rs.wtot[d * 16 + wave_id()] = inc;
            }
        }
        __syncthreads();
        // exclusive prefix over (digit major, wave minor), four of the 256 totals per lane of the first wave
        if (t < WAVE) {
            int x[4], sum = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                x[j] = rs.wtot[4 * t + j];
                sum += x[j];
            }
            int inc = sum;
#pragma unroll
            for (int o = 1; o < WAVE; o <<= 1) {
                const int up = __shfl_up(inc, o, WAVE);
                if (t >= o) {
                    inc += up;
                }
            }
            int at = inc - sum;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                rs.wtot[4 * t + j] = at;
                at += x[j];
            }
        }
        __syncthreads();
#pragma unroll
        for (int d = 0; d < 16; ++d) {
            base_off[d] += rs.wtot[d * 16 + wave_id()];
        }
        __syncthreads();
        // 3. stable scatter
        for (int i = lo; i < hi; ++i) {
            const unsigned long long e = src[i];
            const int                d = (int)((e >> shift) & 0xFull);
            int                      pos = 0;
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                if (q == d) {
                    pos = base_off[q]++;
                }
            }
            dst[pos] = e;
        }
        __threadfence_block();
        __syncthreads();
        unsigned long long* tmp = src;
        src                     = dst;
        dst                     = tmp;
    }
    return src;
}

// Ascending bitonic sort of 64 * R 64-bit keys held R per lane by one wave; key r of lane l has the
// position r * 64 + l. Exchanges inside a register go through lane shuffles, the others stay in the
// lane.
template<int R>
__device__ __forceinline__ void wave_sort_u64(unsigned long long (&v)[R])
{
    const int lane = lane_id();
#pragma unroll
    for (int k = 2; k <= 64 * R; k <<= 1) {
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            if (j < 64) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int                idx   = r * 64 + lane;
                    const unsigned long long other = __shfl_xor(v[r], j, WAVE);
                    const bool               up    = (idx & k) == 0;
                    const bool               lower = (idx & j) == 0;
                    const bool               less  = other < v[r];
                    // the lower position keeps the smaller key in ascending runs
                    v[r] = ((lower == up) == less) ? other : v[r];
                }
            }
            else {
                const int jj = j >> 6;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    if ((r & jj) == 0) {
                        const bool               up = ((r * 64) & k) == 0;
                        const unsigned long long a  = v[r];
                        const unsigned long long b  = v[r | jj];
                        const bool               sw = (a > b) == up;
                        v[r]                        = sw ? b : a;
                        v[r | jj]                   = sw ? a : b;
                    }
                }
            }
        }
    }
}

// One wave sorts buf[s0, s0 + len), len <= 64 * R, and writes the result to out[s0, ...).
template<int R>
__device__ __forceinline__ void wave_sort_group(const unsigned long long* buf, unsigned long long* out, int s0, int len)
{
    const int          lane = lane_id();
    unsigned long long v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = r * 64 + lane;
        v[r]        = i < len ? buf[s0 + i] : ~0ull;
    }
    wave_sort_u64<R>(v);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = r * 64 + lane;
        if (i < len) {
            out[s0 + i] = v[r];
        }
    }
}

constexpr int TPS_DIGITS = 1024;  // bins of the partition inside a segment
constexpr int TPS_GROUP  = 48;    // group boundaries follow multiples of this
constexpr int TPS_EPT    = (TPS_CAP + TP_THREADS - 1) / TP_THREADS;

// The radix path needs 32 KB of digit counters; its small arrays live behind them in the same buffer.
struct ToppSortShared {
    unsigned long long buf[TPS_CAP];
    uint32_t           hist[TPS_DIGITS];  // entries per bin, then the write cursors
    uint32_t           base[TPS_DIGITS];  // first position of a bin
    uint32_t           gend[TPS_DIGITS];  // end of every group of bins
    uint32_t           psum[TP_THREADS];  // running number of segments over a tile of rows
    uint32_t           wtot[TP_THREADS / WAVE];
    uint32_t           red32[16];
    int                big[64];           // groups left to the whole workgroup
    int                nbig;
};
static_assert(sizeof(ToppSortShared) <= 65536, "static LDS");

// Inclusive scan of one value per thread over the TP_THREADS threads; `total` gets the sum. Two barriers.
__device__ __forceinline__ uint32_t block_scan_incl(uint32_t v, uint32_t* wtot, uint32_t& total)
{
    uint32_t inc = v;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        const uint32_t up = __shfl_up(inc, o, WAVE);
        if (lane_id() >= o) {
            inc += up;
        }
    }
    __syncthreads();
    if (lane_id() == WAVE - 1) {
        wtot[wave_id()] = inc;
    }
    __syncthreads();
    total = 0;
    for (int w = 0; w < TP_THREADS / WAVE; ++w) {
        const uint32_t x = wtot[w];
        inc += w < wave_id() ? x : 0u;
        total += x;
    }
    return inc;
}

// Sorts seg[0, n) ascending (descending probability, ascending id among equals), n <= TPS_CAP: the keys
// are spread over TPS_DIGITS bins of equal width between the smallest and the largest, neighbouring
// bins are joined into groups of about TPS_GROUP entries, and every group is sorted by one wave in
// registers. A group too long for that (equal keys land in one bin) is left to the whole workgroup.
__device__ void sort_segment(ToppSortShared& s, unsigned long long* __restrict__ seg, int n)
{
    const int          t = threadIdx.x;
    unsigned long long e[TPS_EPT];
    uint32_t           kmin = 0xFFFFFFFFu, kmax = 0u;
#pragma unroll
    for (int r = 0; r < TPS_EPT; ++r) {
        const int i = t + r * TP_THREADS;
        if (i < n) {
            e[r]             = seg[i];
            const uint32_t h = (uint32_t)(e[r] >> 32);
            kmin             = min(kmin, h);
            kmax             = max(kmax, h);
        }
    }
    s.hist[t] = 0u;  // TPS_DIGITS == TP_THREADS
    if (t == 0) {
        s.nbig = 0;
    }
    kmin = block_min<uint32_t, TP_THREADS / WAVE>(kmin, s.red32, 0xFFFFFFFFu);
    kmax = block_max<uint32_t, TP_THREADS / WAVE>(kmax, s.red32, 0u);
    const uint32_t range = kmax - kmin;
    const int      nbits = range == 0u ? 0 : 32 - __clz(range);
    const int      shift = nbits > 10 ? nbits - 10 : 0;
#pragma unroll
    for (int r = 0; r < TPS_EPT; ++r) {
        if (t + r * TP_THREADS < n) {
            atomicAdd(&s.hist[((uint32_t)(e[r] >> 32) - kmin) >> shift], 1u);
        }
    }
    __syncthreads();
    const uint32_t cnt = s.hist[t];
    uint32_t       total;
    const uint32_t en = block_scan_incl(cnt, s.wtot, total);
    const uint32_t o  = en - cnt;
    s.base[t]         = o;
    s.hist[t]         = 0u;
    const bool     closes = cnt != 0u && (en / TPS_GROUP != o / TPS_GROUP || en == (uint32_t)n);
    uint32_t       ngroups;
    const uint32_t gi = block_scan_incl(closes ? 1u : 0u, s.wtot, ngroups);
    if (closes) {
        s.gend[gi - 1] = en;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < TPS_EPT; ++r) {
        if (t + r * TP_THREADS < n) {
            const uint32_t d   = ((uint32_t)(e[r] >> 32) - kmin) >> shift;
            const uint32_t pos = s.base[d] + atomicAdd(&s.hist[d], 1u);
            s.buf[pos]         = e[r];
        }
    }
    __syncthreads();
    for (int g = wave_id(); g < (int)ngroups; g += TP_THREADS / WAVE) {
        const int s0  = g > 0 ? (int)s.gend[g - 1] : 0;
        const int len = (int)s.gend[g] - s0;
        if (len <= 64) {
            wave_sort_group<1>(s.buf, seg, s0, len);
        }
        else if (len <= 128) {
            wave_sort_group<2>(s.buf, seg, s0, len);
        }
        else if (len <= 256) {
            wave_sort_group<4>(s.buf, seg, s0, len);
        }
        else if (lane_id() == 0) {
            const int slot = atomicAdd(&s.nbig, 1);
            if (slot < 64) {
                s.big[slot] = g;
            }
        }
    }
    __syncthreads();
    const int nbig = s.nbig;
    if (nbig > 64) {
        // cannot happen with more than 256 entries per long group and n <= TPS_CAP; sort everything
        block_sort_u64<TP_THREADS>(s.buf, n);
        for (int i = t; i < n; i += TP_THREADS) {
            seg[i] = s.buf[i];
        }
    }
    else {
        for (int q = 0; q < nbig; ++q) {
            const int g   = s.big[q];
            const int s0  = g > 0 ? (int)s.gend[g - 1] : 0;
            const int len = (int)s.gend[g] - s0;
            block_sort_u64<TP_THREADS>(s.buf + s0, len);
            for (int i = t; i < len; i += TP_THREADS) {
                seg[s0 + i] = s.buf[s0 + i];
            }
        }
    }
    __syncthreads();
}

// Sorts one segment seg[0, n) of a row's prefix by the whole workgroup; `spare` is scratch of the same length.
__device__ __forceinline__ void topp_sort_one(ToppSortShared& s, unsigned long long* seg, unsigned long long* spare, int n)
{
    const int t = threadIdx.x;
    if (n < 2) {
        return;
    }
    if (n <= 256) {
        // one wave, straight from memory (most rows only order a few dozen entries)
        if (wave_id() == 0) {
            if (n <= 64) {
                wave_sort_group<1>(seg, seg, 0, n);
            }
            else {
                wave_sort_group<4>(seg, seg, 0, n);
            }
        }
    }
    else if (n <= TPS_CAP) {
        sort_segment(s, seg, n);
    }
    else {
        RadixScratch        rs{reinterpret_cast<unsigned short*>(s.buf), reinterpret_cast<int*>(s.buf + 4096),
                        reinterpret_cast<unsigned long long*>(s.buf + 4096 + 128)};
        unsigned long long* res = radix_sort_range(seg, spare, n, 0, rs);
        if (res != seg) {
            for (int q = t; q < n; q += TP_THREADS) {
                seg[q] = res[q];
            }
        }
        __threadfence_block();
        __syncthreads();
    }
}

// What the pick kernels keep in LDS besides the digit counters of the fallback's radix sort (TP_DIGITS entries).
constexpr int TP_DIGITS = 4096;
struct TopPScan {
    unsigned long long red64[16];
    uint32_t           red32[16];
    float              agg[TP_ROUND];
    float              carry[TP_ROUND + 1];
    int                wtot[256];
    int                misc[8];
    float              fmisc[4];
};

// One 32-lane group loads the eight items of each of its lanes from tile `tile` of the ordered
// array (entries at or beyond n count as 0).
__device__ __forceinline__ void tile_load(const unsigned long long* __restrict__ src, int n, int tile, int l, float x[8])
{
    const int i0 = tile * TP_TILE + l * 8;
    if (i0 + 8 <= n && ((uintptr_t)src & 15u) == 0u) {
        const ulonglong2* v = reinterpret_cast<const ulonglong2*>(src + i0);  // i0 is a multiple of 8
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const ulonglong2 p = v[j];
            x[2 * j]           = key64_prob(p.x);
            x[2 * j + 1]       = key64_prob(p.y);
        }
    }
    else {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            x[j] = i0 + j < n ? key64_prob(src[i0 + j]) : 0.0f;
        }
    }
}

// x of the lane `D` lanes below within a 32-lane group, for lanes that have one (others get something): shifts inside
// rows of 16 lanes, and across rows the other row's value, rotated. Vector instructions, where a shuffle goes through LDS.
template<int D>
__device__ __forceinline__ float group_shift_up(float x, int l)
{
    static_assert(D == 1 || D == 2 || D == 4 || D == 8 || D == 16, "shifts of the raking");
    constexpr int ROW_SHR = 0x110, ROW_ROR = 0x120;
    const int     bits = __float_as_int(x);
    // (v_permlane16_swap: its first result holds, in odd rows of 16 lanes, the even row in front of them)
    if constexpr (D == 16) {
        return __int_as_float((int)__builtin_amdgcn_permlane16_swap((unsigned)bits, (unsigned)bits, false, false)[0]);
    }
    else {
        const int within = __builtin_amdgcn_update_dpp(bits, bits, ROW_SHR + D, 0xF, 0xF, false);
        const int turned = __builtin_amdgcn_update_dpp(bits, bits, ROW_ROR + D, 0xF, 0xF, false);
        const int across = (int)__builtin_amdgcn_permlane16_swap((unsigned)turned, (unsigned)turned, false, false)[0];
        return __int_as_float((l & 15) >= D ? within : across);
    }
}

// Inclusive raking scan of the lane totals of a tile.
__device__ __forceinline__ float tile_scan(const float x[8], int l)
{
    float seg = x[0];
#pragma unroll
    for (int j = 1; j < 8; ++j) {
        seg = seg + x[j];
    }
    float incl = seg;
    auto  step = [&](auto d) {
        constexpr int D  = decltype(d)::value;
        const float   up = group_shift_up<D>(incl, l);
        if (l >= D) {
            incl = up + incl;
        }
    };
    step(std::integral_constant<int, 1>());
    step(std::integral_constant<int, 2>());
    step(std::integral_constant<int, 4>());
    step(std::integral_constant<int, 8>());
    step(std::integral_constant<int, 16>());
    return incl;
}

// Inclusive sum over the lanes of a wave.
__device__ __forceinline__ uint32_t wave_scan_add(uint32_t x)
{
    constexpr int ROW_SHR = 0x110, ROW_BCAST15 = 0x142, ROW_BCAST31 = 0x143;
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, ROW_SHR + 1, 0xF, 0xF, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, ROW_SHR + 2, 0xF, 0xF, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, ROW_SHR + 4, 0xF, 0xF, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, ROW_SHR + 8, 0xF, 0xF, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, ROW_BCAST15, 0xA, 0xF, false);  // odd rows: the row in front
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, ROW_BCAST31, 0xC, 0xF, false);  // upper half: the lower one
    return x;
}

// One wave: c + a of lane 0, + a of lane 1, ... of `n` lanes, one rounded addition after the other; a lane gets the sum in
// front of it, c becomes the last one. (No a is negative or NaN.) While the sum stays below a power of two, it counts in
// units of its last place and an addition rounds to a whole number of them, whatever the sum is, except that a value halfway
// between two makes the sum even: then what it adds depends on whether the sum in front of it is odd, that is on the last
// such value before it and the odd numbers since. So all of that is worked out side by side and added as whole numbers;
// the additions at which the sum outgrows its power of two are made by themselves. (300 tile totals: 11.2 us with an
// addition per lane in turn, 2.6.)
__device__ __forceinline__ float running_sums(float& c, float a, int n)
{
    const int l      = lane_id();
    float     before = c;
    int       first  = 0;  // lanes in front of it are done
    while (first < n) {
        int stop = first;  // the lane whose addition is made by itself
        if (c > 1e-20f && c < 1e20f) {
            const uint32_t bits  = f2u(c);
            const float    to    = u2f((277u << 23) - (bits & 0x7F800000u));  // 1 / unit
            const float    unit  = u2f((bits & 0x7F800000u) - (23u << 23));
            const uint32_t sum   = (bits & 0x007FFFFFu) | 0x00800000u;
            const float    q     = l >= first && l < n ? a * to : 0.0f;
            const bool     large = !(q < 8388608.0f);
            const uint32_t whole = large ? 0u : (uint32_t)q;
            const float    part  = large ? 0.0f : q - (float)whole;
            const unsigned long long ties = __ballot(part == 0.5f);
            const uint32_t near  = whole + (part > 0.5f ? 1u : 0u);
            const unsigned long long odds  = __ballot((near & 1u) != 0u);
            const unsigned long long below = (1ull << l) - 1ull;
            unsigned long long       since = below;  // lanes whose numbers decide whether the sum in front of this one is odd
            uint32_t                 start = sum;
            if ((ties & below) != 0ull) {
                since = below & ~((2ull << (63 - __builtin_clzll(ties & below))) - 1ull);
                start = 0u;
            }
            const uint32_t odd = (start + (uint32_t)__popcll(odds & since)) & 1u;
            const uint32_t add = near + (part == 0.5f ? (odd + near) & 1u : 0u);
            const uint32_t upto = sum + wave_scan_add(add);
            const unsigned long long over = __ballot(large || upto >= 0x01000000u);
            stop = over != 0ull ? (int)__builtin_ctzll(over) : n;
            const float mine = (float)(upto - add) * unit;
            if (l >= first && l <= stop) {
                before = mine;
            }
            if (stop >= n) {
                c = (float)(uint32_t)__builtin_amdgcn_readlane((int)upto, WAVE - 1) * unit;
                break;
            }
            c = u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(mine), stop));
        }
        else if (l == stop) {
            before = c;
        }
        c     = c + u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(a), stop));
        first = stop + 1;
    }
    return before;
}

// Replays the reference scan over `nt` tiles of an ordered row; load(tile, l, x) gives the eight values lane l of a
// 32-lane group takes from a tile (0 beyond the row's entries); totals(base, n) leaves the totals of tiles
// [base, base + n) in s.agg[0, n). Returns the position the reference would pick (it can lie in the zero padding of the
// last tile) or -1 when the draw is never reached. All threads must call; the result is block-uniform.
template<class LoadTile, class Totals>
__device__ __forceinline__ int scan_tiles(TopPScan& s, int nt, float rand_num, LoadTile&& load, Totals&& totals)
{
    const int t     = threadIdx.x;
    const int group = t >> 5;
    const int l     = t & 31;
    // a tile whose running total stays below this cannot hold the crossing: the prefixes inside a
    // tile and the tile's total differ by rounding only
    const float near = rand_num * (1.0f - 1.0f / 4096.0f);
    float       carry_in = 0.0f;
    for (int base = 0; base < nt; base += TP_ROUND) {
        const int ntr = min(TP_ROUND, nt - base);
        totals(base, ntr);
        __syncthreads();
        if (t < WAVE) {
            float c  = carry_in;
            int   g0 = -1;
            for (int g = 0; g < ntr; g += WAVE) {
                const bool  mine   = g + t < ntr;
                const float a      = mine ? s.agg[g + t] : 0.0f;
                const float before = running_sums(c, a, min(WAVE, ntr - g));
                if (mine) {
                    s.carry[g + t] = before;
                }
                const unsigned long long reach = __ballot(mine && before + a >= near);
                if (g0 < 0 && reach != 0ull) {
                    g0 = g + __builtin_ctzll(reach);
                }
            }
            if (t == 0) {
                s.carry[ntr] = c;
                s.misc[0]    = 0x7FFFFFFF;
                s.misc[1]    = g0;
            }
        }
        __syncthreads();
        const int g0 = s.misc[1];
        if (g0 >= 0) {
            for (int gs = g0; gs < ntr; gs += TP_THREADS / 32) {
                const int g  = gs + group;
                uint32_t  m8 = 0;
                if (g < ntr) {
                    float x[8];
                    load(base + g, l, x);
                    const float incl   = tile_scan(x, l);
                    const float excl   = __shfl_up(incl, 1, 32);
                    const float prefix = s.carry[g];
                    float       a      = l == 0 ? prefix : prefix + excl;
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        a = a + x[j];
                        if (rand_num <= a) {
                            m8 |= 1u << j;
                        }
                    }
                }
                // the reference looks at words of 32 positions, four lanes here: the first that holds a crossing counts
                // from its end
                int c = __popc(m8);
                c += dpp_from<DPP_QUAD_XOR1>(c);
                c += dpp_from<DPP_QUAD_XOR2>(c);
                const uint32_t lanes = (uint32_t)(__ballot(m8 != 0u) >> (lane_id() & 32));
                if (lanes != 0u) {
                    const int first = __builtin_ctz(lanes) >> 2;
                    if (l == first * 4) {
                        atomicMin(&s.misc[0], (base + g) * TP_TILE + first * 32 + (32 - c));
                    }
                }
                __syncthreads();
                const int found = s.misc[0];
                __syncthreads();
                if (found != 0x7FFFFFFF) {
                    return found;
                }
            }
        }
        carry_in = s.carry[ntr];
        __syncthreads();
    }
    return -1;
}

// The same with the totals worked out from load(), Q tiles in flight per 32-lane group.
template<int Q, class LoadTile>
__device__ __forceinline__ int scan_tiles(TopPScan& s, int nt, float rand_num, LoadTile&& load)
{
    return scan_tiles(s, nt, rand_num, load, [&](int base, int n) {
        constexpr int NG    = TP_THREADS / 32;
        const int     group = (int)threadIdx.x >> 5, l = (int)threadIdx.x & 31;
        for (int g = group; g < n; g += Q * NG) {
            float x[Q][8];
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                if (g + q * NG < n) {
                    load(base + g + q * NG, l, x[q]);
                }
            }
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                if (g + q * NG < n) {
                    const float incl = tile_scan(x[q], l);
                    if (l == 31) {
                        s.agg[g + q * NG] = incl;
                    }
                }
            }
        }
    });
}
// id of the `nth` (0-based) entry whose probability is not positive, in ascending id order: what a stable descending
// sort leaves behind the positive entries. prob(v) gives the probability of column v. Single thread; reached only when
// a draw lands within rounding distance of the total mass.
template<class P>
__device__ int nth_zero_entry(P&& prob, int vocab, int nth)
{
    int seen = 0, last = vocab - 1;
    for (int v = 0; v < vocab; ++v) {
        if (order_key(prob(v)) <= ZERO_KEY) {
            last = v;
            if (seen == nth) {
                return v;
            }
            seen++;
        }
    }
    return last;
}
// What the sampler leaves behind for one row. Called by a single thread.
struct TopPEmit {
    int*       ids;
    int*       sequence_length;
    bool*      finished;
    float*     cum_log_probs;
    float*     output_log_probs;
    const int* end_ids;
    int        row;
    __device__ __forceinline__ void operator()(int id, float prob) const
    {
        ids[row] = id;
        if (cum_log_probs != nullptr || output_log_probs != nullptr) {
            const float lp = det_logf(prob);
            if (cum_log_probs != nullptr) {
                cum_log_probs[row] += lp;
            }
            if (output_log_probs != nullptr) {
                output_log_probs[row] = lp;
            }
        }
        if (sequence_length != nullptr && finished != nullptr) {
            sequence_length[row] = finished[row] ? sequence_length[row] : sequence_length[row] + 1;
            finished[row]        = id == end_ids[row];
        }
    }
};

// The exact way out: every entry of a row with a positive probability, compacted in id order, and a stable radix sort
// on the key bits. Returns where the result is (A or B); s.misc[2] holds the number of entries. Every thread calls.
template<class P>
__device__ __forceinline__ const unsigned long long* sort_whole_row(TopPScan& s, unsigned long long* digits, P&& prob_at,
                                                                    int vocab, unsigned long long* A,
                                                                    unsigned long long* B)
{
    const int t = threadIdx.x;
    if (t == 0) {
        s.misc[2] = 0;
    }
    __syncthreads();
    for (int base = 0; base < vocab; base += TP_THREADS) {
        const int                v    = base + t;
        const uint32_t           k    = v < vocab ? order_key(prob_at(v)) : 0u;
        const bool               keep = k > ZERO_KEY;
        const unsigned long long bal  = __ballot(keep);
        const int                below = __popcll(bal & ((1ull << lane_id()) - 1ull));
        if (lane_id() == 0) {
            s.red32[wave_id()] = (uint32_t)__popcll(bal);
        }
        __syncthreads();
        int off = s.misc[2];
        for (int w = 0; w < wave_id(); ++w) {
            off += (int)s.red32[w];
        }
        if (keep) {
            A[off + below] = ((unsigned long long)(~k) << 32) | (uint32_t)v;
        }
        __syncthreads();
        if (t == 0) {
            int tot = 0;
            for (int w = 0; w < TP_THREADS / WAVE; ++w) {
                tot += (int)s.red32[w];
            }
            s.misc[2] += tot;
        }
        __syncthreads();
    }
    const int n_all = s.misc[2];
    __threadfence_block();
    __syncthreads();
    RadixScratch rs{reinterpret_cast<unsigned short*>(digits), s.wtot, s.red64};
    return radix_sort_range(A, B, n_all, 32, rs);
}

// What computeToppDecay (:1381-1412) does to one row; the fused step runs it at the end of the row's pick.
struct ToppDecayArgs {
    float*         runtime_top_p;  // NULL: no decay
    const float*   initial_top_p;
    const float*   decay;
    const float*   top_p_min;
    const int32_t* reset_ids;
};

// One thread, after the row's id is there (the reference reads it back the same way).
__device__ __forceinline__ void topp_decay_row(const ToppDecayArgs& dec, int row, int id)
{
    if (id == dec.reset_ids[row]) {
        dec.runtime_top_p[row] = dec.initial_top_p[row];
    }
    else {
        dec.runtime_top_p[row] = __builtin_fmaxf(dec.runtime_top_p[row] * dec.decay[row], dec.top_p_min[row]);
    }
}

// The draw of row `b` without consuming it (the pick kernel consumes it).
__device__ __forceinline__ float row_uniform_peek(const RngState* rng, const float* injected, int b)
{
    if (injected != nullptr) {
        return injected[b];
    }
    RngState copy = rng[b];
    return rng_next_uniform(&copy);
}

}  // namespace ftk
