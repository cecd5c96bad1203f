// T(exp(y - max)) for the 16-bit types, two values at a time: the bits that det_expf and one rounding to T give.
//
// The softmax of the reference rounds every numerator to T (src/fastertransformer/kernels/sampling_topp_kernels.cu:1332),
// so of det_expf's 24 bits only those that decide the rounding matter. The hardware's exponential of
// t = y log2 e - max log2 e (one fused multiply-add) is within a known relative error of det_expf; where both ends of
// that interval round to the same T, that is the result. Where they differ det_expf decides: the caller collects
// `redo` over a few pairs and looks at it once (undecided()).
#pragma once
#include "ftk_device.cuh"

namespace ftk {

template<int DT>
struct ExpPairs {
    static_assert(DT == DT_F16 || DT == DT_BF16, "16-bit types");
    typedef Storage<DT> S;
    typedef float       f32x2 __attribute__((ext_vector_type(2)));
    typedef _Float16    f16x2 __attribute__((ext_vector_type(2)));
    typedef __bf16      bf16x2 __attribute__((ext_vector_type(2)));
    static constexpr float LOG2E = 1.44269502162933349609375f;
    // t carries SHIFT more than the argument: its rounding is finest where it is small, SHIFT / log2 e below the maximum.
    // (bfloat16: with it nothing is flushed either that does not round to zero)
    static constexpr float SHIFT = DT == DT_F16 ? 13.0f : 24.0f, UNSHIFT = DT == DT_F16 ? 0x1p-13f : 0x1p-24f;
    // How far det_expf can lie above / below the hardware's value: a share of it and an absolute part, for where the
    // roundings of t and of det_expf's y - max are larger. Largest distances over every pair of values y <= max of the type:
    // binary16 6.0e-7 / 8.0e-7 and 7.7e-13; bfloat16 1.34e-6 / 1.75e-6 and 2.4e-19. The factors' own rounding comes on top
    // (a test goes through all pairs). Wider bounds cost time, not bits: more pairs are evaluated twice. (bfloat16, normal
    // logits at temperatures of 0.7 to 2: a pair in 12.5 % of the groups of 512 columns, with a SHIFT of 16 in 13.7 %, of 28
    // in 16.4 %: the e of near columns lie close to where the type rounds more often than by chance, so that t has to be
    // good there)
    static constexpr float UP    = DT == DT_F16 ? 6.7e-7f : 1.4e-6f;
    static constexpr float DOWN  = DT == DT_F16 ? 8.7e-7f : 1.82e-6f;
    static constexpr float FLOOR = DT == DT_F16 ? 8.0e-13f : 3.0e-19f;
    // bfloat16, columns more than some 30 below the maximum (e below FAR): there the absolute part tells, and soon is as
    // large as the value, so that nothing is decided. Bounds that grow with |t| hold everywhere (largest distances beyond the
    // growing parts 8.6e-7 / 1.31e-6) and need none, apart from the last bits of subnormal numbers. They take three more
    // operations a column.
    static constexpr float WIDE_UP = 9.4e-7f, WIDE_UP_T = 8.0e-8f, WIDE_DOWN = 1.38e-6f, WIDE_DOWN_T = 1.0e-7f;
    static constexpr float WIDE_LAST = 0x1p-147f;
    static constexpr uint32_t FAR = (127 - 43) << 7;  // 2^-43
    float    max;
    float    c, hi, lo, one;
    float    wide_hi, wide_lo, wide_hi_t, wide_lo_t;
    uint32_t never;  // redo from the start: a maximum so large that c says little about it

    // `row_max` is the same for every lane
    __device__ __forceinline__ explicit ExpPairs(float row_max)
    {
        max   = row_max;
        never = __builtin_fabsf(row_max) < 1048576.0f ? 0u : 1u;
        // c = SHIFT - max log2 e; what its two roundings took goes into the factors
        const float m = row_max * LOG2E, m_low = fma_rn(row_max, LOG2E, -m);
        const float sum = SHIFT - m, part = sum - SHIFT;
        const float sum_low = (SHIFT - (sum - part)) + (-m - part);
        const float scale   = __builtin_amdgcn_exp2f(sum_low - m_low) * UNSHIFT;
        c                   = uniform_f(sum);
        hi                  = uniform_f(fma_rn(scale, UP, scale));
        lo                  = uniform_f(fma_rn(scale, -DOWN, scale));
        if constexpr (DT == DT_BF16) {
            wide_hi   = uniform_f(fma_rn(scale, WIDE_UP, scale));
            wide_lo   = uniform_f(fma_rn(scale, -WIDE_DOWN, scale));
            wide_hi_t = uniform_f(scale * WIDE_UP_T);
            wide_lo_t = uniform_f(scale * -WIDE_DOWN_T);
        }
        one                 = 1.0f;
        asm("" : "+s"(one));  // (a multiplication by a visible 1 would be taken out, and with it the fused conversion)
    }
    static __device__ __forceinline__ float low(uint32_t w)
    {
        if constexpr (DT == DT_F16) {
            return (float)__builtin_bit_cast(f16x2, w).x;
        }
        else {
            return u2f(w << 16);
        }
    }
    static __device__ __forceinline__ float high(uint32_t w)
    {
        if constexpr (DT == DT_F16) {
            return (float)__builtin_bit_cast(f16x2, w).y;
        }
        else {
            return u2f(w & 0xFFFF0000u);
        }
    }
    static __device__ __forceinline__ uint32_t pack(float a, float b)
    {
        const f32x2 v = {a, b};
        if constexpr (DT == DT_F16) {
            return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
        }
        else {
            return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
        }
    }
    // two values after temperature and penalties -> their two e
    __device__ __forceinline__ uint32_t operator()(uint32_t y, uint32_t& redo) const
    {
        const float a = __builtin_amdgcn_exp2f(fma_rn(low(y), LOG2E, c));
        const float b = __builtin_amdgcn_exp2f(fma_rn(high(y), LOG2E, c));
        const uint32_t up   = pack(fma_rn(a, hi, FLOOR), fma_rn(b, hi, FLOOR));
        const uint32_t down = pack(fma_rn(a, lo, -FLOOR), fma_rn(b, lo, -FLOOR));
        redo |= up ^ down;
        return up;
    }
    // the same with the bounds that hold at any distance (bfloat16)
    __device__ __forceinline__ uint32_t wide(uint32_t y, uint32_t& redo) const
    {
        float up[2], down[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float t = fma_rn(h == 0 ? low(y) : high(y), LOG2E, c);
            const float a = __builtin_amdgcn_exp2f(t);
            const float d = __builtin_fminf(__builtin_fabsf(t), 256.0f);  // (zero times infinity)
            up[h]         = fma_rn(a, fma_rn(d, wide_hi_t, wide_hi), WIDE_LAST);
            down[h]       = fma_rn(a, fma_rn(d, wide_lo_t, wide_lo), -WIDE_LAST);
        }
        const uint32_t e = pack(up[0], up[1]);
        redo |= e ^ pack(down[0], down[1]);
        return e;
    }
    // Whether what the calls above collected asks for det_expf. Where the absolute part rounds to zero (binary16, and the wide
    // bounds) the lower end of a value near zero rounds to -0, which is no difference; where it does not, a change of sign is
    // one.
    static __device__ __forceinline__ bool undecided(uint32_t redo, bool of_wide = false)
    {
        return DT == DT_F16 || of_wide ? (redo & 0x7FFF7FFFu) != 0u : redo != 0u;
    }
    // the same by det_expf
    __device__ __forceinline__ uint32_t exact(uint32_t y) const
    {
        return pack(det_expf_nonpos(low(y) - max), det_expf_nonpos(high(y) - max));
    }
    // e of P pairs, exactly: all of them in a straight line, then one look for pairs that are not decided, in a branch that
    // the whole wave takes, and one at each pair (1024 x 32000 binary16 at temperature 2, where nearly every group of 512
    // columns holds an undecided one: 49.0 us a step with two pairs each, 46.1). `far`: lanes with a column so far below the maximum that the
    // wide bounds are the better ones are added.
    template<int P>
    __device__ __forceinline__ void numerators(const uint32_t* y, uint32_t* e, unsigned long long& far) const
    {
        uint32_t redo[P], any = 0u;
#pragma unroll
        for (int i = 0; i < P; ++i) {
            redo[i] = never;
            e[i]    = (*this)(y[i], redo[i]);
            any |= redo[i];
        }
        if (__builtin_expect(__ballot(undecided(any)) != 0ull, 0)) {
            if constexpr (DT == DT_BF16) {
                typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
                u16x2                  least = {0x7FFF, 0x7FFF};
#pragma unroll
                for (int i = 0; i < P; ++i) {
                    least = __builtin_elementwise_min(least, __builtin_bit_cast(u16x2, e[i] & 0x7FFF7FFFu));
                }
                far |= __ballot(min(least.x, least.y) < FAR);
            }
            redone<P>(y, e, redo, false);
        }
    }
    // the same with the wide bounds
    template<int P>
    __device__ __forceinline__ void wide_numerators(const uint32_t* y, uint32_t* e) const
    {
        uint32_t redo[P], any = 0u;
#pragma unroll
        for (int i = 0; i < P; ++i) {
            redo[i] = never;
            e[i]    = wide(y[i], redo[i]);
            any |= redo[i];
        }
        if (__ballot(undecided(any, true)) != 0ull) {
            redone<P>(y, e, redo, true);
        }
    }
    // e of the pairs that are not decided, by det_expf
    template<int P>
    __device__ __forceinline__ void redone(const uint32_t* y, uint32_t* e, const uint32_t* redo, bool of_wide) const
    {
#pragma unroll
        for (int i = 0; i < P; ++i) {
            if (__ballot(undecided(redo[i], of_wide)) != 0ull) {
                e[i] = exact(y[i]);
            }
        }
    }
    // sum + the first / second value of a pair, rounded once
    __device__ __forceinline__ float add_low(float sum, uint32_t e) const
    {
        return fma_rn(low(e), one, sum);
    }
    __device__ __forceinline__ float add_high(float sum, uint32_t e) const
    {
        return fma_rn(high(e), one, sum);
    }
    // y times a T, rounded to T
    static __device__ __forceinline__ uint32_t times(uint32_t y, float by)
    {
        if constexpr (DT == DT_F16) {
            const _Float16 m = (_Float16)by;
            const f16x2    v = {m, m};
            return __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, y) * v);
        }
        else {
            return pack(low(y) * by, high(y) * by);
        }
    }
};

}  // namespace ftk
