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
    // t carries 16 more than the argument: where most columns of a row lie (e^-11 and around it) t is then small and
    // its rounding finer.
    static constexpr float SHIFT = 16.0f, UNSHIFT = 1.52587890625e-05f;
    // How far det_expf can lie above / below the hardware's value: a share of it and an absolute part, which takes over
    // far from the maximum, where the rounding of y - max in det_expf's argument counts. Largest distances over every
    // pair of values y <= max of the type: binary16 7.8e-7 / 9.2e-7 down to 2^-20 and 1.3e-6 / 1.7e-6 down to 2^-32,
    // bfloat16 1.2e-6 / 1.7e-6 down to 2^-32; the factors' own rounding comes on top (a test goes through all pairs).
    // Wider bounds cost time, not bits: more pairs are evaluated twice.
    static constexpr float UP    = DT == DT_F16 ? 1.0e-6f : 1.4e-6f;
    static constexpr float DOWN  = DT == DT_F16 ? 1.1e-6f : 1.9e-6f;
    static constexpr float FLOOR = DT == DT_F16 ? 8.0e-13f : 1.5e-16f;  // (bfloat16: also what the hardware flushes)
    float    max;
    float    c, hi, lo, one;
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
        hi                  = uniform_f(scale * (1.0f + UP));
        lo                  = uniform_f(scale * (1.0f - DOWN));
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
    // whether what the calls above collected asks for det_expf (binary16: below zero the lower end rounds to -0)
    static __device__ __forceinline__ bool undecided(uint32_t redo)
    {
        return DT == DT_F16 ? (redo & 0x7FFF7FFFu) != 0u : redo != 0u;
    }
    // the same by det_expf
    __device__ __forceinline__ uint32_t exact(uint32_t y) const
    {
        return pack(det_expf_nonpos(low(y) - max), det_expf_nonpos(high(y) - max));
    }
    // e of P pairs, exactly: all of them in a straight line, then one look for pairs that are not decided, in a branch that
    // the whole wave takes, and a closer one at two pairs each.
    template<int P>
    __device__ __forceinline__ void numerators(const uint32_t* y, uint32_t* e) const
    {
        static_assert(P % 2 == 0, "two pairs at a time");
        uint32_t redo[P / 2], any = 0u;
#pragma unroll
        for (int i = 0; i < P / 2; ++i) {
            redo[i]      = never;
            e[2 * i]     = (*this)(y[2 * i], redo[i]);
            e[2 * i + 1] = (*this)(y[2 * i + 1], redo[i]);
            any |= redo[i];
        }
        if (__builtin_expect(__ballot(undecided(any)) != 0ull, 0)) {
#pragma unroll
            for (int i = 0; i < P / 2; ++i) {
                if (DT == DT_BF16 && never == 0u) {
                    // masked columns: -inf has e = 0, whatever the absolute part of the bounds says
                    const uint32_t a = infinite(y[2 * i]), b = infinite(y[2 * i + 1]);
                    e[2 * i] &= ~a;
                    e[2 * i + 1] &= ~b;
                    redo[i] &= ~(a & b);
                }
                if (__ballot(undecided(redo[i])) != 0ull) {
                    e[2 * i]     = exact(y[2 * i]);
                    e[2 * i + 1] = exact(y[2 * i + 1]);
                }
            }
        }
    }
    // all ones in the halves that are -inf
    static __device__ __forceinline__ uint32_t infinite(uint32_t y)
    {
        const uint32_t x = Storage<DT>::st(-__builtin_inff());
        return ((y & 0xFFFFu) == x ? 0xFFFFu : 0u) | ((y >> 16) == x ? 0xFFFF0000u : 0u);
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
    static __device__ __forceinline__ uint32_t scale(uint32_t y, float by)
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
