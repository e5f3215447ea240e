// Row reductions over groups of lanes and the Softmax arithmetic of one row piece, shared by the
// Softmax kernels and by the attention kernel that applies Softmax to scores it has just computed:
// both must round alike, sums included, so both call these.
#pragma once
#include <cmath>

#include "hipq_common.h"

namespace hipq
{
    typedef float row_f4 __attribute__((ext_vector_type(4)));

    // Reductions over aligned groups of W lanes of a wavefront: a butterfly whose distance halves from W / 2
    // down, every lane ending with the result.  Data-parallel-primitive moves and the half-wavefront swaps
    // instead of shuffles: a shuffle goes through LDS, and the six of a row in sequence are what a short row
    // waits for (LayerNorm of 128 rows of 768: 4.37 us with shuffles, 4.11 so; Softmax of 7880 rows of 197,
    // with its single pass over unaligned rows: 7.30, 6.10).
    template <int CTRL>
    __device__ __forceinline__ float dpp_move(float v)
    {
        const int x = __builtin_bit_cast(int, v);
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(x, x, CTRL, 0xf, 0xf, false));
    }
    template <int W, typename F>
    __device__ __forceinline__ float butterfly(float v, F combine)
    {
        // distances 32 and 16: v_permlane*_swap of two copies leaves the lower halves in one register and the
        // upper ones in the other (the two wait states are the ones a freshly written operand needs)
        if (W >= 64)
        {
            float a = v, b = v;
            asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
            v = combine(a, b);
        }
        if (W >= 32)
        {
            float a = v, b = v;
            asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
            v = combine(a, b);
        }
        // distance 8: a rotation within 16 lanes; 4: the same, since what the lanes hold has period 8 by then. In
        // groups of 8 a mirror of eight lanes and one of four
        if (W >= 16)
        {
            v = combine(v, dpp_move<0x128>(v)); // row_ror:8
            v = combine(v, dpp_move<0x124>(v)); // row_ror:4
        }
        else if (W == 8)
            v = combine(v, dpp_move<0x1b>(dpp_move<0x141>(v))); // row_half_mirror (l ^ 7), then quad_perm:[3,2,1,0] (l ^ 3)
        if (W >= 4)
            v = combine(v, dpp_move<0x4e>(v)); // quad_perm:[2,3,0,1]
        return combine(v, dpp_move<0xb1>(v));  // quad_perm:[1,0,3,2]
    }
    template <int W = 64>
    __device__ __forceinline__ float wave_max(float v)
    {
        return butterfly<W>(v, [](float a, float b) { return fmaxf(a, b); });
    }
    template <int W = 64>
    __device__ __forceinline__ float wave_sum(float v)
    {
        return butterfly<W>(v, [](float a, float b) { return a + b; });
    }

    // a / b rounded as the division rounds it, from r = fl(1 / b): q0 = a r, e = a - b q0 (exact in a fused
    // multiply-add), q = q0 + e r -- three instructions where the division sequence takes eleven.
    // (Markstein's correction: with a correctly rounded reciprocal the result is the correctly rounded
    // quotient as long as nothing overflows or goes subnormal; checked on the CPU against the division
    // for all 2^23 mantissas of a with b = float(sqrt(2)), and for 2 x 10^8 random pairs.)  Callers keep
    // infinities and zero divisors away from it.
    __device__ __forceinline__ float div_by_reciprocal(float a, float b, float r)
    {
        const float q0 = __fmul_rn(a, r);
        return fmaf(fmaf(-b, q0, a), r, q0);
    }

    // Softmax of a row held in 16-byte pieces by W neighbouring lanes, lane l pieces l, l + W, ..
    // (src/ngraph/runtime/reference/softmax.hpp:31-57): exp(x - max) / sum(exp(x - max)); with `scaled`
    // the input is Multiply(x, c), the product rounded to f32 as the Multiply op rounds it.  `live` of the
    // row's elements exist (the others come out as zero, or NaN in a row that is NaN throughout).  The sum is
    // the one that 64 lanes get, whatever W is: of rows in whole pieces (and of any with W = 64) lane l sums
    // pieces l, l + 64, .., of other rows elements l, l + 64, .., and the butterfly of wave_sum adds the 64 sums.
    // So a row's result does not depend on the kernel that takes it; the longer way costs nothing seen
    // (a pass of an encoder of 4 layers, 8 heads on 5 x 197 tokens 310 us before, 308 so).
    template <int W, int P>
    __device__ __forceinline__ void softmax_row(row_f4 (&v)[P], int lane, int live, bool scaled, float c)
    {
        float m = -INFINITY;
#pragma unroll
        for (int i = 0; i < P; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
            {
                const float x = scaled ? __fmul_rn(v[i][e], c) : v[i][e];
                v[i][e] = 4 * (W * i + lane) + e < live ? x : -INFINITY;
                m = fmaxf(m, v[i][e]);
            }
        m = wave_max<W>(m);
#pragma unroll
        for (int i = 0; i < P; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                v[i][e] = expf(v[i][e] - m);
        float s;
        if (W == 64 || (live & 3) == 0) // (the lanes of a row agree)
        {
            float even = 0.0f, odd = 0.0f; // W == 32: pieces l, l + 64, .. and l + 32, l + 96, ..
#pragma unroll
            for (int i = 0; i < P; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    (W == 32 && (i & 1) ? odd : even) += v[i][e];
            s = wave_sum<W>(W == 32 ? even + odd : even);
        }
        else
        {
            float t[4] = {0.0f, 0.0f, 0.0f, 0.0f}; // elements 4 l + e (mod 64), in order
#pragma unroll
            for (int i = 0; i < P; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                {
                    float lower = v[i][e], upper = v[i][e];
                    if (W == 32)
                    {
                        asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(lower), "+v"(upper));
                        t[e] = (t[e] + lower) + upper;
                    }
                    else
                        t[e] += lower;
                }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                t[e] = wave_sum<(W < 16 ? W : 16)>(t[e]);
            s = (t[0] + t[2]) + (t[1] + t[3]);
        }
        // The divisions through one reciprocal a row where that gives the division's own result: the sum is 1 to the row's
        // length (a row with an infinity or a NaN has none), and a remainder is exact while the dividend is zero or not
        // below 2^-100.  (Zero less one is the largest unsigned number.)  An element is five instructions instead of the
        // division's eleven, three of them slow: attention of 36 heads of 384 x 384 40.7 -> 39.3 us, of 40 of 197 x 197 20.6 -> 20.3, of 384
        // of 128 x 128 38.7 -> 38.1; of a whole encoder that is 0.2 to 0.4 %.
        uint32_t least = 0xffffffffu;
#pragma unroll
        for (int i = 0; i < P; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                least = min(least, __float_as_uint(v[i][e]) - 1u);
        if (__all(least >= 0x0d800000u - 1u && s < 65536.0f)) // uniform
        {
            const float r = __fdiv_rn(1.0f, s);
#pragma unroll
            for (int i = 0; i < P; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[i][e] = div_by_reciprocal(v[i][e], s, r);
        }
        else
        {
#pragma unroll
            for (int i = 0; i < P; ++i)
                v[i] = row_f4{v[i][0] / s, v[i][1] / s, v[i][2] / s, v[i][3] / s};
        }
    }

    // Gelu as the reference decomposes it (src/ngraph/op/gelu.cpp:46-60):
    // (0.5 * x) * (1 + erf(x / float(sqrt(2.0)))), every step rounded to f32.  Shared by the Gelu
    // kernel and by the GEMM epilogue that applies Gelu to what it has just computed.
    __device__ __forceinline__ float gelu1(float x)
    {
        const float sqrt_two = 1.41421354f; // float(std::sqrt(2.0))
        const float r = 0.70710677f;        // fl(1 / sqrt_two)
        // x / sqrt_two, bit for bit; an infinite x stays itself, and where the quotient would be
        // subnormal erf's argument is so small that 1 + erf is 1 either way
        const float t = __builtin_isinf(x) ? x : div_by_reciprocal(x, sqrt_two, r);
        return __fmul_rn(__fmul_rn(0.5f, x), __fadd_rn(1.0f, erff(t)));
    }

}
