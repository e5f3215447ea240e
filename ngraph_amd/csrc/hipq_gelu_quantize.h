// Quantize(Gelu(x)) of four elements, for the kernels that apply both to what they have just computed or read: the
// bytes of the two ops one after the other (gelu1, then quantize4 / quantize_one), at about half their instructions.
#pragma once
#include "hipq_quant_math.h"
#include "hipq_row_math.h"

namespace hipq
{
    // A byte needs gelu(x) / scale only to the nearest integer.  gelu(x) = max(x, 0) - |x| phi(-|x|) (phi: the normal
    // distribution), and |x| phi(-|x|) is a polynomial of degree 14 in |x| on [0, 5.2] to 5.4e-7 (least squares at Chebyshev
    // nodes, reweighted to the smallest largest error; in u = |x| / 2.6 - 1, where its f32 evaluation is well conditioned) and stays below
    // that from there on.  The difference from gelu1 is at most 9.6e-7 (every float up to 64 in magnitude tried on the device; beyond,
    // both are x or within the bound of 0).  Where the quotient lies further from every half than what that and
    // the roundings of reciprocal, product and division amount to, both round to the same integer; the other elements
    // (one group of 64 x 4 in 23 has one at a scale of 0.0175), a NaN or an infinity are computed as the ops do.
    // erff's two branches, the division and their fix-ups are about 60 instructions an element; these 24, which still bound the epilogue: a
    // SIMD starts one in 2.2 cycles, 12.6 M elements are 8 us.  Projection 4096 x 768 x 3072 with Gelu and Quantize in its
    // epilogue: 31.8 -> 26.3 us (2048 x 1024 x 4096 23.6 -> 19.8, 985 x 512 x 2048 10.4 -> 8.1).
    struct GeluQuantize
    {
        float scale, zp;
        float far;    // from here on the polynomial's last value
        float r, zz;  // reciprocal of the scale, zero point (128 more for signed bytes)
        float limit;  // distance from the nearest integer up to which the fast result is the ops'; negative: never
        int32_t zp_i, quant_t, mode;
    };
    __device__ __forceinline__ GeluQuantize gelu_quantize_of(float scale, int32_t zp, int32_t quant_t, int32_t mode)
    {
        GeluQuantize q;
        q.scale = scale;
        q.far = 5.2f;
        q.zp = static_cast<float>(zp);
        q.zp_i = zp;
        q.quant_t = quant_t;
        q.mode = mode;
        float r = __builtin_amdgcn_rcpf(scale);
        r = __builtin_fmaf(__builtin_fmaf(-scale, r, 1.0f), r, r);
        q.r = r;
        q.zz = quant_t == HIPQ_U8 ? q.zp : q.zp + 128.0f;
        // quotients that do not saturate are at most `reach` in magnitude; reciprocal, product and division round once each
        const float reach = quant_t == HIPQ_U8 ? fmaxf(q.zp, 255.0f - q.zp) + 1.0f : fmaxf(q.zp + 128.0f, 127.0f - q.zp) + 1.0f;
        const float a = __builtin_fabsf(scale);
        const bool plain = mode == HIPQ_ROUND_NEAREST_TOWARD_EVEN && __builtin_amdgcn_fmed3f(a, 9.31322574615478515625e-10f, 1073741824.0f) == a;
        q.limit = plain ? 0.5f - (1.0e-6f * __builtin_fabsf(r) + 3.0e-7f * reach) : -1.0f;
        return q;
    }

    __device__ __forceinline__ uint32_t gelu_quantize4(f32x4 x, const GeluQuantize& q)
    {
        const bool is_signed = q.quant_t != HIPQ_U8; // uniform
        constexpr float c[15] = {0.0121195605f,  -0.0796987563f, 0.218476549f,   -0.285643339f, 0.0626382008f,  0.374073148f,   -0.565343797f, 0.214285165f,
                                 0.307422817f, -0.367647082f,  0.00617902679f, 0.17760843f,   -0.0571440049f, -0.0329778343f, 0.0156519208f};
        uint32_t packed = 0;
        bool sure[4];
        // (the four side by side: one chain of dependent multiply-adds would wait for itself)
        float u[4], p[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
        {
            asm("v_min_f32 %0, |%1|, %2" : "=v"(u[e]) : "v"(x[e]), "v"(q.far));
            u[e] = __builtin_fmaf(u[e], 1.0f / 2.6f, -1.0f);
            p[e] = c[14];
        }
#pragma unroll
        for (int k = 13; k >= 0; --k)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                p[e] = __builtin_fmaf(p[e], u[e], c[k]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
        {
            // (x + |x| is infinite or NaN where x is an infinity of either sign or a NaN: not sure)
            const float v = __fmul_rn(__builtin_fmaf(0.5f, __fadd_rn(x[e], __builtin_fabsf(x[e])), -p[e]), q.r);
            const float t = __builtin_rintf(v);
            sure[e] = __builtin_fabsf(__fsub_rn(v, t)) < q.limit;
            packed = __builtin_amdgcn_cvt_pk_u8_f32(__fadd_rn(t, q.zz), e, packed); // saturates to 0..255 and packs
        }
        packed ^= is_signed ? 0x80808080u : 0u;
        if (!__builtin_expect(__all(sure[0] & sure[1] & sure[2] & sure[3]), 1))
        {
            // (an element at a time, as a rule one: a chain of 150 instructions each, the same ones for all)
            const uint64_t doubt[4] = {__ballot(!sure[0]), __ballot(!sure[1]), __ballot(!sure[2]), __ballot(!sure[3])};
#pragma unroll 1
            for (int k = 0; k < 4; ++k)
            {
                if ((k == 0 ? doubt[0] : k == 1 ? doubt[1] : k == 2 ? doubt[2] : doubt[3]) == 0) // uniform
                    continue;
                const float g = gelu1(k == 0 ? x[0] : k == 1 ? x[1] : k == 2 ? x[2] : x[3]);
                uint32_t byte;
                if (q.mode == HIPQ_ROUND_NEAREST_TOWARD_EVEN) // uniform; as quantize4
                {
                    const float lo = is_signed ? -128.0f : 0.0f, hi = is_signed ? 127.0f : 255.0f;
                    float v = __fadd_rn(rintf(__fdiv_rn(g, q.scale)), q.zp);
                    v = (v < lo) ? lo : v;
                    v = (hi < v) ? hi : v;
                    byte = static_cast<uint32_t>(static_cast<int32_t>(v)) & 0xFFu;
                }
                else if (is_signed)
                    byte = static_cast<uint32_t>(static_cast<uint8_t>(quantize_one<float, int8_t>(g, q.scale, static_cast<int8_t>(q.zp_i), q.mode)));
                else
                    byte = static_cast<uint32_t>(quantize_one<float, uint8_t>(g, q.scale, static_cast<uint8_t>(q.zp_i), q.mode));
                packed = (packed & ~(0xFFu << (8 * k))) | (byte << (8 * k));
            }
        }
        return packed;
    }
}
