// Quantize(Gelu(x)) of four elements, for the kernels that apply both to what they have just computed or read: the
// bytes of the two ops one after the other (gelu1, then quantize4 / quantize_one), at about half their instructions.
#pragma once
#include "hipq_quant_math.h"
#include "hipq_row_math.h"

namespace hipq
{
    // A byte needs gelu(x) / scale only to the nearest integer.  gelu(x) = max(x, 0) - |x| phi(-|x|) (phi: the normal
    // distribution), and phi(-a) is 2 to a polynomial of degree 7 in a (least squares on log2 phi, weighted by what an error
    // there does to the product and reweighted to the smallest largest error: 7.3e-8, the leading coefficient held below
    // zero so that it falls for good beyond the range that counts).  The difference from gelu1, mostly gelu1's own
    // roundings, is at most 2.4e-7 + 1.8e-7 |gelu(x)| (the largest seen when it was fitted; the bytes that rest on it are held
    // next to every rounding step and for every 127th float by tests/test_gelu_quantize.py).  Where the quotient lies
    // further from every half than what that and the roundings of reciprocal, product and division amount to, both
    // round to the same integer; the other elements (about one in 15 000 at a scale of 0.0175: each holds up its
    // workgroup for 0.8 us), a NaN or an infinity are computed as the ops do.
    // erff's two branches, the division and their fix-ups are about 60 instructions an element; these 18, one of them an
    // exponential, which still bound the epilogue: a SIMD starts one in 2.2 cycles.  Projection 4096 x 768 x 3072 with Gelu
    // and Quantize in its epilogue: 31.8 us with the ops' own arithmetic, 22.7 so (128 x 192 tiles in both: 26.1).
    // the difference from gelu1: at most kGeluAbsolute + 1.8e-7 |gelu(x)|; reciprocal, product and division round once each
    constexpr float kGeluAbsolute = 3.0e-7f, kGeluRelative = 1.8e-7f + 2.5e-7f;
    struct GeluQuantize
    {
        float scale, zp;
        float r, zz;  // reciprocal of the scale, zero point (128 more for signed bytes)
        float limit;  // distance from the nearest integer up to which the fast result is the ops'; negative: never
        int32_t zp_i, quant_t, mode;
    };
    __device__ __forceinline__ GeluQuantize gelu_quantize_of(float scale, int32_t zp, int32_t quant_t, int32_t mode)
    {
        GeluQuantize q;
        q.scale = scale;
        q.zp = static_cast<float>(zp);
        q.zp_i = zp;
        q.quant_t = quant_t;
        q.mode = mode;
        float r = __builtin_amdgcn_rcpf(scale);
        r = __builtin_fmaf(__builtin_fmaf(-scale, r, 1.0f), r, r);
        q.r = r;
        q.zz = quant_t == HIPQ_U8 ? q.zp : q.zp + 128.0f;
        const float a = __builtin_fabsf(scale);
        const bool plain = mode == HIPQ_ROUND_NEAREST_TOWARD_EVEN && __builtin_amdgcn_fmed3f(a, 9.31322574615478515625e-10f, 1073741824.0f) == a;
        q.limit = plain ? 0.5f - (kGeluAbsolute * __builtin_fabsf(r) + kGeluRelative) : -1.0f;
        return q;
    }

    // gelu(x) to the bound above; NaN where x is an infinity or a NaN
    template <int COUNT>
    __device__ __forceinline__ void gelu_near(const float (&x)[COUNT], float (&g)[COUNT])
    {
        constexpr float c[8] = {-9.99990471e-01f, -1.1512332f, -4.58648141e-01f, -5.36282689e-02f, 8.27510651e-03f, -8.61299051e-04f, 5.48178113e-05f, -2.0e-06f};
        // (side by side: one chain of dependent multiply-adds would wait for itself)
#pragma unroll
        for (int e = 0; e < COUNT; ++e)
            g[e] = __builtin_fmaf(c[7], __builtin_fabsf(x[e]), c[6]);
#pragma unroll
        for (int k = 5; k >= 0; --k)
#pragma unroll
            for (int e = 0; e < COUNT; ++e)
                g[e] = __builtin_fmaf(g[e], __builtin_fabsf(x[e]), c[k]);
#pragma unroll
        for (int e = 0; e < COUNT; ++e)
            g[e] = __builtin_fmaf(-__builtin_fabsf(x[e]), __builtin_amdgcn_exp2f(g[e]), __builtin_fmaxf(x[e], 0.0f));
    }

    // byte e of `packed` (signed ones still to be flipped), and whether it is the ops'
    __device__ __forceinline__ void gelu_byte(float g, const GeluQuantize& q, int e, uint32_t* packed, bool* sure)
    {
        const float v = __fmul_rn(g, q.r);
        const float t = __builtin_rintf(v);
        *sure = __builtin_fmaf(__builtin_fabsf(t), kGeluRelative, __builtin_fabsf(__fsub_rn(v, t))) < q.limit;
        *packed = __builtin_amdgcn_cvt_pk_u8_f32(__fadd_rn(t, q.zz), e, *packed); // saturates to 0..255 and packs
    }

    __device__ __forceinline__ uint32_t gelu_quantize4(f32x4 x, const GeluQuantize& q)
    {
        const bool is_signed = q.quant_t != HIPQ_U8; // uniform
        uint32_t packed = 0;
        bool sure[4];
        const float xs[4] = {x[0], x[1], x[2], x[3]};
        float g[4];
        gelu_near(xs, g);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            gelu_byte(g[e], q, e, &packed, &sure[e]);
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
                const float exact = gelu1(k == 0 ? x[0] : k == 1 ? x[1] : k == 2 ? x[2] : x[3]);
                uint32_t byte;
                if (q.mode == HIPQ_ROUND_NEAREST_TOWARD_EVEN) // uniform; as quantize4
                {
                    const float lo = is_signed ? -128.0f : 0.0f, hi = is_signed ? 127.0f : 255.0f;
                    float v = __fadd_rn(rintf(__fdiv_rn(exact, q.scale)), q.zp);
                    v = (v < lo) ? lo : v;
                    v = (hi < v) ? hi : v;
                    byte = static_cast<uint32_t>(static_cast<int32_t>(v)) & 0xFFu;
                }
                else if (is_signed)
                    byte = static_cast<uint32_t>(static_cast<uint8_t>(quantize_one<float, int8_t>(exact, q.scale, static_cast<int8_t>(q.zp_i), q.mode)));
                else
                    byte = static_cast<uint32_t>(quantize_one<float, uint8_t>(exact, q.scale, static_cast<uint8_t>(q.zp_i), q.mode));
                packed = (packed & ~(0xFFu << (8 * k))) | (byte << (8 * k));
            }
        }
        return packed;
    }
}
