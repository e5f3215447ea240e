// The tiles that fit the chip (hipq_igemm_ring.h) for what hipq_igemm_ring.hip does not take: any number of output channels, any
// multiple of 16 input channels, outputs of either layout.
//
// What these calls spent their time on before: the kernels that take their fragments straight from memory take half of every
// cache line, and are bound by what a compute unit takes in; the ones that stage through registers wait for each slice, and
// write ragged columns a byte at a time.  Here the operands come as in the other tiles; a lane's chunk of a
// window has a cursor of its own (a slice may lie across taps), and rows leave 16 bytes a lane at whatever address
// they have, the last columns of an odd width by dword and byte.  [image][channel][pixel] outputs: a 4 x 4 byte transposition
// inside each quad of lanes, then four pixels a store.  No count of stores is sure, so a tile's first wait is for all of the
// tile before.  Figures and limits at ring_any_preferred; what is left above the floor is the slice's intake (an
// unaligned 128-byte slice of a pixel is two lines) and the epilogue.
#include "hipq_igemm_ring.h"

namespace hipq
{
    namespace
    {
        // (as kRingQ8 ...; over 95 sizes the tile picked is 1.1 % slower than the best one)
        constexpr RingTile kAny[] = {{128, 128, 0.45f, 3.0f}, {64, 128, 0.335f, 2.0f}, {64, 64, 0.29f, 1.2f}, {256, 64, 0.56f, 2.8f}};

        template <class XL, int MODE, bool HAS_SUM, int KIND>
        int launch_any(const XL& xl, const int8_t* w, const int32_t* wsum, int64_t M, int32_t N, int32_t Kred, int x_unsigned, const ZeroPoints& zp, const Epilogue& epi, const RingMap& map, void* out,
                       hipStream_t s, const char* name)
        {
#define RING(WM_, WN_, A_, B_, NB_) launch_ring_tile<XL, WM_, WN_, A_, B_, NB_, MODE, HAS_SUM, KIND, true>(xl, w, wsum, M, N, Kred, x_unsigned, zp, epi, map, out, s, name)
            switch (ring_choose(kAny, M, N, Kred))
            {
            case 0: return RING(4, 2, 2, 4, 4);
            case 1: return RING(4, 2, 1, 4, 6);
            case 2: return RING(4, 2, 1, 2, 8);
            case 3: return RING(8, 1, 2, 4, 3);
            default: return HIPQ_ERR_UNSUPPORTED;
            }
#undef RING
        }

        template <class XL>
        int launch_any_of(const XL& xl, const int8_t* w, const int32_t* wsum, int64_t M, int32_t N, int32_t Kred, int x_unsigned, const ZeroPoints& zp, const Epilogue& epi, const RingMap& map, void* out,
                          hipStream_t s, const char* name)
        {
            const bool q8 = epi.out_t == HIPQ_U8 || epi.out_t == HIPQ_I8;
            if (N > (1 << 20) || Kred >= 65536 || epi.post_scale)
                return HIPQ_ERR_UNSUPPORTED;
            if (epi.mode == EPI_INTERP)
            {
                if (epi.sum_in)
                    return HIPQ_ERR_UNSUPPORTED;
                if (q8)
                    return launch_any<XL, EPI_INTERP, false, OUT_Q8>(xl, w, wsum, M, N, Kred, x_unsigned, zp, epi, map, out, s, name);
                return epi.out_t == HIPQ_I32 ? launch_any<XL, EPI_INTERP, false, OUT_I32>(xl, w, wsum, M, N, Kred, x_unsigned, zp, epi, map, out, s, name) : HIPQ_ERR_UNSUPPORTED;
            }
            if (q8)
                return epi.sum_in ? launch_any<XL, EPI_FUSED, true, OUT_Q8>(xl, w, wsum, M, N, Kred, x_unsigned, zp, epi, map, out, s, name)
                                  : launch_any<XL, EPI_FUSED, false, OUT_Q8>(xl, w, wsum, M, N, Kred, x_unsigned, zp, epi, map, out, s, name);
            if constexpr (!XL::kConv)
                if (epi.out_t == HIPQ_F32 && !epi.sum_in && !map.ncx)
                    return launch_any<XL, EPI_FUSED, false, OUT_F32>(xl, w, wsum, M, N, Kred, x_unsigned, zp, epi, map, out, s, name);
            return HIPQ_ERR_UNSUPPORTED;
        }
    }

    int launch_rows_ring_any(const void* a, int a_unsigned, const int8_t* w, const int32_t* wsum, int64_t M, int32_t N, int32_t K, const ZeroPoints& zp, const Epilogue& epi, void* out, hipStream_t s,
                             const char* name)
    {
        return launch_any_of(RingRows{static_cast<const uint8_t*>(a), static_cast<uint32_t>(M * K), K}, w, wsum, M, N, K, a_unsigned, zp, epi, RingMap{}, out, s, name);
    }

    int launch_conv_ring_any(const ConvX& cx, const int8_t* w, const int32_t* wsum, int64_t M, int32_t N, int32_t K, int x_unsigned, const ZeroPoints& zp, const Epilogue& epi, bool ncx, void* out,
                             hipStream_t s, const char* name)
    {
        if (cx.R * cx.S > 32 || M >= (1ll << 31) - 1024)
            return HIPQ_ERR_UNSUPPORTED;
        const RingMap map{ncx ? 1 : 0, static_cast<int32_t>(cx.PQ), cx.by_pq};
        if (cx.every_pixel())
            return launch_any_of(RingRows{cx.x, cx.bytes, cx.C}, w, wsum, M, N, K, x_unsigned, zp, epi, map, out, s, name);
        RingConvAny xl;
        static_cast<RingWindow&>(xl) = ring_window(cx);
        xl.by_c = cx.by_c;
        xl.by_s = cx.by_s;
        xl.taps = SL / cx.C;
        xl.cols = xl.taps % cx.S;
        xl.rest = SL % cx.C;
        xl.step = xl.taps / cx.S * cx.dh * cx.W * cx.C + xl.cols * cx.dw * cx.C + xl.rest;
        xl.tap_step = cx.dw * cx.C - cx.C;
        xl.row_step = cx.dh * cx.W * cx.C - cx.S * cx.dw * cx.C;
        return launch_any_of(xl, w, wsum, M, N, K, x_unsigned, zp, epi, map, out, s, name);
    }
}
