// The tiles that fit the chip (hipq_igemm_ring.h) for outputs in whole 16-byte pieces, and the rule that gives calls to them.
#include "hipq_igemm_ring.h"

namespace hipq
{
    namespace
    {
        // The tiles of each kind of call, with what a slice and a round (first fragments, epilogue, stores) cost: a call
        // takes about 2.6 us and, for each tile a compute unit has in turn, slices x slice + round (us; least squares over
        // 3 600 timings of 330 sizes, 5 % off on average, so that the tile picked is 1 % slower than the best one).  What
        // bounds a slice: 128 x 256 tiles the matrix cores (1024 cycles of 1414 at the 1.95 GHz that random bytes leave
        // them), the small ones what a compute unit takes in (16 KB in 0.25 us).  The rings are as deep as the LDS
        // allows: looped on its own a layer finds its operands in the L2s and does as well with two slices, behind
        // other layers it does not (256 -> 256 channels 3 x 3 on 128 x 14 x 14 pixels inside ResNet-50: 28.0 us with two, 24.0
        // with three; the register- or line-limited kernels before these 28.9).
        constexpr RingTile kRingQ8[] = {{128, 256, 0.77f, 2.2f}, {256, 128, 0.80f, 3.0f}, {128, 128, 0.435f, 2.0f}, {64, 128, 0.321f, 1.2f}, {64, 64, 0.273f, 0.77f}, {256, 64, 0.55f, 1.8f}};
        constexpr RingTile kRingSum[] = {{128, 256, 0.795f, 3.29f}, {256, 128, 0.85f, 3.8f}, {128, 128, 0.461f, 2.62f}, {64, 128, 0.335f, 1.93f}};
        constexpr RingTile kRingInterp[] = {{128, 256, 0.77f, 2.4f}, {256, 128, 0.80f, 3.2f}, {128, 128, 0.435f, 2.2f}, {64, 128, 0.321f, 1.3f}};
        constexpr RingTile kRingF32[] = {{256, 144, 0.873f, 6.2f}, {256, 192, 0.989f, 7.6f}, {128, 192, 0.589f, 5.1f}, {128, 128, 0.408f, 3.4f},
                                         {128, 96, 0.390f, 2.9f},  {64, 128, 0.294f, 2.4f},  {64, 96, 0.293f, 2.1f},   {64, 64, 0.251f, 1.7f}};
        // Gelu and Quantize: a third of a tile's time or more is its epilogue, vector work that two workgroups a compute unit
        // overlap with each other's products where the tiles come in pairs (128 x 128 alone 4.6 us a tile beyond its
        // slices, two together 6.4), and fewer, larger tiles spend on fewer rounds (4096 x 768 x 3072: 128 x 192 in two
        // rounds 26.1 us, 256 x 192 in one 22.7; 2048 x 1024 x 4096: 128 x 256 18.5, 128 x 128 in pairs 17.6; fitted to 90 sizes,
        // the tile picked is 0.8 % slower than the best one).  The other kinds gain in a loop and lose behind other layers,
        // where two buffers are too few (256 x 192 for 256 -> 512 channels 3 x 3 on 128 x 56 x 56 pixels 36.8 -> 41.4 us in
        // ResNet-50, pairs for 512 -> 256 36.5 -> 39.8).
        constexpr RingTile kRingGelu[] = {{128, 256, 0.783f, 7.77f}, {128, 192, 0.635f, 6.10f}, {128, 128, 0.507f, 4.15f}, {64, 128, 0.380f, 2.38f},
                                          {256, 192, 1.033f, 10.58f}, {128, 128, 0.513f, 4.63f, 1.084f, 6.39f}, {128, 96, 0.477f, 4.03f, 0.928f, 4.87f}};

        template <class XL>
        int launch_ring(const XL& xl, const int8_t* w, const int32_t* wsum, int64_t M, int32_t N, int32_t Kred, int x_unsigned, const ZeroPoints& zp, const Epilogue& epi, void* out, hipStream_t s,
                        const char* name)
        {
            const bool q8 = epi.out_t == HIPQ_U8 || epi.out_t == HIPQ_I8;
            const bool f32 = epi.out_t == HIPQ_F32 && epi.mode == EPI_FUSED && epi.sum_in == nullptr && !XL::kConv;
            auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
            // (offsets inside a tile of rows are 32 bits, wsum fits 24)
            // (residuals over two or three slices and more than one round: 256 -> 1024 channels on 128 x 14 x 14 pixels 24.0 us here,
            // 22.5 on the kernel that has three workgroups a compute unit; 512 -> 2048 on 7 x 7 18.9 and 21.7)
            if (epi.sum_in != nullptr && Kred < 4 * SL && getenv("HIPQ_RING_TILE") == nullptr && ((M + 63) / 64) * ((N + 127) / 128) > 2 * device_compute_units())
                return HIPQ_ERR_UNSUPPORTED;
            if ((!q8 && !f32) || N % 16 != 0 || N > (1 << 20) || Kred < 2 * SL || Kred >= 65536 || !aligned(out) || !aligned(epi.sum_in))
                return HIPQ_ERR_UNSUPPORTED;
#define RING2(WM_, WN_, A_, B_, NB_, MODE_, SUM_, KIND_) launch_ring_tile<XL, WM_, WN_, A_, B_, NB_, MODE_, SUM_, KIND_, false, 2>(xl, w, wsum, M, N, Kred, x_unsigned, zp, epi, RingMap{}, out, s, name)
#define RING(WM_, WN_, A_, B_, NB_, MODE_, SUM_, KIND_) launch_ring_tile<XL, WM_, WN_, A_, B_, NB_, MODE_, SUM_, KIND_>(xl, w, wsum, M, N, Kred, x_unsigned, zp, epi, RingMap{}, out, s, name)
            if constexpr (!XL::kConv)
            {
                if (f32 && epi.post_scale)
                    switch (ring_choose(kRingGelu, M, N, Kred))
                    {
                    case 0: return RING(2, 4, 4, 4, 3, EPI_FUSED, false, OUT_GELU_Q8);
                    case 1: return RING(2, 4, 4, 3, 3, EPI_FUSED, false, OUT_GELU_Q8);
                    case 2: return RING(4, 2, 2, 4, 4, EPI_FUSED, false, OUT_GELU_Q8);
                    case 3: return RING(4, 2, 1, 4, 6, EPI_FUSED, false, OUT_GELU_Q8);
                    case 4: return RING(4, 2, 4, 6, 2, EPI_FUSED, false, OUT_GELU_Q8);
                    case 5: return RING2(4, 2, 2, 4, 2, EPI_FUSED, false, OUT_GELU_Q8);
                    case 6: return RING2(4, 2, 2, 3, 2, EPI_FUSED, false, OUT_GELU_Q8);
                    default: return HIPQ_ERR_UNSUPPORTED;
                    }
                if (f32)
                    switch (ring_choose(kRingF32, M, N, Kred))
                    {
                    case 0: return RING(8, 1, 2, 9, 2, EPI_FUSED, false, OUT_F32);
                    case 1: return RING(4, 2, 4, 6, 2, EPI_FUSED, false, OUT_F32);
                    case 2: return RING(2, 4, 4, 3, 3, EPI_FUSED, false, OUT_F32);
                    case 3: return RING(4, 2, 2, 4, 4, EPI_FUSED, false, OUT_F32);
                    case 4: return RING(4, 2, 2, 3, 4, EPI_FUSED, false, OUT_F32);
                    case 5: return RING(4, 2, 1, 4, 6, EPI_FUSED, false, OUT_F32);
                    case 6: return RING(4, 2, 1, 3, 6, EPI_FUSED, false, OUT_F32);
                    case 7: return RING(4, 2, 1, 2, 8, EPI_FUSED, false, OUT_F32);
                    default: return HIPQ_ERR_UNSUPPORTED;
                    }
            }
            if (!q8)
                return HIPQ_ERR_UNSUPPORTED;
            if (epi.mode == EPI_INTERP)
                switch (ring_choose(kRingInterp, M, N, Kred))
                {
                case 0: return RING(2, 4, 4, 4, 3, EPI_INTERP, false, OUT_Q8);
                case 1: return RING(4, 2, 4, 4, 3, EPI_INTERP, false, OUT_Q8);
                case 2: return RING(4, 2, 2, 4, 4, EPI_INTERP, false, OUT_Q8);
                case 3: return RING(4, 2, 1, 4, 6, EPI_INTERP, false, OUT_Q8);
                default: return HIPQ_ERR_UNSUPPORTED;
                }
            if (epi.sum_in)
                switch (ring_choose(kRingSum, M, N, Kred))
                {
                case 0: return RING(2, 4, 4, 4, 2, EPI_FUSED, true, OUT_Q8);
                case 1: return RING(4, 2, 4, 4, 2, EPI_FUSED, true, OUT_Q8);
                case 2: return RING(4, 2, 2, 4, 3, EPI_FUSED, true, OUT_Q8);
                case 3: return RING(4, 2, 1, 4, 3, EPI_FUSED, true, OUT_Q8);
                default: return HIPQ_ERR_UNSUPPORTED;
                }
            switch (ring_choose(kRingQ8, M, N, Kred))
            {
            case 0: return RING(2, 4, 4, 4, 3, EPI_FUSED, false, OUT_Q8);
            case 1: return RING(4, 2, 4, 4, 3, EPI_FUSED, false, OUT_Q8);
            case 2: return RING(4, 2, 2, 4, 4, EPI_FUSED, false, OUT_Q8);
            case 3: return RING(4, 2, 1, 4, 6, EPI_FUSED, false, OUT_Q8);
            case 4: return RING(4, 2, 1, 2, 8, EPI_FUSED, false, OUT_Q8);
            case 5: return RING(8, 1, 2, 4, 3, EPI_FUSED, false, OUT_Q8);
            default: return HIPQ_ERR_UNSUPPORTED;
            }
#undef RING
#undef RING2
        }

        bool ring_enabled()
        {
            // (the switches that name a kernel of another family mean that family)
            for (const char* name : {"HIPQ_NO_RING", "HIPQ_SPLIT_K", "HIPQ_NO_DMA", "HIPQ_NO_PIPE", "HIPQ_NO_CONV_DMA", "HIPQ_NO_HALF_TILES", "HIPQ_NO_DEEP_SLICES", "HIPQ_NO_TILE_GROUPS"})
                if (getenv(name) != nullptr)
                    return false;
            return true;
        }
    }

    // The lines against the kernels that split a reduction inside a workgroup: from how many 64-byte steps on the tiles here are
    // ahead, by 32 x 32 tiles a compute unit (from 5/8, 1, 2, 3, 4, 6 and 9 on).  Few tiles leave units idle here and few
    // steps the fill of the ring exposed, where those kernels wait for less; many of both they pay for reading their operands
    // more times.  At most 32 columns count half, since the tiles here are 64 wide and more.  Read off 34 400 drawn sizes that
    // both families take, looped, three in four between 1 500 and 30 000 tiles x steps: the side taken is 0.6 % behind the better
    // one on average (lines linear in tiles x steps, fitted to fewer and wider sizes, before: 1.9 %; sizes that take more than
    // 1.1 times as long here as there 1 600, now 288; the other way round 921, now 420).  The first columns of kLineRows and
    // kLineWindow are a little early for a loop: behind other layers these tiles, which load a ring ahead, gain (ResNet-50 of
    // five images 388 us so, 405 with 20 for rows and 256 -> 256 channels 3 x 3 on 14 x 14 pixels on the other kernels).  us,
    // those kernels and these, of sizes that the lines before gave to the wrong side: 1012 x 464 x 464 with Gelu 5.0 and 8.2,
    // 1329 x 2320 x 192 8.0 and 12.7; 3 x 3 over 384 channels on 4800 pixels -> 16, INTERPRETER policy, 10.2 and 15.5;
    // 368 x 3040 x 704 8.1 and 10.8; 1 x 1 over 32 channels on 3 x 74 x 59 pixels -> 226, [image][channel][pixel], 16.5 and
    // 9.1.  Of the right one: 985 x 4096 x 768 27.6 and 12.7.  Gelu and Quantize are an epilogue of 4 us and more that nothing
    // overlaps; in windows of the INTERPRETER policy taps in a padding become the zero point in LDS, a third of a slice more.
    struct RingLine
    {
        int16_t least[7];
        bool reached(int64_t M, int64_t N, int64_t steps, bool halve) const
        {
            const int64_t tiles = ((M + 31) / 32) * ((N + 31) / 32) / (halve ? 2 : 1), units = device_compute_units(), per = tiles / units;
            if (tiles * 8 < units * 5)
                return false;
            return steps >= least[per < 4 ? per : per < 6 ? 4 : per < 9 ? 5 : 6];
        }
    };
    constexpr int16_t kNever = 0x7fff; // (a reduction is shorter)
    constexpr RingLine kLineRows = {{kNever, 16, 8, 4, 4, 3, 1}}, kLineGelu = {{kNever, kNever, 28, 5, 5, 5, 5}}, kLineWindow = {{32, 16, 8, 5, 5, 3, 1}},
                       kLineNarrowWindow = {{kNever, 32, 32, 32, 32, 32, 32}}, kLineFilled = {{kNever, 32, 12, 8, 8, 5, 5}};
    constexpr RingLine kLineAnyRows = {{kNever, 20, 10, 5, 4, 3, 2}}, kLineAnyWindow = {{kNever, 48, 16, 12, 5, 5, 3}}, kLineAnyFilled = {{kNever, kNever, 96, 16, 12, 6, 4}};
    constexpr RingLine kLineNcxRows = {{kNever, 5, 3, 2, 1, 1, 1}}, kLineNcxWindow = {{kNever, 20, 12, 3, 3, 1, 1}}, kLineNcxFilled = {{kNever, kNever, 20, 16, 12, 5, 3}};

    // Calls that the kernels for small products do not take are better off here than on the other tile kernels (5 250 of those
    // sizes: 0.66 of the time, 76 of them more than 1.03 times as long, the worst 1.3: 3981 x 288 x 2400 12.2 us there, 15.9 here).
    bool ring_preferred(int64_t M, int64_t N, int64_t K, const Epilogue& epi, bool window)
    {
        const int64_t steps = (K + 63) / 64;
        const bool switched = library_switched(), narrow = N <= 32;
        if (switched && !ring_enabled())
            return false;
        if (switched && getenv("HIPQ_RING_TILE") != nullptr)
            return true;
        if (!wk_fits(M, N, steps, true, 0))
        {
            // (but for rows of the INTERPRETER policy into at most 64 columns, for which its tiles here are twice as wide: in a
            // second round of the 256-row ones that costs more than the slices save on short reductions; 68 970 x 384 x 64
            // 9.9 us there, 13.1 here, 230 sizes of fewer than 16 steps 1.15 times as long on average)
            return epi.mode == EPI_FUSED || window || N > 64 || steps >= 16 || M <= 256 * static_cast<int64_t>(device_compute_units());
        }
        if (window && epi.mode == EPI_FUSED)
            return (narrow ? kLineNarrowWindow : kLineWindow).reached(M, N, steps, false);
        return (epi.post_scale ? kLineGelu : window ? kLineFilled : kLineRows).reached(M, N, steps, narrow);
    }

    // The tiles for any width (hipq_igemm_ring_any.hip).  Rows of whole 16-byte columns are taken, or refused, above, and so
    // are windows over multiples of 128 channels; windows over 64, 192, 320 ... channels into whole columns stay on the kernel that
    // loads 64-byte slices.  (Not because that is faster in a loop: 1 050 such sizes took 0.70 of its time here, the worst 1.54.
    // Inside a pass, where the ring kernels lose some of that, it has not been measured.)
    // us, before and here: 2044 x 1379 x 1017 product 33.2 and 12.7, 2836 x 727 x 3157 f32 50.8 and 26.4, 2304 x 1344 x 1001 without
    // a bias 23.7 and 11.4; 3 x 3 windows, 80 -> 412 channels on 30 x 19 x 7 pixels 12.3 and 8.3, 240 -> 704 on 6 x 25 x 25 of the
    // INTERPRETER policy 32.8 and 20.3, [image][channel][pixel] 335 -> 460 on 43 x 59 32.0 and 20.3.
    bool ring_any_preferred(int64_t M, int64_t N, int64_t K, int64_t C, const Epilogue& epi, bool window, bool ncx)
    {
        const int64_t steps = (K + 63) / 64;
        const bool switched = library_switched(), q8 = epi.out_t == HIPQ_U8 || epi.out_t == HIPQ_I8, narrow = N <= 32;
        if (switched && !ring_enabled())
            return false;
        if (switched && getenv("HIPQ_RING_TILE") != nullptr)
            return true;
        if (N % 16 == 0 && !ncx && (q8 || epi.mode == EPI_FUSED) && (!window || C % 64 == 0))
            return false;
        const bool interp = epi.mode == EPI_INTERP, filled = window && interp;
        // More tiles than the kernels for small products take: here, but for channels-last outputs of at most 32 columns and few
        // steps, which the other tile kernels have tiles of 512 rows for (16 -> 36 channels 1 x 1 on 79 x 112 x 26 pixels,
        // INTERPRETER policy, 12.2 us there, 17.3 here; 217 such sizes take 1.26 times as long here on average, 2 100 others 0.55).
        if (!wk_fits(M, N, steps, false, 9))
            return ncx || !narrow || steps > (filled ? 7 : interp ? 2 : 1);
        const RingLine& line = ncx ? (filled ? kLineNcxFilled : window ? kLineNcxWindow : kLineNcxRows) : (filled ? kLineAnyFilled : window ? kLineAnyWindow : kLineAnyRows);
        return line.reached(M, N, steps, narrow);
    }

    int launch_rows_ring(const void* a, int a_unsigned, const int8_t* w, const int32_t* wsum, int64_t M, int32_t N, int32_t K, const ZeroPoints& zp, const Epilogue& epi, void* out, hipStream_t s,
                         const char* name)
    {
        return launch_ring(RingRows{static_cast<const uint8_t*>(a), static_cast<uint32_t>(M * K), K}, w, wsum, M, N, K, a_unsigned, zp, epi, out, s, name);
    }

    int launch_conv_ring(const ConvX& cx, const int8_t* w, const int32_t* wsum, int64_t M, int32_t N, int32_t K, int x_unsigned, const ZeroPoints& zp, const Epilogue& epi, void* out, hipStream_t s,
                         const char* name)
    {
        if (cx.C % SL != 0 || cx.R * cx.S > 32 || M >= (1ll << 31))
            return HIPQ_ERR_UNSUPPORTED;
        RingConv xl;
        static_cast<RingWindow&>(xl) = ring_window(cx);
        return launch_ring(xl, w, wsum, M, N, K, x_unsigned, zp, epi, out, s, name);
    }
}
