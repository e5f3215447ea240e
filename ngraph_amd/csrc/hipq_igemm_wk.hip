// int8 products and implicit-GEMM convolutions too small to fill the chip with the tile kernels of
// hipq_igemm.h: few output pixels or rows, where a launch lasts as long as its slowest chain of
// dependent steps and not as long as its arithmetic.
//
// What bounds them: the tile kernels walk a tile's reduction slice by slice -- global memory to LDS,
// barrier, LDS to registers, MFMA -- and a workgroup that is alone on its compute unit takes about
// 400 ns a slice, nearly all of it latency (a 256 -> 256 3 x 3 layer on 14 x 14 pixels is 36 slices).
// Here a workgroup owns a small output tile (MT x NT blocks of 16 x 16) and the whole reduction, its
// wavefronts take a part of the reduction each, and a wavefront asks for the
// v_mfma_i32_16x16x64_i8 fragments of all its steps at once, straight into registers: one memory
// latency instead of one a slice, no LDS and no barrier in front of the MFMAs.  The partial tiles meet
// in LDS once.  Fragment loads from a row-major matrix take half of every cache line they touch, so
// a compute unit takes operands in at about half of its best rate: the launcher gives these kernels
// only what that costs less for than the slices would (4012 of 5000 sizes of up to 24 tiles of 32 x 32 a
// compute unit, 2.65 times as fast on average as without them).
//
// Measured, one launch of a replayed graph: 256 -> 256 3 x 3 on one 14 x 14 picture 17.4 -> 6.1 us,
// 512 -> 512 3 x 3 on 7 x 7 (an unrolled copy and a skinny product before) 16.3 -> 8.3, 1024 -> 256
// 1 x 1 on 14 x 14 10.7 -> 4.9, 128 x 768 x 768 with float outputs 8.5 -> 3.8; a launch that does
// nothing takes 1.7.
//
// A launch of a single picture's layer is mostly the way to its first operands: the arguments' lines are touched at once
// (touch_arguments), operands are asked for before anything that the epilogue needs, and a window's steps follow
// from each other (ConvStepX) instead of two divisions each.  With that and the row loader for 1 x 1 filters ResNet-50
// on one picture 340 -> 275 us (306 with the row loader alone), the encoder of one sequence 457 -> 442, u8 [8,90,35,29] x
// i8 [150,90,3,3] 13.1 -> 12.5.
//
// Rows and pixels that are no multiple of 16 bytes are read where they lie (ragged_preferred): u8
// [8,90,35,29] x i8 [150,90,3,3] 14.4 -> 13.1 us, 77 x 1000 x 1003 8.2 -> 4.1 with the copy's launch gone.
#include <cstdlib>
#include <cstring>


#include "hipq_igemm.h"

namespace hipq
{
    typedef int v4acc __attribute__((ext_vector_type(4)));
    // (global loads and stores need no alignment on this chip)
    typedef v4i v4i_any __attribute__((aligned(1)));
    typedef uint32_t u32_any __attribute__((aligned(1)));
    typedef v4i v4i_word __attribute__((aligned(4)));

    struct WkParams
    {
        const int8_t* w;      // weights: [N][Kred] rows, or 1 KB blocks in fragment order
        const int8_t* w_rows; // the [N][Kred] rows in either case
        const int32_t* wsum;
        uint32_t w_bytes;
        int32_t w_row;        // bytes from one 16-row block's lane to its next row (rows) / 0 (fragments)
        int32_t w_block;      // bytes between column blocks of 16
        int32_t w_step;       // bytes between 64-byte reduction steps
        int32_t w_lane_chunk; // bytes between a lane's 16-byte chunks of a step (rows: 16, fragments: 256)
        int32_t fragments;
        int64_t M;
        int32_t Kred;
        int32_t x_unsigned;
        int32_t inner;        // tiles along the inner dimension of the tile order
        int32_t m_inner;      // 1: consecutive tiles share a column block, 0: a row block
    };

    // KW wavefronts split the reduction of a tile of MT x NT blocks, TW such tiles (one below the other)
    // make a workgroup; U: reduction steps of 64 bytes a wavefront has in flight.
    // X_ON_A: the activations are MFMA source A, so that a lane's four accumulators are four consecutive
    // pixels of one channel (NCHW outputs); otherwise four consecutive channels of one pixel
    // Short reductions over ragged rows are launches of many workgroups, which live on how many a compute unit holds: they
    // are held to the registers of five wavefronts a SIMD (left to itself the compiler takes 97: four; 9320 x 71 x 1683 26.2 us,
    // with five 22.4).
    template <class XL, int MT, int NT, int KW, int TW, int U, bool X_ON_A>
    __global__ __launch_bounds__(KW * TW * 64, (std::is_same<XL, GemmRaggedX>::value && KW == 1 ? 5 : 0)) void igemm_wk_kernel(XL arg, WkParams p, ZeroPoints zp, Epilogue epi, OutMap om, void* __restrict__ out)
    {
        using Loader = typename std::conditional<std::is_same<XL, ConvX>::value, ConvStepX, XL>::type;
        Loader xl;
        static_cast<XL&>(xl) = arg;
        constexpr int BM = MT * 16, BN = NT * 16;
        constexpr int BLOCKS = MT * NT;
        static_assert(BLOCKS % KW == 0 || KW % BLOCKS == 0, "the wavefronts of a tile share its blocks evenly");
        constexpr int ITER = BLOCKS >= KW ? BLOCKS / KW : 1; // blocks a wavefront finishes
        __shared__ v4acc red[KW > 1 ? KW * TW * BLOCKS * 64 : 1];
        __shared__ __attribute__((aligned(16))) int32_t col_corr[BN];
        __shared__ __attribute__((aligned(16))) float col_bias[BN], col_scale[BN];

        touch_arguments<sizeof(XL) + sizeof(WkParams) + sizeof(ZeroPoints) + sizeof(Epilogue) + sizeof(OutMap) + sizeof(void*) + 8>(); // (8: the grid, behind them)
        const int tid = threadIdx.x;
        const int lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int kw = wave % KW, tw = wave / KW;
        const int r16 = lane & 15, kc = lane >> 4;
        const int N = om.N;
        const bool fused = epi.mode == EPI_FUSED;
        // workgroups are dealt round robin to the eight compute dies: a die gets consecutive tiles, which
        // share the operand that is the larger one
        const int grid = static_cast<int>(gridDim.x);
        const int id = (grid & 7) == 0 ? (static_cast<int>(blockIdx.x) & 7) * (grid >> 3) + (static_cast<int>(blockIdx.x) >> 3) : static_cast<int>(blockIdx.x);
        const int outer_i = id / p.inner, inner_i = id - outer_i * p.inner; // (a multiplication by a reciprocal from the host takes longer: the encoder of one sequence 513 us so, 527 with it)
        const int64_t m0 = (static_cast<int64_t>(p.m_inner ? inner_i : outer_i) * TW + tw) * BM;
        const int n0 = (p.m_inner ? outer_i : inner_i) * BN;

        // ---- operands: fragments of this wavefront's steps
        const int steps = (p.Kred + 63) >> 6;
        const int per = (steps + KW - 1) / KW;
        const int s_begin = ((kw + id) & (KW - 1)) * per;
        static_assert((KW & (KW - 1)) == 0, "wavefronts on a reduction");
        const int s_end = min(steps, s_begin + per);
        const __amdgpu_buffer_rsrc_t xrs = make_rsrc(xl.x, xl.bytes);
        const __amdgpu_buffer_rsrc_t wrs = make_rsrc(p.w, p.w_bytes);
        typename Loader::Row xr[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i)
            xl.init_row(xr[i], m0 + i * 16 + r16, p.M);
        typename Loader::Cursor cur; // kWalk: of the next step to load
        if constexpr (Loader::kWalk != 0)
            xl.init_cursor(cur, s_begin * 64 + kc * 16);
        int32_t woff[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j)
        {
            const int n = n0 + j * 16 + r16;
            // (a block of the fragment-ordered copy holds zeros beyond N)
            const bool ok = p.fragments ? n0 + j * 16 < N : n < N;
            woff[j] = ok ? ((n0 >> 4) + j) * p.w_block + r16 * p.w_row + kc * p.w_lane_chunk : kOob;
        }
        v4i xf[U][MT], wf[U][NT];
        uint32_t pads = 0; // bit u * MT + i: the data fragment lies in the padding
        // Ragged data: a chunk that would run past the tensor's last byte is read as far to the front as it
        // takes to end there; the bytes it starts late by, four bits a step in flight
        const int32_t x_last = static_cast<int32_t>(xl.bytes) - 16;
        uint32_t late[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i)
            late[i] = 0;
        auto load = [&](int u, int s) {
            const int kbyte = s * 64 + kc * 16;
            const bool in_k = (s < s_end) & (kbyte < p.Kred);
            if constexpr (Loader::kWalk == 0)
                xl.init_cursor(cur, kbyte);
#pragma unroll
            for (int i = 0; i < MT; ++i)
            {
                const int32_t off = in_k ? xl.offset(xr[i], cur) : kOob;
                if (XL::kPadded)
                    pads = (pads & ~(1u << (u * MT + i))) | ((off == kOob ? 1u : 0u) << (u * MT + i));
                if constexpr (XL::kRagged)
                {
                    // (a fragment that does not exist is whatever the tensor starts with: its weights are zeros,
                    // its row is not stored, or the padding replaces it)
                    const int32_t at = min(max(off, 0), x_last);
                    late[i] = (late[i] & ~(15u << (4 * u))) | static_cast<uint32_t>(max(off, at) - at) << (4 * u);
                    xf[u][i] = *reinterpret_cast<const v4i_any*>(xl.x + static_cast<uint32_t>(at));
                }
                else
                    xf[u][i] = buffer_load16(xrs, off);
            }
#pragma unroll
            for (int j = 0; j < NT; ++j)
                wf[u][j] = buffer_load16(wrs, (in_k && woff[j] != kOob) ? woff[j] + s * p.w_step : kOob);
            if constexpr (Loader::kWalk != 0)
                xl.advance(cur, 64);
        };
        // The byte of the padding, which a window of the INTERPRETER policy waits for before its first product: in front of the
        // operands where a tile is 16 rows, as a trip of its own behind them it was 0.4 us of a launch of 4.4 (213 drawn
        // sizes of one and two steps, channels-last: 1.05 times the time that they took when the operands came behind the epilogue's
        // words, so 0.96; 1457 others 0.97 of it behind).  Tiles of 32 rows, sixteen wavefronts and 16 x 16 tiles
        // of [image][channel][pixel] outputs lose by it, up to 1.1 times.
        constexpr bool kByteFirst = Loader::kWalk != 0 && MT == 1 && KW <= 8 && (NT == 2 || !X_ON_A);
        int32_t xzp_early = 0;
        if constexpr (XL::kPadded && kByteFirst)
            xzp_early = load_zp(zp.data_zp, zp.data_t);
#pragma unroll
        for (int u = 0; u < U; ++u)
            load(u, s_begin + u);
        // what the epilogue needs from memory is asked for behind the operands, none of it looked at
        // before the reduction is done: per-channel constants, the scalars, the residual
        const bool with_bias = fused && epi.bias != nullptr, per_channel = fused && epi.per_channel != 0;
        // (every thread, of which BN are listened to: behind a branch the values are waited for where it ends)
        const int n_of = tid < BN && n0 + tid < N ? n0 + tid : 0;
        const int32_t raw_wsum = p.wsum[n_of];
        const int32_t raw_bias = (with_bias ? epi.bias : p.wsum)[n_of];
        const float raw_scale = (per_channel ? epi.scale : reinterpret_cast<const float*>(p.wsum))[n_of];
        HeadWords hw = head_scalars_load(zp, epi, p.wsum);
        // this wavefront finishes blocks it * KW + kw of its tile, a group of four outputs a lane
        const bool has_sum = fused && epi.sum_in != nullptr;
        const bool vec_ok = !X_ON_A || !om.ncx || (om.PQ & 3) == 0; // the group is contiguous (rows of N may start anywhere)
        int64_t o_at[ITER];
        int o_left[ITER]; // outputs of the group that exist
        uint32_t res[ITER];
#pragma unroll
        for (int it = 0; it < ITER; ++it)
        {
            const int blk = it * KW + kw;
            const int mi = blk / NT, ni = blk % NT;
            const int64_t m = m0 + mi * 16 + (X_ON_A ? 4 * kc : r16);
            const int n = n0 + ni * 16 + (X_ON_A ? r16 : 4 * kc);
            const bool live = blk < BLOCKS && m < p.M && n < N;
            o_left[it] = !live ? 0 : X_ON_A ? static_cast<int>(p.M - m < 4 ? p.M - m : 4) : (N - n < 4 ? N - n : 4);
            o_at[it] = live ? om.index(m, n) : 0;
            res[it] = 0;
            if (has_sum && o_left[it] > 0)
            {
                if (vec_ok && o_left[it] == 4)
                    res[it] = *reinterpret_cast<const u32_any*>(static_cast<const uint8_t*>(epi.sum_in) + o_at[it]);
                else
                {
                    for (int e = 0; e < o_left[it]; ++e)
                        res[it] |= static_cast<uint32_t>(static_cast<const uint8_t*>(epi.sum_in)[X_ON_A ? om.index(m + e, n) : o_at[it] + e]) << (8 * e);
                }
            }
        }

        const int xor_mask = p.x_unsigned ? static_cast<int>(0x80808080u) : 0;
        if constexpr (XL::kPadded && !kByteFirst)
            xzp_early = load_zp(zp.data_zp, zp.data_t);
        const int fill = (xzp_early & 0xFF) * 0x01010101;
        v4acc acc[MT][NT];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
                acc[i][j] = v4acc{0, 0, 0, 0};
        auto multiply = [&](int u) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
            {
                v4i x = xf[u][i];
                if constexpr (XL::kRagged)
                {
                    const uint32_t n = (late[i] >> (4 * u)) & 15u;
                    if (__builtin_amdgcn_ballot_w64(n != 0) != 0) // uniform, and rare
                    {
                        const int q = static_cast<int>(n >> 2);
                        const int d[8] = {x[0], x[1], x[2], x[3], 0, 0, 0, 0};
                        int y[5];
#pragma unroll
                        for (int e = 0; e < 5; ++e)
                            y[e] = q == 0 ? d[e] : q == 1 ? d[e + 1] : q == 2 ? d[e + 2] : d[e + 3];
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            x[e] = static_cast<int>(__builtin_amdgcn_alignbyte(static_cast<uint32_t>(y[e + 1]), static_cast<uint32_t>(y[e]), n & 3u));
                    }
                }
                if (XL::kPadded && (XL::kRagged || fill != 0)) // uniform: padding taps hold the data zero point
                {
                    const bool pad = (pads >> (u * MT + i)) & 1u;
                    x = v4i{pad ? fill : x[0], pad ? fill : x[1], pad ? fill : x[2], pad ? fill : x[3]};
                }
                // (steps past the reduction read zero weights, which cancel whatever is here)
                x = v4i{x[0] ^ xor_mask, x[1] ^ xor_mask, x[2] ^ xor_mask, x[3] ^ xor_mask};
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j] = X_ON_A ? __builtin_amdgcn_mfma_i32_16x16x64_i8(x, wf[u][j], acc[i][j], 0, 0, 0) : __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[u][j], x, acc[i][j], 0, 0, 0);
            }
        };
        for (int s = s_begin; s + U < s_end; s += U) // (uniform; most launches ask for everything above)
        {
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                multiply(u);
                load(u, s + U + u);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            multiply(u);

        head_scalars_settle(hw);
        const HeadScalars hs = head_scalars_finish(hw, zp, epi);
        if (hs.wzp != 0) // uniform; w - wzp does not fit a signed byte: exact, slow
        {
            slow_tile(xl, p.w_rows, p.M, p.Kred, p.x_unsigned, hs.xzp, hs.wzp, epi, om, out, m0 - tw * BM, n0, TW * BM, BN);
            return;
        }
        // ---- the partial tiles meet in LDS
        if constexpr (KW > 1)
        {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    red[(wave * BLOCKS + i * NT + j) * 64 + lane] = acc[i][j];
        }
        if (tid < BN)
        {
            col_corr[tid] = ((p.x_unsigned ? 128 : 0) - hs.xzp) * raw_wsum;
            col_bias[tid] = with_bias ? static_cast<float>(raw_bias) : 0.0f;
            col_scale[tid] = per_channel ? raw_scale : hs.ec.scale;
        }
        const EpiConst ec = hs.ec;
        const bool relu = epi.relu != 0;
        const bool gelu = epi.post_scale != nullptr;
        const float post_scale = gelu ? *epi.post_scale : 1.0f;
        const int32_t post_zp = gelu ? load_zp(epi.post_zp, epi.post_t) : 0;
        __syncthreads();
        // (one instantiation of the arithmetic a policy and output kind, chosen by uniform branches: the kernel
        // runs it once)
        auto finish = [&](auto mode_c, auto kind_c) {
            constexpr int MODE = decltype(mode_c)::value;
            constexpr int KIND = decltype(kind_c)::value;
#pragma unroll
            for (int it = 0; it < ITER; ++it)
            {
                if (o_left[it] == 0)
                    continue;
                const int blk = it * KW + kw;
                v4acc a;
                if constexpr (KW > 1)
                {
                    a = red[(tw * KW * BLOCKS + blk) * 64 + lane];
#pragma unroll
                    for (int v = 1; v < KW; ++v)
                        a += red[((tw * KW + v) * BLOCKS + blk) * 64 + lane];
                }
                else
                    a = acc[it / NT][it % NT];
                const int nl = (blk % NT) * 16 + (X_ON_A ? r16 : 4 * kc); // column within the tile
                int32_t v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                {
                    const int c = X_ON_A ? nl : nl + e;
                    const int32_t sum = a[e] + col_corr[c];
                    const uint32_t rb = (res[it] >> (8 * e)) & 0xFFu;
                    const float sv = epi.sum_t == HIPQ_I8 ? static_cast<float>(static_cast<int8_t>(rb)) : static_cast<float>(rb);
                    v[e] = MODE == EPI_INTERP ? epi_interp<KIND>(ec, sum) : epi_fused<KIND == OUT_GELU_Q8 ? OUT_F32 : KIND>(ec, sum, col_bias[c], col_scale[c], has_sum, sv, relu);
                }
                if constexpr (KIND == OUT_GELU_Q8)
                {
                    // Gelu and Quantize with the arithmetic of their own kernels: the bytes equal the three launches'.  (Not
                    // gelu_quantize4: a lane has four elements, and its constants and checks take longer to fetch than they spare: the encoder
                    // of one sequence 457 us so, 462 with it.)
                    const f32x4 r4 = f32x4{gelu1(__int_as_float(v[0])), gelu1(__int_as_float(v[1])), gelu1(__int_as_float(v[2])), gelu1(__int_as_float(v[3]))};
                    uint32_t packed = 0;
                    if (epi.post_mode == HIPQ_ROUND_NEAREST_TOWARD_EVEN) // uniform
                        packed = epi.post_t == HIPQ_U8 ? quantize4<uint8_t, true>(r4, post_scale, static_cast<float>(post_zp), epi.post_mode)
                                                       : quantize4<int8_t, true>(r4, post_scale, static_cast<float>(post_zp), epi.post_mode);
                    else
                    {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            packed |= (epi.post_t == HIPQ_U8 ? static_cast<uint32_t>(quantize_one<float, uint8_t>(r4[e], post_scale, static_cast<uint8_t>(post_zp), epi.post_mode))
                                                             : static_cast<uint32_t>(static_cast<uint8_t>(quantize_one<float, int8_t>(r4[e], post_scale, static_cast<int8_t>(post_zp), epi.post_mode))))
                                      << (8 * e);
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        v[e] = static_cast<int32_t>((packed >> (8 * e)) & 0xFFu);
                }
                if (vec_ok && o_left[it] == 4)
                {
                    if (KIND == OUT_Q8 || KIND == OUT_GELU_Q8)
                        *reinterpret_cast<u32_any*>(static_cast<uint8_t*>(out) + o_at[it]) = pack4(v);
                    else
                        *reinterpret_cast<v4i_word*>(static_cast<int32_t*>(out) + o_at[it]) = v4i{v[0], v[1], v[2], v[3]};
                }
                else
                {
                    const int64_t m = m0 + (blk / NT) * 16 + 4 * kc;
                    for (int e = 0; e < o_left[it]; ++e)
                        store_out(out, KIND == OUT_Q8 || KIND == OUT_GELU_Q8 ? HIPQ_U8 : HIPQ_I32, X_ON_A ? om.index(m + e, n0 + nl) : o_at[it] + e, e == 0 ? v[0] : e == 1 ? v[1] : e == 2 ? v[2] : v[3]);
                }
            }
        };
        using std::integral_constant;
        const bool q8 = epi.out_t == HIPQ_U8 || epi.out_t == HIPQ_I8;
        if (!fused)
        {
            if (q8)
                finish(integral_constant<int, EPI_INTERP>{}, integral_constant<int, OUT_Q8>{});
            else
                finish(integral_constant<int, EPI_INTERP>{}, integral_constant<int, OUT_I32>{});
        }
        else if (q8)
            finish(integral_constant<int, EPI_FUSED>{}, integral_constant<int, OUT_Q8>{});
        else if constexpr (!X_ON_A && !XL::kPadded)
        {
            if (gelu)
                finish(integral_constant<int, EPI_FUSED>{}, integral_constant<int, OUT_GELU_Q8>{});
            else
                finish(integral_constant<int, EPI_FUSED>{}, integral_constant<int, OUT_F32>{});
        }
    }

    enum class WkShape
    {
        kTile1181, // 16 x 16, eight wavefronts on the reduction
        kTile11161, // the same, sixteen
        kTile1241, // 16 x 32, four
        kTile2241, // 32 x 32, four
        kTile2222, // two tiles of 32 x 32, two wavefronts each
        kTile2214  // four tiles of 32 x 32, a wavefront each
    };
    static int64_t wk_tiles(int64_t M, int64_t N, int bm, int bn) { return (M + bm - 1) / bm * ((N + bn - 1) / bn); }

    // Which tile: the largest that still gives every compute unit work.  From three 32 x 32 tiles for two
    // compute units on those; their reduction is worth splitting over all four wavefronts unless it is
    // short and there are many of them.  Fewer tiles: 16 x 32, and where even those leave half of the chip
    // idle on a reduction of eight steps or more, 16 x 16 with eight wavefronts on it.  (2000 products and
    // convolutions of up to six tiles a unit, each timed in all six shapes: 1.024 times the best shape of each on
    // average; 16 x 32 with 49 steps and more 1.10 times, 106 x 4128 x 1344 13.6 us, 8.8 with sixteen wavefronts.)
    // Reductions that eight wavefronts cannot ask for at once (more than 48 steps) and sixteen ask for in four
    // loads each take sixteen: 40 x 4096 x 512 5.6 -> 5.3 us, 100 x 4004 x 200 5.6 -> 5.1, 400 -> 400 3 x 3 on 9 x 9
    // 6.8 -> 6.2; from five loads on the larger exchange costs more (512 -> 512 3 x 3 on 7 x 7 8.0 -> 8.2).
    static WkShape wk_shape(int64_t M, int64_t N, int64_t Kred)
    {
        const int64_t t22 = wk_tiles(M, N, 32, 32), steps = (Kred + 63) / 64, units = device_compute_units();
        if (t22 * 2 >= units * 3)
        {
            if (t22 < units * 3 || steps > 6)
                return WkShape::kTile2241;
            return steps <= 2 ? WkShape::kTile2214 : WkShape::kTile2222;
        }
        if (wk_tiles(M, N, 16, 32) * 2 >= units || steps < 8)
            return WkShape::kTile1241;
        return steps > 48 && steps <= 64 ? WkShape::kTile11161 : WkShape::kTile1181;
    }

    // Whether these kernels are the better ones.  Against the kernels that load straight into LDS (`dma`: 8-bit
    // or fused float rows in whole 16-byte pieces, channels in whole 64-byte slices) up to three 32 x 32
    // tiles a compute unit: above that those kernels' whole-line loads and larger tiles win (985 x 512 x
    // 1536: 8.6 us there, 9.9 us here; 985 x 512 x 512: 7.9, 5.5); up to four on reductions of at most 256
    // bytes and seven on those of one step, where their larger tiles wait for one slice as long as these do
    // and leave compute units idle (784 x 256 x 1024 6.4, 5.6; 3136 x 64 x 256 6.4, 5.2; 6272 x 64 x 256 6.8, 5.9;
    // but 1568 x 256 x 1024, six tiles a unit: 6.8, 7.9; looped on hot inputs 49 sizes of one step and four to
    // seven tiles take 1.06 times as long here, inside a pass they gain: ResNet-50 of two images 390 us, with a
    // line at four 395).  Not for at most 64 outputs (12544 x 256 x 64: 6.4,
    // 6.7).  Against the register-staged ones up to sixteen; nine on reductions of more than 20 steps, where their
    // larger tiles read each operand fewer times (of 14 500 sizes 136 lie above that line, 1.27 times as fast there on average:
    // 28 x 12 x 12 pixels of 512 -> 788 3 x 3, twelve tiles: 61 us there, 108 here; 985 x 5888 x 2971, eleven: 72, 127;
    // on shorter ones as many would lose: 806 x 960 x 4593, fifteen: 35, 21).  Sixteen all the same for at most 64 outputs,
    // which leave most units idle there (42 x 32 x 32 of 288 -> 46 3 x 3, ten: 79, 45), for at most 512 rows, which
    // wait for weights out of HBM there, on the tile kernels and on those that stream them past up to 256 rows
    // (137 x 2192 x 23255, fourteen: 157, 66; 128 x 4096 x 20001, ten: 93, 55), and where Gelu is a launch of its
    // own there (`alone` unset).
    static bool wk_enabled()
    {
        if (!library_switched())
            return true;
        // (the switches that name a kernel of the other family mean that family)
        for (const char* name : {"HIPQ_NO_WK", "HIPQ_SPLIT_K", "HIPQ_NO_DMA", "HIPQ_NO_PIPE", "HIPQ_NO_CONV_DMA", "HIPQ_NO_HALF_TILES", "HIPQ_NO_REGW"})
            if (getenv(name) != nullptr)
                return false;
        return true;
    }
    // long_limit: tiles a compute unit on long reductions
    bool wk_fits(int64_t M, int64_t N, int64_t steps, bool dma, int64_t long_limit)
    {
        // (the entry point that allocates nothing keeps sixteen: the tile kernels may want more scratch than it has)
        const bool few = N <= 64 || M <= 512 || steps <= 20 || !workspace_holds(SIZE_MAX);
        const int64_t limit = dma ? (N <= 64 || steps > 4 ? 3 : steps > 1 ? 4 : 7) : (few ? 16 : long_limit);
        return wk_tiles(M, N, 32, 32) <= static_cast<int64_t>(device_compute_units()) * limit;
    }
    bool wk_preferred(int64_t M, int64_t N, int64_t steps, bool dma, bool alone) { return wk_fits(M, N, steps, dma, alone ? 9 : 16) && wk_enabled(); }

    // Whether rows (pixels) of `row_bytes` that are no multiple of 16 are read where they lie, instead of
    // through a copy padded to whole chunks (a launch, 2.5 us and more, and rows a power of two apart).
    // Chunks then start at any byte.  On rows of whole dwords that costs nothing seen (4096 x 1500 x 1003:
    // copy and product 58.5 us, in place 39.5; 16 x 1000 x 1003: 6.6, 3.7); on others a chunk takes about
    // twice its time in the memory path, so only while there are few of them: 32 steps of 64 bytes (40 with a
    // window's taps, which hit the same lines) and 8192 step-tiles (24576 with taps or up to six steps):
    // 77 x 2001 x 1003 7.1 there, 6.2 in place; 600 x 1301 x 1003 12.0, 14.4; 16 x 4001 x 150 6.7, 8.7;
    // 90 -> 150 channels 3 x 3 on 8 x 35 x 35 pixels 15.4, 14.8, on 64 x 35 x 35 68, 82.  Of 3974 sizes 2792 stay in
    // place, 1.52 times as fast as with the copy; 17 of them more than 5 % slower, at worst 1.34 times (20 x 10 x 10 of
    // 261 -> 304 3 x 3: 16.0, 21.4).
    // Where no kernel that loads straight into LDS would take the call, short reductions stay here beyond
    // the sizes of wk_preferred: 90 -> 150 channels 1 x 1 on 128 x 56 x 56 179 there, 79 in place.
    bool ragged_preferred(int64_t M, int64_t N, int64_t row_bytes, int64_t steps, bool dma, bool pointwise)
    {
        const int64_t tiles = wk_tiles(M, N, 32, 32), units = device_compute_units();
        const bool few_steps = !dma && pointwise && (steps <= 3 || (steps <= 6 && tiles <= units * 40));
        const bool few_bytes = row_bytes % 4 == 0 ? pointwise || steps <= 40 : steps <= (pointwise ? 32 : 40) && tiles * steps <= (steps <= 6 || !pointwise ? 24576 : 8192);
        return (few_steps || (few_bytes && wk_fits(M, N, steps, dma, 12))) && wk_enabled(); // (12: the copy is spared as well)
    }

    template <class XL, int MT, int NT, int KW, int TW, int U, bool X_ON_A>
    static int launch_wk_tile(const XL& xl, WkParams p, const ZeroPoints& zp, const Epilogue& epi, const OutMap& om, void* out, hipStream_t s, const char* name)
    {
        const int64_t m_tiles = (p.M + TW * MT * 16 - 1) / (TW * MT * 16), n_tiles = (om.N + NT * 16 - 1) / (NT * 16);
        HIPQ_REQUIRE(fits_i32(m_tiles * n_tiles), "too many tiles");
        p.m_inner = p.M <= om.N ? 1 : 0; // the larger operand is the one that consecutive tiles share
        p.inner = static_cast<int32_t>(p.m_inner ? m_tiles : n_tiles);
        igemm_wk_kernel<XL, MT, NT, KW, TW, U, X_ON_A><<<static_cast<unsigned>(m_tiles * n_tiles), KW * TW * 64, 0, s>>>(xl, p, zp, epi, om, out);
        return check_launch(name);
    }

    // as many steps in flight as a wavefront has, up to what its registers hold (the last of UPS): a load that
    // has no step would still take its turn in the texture path, which is what bounds these kernels
    template <class XL, bool X_ON_A, int MT, int NT, int KW, int TW, int U, int... UPS>
    static int launch_wk_steps(const XL& xl, const WkParams& p, const ZeroPoints& zp, const Epilogue& epi, const OutMap& om, void* out, hipStream_t s, const char* name)
    {
        if constexpr (sizeof...(UPS) > 0)
            if (((p.Kred + 63) / 64 + KW - 1) / KW > U)
                return launch_wk_steps<XL, X_ON_A, MT, NT, KW, TW, UPS...>(xl, p, zp, epi, om, out, s, name);
        return launch_wk_tile<XL, MT, NT, KW, TW, U, X_ON_A>(xl, p, zp, epi, om, out, s, name);
    }

    template <class XL, bool X_ON_A>
    static int launch_wk(const XL& xl, const WkParams& p, const ZeroPoints& zp, const Epilogue& epi, const OutMap& om, void* out, hipStream_t s, const char* name)
    {
        const bool q8 = epi.out_t == HIPQ_U8 || epi.out_t == HIPQ_I8;
        if (epi.mode == EPI_FUSED && !q8 && (X_ON_A || XL::kPadded || epi.out_t != HIPQ_F32))
            return HIPQ_ERR_UNSUPPORTED;
        // (of each shape the step counts that wk_shape gives it)
        switch (wk_shape(p.M, om.N, p.Kred))
        {
        case WkShape::kTile1181: return launch_wk_steps<XL, X_ON_A, 1, 1, 8, 1, 1, 2, 3, 4, 6>(xl, p, zp, epi, om, out, s, name);
        case WkShape::kTile11161: return launch_wk_steps<XL, X_ON_A, 1, 1, 16, 1, 4>(xl, p, zp, epi, om, out, s, name);
        case WkShape::kTile1241: return launch_wk_steps<XL, X_ON_A, 1, 2, 4, 1, 1, 2, 3, 4, 6>(xl, p, zp, epi, om, out, s, name);
        case WkShape::kTile2214:
            if constexpr (std::is_same<XL, GemmRaggedX>::value) // (65 bytes and more, padded to whole steps)
                return launch_wk_steps<XL, X_ON_A, 2, 2, 1, 4, 2>(xl, p, zp, epi, om, out, s, name);
            else
                return launch_wk_steps<XL, X_ON_A, 2, 2, 1, 4, 1, 2>(xl, p, zp, epi, om, out, s, name);
        case WkShape::kTile2222: return launch_wk_steps<XL, X_ON_A, 2, 2, 2, 2, 2, 3>(xl, p, zp, epi, om, out, s, name);
        case WkShape::kTile2241: return launch_wk_steps<XL, X_ON_A, 2, 2, 4, 1, 1, 2, 3, 4, 5>(xl, p, zp, epi, om, out, s, name);
        }
        return HIPQ_ERR_UNSUPPORTED; // (not reached)
    }

    static WkParams wk_params(const int8_t* w_nk, const void* w_frag, const int32_t* wsum, int64_t M, int32_t N, int32_t K, int x_unsigned)
    {
        WkParams p;
        p.fragments = w_frag != nullptr;
        p.w = w_frag ? static_cast<const int8_t*>(w_frag) : w_nk;
        p.w_rows = w_nk;
        p.wsum = wsum;
        p.w_bytes = w_frag ? static_cast<uint32_t>((N + 15) / 16) * static_cast<uint32_t>(K / 64) * 1024u : static_cast<uint32_t>(N) * static_cast<uint32_t>(K);
        p.w_row = w_frag ? 16 : K;
        p.w_block = w_frag ? (K / 64) * 1024 : 16 * K;
        p.w_step = w_frag ? 1024 : 64;
        p.w_lane_chunk = w_frag ? 256 : 16;
        p.M = M;
        p.Kred = K;
        p.x_unsigned = x_unsigned;
        p.inner = p.m_inner = 1;
        return p;
    }

    template <class XL>
    static XL rows_of(const void* a, int64_t M, int32_t row_bytes)
    {
        XL xl;
        xl.x = static_cast<const uint8_t*>(a);
        xl.K = row_bytes;
        xl.bytes = static_cast<uint32_t>(M * row_bytes);
        return xl;
    }

    int launch_rows_wk(const void* a, bool a_unsigned, const int8_t* w_nk, const void* w_frag, const int32_t* wsum, int64_t M, int32_t N, int32_t K, const ZeroPoints& zp, const Epilogue& epi,
                       void* out, hipStream_t s, const char* name)
    {
        const OutMap om{0, N, 1};
        return launch_wk<GemmX, false>(rows_of<GemmX>(a, M, K), wk_params(w_nk, w_frag, wsum, M, N, K, a_unsigned ? 1 : 0), zp, epi, om, out, s, name);
    }

    int launch_rows_wk_ragged(const void* a, int32_t a_row, bool a_unsigned, const int8_t* w_nk, const void* w_frag, const int32_t* wsum, int64_t M, int32_t N, int32_t K, const ZeroPoints& zp,
                              const Epilogue& epi, void* out, hipStream_t s, const char* name)
    {
        const OutMap om{0, N, 1};
        return launch_wk<GemmRaggedX, false>(rows_of<GemmRaggedX>(a, M, a_row), wk_params(w_nk, w_frag, wsum, M, N, K, a_unsigned ? 1 : 0), zp, epi, om, out, s, name);
    }

    int launch_conv_wk_ragged(const ConvRaggedX& xl, const int8_t* w, const int32_t* wsum, int64_t M, int32_t N, int32_t K, int x_unsigned, const ZeroPoints& zp, const Epilogue& epi,
                              const OutMap& om, void* out, hipStream_t s, const char* name)
    {
        const WkParams p = wk_params(w, nullptr, wsum, M, N, K, x_unsigned);
        if (om.ncx)
            return launch_wk<ConvRaggedX, true>(xl, p, zp, epi, om, out, s, name);
        return launch_wk<ConvRaggedX, false>(xl, p, zp, epi, om, out, s, name);
    }

    int launch_conv_wk(const ConvX& xl, const int8_t* w, const int32_t* wsum, int64_t M, int32_t N, int32_t K, int x_unsigned, const ZeroPoints& zp, const Epilogue& epi, const OutMap& om, void* out,
                       hipStream_t s, const char* name)
    {
        if (M >= (1ll << 31))
            return HIPQ_ERR_UNSUPPORTED;
        const WkParams p = wk_params(w, nullptr, wsum, M, N, K, x_unsigned);
        if (om.ncx)
            return launch_wk<ConvX, true>(xl, p, zp, epi, om, out, s, name);
        return launch_wk<ConvX, false>(xl, p, zp, epi, om, out, s, name);
    }
}
