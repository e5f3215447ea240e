// A bottleneck block's last layer and the next block's first one in one launch, at the stages of a ResNet whose layers move
// more bytes than they compute on: the 1 x 1 convolution that widens 64 or 128 channels to 256 or 512 (with the residual input,
// or with the residual itself: the projection shortcut, a 1 x 1 convolution of the same pixels) and the 1 x 1 convolution that
// narrows its result again.  One launch a layer writes the wide tensor, reads it again for the narrow layer and, with a
// projection, writes and reads a second one; here the wide tensor is written once and the projection never.
//
// A workgroup takes 16 pixels at a time and has a wavefront for every 64 channels of the wide result, whose weights and
// constants stay in its registers.  v_mfma_i32_16x16x64_i8 with the weights as its first operand leaves lane (pixel r = lane %
// 16, k = lane / 16) four rows of the weights: rows 16 (r / 4) + 4 b + r % 4 of the 64 are laid out as block b, so that after four
// blocks the lane holds channels 16 k .. 16 k + 15 of its pixel.  That is 16 bytes of output, 16 bytes of residual, and exactly
// the second operand of the narrow layer's instruction for these 64 channels: the requantized dwords go through LDS as they are, a
// lane's to the same lane of every wavefront, each of which has its share of the narrow layer's weights in registers as well.
// Data and residual arrive by loads straight into LDS, a lane's bytes where that lane reads them.  One barrier a tile.
//
// Bound by HBM and by vector instructions (the requantization of the wide result), which add up to about four fifths: 64 -> 256 -> 64
// over 401 408 pixels moves 257 MB (38 us at the rate of a copy), its arithmetic alone takes 32, together 52 looped and 54 inside
// ResNet-50 of 128 images; with the projection 180 MB, 46 and 48.  us, separate launches and one, looped (64 -> 256 -> 64 with
// the projection; with a residual; 64 -> 256 -> 128; 128 -> 512 -> 128 on a quarter of the pixels; 128 -> 512 -> 256 likewise):
//   401 408 pixels  96.2 -> 47.9   64.0 -> 51.8   72.2 -> 66.9   45.3 -> 30.6   57 -> 35.9
//    25 088         21.9 -> 10.1   15.2 ->  8.2   12.6 ->  9.7   12.2 ->  9.4   14 -> 11.9
//     3 136         13.1 ->  6.8    8.5 ->  6.1    8.7 ->  6.7    8.4 ->  8.2  8.7 -> 10.2
// Tried and taken back: a wavefront that takes all channels of its pixels, with the weights in LDS and no barrier (72 to 112 reads a
// tile: 47, 43-59, 64, 30; the small ones 2 to 4 us more, for the weights have to be laid out first); tiles of 32 and 64 pixels (no
// faster, 1 to 4 us more for few pixels); the narrow layer a tile behind, beside the wide one's instructions; three or four
// wavefronts a SIMD (no faster where their registers fit); stores that bypass the caches (inside a pass the next layers miss them).
//
// Arithmetic: that of the tile kernels' fused epilogue (hipq_igemm.h), see hipq_conv_pw.hip; the bytes equal the separate calls'.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "hipq_igemm.h"

namespace hipq
{
    namespace
    {
        typedef int v4i_at4 __attribute__((ext_vector_type(4), aligned(4)));
        typedef int v2i __attribute__((ext_vector_type(2)));
        struct ChainLayer
        {
            const int8_t* w; // [N][C]
            const int32_t* wsum;
            const int32_t* bias; // or null
            const float* scale;
            int32_t per_channel, x_unsigned;
        };
        struct ChainParams
        {
            const uint8_t* x;   // [M][C]
            const uint8_t* sum; // [M][N1], or the shortcut's data [M][64]
            uint8_t* out;       // [M][N1]
            uint8_t* narrow;    // [M][N2]
            const float* sum_scale;
            ChainLayer l1, ls, l2;
            int32_t M, tiles;
            int32_t short_relu;
        };

        constexpr int kChainShort = 64; // channels of a shortcut's data
        // LDS: two tiles of operands (data, residual or the shortcut's data; three or four of them gain nothing, 401 408 pixels 64 ->
        // 256 -> 64 52.1, 54.8 and 54.9 us), two of the wide result, and a place for loads of nothing
        constexpr int chain_tile(int C, int N1, bool shortcut) { return 16 * (C + (shortcut ? kChainShort : N1)); }
        constexpr size_t chain_lds(int C, int N1, bool shortcut) { return 2 * static_cast<size_t>(chain_tile(C, N1, shortcut)) + 2 * static_cast<size_t>(16) * N1 + 1024; }

        // N1 / 64 wavefronts.  I8: the wide result (after its ReLU) and the residual are i8, else both u8
        template <int C, int N1, int N2, bool SHORT, bool I8>
        __global__ __launch_bounds__(N1, 2) void conv_chain_kernel(const ChainParams p)
        {
            touch_arguments<sizeof(ChainParams)>();
            constexpr int G = N1 / 64, KS = C / 64, CS = kChainShort;
            constexpr int OUTW = N2 / G, NB2 = OUTW / 16; // channels of the narrow layer a wavefront, and blocks of 16 of them
            static_assert(OUTW % 16 == 0, "whole blocks");
            constexpr int TILE = chain_tile(C, N1, SHORT);
            constexpr int SHARED = KS + (SHORT ? 1 : 0); // pieces of 1 KB that every wavefront reads
            static_assert(SHARED <= G, "a wavefront asks for one of them");
            extern __shared__ __attribute__((aligned(16))) uint8_t lds[]; // [2][shared pieces | residual: group][64 lanes][16 bytes], [2][group][the same], nothing
            uint8_t* const wide = lds + 2 * TILE;
            const int tid = static_cast<int>(threadIdx.x);
            const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
            const int r16 = lane & 15, kc = lane >> 4;
            const int first = static_cast<int>(blockIdx.x), stride = static_cast<int>(gridDim.x);

            // ---- loads: of the first tile before anything else --------------------------------------------
            const __amdgpu_buffer_rsrc_t ors = make_rsrc(p.out, static_cast<uint32_t>(p.M) * N1);
            const __amdgpu_buffer_rsrc_t nrs = make_rsrc(p.narrow, static_cast<uint32_t>(p.M) * N2);
            // the loads of the workgroup's tile j go to slot j % 2, a lane's 16 bytes where the same lane reads them.  (Beyond
            // the last tile every pixel is beyond M: nothing is read, zeros arrive, the counts stay the same)
            const v4i xw = rsrc_words(p.x, static_cast<uint32_t>(p.M) * C), sw = rsrc_words(p.sum, static_cast<uint32_t>(p.M) * (SHORT ? CS : N1));
            const uint32_t lds_at = lds_address(lds);
            auto pixel = [&](int t) { return t * 16 + r16; };
            const bool second = SHORT && wave >= KS; // uniform, as is everything of the wavefront: its shared piece is the shortcut's data
            auto issue = [&](int t, int slot) {
                const uint32_t to = lds_at + static_cast<uint32_t>(slot) * TILE;
                const int m = pixel(t);
                const int off = wave < SHARED && m < p.M ? m * (second ? CS : C) + (second ? 0 : wave * 64) + kc * 16 : kOob;
                lds_dma16_unfenced(second ? sw : xw, off, __builtin_amdgcn_readfirstlane(wave < SHARED ? to + wave * 1024 : lds_at + 2 * TILE + 2 * 16 * N1));
                if constexpr (!SHORT)
                    lds_dma16_unfenced(sw, m < p.M ? m * N1 + wave * 64 + kc * 16 : kOob, __builtin_amdgcn_readfirstlane(to + (SHARED + wave) * 1024));
            };
            issue(first, 0);
            issue(first + stride, 1);

            // ---- weights and constants --------------------------------------------------------------------
            // the lane's channels 4 b .. + 3 of the wavefront's, of each layer
            const int n1 = wave * 64 + kc * 16, o2 = wave * OUTW, n2 = o2 + kc * 4 * NB2;
            auto words = [](const void* from, int at) { return *reinterpret_cast<const v4i_at4*>(static_cast<const int32_t*>(from) + at); };
            // rows first + 4 BLOCKS (r / 4) + 4 b + r % 4 of a layer's weights, STEPS x 64 bytes of them, as fragments
            auto fragment = [&](const int8_t* w, int cols, int row0, int blocks, int b, int step) {
                return *reinterpret_cast<const v4i*>(w + (row0 + 4 * blocks * (r16 >> 2) + 4 * b + (r16 & 3)) * cols + step * 64 + kc * 16);
            };
            v4i w1[4][KS], ws[4], w2[NB2][G];
#pragma unroll
            for (int b = 0; b < 4; ++b)
            {
#pragma unroll
                for (int k = 0; k < KS; ++k)
                    w1[b][k] = fragment(p.l1.w, C, wave * 64, 4, b, k);
                if constexpr (SHORT)
                    ws[b] = fragment(p.ls.w, CS, wave * 64, 4, b, 0);
            }
#pragma unroll
            for (int b = 0; b < NB2; ++b)
#pragma unroll
                for (int g = 0; g < G; ++g)
                    w2[b][g] = fragment(p.l2.w, N1, o2, NB2, b, g);
            // (A bias of up to 2^24 is carried in the accumulators: as the sums of up to 512 products are exact as floats, float(sum + bias)
            // rounds once, as float(sum) + float(bias) does)
            static_assert(N1 * 255 * 128 <= (1 << 24) && C <= N1 && CS <= N1, "sums of products that are exact as floats");
            bool small = true;
            auto look = [&](const ChainLayer& l, int n) {
                if (l.bias && tid < n) // (no more channels than threads)
                    small = small && l.bias[tid] >= -(1 << 24) && l.bias[tid] <= (1 << 24);
            };
            look(p.l1, N1);
            look(p.l2, N2);
            if constexpr (SHORT)
                look(p.ls, N1);
            wait_vmcnt<0>(); // the first tiles have landed, behind the barrier everyone's
            const bool fold = __syncthreads_and(small) != 0;
            auto start_of = [&](const ChainLayer& l, int n) {
                v4i r = l.x_unsigned ? 128 * words(l.wsum, n) : v4i{0, 0, 0, 0}; // uniform
                return fold && l.bias ? r + words(l.bias, n) : r;               // uniform
            };
            auto scale_of = [&](const ChainLayer& l, int n) {
                const float one = l.scale[0];
                return l.per_channel ? __builtin_bit_cast(v4f, words(l.scale, n)) : v4f{one, one, one, one}; // uniform
            };
            v4i start1[4], starts[4], start2[NB2];
            v4f scale1[4], scales[4], scale2[NB2];
#pragma unroll
            for (int b = 0; b < 4; ++b)
            {
                start1[b] = start_of(p.l1, n1 + 4 * b);
                scale1[b] = scale_of(p.l1, n1 + 4 * b);
                if constexpr (SHORT)
                {
                    starts[b] = start_of(p.ls, n1 + 4 * b);
                    scales[b] = scale_of(p.ls, n1 + 4 * b);
                }
            }
#pragma unroll
            for (int b = 0; b < NB2; ++b)
            {
                start2[b] = start_of(p.l2, n2 + 4 * b);
                scale2[b] = scale_of(p.l2, n2 + 4 * b);
            }
            const int x_mask = p.l1.x_unsigned ? static_cast<int>(0x80808080u) : 0, s_mask = p.ls.x_unsigned ? static_cast<int>(0x80808080u) : 0,
                      n_mask = p.l2.x_unsigned ? static_cast<int>(0x80808080u) : 0;
            const float sum_scale = *p.sum_scale;
            const float short_lo = p.short_relu ? 0.0f : -128.0f;
            auto flip = [](v4i v, int mask) { return v4i{v[0] ^ mask, v[1] ^ mask, v[2] ^ mask, v[3] ^ mask}; };

            auto run = [&](auto folded) {
                constexpr bool FOLD = decltype(folded)::value;
                // (a bias beyond 2^24 is read again where it is used: it is in nobody's way otherwise)
                auto scaled = [&](const v4i& a, const v4f& scale, const ChainLayer& l, int n, int e) {
                    const float f = static_cast<float>(a[e]);
                    return __fmul_rn(FOLD ? f : __fadd_rn(f, l.bias ? static_cast<float>(l.bias[n + e]) : 0.0f), scale[e]);
                };
                // float -> byte with saturation (the ReLU is the lower bound) and round half to even
                auto pack = [](float v, int e, uint32_t packed) { return __builtin_amdgcn_cvt_pk_u8_f32(v, e, packed); };
                int buf = 0;
                for (int t = first; t < p.tiles; t += stride, buf ^= 1)
                {
                    uint8_t* const ys = wide + buf * (16 * N1) + lane * 16;
                    const uint8_t* const in = lds + buf * TILE + lane * 16;
                    const int m = pixel(t);
                    v4i acc[4], accs[4];
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                        acc[b] = start1[b];
#pragma unroll
                    for (int k = 0; k < KS; ++k)
                    {
                        const v4i xf = flip(*reinterpret_cast<const v4i*>(in + k * 1024), x_mask);
#pragma unroll
                        for (int b = 0; b < 4; ++b)
                            acc[b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1[b][k], xf, acc[b], 0, 0, 0);
                    }
                    // the residual's bytes, or the shortcut's data
                    const v4i res = *reinterpret_cast<const v4i*>(in + (SHORT ? KS : SHARED + wave) * 1024);
                    if constexpr (SHORT)
                    {
                        const v4i sf = flip(res, s_mask);
#pragma unroll
                        for (int b = 0; b < 4; ++b)
                            accs[b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ws[b], sf, starts[b], 0, 0, 0);
                    }
                    v4i y;
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                    {
                        uint32_t packed = 0;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                        {
                            float r;
                            if constexpr (SHORT)
                                r = rintf(__builtin_amdgcn_fmed3f(scaled(accs[b], scales[b], p.ls, n1 + 4 * b, e), short_lo, 127.0f));
                            else
                            {
                                const uint32_t byte = (static_cast<uint32_t>(res[b]) >> (8 * e)) & 0xFFu;
                                r = I8 ? static_cast<float>(static_cast<int8_t>(byte)) : static_cast<float>(byte);
                            }
                            packed = pack(fmaf(sum_scale, r, scaled(acc[b], scale1[b], p.l1, n1 + 4 * b, e)), e, packed);
                        }
                        if constexpr (I8) // 127 at most
                        {
                            const uint32_t high = packed & 0x80808080u;
                            packed = (packed | (high - (high >> 7))) & 0x7f7f7f7fu;
                        }
                        y[b] = static_cast<int>(packed);
                    }
                    __builtin_amdgcn_raw_buffer_store_b128(y, ors, m < p.M ? m * N1 + n1 : kOob, 0, 0);
                    *reinterpret_cast<v4i*>(ys + wave * 1024) = flip(y, n_mask); // (the readers of two tiles ago are behind the barrier of the last one)
                    // the next tile's loads have landed (the two stores since may still be in flight), and behind the barrier
                    // everyone's; everyone has read this tile, whose slot is free
                    asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)\n\ts_barrier" ::: "memory");
                    issue(t + 2 * stride, buf);
                    v4i acc2[NB2];
#pragma unroll
                    for (int b = 0; b < NB2; ++b)
                        acc2[b] = start2[b];
#pragma unroll
                    for (int g = 0; g < G; ++g)
                    {
                        const v4i yf = *reinterpret_cast<const v4i*>(ys + g * 1024);
#pragma unroll
                        for (int b = 0; b < NB2; ++b)
                            acc2[b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w2[b][g], yf, acc2[b], 0, 0, 0);
                    }
                    int z[NB2];
#pragma unroll
                    for (int b = 0; b < NB2; ++b)
                    {
                        uint32_t packed = 0;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            packed = pack(scaled(acc2[b], scale2[b], p.l2, n2 + 4 * b, e), e, packed);
                        z[b] = static_cast<int>(packed);
                    }
                    const int at = m < p.M ? m * N2 + n2 : kOob;
                    if constexpr (NB2 == 2)
                        __builtin_amdgcn_raw_buffer_store_b64(v2i{z[0], z[1]}, nrs, at, 0, 0);
                    else
                        __builtin_amdgcn_raw_buffer_store_b32(z[0], nrs, at, 0, 0);
                }
            };
            if (fold) // uniform
                run(std::true_type{});
            else
                run(std::false_type{});
            wait_vmcnt<0>(); // nothing may still be on its way into LDS when the wavefront ends
        }

        template <int C, int N1, int N2, bool SHORT, bool I8>
        int launch_chain(ChainParams p, hipStream_t s)
        {
            constexpr size_t bytes = chain_lds(C, N1, SHORT);
            static_assert(bytes + 512 <= 64 * 1024, "what a workgroup may have without asking (512 bytes are the barrier's that counts votes)");
            p.tiles = (p.M + 15) / 16;
            const int grid = std::min(device_compute_units() * (512 / N1), p.tiles); // (two wavefronts a SIMD)
            conv_chain_kernel<C, N1, N2, SHORT, I8><<<static_cast<unsigned>(grid), N1, bytes, s>>>(p);
            return check_launch("conv_chain_i8_16x16x64");
        }

        // ---- 256 -> 1024 -> 256 channels --------------------------------------------------------------------
        // Both layers' weights are 512 KB: no wavefronts hold them.  A workgroup takes all channels of 16 (P0 + P1) pixels, whose data
        // stay in LDS, and streams the weights past them once, in slices of 256 rows x 128 bytes through a ring of three in LDS: for
        // every 256 channels of the wide result two slices of the widening layer, then (requantized, through LDS) two of the narrow
        // one, whose sums stay in registers to the end.  A wavefront has 64 channels of half of the pixels (four blocks of 16 and three
        // for 112 pixels: the two halves share each SIMD); rows of weights are dealt to lanes as above.  The residual arrives where the
        // wide bytes will stand, a lane's bytes in place of its own.  One barrier a slice; loads two slices ahead.
        //
        // Bound by the matrix cores and the LDS reads that feed them, which a barrier a slice keeps from overlapping: 25 088 pixels are
        // 26 GOP and 64 MB (10 us each way); a workgroup of 112 pixels takes 4.0 us for 256 channels of the wide result, 1.4 for a
        // block of 16 pixels and 5.2 before and after them.  Two launches and one, looped: 25 088 pixels 32.4 -> 25.0 us, 12 544
        // 23.0 -> 16.6, 6 272 15.2 -> 12.9.  ResNet-50 of 128 images 1222 -> 1179 us, of 64 806 -> 773, of 32 578 -> 569.
        // Tried and taken back: all fragments of a slice read ahead of its products, with the wavefront's priority raised or not (no
        // faster).  Without the loads of weights the same time, without the requantization 0.8 us less.
        constexpr int kBlockC = 256, kBlockN1 = 1024, kBlockN2 = 256;
        constexpr int kBlockSlice = 256 * 128; // bytes of a slice of weights
        constexpr size_t chain_block_lds(int blocks) { return 2 * static_cast<size_t>(blocks) * 4096 + 3 * static_cast<size_t>(kBlockSlice) + 4096; }

        template <int P0, int P1, bool I8>
        __global__ __launch_bounds__(512, 2) void conv_chain_block_kernel(const ChainParams p)
        {
            touch_arguments<sizeof(ChainParams)>();
            constexpr int PB = P0 + P1;
            constexpr int PIECES = PB * 4;                     // of the data: 16 pixels x 64 channels, as the lanes read them
            extern __shared__ __attribute__((aligned(16))) uint8_t lds[]; // [PB][4][1024] data, [PB][4][1024] wide, [3] slices, [3][256] wsum, bias, scale, 1 KB for loads of nothing
            uint8_t* const xs = lds;
            uint8_t* const ys = lds + PB * 4096;
            uint8_t* const ring = lds + 2 * PB * 4096;
            const uint8_t* const params = ring + 3 * kBlockSlice;
            const int tid = static_cast<int>(threadIdx.x);
            const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
            const int r16 = lane & 15, kc = lane >> 4;
            const int wm = wave >> 2, wn = wave & 3;
            const int m0 = static_cast<int>(blockIdx.x) * 16 * PB;
            const int channel = wn * 64 + kc * 16; // the lane's first channel within 256

            // ---- constants of the narrow layer, and whether the widening layer's bias goes into the accumulators (as above; the narrow
            // layer's sums reach 1024 * 255 * 128 > 2^24: float(sum) rounds before float(bias) is added, so they are never folded) ------
            static_assert(kBlockC * 255 * 128 <= (1 << 24), "sums of products that are exact as floats");
            auto words = [](const void* from, int at) { return *reinterpret_cast<const v4i_at4*>(static_cast<const int32_t*>(from) + at); };
            bool small = true;
            auto look = [&](const int32_t* bias, int n) {
                if (bias && n >= 0)
                    small = small && bias[n] >= -(1 << 24) && bias[n] <= (1 << 24);
            };
            look(p.l1.bias, tid);
            look(p.l1.bias, tid + 512);
            v4i wsum2[4];
#pragma unroll
            for (int b = 0; b < 4; ++b)
                wsum2[b] = words(p.l2.wsum, channel + 4 * b);
            const float sum_scale = *p.sum_scale, one1 = p.l1.scale[0], one2 = p.l2.scale[0];

            // ---- loads ---------------------------------------------------------------------------------------
            const v4i xw = rsrc_words(p.x, static_cast<uint32_t>(p.M) * kBlockC), sw = rsrc_words(p.sum, static_cast<uint32_t>(p.M) * kBlockN1);
            const v4i w1 = rsrc_words(p.l1.w, kBlockN1 * kBlockC), w2 = rsrc_words(p.l2.w, kBlockN2 * kBlockN1);
            const __amdgpu_buffer_rsrc_t ors = make_rsrc(p.out, static_cast<uint32_t>(p.M) * kBlockN1);
            const __amdgpu_buffer_rsrc_t nrs = make_rsrc(p.narrow, static_cast<uint32_t>(p.M) * kBlockN2);
            const uint32_t xs_at = lds_address(xs), ys_at = lds_address(ys), ring_at = lds_address(ring), params_at = lds_address(params);
            auto dma4 = [](v4i rsrc, int32_t off, uint32_t to) {
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"s"(to), "v"(off), "s"(rsrc));
            };
            // wsum, bias, scale of 256 channels from `first` (zeros for absent arrays): twelve pieces of 64
            auto load_params = [&](const ChainLayer& l, int first) {
#pragma unroll
                for (int j = 0; j < 2; ++j)
                {
                    const int piece = j * 8 + wave, array = piece >> 2; // uniform
                    const void* const from = array == 0 ? static_cast<const void*>(l.wsum) : array == 1 ? static_cast<const void*>(l.bias) : static_cast<const void*>(l.scale);
                    const bool there = array == 0 || (array == 1 && l.bias != nullptr) || (array == 2 && l.per_channel != 0);
                    dma4(rsrc_words(from, there ? kBlockN1 * 4u : 0u), (first + (piece & 3) * 64 + lane) * 4, __builtin_amdgcn_readfirstlane(params_at + piece * 256));
                }
            };
            // a load of the workgroup covers 64 rows of a slice, eight lanes a row: whole lines.  Chunk c of row r stands at position
            // c ^ (r % 4 / 2 + r / 16 % 4 * 2) of the row: sixteen lanes of a fragment meet sixteen columns of the banks
            const int lrow = wave * 8 + (lane >> 3);
            const int chunk = ((lane & 7) ^ (((lrow >> 1) & 1) | (((lrow >> 4) & 3) << 1))) * 16;
            const int at1 = lrow * kBlockC + chunk, at2 = lrow * kBlockN1 + chunk;
            // slice j % 4 of channels 256 (j / 4) ..: two of the widening layer's rows, two of the narrow layer's columns.  (Beyond
            // the last: rows beyond the weights, zeros)
            auto load_widen = [&](int blk, int half, int slot) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    lds_dma16_unfenced(w1, at1 + (blk * 256 + i * 64) * kBlockC + half * 128, __builtin_amdgcn_readfirstlane(ring_at + slot * kBlockSlice + i * 8192 + wave * 1024));
            };
            auto load_narrow = [&](int blk, int half, int slot) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    lds_dma16_unfenced(w2, at2 + i * 64 * kBlockN1 + blk * 256 + half * 128, __builtin_amdgcn_readfirstlane(ring_at + slot * kBlockSlice + i * 8192 + wave * 1024));
            };
            // The workgroups of a compute die (consecutive ones go to the eight of them in turn) touch a line of the weights a lane, all of
            // them together: what the ring asks for later is then on its way into their L2, or there.  ResNet-50, where other layers have
            // been through it, with the touch over without, both in turn, 29 numbers of images: 0.97 to 0.998 for each with one round of
            // 148 workgroups or more (30 images 548 -> 530 us, 64 776 -> 770, 128 1190 -> 1183), 1.00 for two rounds.  Below, with 32
            // pixels a workgroup, mixed: 129 workgroups 1.015, 135 0.988, 141 1.005, 147 0.993.  (With 64 pixels 129 to 147 workgroups gain
            // 1 %, which the line leaves)
            if (gridDim.x >= 148) // uniform
            {
                constexpr int parts = 2 * kBlockN1 * kBlockC / (64 * 128); // of 64 lines
                const int each = (parts + (static_cast<int>(gridDim.x) >> 3) - 1) / (static_cast<int>(gridDim.x) >> 3);
                const int part = static_cast<int>(blockIdx.x >> 3) * each + wave; // uniform
                const bool second = part >= parts / 2;
                dma4(second ? w2 : w1, wave < each && part < parts ? (part - (second ? parts / 2 : 0)) * (64 * 128) + lane * 128 : kOob, __builtin_amdgcn_readfirstlane(params_at + 3072));
            }
#pragma unroll
            for (int j = 0; j < (PIECES + 7) / 8; ++j)
            {
                const int piece = j * 8 + wave; // uniform
                const int m = m0 + (piece >> 2) * 16 + r16;
                lds_dma16_unfenced(xw, piece < PIECES && m < p.M ? m * kBlockC + (piece & 3) * 64 + kc * 16 : kOob,
                                   __builtin_amdgcn_readfirstlane(piece < PIECES ? xs_at + piece * 1024 : params_at + 3072));
            }
            load_params(p.l1, 0);
            load_widen(0, 0, 0);
            load_widen(0, 1, 1);
            wait_vmcnt<8>(); // data and constants
            auto flip = [](v4i v, int mask) { return v4i{v[0] ^ mask, v[1] ^ mask, v[2] ^ mask, v[3] ^ mask}; };
            const int n_mask = p.l2.x_unsigned ? static_cast<int>(0x80808080u) : 0;
            if (p.l1.x_unsigned) // uniform
#pragma unroll
                for (int j = 0; j < (PIECES + 7) / 8; ++j)
                    if (j * 8 + wave < PIECES) // uniform; the lane's own bytes
                    {
                        v4i* const at = reinterpret_cast<v4i*>(xs + (j * 8 + wave) * 1024 + lane * 16);
                        *at = flip(*at, static_cast<int>(0x80808080u));
                    }
            const bool fold = __syncthreads_and(small) != 0;

            // fragments of a slice: rows 64 wn + 16 (r / 4) + 4 b + r % 4, 64 bytes
            const int f_row = (wn * 64 + 16 * (r16 >> 2) + (r16 & 3)) * 128;
            const int f_at[2] = {f_row + ((kc ^ (r16 >> 1)) << 4), f_row + (((4 + kc) ^ (r16 >> 1)) << 4)};

            auto run = [&](auto folded, auto blocks) {
                constexpr bool FOLD = decltype(folded)::value;
                constexpr int P = decltype(blocks)::value; // the wavefront's blocks of pixels
                const int px0 = wm * P0;
                const uint8_t* const xl = xs + px0 * 4096 + lane * 16;
                uint8_t* const yl = ys + px0 * 4096 + lane * 16;
                auto pixel = [&](int i) { return m0 + (px0 + i) * 16 + r16; };
                auto pack = [](float v, int e, uint32_t packed) { return __builtin_amdgcn_cvt_pk_u8_f32(v, e, packed); };
                v4i acc1[P][4], acc2[P][4];
#pragma unroll
                for (int b = 0; b < 4; ++b)
                {
                    const v4i start = p.l2.x_unsigned ? 128 * wsum2[b] : v4i{0, 0, 0, 0}; // uniform
#pragma unroll
                    for (int i = 0; i < P; ++i)
                        acc2[i][b] = start;
                }
                // 128 bytes of the reduction: `from` is the lane's place in the first of their two pieces of the data
                auto multiply = [&](v4i (&acc)[P][4], const uint8_t* from, int slot) {
#pragma unroll
                    for (int k = 0; k < 2; ++k)
                    {
                        v4i wf[4], xf[P];
#pragma unroll
                        for (int b = 0; b < 4; ++b)
                            wf[b] = *reinterpret_cast<const v4i*>(ring + slot * kBlockSlice + f_at[k] + b * 512);
#pragma unroll
                        for (int i = 0; i < P; ++i)
                            xf[i] = *reinterpret_cast<const v4i*>(from + i * 4096 + k * 1024);
#pragma unroll
                        for (int i = 0; i < P; ++i)
#pragma unroll
                            for (int b = 0; b < 4; ++b)
                                acc[i][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[b], xf[i], acc[i][b], 0, 0, 0);
                    }
                };
                // the slice's loads have landed (LATER loads and stores of this wavefront since may be in flight), and behind the
                // barrier everyone's; everyone has read the slice before, whose place the loads two slices ahead take
                auto next_slice = [](auto later) { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(decltype(later)::value) : "memory"); };
                auto after = [](int slot, int n) { return slot + n >= 3 ? slot + n - 3 : slot + n; };
                int slot = 0;
                for (int blk = 0; blk < kBlockN1 / 256; ++blk)
                {
                    next_slice(std::integral_constant<int, 4>{});
#pragma unroll
                    for (int i = 0; i < P; ++i)
                        lds_dma16_unfenced(sw, pixel(i) < p.M ? pixel(i) * kBlockN1 + blk * 256 + channel : kOob, __builtin_amdgcn_readfirstlane(ys_at + (px0 + i) * 4096 + wn * 1024));
                    load_narrow(blk, 0, after(slot, 2));
                    const v4i* const constants = reinterpret_cast<const v4i*>(params + channel * 4);
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                    {
                        const v4i start = (p.l1.x_unsigned ? 128 * constants[b] : v4i{0, 0, 0, 0}) + (FOLD ? constants[64 + b] : v4i{0, 0, 0, 0});
#pragma unroll
                        for (int i = 0; i < P; ++i)
                            acc1[i][b] = start;
                    }
                    multiply(acc1, xl, slot);
                    slot = after(slot, 1);
                    next_slice(std::integral_constant<int, 4 + P>{});
                    load_narrow(blk, 1, after(slot, 2));
                    multiply(acc1, xl + 2048, slot);
                    slot = after(slot, 1);
                    wait_vmcnt<8>(); // the residual, the lane's own bytes
#pragma unroll
                    for (int i = 0; i < P; ++i)
                    {
                        v4i* const place = reinterpret_cast<v4i*>(yl + i * 4096 + wn * 1024);
                        const v4i res = *place;
                        v4i y;
#pragma unroll
                        for (int b = 0; b < 4; ++b)
                        {
                            const v4f scale = p.l1.per_channel ? __builtin_bit_cast(v4f, constants[128 + b]) : v4f{one1, one1, one1, one1};
                            const v4i bias = FOLD ? v4i{0, 0, 0, 0} : constants[64 + b];
                            uint32_t packed = 0;
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                            {
                                const uint32_t byte = (static_cast<uint32_t>(res[b]) >> (8 * e)) & 0xFFu;
                                const float r = I8 ? static_cast<float>(static_cast<int8_t>(byte)) : static_cast<float>(byte);
                                const float f = static_cast<float>(acc1[i][b][e]);
                                packed = pack(fmaf(sum_scale, r, __fmul_rn(FOLD ? f : __fadd_rn(f, static_cast<float>(bias[e])), scale[e])), e, packed);
                            }
                            if constexpr (I8) // 127 at most
                            {
                                const uint32_t high = packed & 0x80808080u;
                                packed = (packed | (high - (high >> 7))) & 0x7f7f7f7fu;
                            }
                            y[b] = static_cast<int>(packed);
                        }
                        __builtin_amdgcn_raw_buffer_store_b128(y, ors, pixel(i) < p.M ? pixel(i) * kBlockN1 + blk * 256 + channel : kOob, 0, 0);
                        *place = flip(y, n_mask);
                    }
                    next_slice(std::integral_constant<int, 4 + P>{});
                    load_params(blk + 1 < kBlockN1 / 256 ? p.l1 : p.l2, (blk + 1) % (kBlockN1 / 256) * 256);
                    load_widen(blk + 1, 0, after(slot, 2));
                    multiply(acc2, yl, slot);
                    slot = after(slot, 1);
                    next_slice(std::integral_constant<int, 6 + P>{});
                    load_widen(blk + 1, 1, after(slot, 2));
                    multiply(acc2, yl + 2048, slot);
                    slot = after(slot, 1);
                }
                next_slice(std::integral_constant<int, 4>{}); // the narrow layer's constants
#pragma unroll
                for (int i = 0; i < P; ++i)
                {
                    const v4i* const constants = reinterpret_cast<const v4i*>(params + channel * 4);
                    v4i z;
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                    {
                        const v4f scale = p.l2.per_channel ? __builtin_bit_cast(v4f, constants[128 + b]) : v4f{one2, one2, one2, one2};
                        const v4i bias = constants[64 + b];
                        uint32_t packed = 0;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                        {
                            packed = pack(__fmul_rn(__fadd_rn(static_cast<float>(acc2[i][b][e]), static_cast<float>(bias[e])), scale[e]), e, packed);
                        }
                        z[b] = static_cast<int>(packed);
                    }
                    __builtin_amdgcn_raw_buffer_store_b128(z, nrs, pixel(i) < p.M ? pixel(i) * kBlockN2 + channel : kOob, 0, 0);
                }
            };
            auto half = [&](auto folded) {
                if (P0 == P1 || wm == 0) // uniform over the wavefront; both sides meet the same barriers
                    run(folded, std::integral_constant<int, P0>{});
                else
                    run(folded, std::integral_constant<int, P1>{});
            };
            if (fold) // uniform
                half(std::true_type{});
            else
                half(std::false_type{});
            wait_vmcnt<0>(); // nothing may still be on its way into LDS when the wavefront ends
        }

        template <int P0, int P1, bool I8>
        int launch_chain_block(const ChainParams& p, hipStream_t s)
        {
            constexpr size_t bytes = chain_block_lds(P0 + P1);
            static_assert(bytes + 512 <= 160 * 1024, "512 bytes are the barrier's that counts votes");
            const auto kernel = conv_chain_block_kernel<P0, P1, I8>;
            static bool configured[16] = {};
            int dev = 0;
            HIPQ_HIP(hipGetDevice(&dev));
            if (dev >= 0 && dev < 16 && !configured[dev])
            {
                HIPQ_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)));
                configured[dev] = true;
            }
            kernel<<<static_cast<unsigned>((p.M + 16 * (P0 + P1) - 1) / (16 * (P0 + P1))), 512, bytes, s>>>(p);
            return check_launch("conv_chain_block_i8_16x16x64");
        }

        // pixels of a workgroup, 0: two launches are as fast.  us, 32 / 64 / 112 pixels a workgroup and two launches:
        //    3 136 pixels  12.3  15.6  21.1  12.4      16 384  25.6  18.7  23.8  27.7      32 768  48.7  35.2  43.6  38.0      57 344  84  66  51.8  57.6
        //    4 704         12.7  15.8  21.3  14.9      25 088  45.9  31.6  25.0  32.4      33 712  58.9  47.7  43.6  42.8      65 536  96  69  70.6  61.1
        //    8 192         13.4  16.2  21.6  15.7      28 672  47.1  32.9  28.1  35.3      40 000  60.0  48.4  44.3  46.5     100 352 153 115  95.8  92.6
        // A round takes what it takes: the fewest pixels with one round to them, then the two sizes with two
        int block_pixels(int64_t M)
        {
            const int64_t units = device_compute_units();
            if (M < 16 * units || M > 224 * units || (M > 128 * units && M < 144 * units))
                return 0;
            return M <= 32 * units ? 32 : M <= 64 * units || (M > 112 * units && M <= 128 * units) ? 64 : 112;
        }

        bool pointwise(const ConvGeom& g)
        {
            if (g.in[0] != 1 || g.taps() != 1)
                return false;
            for (int i = 0; i < 3; ++i)
                if (g.dd[i] != 1 || g.dl[i] != 1 || g.st[i] != 1 || g.pb[i] != 0 || g.out[i] != g.in[i])
                    return false;
            return g.filter_t == HIPQ_I8 && (g.data_t == HIPQ_U8 || g.data_t == HIPQ_I8) && g.data_layout == HIPQ_LAYOUT_NXC && g.out_layout == HIPQ_LAYOUT_NXC;
        }
    }

    bool conv_chain_eligible(const ConvGeom& g1, const Epilogue& e1, const ConvGeom* gs, const Epilogue* es, const ConvGeom& g2, const Epilogue& e2)
    {
        if (!pointwise(g1) || !pointwise(g2) || (gs && !pointwise(*gs)))
            return false;
        auto same_pixels = [&](const ConvGeom& g) { return g.N == g1.N && g.in[1] == g1.in[1] && g.in[2] == g1.in[2]; };
        if (!same_pixels(g2) || (gs && !same_pixels(*gs)) || g2.C != g1.K)
            return false;
        // the wide result after a ReLU, of the residual's type; the narrow layer reads its bytes as either type
        if (!e1.sum_in || !e1.relu || (e1.out_t != HIPQ_U8 && e1.out_t != HIPQ_I8) || e1.sum_t != e1.out_t)
            return false;
        if (e2.sum_in || e2.out_t != HIPQ_U8)
            return false;
        if (gs && (es->sum_in || es->out_t != HIPQ_I8 || e1.out_t != HIPQ_I8 || gs->C != kChainShort || gs->K != g1.K))
            return false;
        const int64_t M = g1.N * g1.in[1] * g1.in[2];
        if (M < 1 || M * g1.K >= (1ll << 31))
            return false;
        if (gs)
            return g1.C == 64 && g1.K == 256 && g2.K == 64;
        // (256 channels of 512 for few pixels: 128 KB of weights are too many for a unit that has one tile.  One launch and two, looped, by
        // pixels: 512 10.2 and 7.2 us, 1024 10.2 and 7.9, 1536 10.3 and 9.4, 2048 10.4 and 9.7, 2304 10.4 and 10.9, 3072 10.6 and 10.8,
        // 6272 12.0 and 12.5, 12 544 14.0 and 13.6.  In a pass of ResNet-50, whose next stage begins with this pair: 784 pixels 1.012 times
        // the two launches' time, 1568 0.996, 2352 and more, up to 12 544, 0.991 to 0.995)
        if (g1.C == 128 && g2.K == 256 && M < 8 * device_compute_units())
            return false;
        if (g1.C == kBlockC && g1.K == kBlockN1 && g2.K == kBlockN2)
            return block_pixels(M) != 0;
        return (g1.C == 64 && g1.K == 256 && (g2.K == 64 || g2.K == 128)) || (g1.C == 128 && g1.K == 512 && (g2.K == 128 || g2.K == 256));
    }

    int launch_conv_chain(const ConvGeom& g1, const Epilogue& e1, const void* data, const void* packed1, const ConvGeom* gs, const Epilogue* es, const void* packed_s, const ConvGeom& g2,
                          const Epilogue& e2, const void* packed2, void* out, void* narrow, hipStream_t s)
    {
        ChainParams p;
        memset(&p, 0, sizeof(p));
        auto layer = [](const ConvGeom& g, const Epilogue& e, const void* packed) {
            return ChainLayer{static_cast<const int8_t*>(packed), reinterpret_cast<const int32_t*>(static_cast<const uint8_t*>(packed) + align_up(static_cast<size_t>(g.K * g.C), 256)), e.bias, e.scale,
                              e.per_channel, g.data_t == HIPQ_U8 ? 1 : 0};
        };
        p.x = static_cast<const uint8_t*>(data);
        p.sum = static_cast<const uint8_t*>(e1.sum_in);
        p.out = static_cast<uint8_t*>(out);
        p.narrow = static_cast<uint8_t*>(narrow);
        p.sum_scale = e1.sum_scale;
        p.l1 = layer(g1, e1, packed1);
        p.l2 = layer(g2, e2, packed2);
        if (gs)
        {
            p.ls = layer(*gs, *es, packed_s);
            p.short_relu = es->relu;
        }
        p.M = static_cast<int32_t>(g1.N * g1.in[1] * g1.in[2]);
        const bool i8 = e1.out_t == HIPQ_I8;
        if (gs)
            return launch_chain<64, 256, 64, true, true>(p, s);
        if (g1.C == kBlockC)
        {
            switch (block_pixels(p.M))
            {
            case 112: return i8 ? launch_chain_block<4, 3, true>(p, s) : launch_chain_block<4, 3, false>(p, s);
            case 64: return i8 ? launch_chain_block<2, 2, true>(p, s) : launch_chain_block<2, 2, false>(p, s);
            default: return i8 ? launch_chain_block<1, 1, true>(p, s) : launch_chain_block<1, 1, false>(p, s);
            }
        }
        if (g1.C == 64 && g2.K == 64)
            return i8 ? launch_chain<64, 256, 64, false, true>(p, s) : launch_chain<64, 256, 64, false, false>(p, s);
        if (g1.C == 64)
            return i8 ? launch_chain<64, 256, 128, false, true>(p, s) : launch_chain<64, 256, 128, false, false>(p, s);
        if (g2.K == 256)
            return i8 ? launch_chain<128, 512, 256, false, true>(p, s) : launch_chain<128, 512, 256, false, false>(p, s);
        return i8 ? launch_chain<128, 512, 128, false, true>(p, s) : launch_chain<128, 512, 128, false, false>(p, s);
    }
}
