// 1 x 1 convolutions of 64, 128, 256 or 512 channels over many channels-last pixels, any stride, fused policy, optionally with
// the residual input: short reductions, whose tiles are mostly loads, requantization and stores.  On the tile kernels these
// follow each other for everything a workgroup has; here a workgroup keeps the weights of its columns in registers for the whole
// launch and a tile is 16 pixels, so that eight wavefronts a compute unit are at different points of it.
//
// A wavefront has 64 output channels: rows 16 (r / 4) + 4 b + r % 4 of them are block b of v_mfma_i32_16x16x64_i8's first
// operand, which leaves lane (pixel r = lane % 16, k = lane / 16) channels 16 k .. 16 k + 15 after four blocks: 16 bytes of
// output and of residual, 64 bytes of a pixel by four lanes.  Data (shared by the workgroup's wavefronts) and residual arrive by
// loads straight into LDS, a lane's bytes where that lane reads them, two tiles ahead; one barrier a tile.
//
// Bound by HBM where the reduction is 64 or 128, by that and the weights' way into the registers (64 bytes of a row at a time)
// where it is longer.  us, looped, before and here: 64 -> 64 over 401 408 pixels 13.9 -> 11.0, 64 -> 192 29.0 -> 20.4, 64 -> 320 with
// a residual 91 -> 63, 128 -> 192 36.4 -> 27.7, 256 -> 512 at stride 2 to 100 352 pixels 30.5 -> 24.1, 256 -> 1024 with a residual
// over 25 088 21.7 -> 19.5, 512 -> 2048 over 50 176 68.1 -> 57.2; ResNet-50 of 128 images 1241 -> 1222.  Tiles of 32 pixels and
// rings of three and four tiles are within 3 % of this.
//
// Arithmetic: that of the tile kernels' fused epilogue (hipq_igemm.h), see hipq_conv_pw.hip.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <type_traits>

#include "hipq_igemm.h"

namespace hipq
{
    namespace
    {
        typedef int v4i_at4 __attribute__((ext_vector_type(4), aligned(4)));
        struct StreamParams
        {
            const uint8_t* x; // [images][H][W][C]
            const int8_t* w;  // [N][C]
            const int32_t* wsum;
            uint8_t* out;       // [M][N]
            const uint8_t* sum; // [M][N] or null
            const int32_t* bias;
            const float* scale;
            const float* sum_scale;
            uint32_t x_bytes;
            int32_t M, N, tiles, col_tiles, xcds;
            int32_t x_unsigned, per_channel, relu, out_t, sum_t;
            // strided: pixel m of the output is pixel (p sh, q sw) of its image
            FastDiv by_pq, by_q;
            int32_t PQ, Q, row_step, col_step, image; // bytes
        };

        constexpr int stream_tile(int C, int waves, bool sum) { return 16 * (C + (sum ? waves * 64 : 0)); }
        constexpr size_t stream_lds(int C, int waves, bool sum) { return 2 * static_cast<size_t>(stream_tile(C, waves, sum)) + 1024; }

        // a workgroup: WAVES x 64 output channels
        template <int C, int WAVES, bool SUM, bool GATHER>
        __global__ __launch_bounds__(WAVES * 64, 2) void conv_stream_kernel(const StreamParams p)
        {
            touch_arguments<sizeof(StreamParams)>();
            constexpr int KS = C / 64, MINE = (KS + WAVES - 1) / WAVES; // pieces of 1 KB of data that every wavefront reads, and that a wavefront asks for
            constexpr int TILE = stream_tile(C, WAVES, SUM);
            extern __shared__ __attribute__((aligned(16))) uint8_t lds[]; // [2][piece of data | residual: wavefront][64 lanes][16 bytes], nothing
            const int tid = static_cast<int>(threadIdx.x);
            const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
            const int r16 = lane & 15, kc = lane >> 4;
            // a workgroup keeps its columns; those of one tile are on one die where the grid allows it
            const int b = static_cast<int>(blockIdx.x), xcd = b % p.xcds, along = b / p.xcds;
            const int col = along % p.col_tiles, first = along / p.col_tiles * p.xcds + xcd;
            const int stride = static_cast<int>(gridDim.x) / p.col_tiles;
            const int n_wave = (col * WAVES + wave) * 64, n0 = n_wave + kc * 16;

            const __amdgpu_buffer_rsrc_t ors = make_rsrc(p.out, static_cast<uint32_t>(p.M) * static_cast<uint32_t>(p.N));
            // (the compiler does not see that these are uniform where the loop is large)
            auto uniform = [](v4i r) { return v4i{__builtin_amdgcn_readfirstlane(r[0]), __builtin_amdgcn_readfirstlane(r[1]), __builtin_amdgcn_readfirstlane(r[2]), __builtin_amdgcn_readfirstlane(r[3])}; };
            const v4i xw = uniform(rsrc_words(p.x, p.x_bytes)), sw = uniform(rsrc_words(p.sum, SUM ? static_cast<uint32_t>(p.M) * static_cast<uint32_t>(p.N) : 0u));
            const uint32_t lds_at = lds_address(lds);
            auto pixel = [&](int t) { return t * 16 + r16; };
            auto data_at = [&](int m) -> int {
                if (!GATHER)
                    return m * C;
                const int img = static_cast<int>(p.by_pq.div(static_cast<uint32_t>(m)));
                const int rem = m - img * p.PQ, row = static_cast<int>(p.by_q.div(static_cast<uint32_t>(rem)));
                return img * p.image + row * p.row_step + (rem - row * p.Q) * p.col_step;
            };
            // (beyond the last tile every pixel is beyond M: nothing is read, zeros arrive, the counts stay the same)
            auto issue = [&](int t, int slot) {
                const uint32_t to = lds_at + static_cast<uint32_t>(slot) * TILE;
                const int m = pixel(t);
                const int at = data_at(m);
#pragma unroll
                for (int i = 0; i < MINE; ++i)
                {
                    const int piece = i * WAVES + wave; // uniform
                    lds_dma16_unfenced(xw, piece < KS && m < p.M ? at + piece * 64 + kc * 16 : kOob, __builtin_amdgcn_readfirstlane(piece < KS ? to + piece * 1024 : lds_at + 2 * TILE));
                }
                if constexpr (SUM)
                    lds_dma16_unfenced(sw, m < p.M ? m * p.N + n0 : kOob, __builtin_amdgcn_readfirstlane(to + (KS + wave) * 1024));
            };
            issue(first, 0);
            issue(first + stride, 1);

            auto words = [](const void* from, int at) { return *reinterpret_cast<const v4i_at4*>(static_cast<const int32_t*>(from) + at); };
            v4i wf[4][KS];
#pragma unroll
            for (int b4 = 0; b4 < 4; ++b4)
#pragma unroll
                for (int k = 0; k < KS; ++k)
                    wf[b4][k] = *reinterpret_cast<const v4i*>(p.w + (n_wave + 16 * (r16 >> 2) + 4 * b4 + (r16 & 3)) * C + k * 64 + kc * 16);
            static_assert(C * 255 * 128 <= (1 << 24), "sums of products that are exact as floats: float(sum + bias) rounds once, as float(sum) + float(bias) does");
            bool small = true;
            if (p.bias)
            {
                const int32_t v = p.bias[col * (WAVES * 64) + tid];
                small = v >= -(1 << 24) && v <= (1 << 24);
            }
            wait_vmcnt<0>(); // the first tiles have landed, behind the barrier everyone's
            const bool fold = __syncthreads_and(small) != 0;
            v4i start[4];
            v4f scale[4];
#pragma unroll
            for (int b4 = 0; b4 < 4; ++b4)
            {
                start[b4] = p.x_unsigned ? 128 * words(p.wsum, n0 + 4 * b4) : v4i{0, 0, 0, 0}; // uniform
                if (fold && p.bias)                                                          // uniform
                    start[b4] += words(p.bias, n0 + 4 * b4);
                const float one = p.scale[0];
                scale[b4] = p.per_channel ? __builtin_bit_cast(v4f, words(p.scale, n0 + 4 * b4)) : v4f{one, one, one, one}; // uniform
            }
            const int x_mask = p.x_unsigned ? static_cast<int>(0x80808080u) : 0;
            const float sum_scale = SUM ? *p.sum_scale : 0.0f;
            const bool u8 = p.out_t == HIPQ_U8;
            const float clamp_lo = p.relu || u8 ? 0.0f : -128.0f, hi = u8 ? 255.0f : 127.0f;
            const bool sum_i8 = p.sum_t == HIPQ_I8;
            const float magic = 12582912.0f; // 1.5 * 2^23: adding it rounds half to even into the low mantissa bits

            auto run = [&](auto folded, auto to_u8) {
                constexpr bool FOLD = decltype(folded)::value, PK_U8 = decltype(to_u8)::value;
                int buf = 0;
                for (int t = first; t < p.tiles; t += stride, buf ^= 1)
                {
                    const uint8_t* const in = lds + buf * TILE + lane * 16;
                    v4i acc[4];
#pragma unroll
                    for (int b4 = 0; b4 < 4; ++b4)
                        acc[b4] = start[b4];
#pragma unroll
                    for (int k = 0; k < KS; ++k)
                    {
                        const v4i x = *reinterpret_cast<const v4i*>(in + k * 1024);
                        const v4i xf = v4i{x[0] ^ x_mask, x[1] ^ x_mask, x[2] ^ x_mask, x[3] ^ x_mask};
#pragma unroll
                        for (int b4 = 0; b4 < 4; ++b4)
                            acc[b4] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[b4][k], xf, acc[b4], 0, 0, 0);
                    }
                    const v4i res = SUM ? *reinterpret_cast<const v4i*>(in + (KS + wave) * 1024) : v4i{0, 0, 0, 0};
                    v4i y;
#pragma unroll
                    for (int b4 = 0; b4 < 4; ++b4)
                    {
                        uint32_t packed = 0;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                        {
                            const float f = static_cast<float>(acc[b4][e]);
                            // (a bias beyond 2^24 is read again where it is used: it is in nobody's way otherwise)
                            float v = __fmul_rn(FOLD ? f : __fadd_rn(f, static_cast<float>(p.bias[n0 + 4 * b4 + e])), scale[b4][e]);
                            if constexpr (SUM)
                            {
                                const uint32_t byte = (static_cast<uint32_t>(res[b4]) >> (8 * e)) & 0xFFu;
                                v = fmaf(sum_scale, sum_i8 ? static_cast<float>(static_cast<int8_t>(byte)) : static_cast<float>(byte), v);
                            }
                            if constexpr (PK_U8)
                            {
                                packed = __builtin_amdgcn_cvt_pk_u8_f32(v, e, packed); // saturates, rounds half to even, packs (the ReLU is the lower bound)
                                continue;
                            }
                            v = __builtin_amdgcn_fmed3f(v, clamp_lo, hi);
                            if (e == 0)
                                packed = __float_as_uint(__fadd_rn(v, magic)); // the bytes above are replaced below
                            else if (e == 1)
                                asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_1 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD" : "+v"(packed) : "v"(v), "v"(magic));
                            else if (e == 2)
                                asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_2 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD" : "+v"(packed) : "v"(v), "v"(magic));
                            else
                                asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_3 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD" : "+v"(packed) : "v"(v), "v"(magic));
                        }
                        y[b4] = static_cast<int>(packed);
                    }
                    const int m = pixel(t);
                    __builtin_amdgcn_raw_buffer_store_b128(y, ors, m < p.M ? m * p.N + n0 : kOob, 0, 0);
                    // the next tile's loads have landed (the store since may still be in flight), and behind the barrier
                    // everyone's; everyone has read this tile, whose slot is free
                    asm volatile("s_waitcnt vmcnt(1) lgkmcnt(0)\n\ts_barrier" ::: "memory");
                    issue(t + 2 * stride, buf);
                }
            };
            if (fold && u8) // uniform
                run(std::true_type{}, std::true_type{});
            else if (fold)
                run(std::true_type{}, std::false_type{});
            else if (u8)
                run(std::false_type{}, std::true_type{});
            else
                run(std::false_type{}, std::false_type{});
            wait_vmcnt<0>(); // nothing may still be on its way into LDS when the wavefront ends
        }

        template <int C, int WAVES, bool SUM, bool GATHER>
        int launch_stream_kernel(const StreamParams& p0, hipStream_t s)
        {
            StreamParams p = p0;
            constexpr size_t bytes = stream_lds(C, WAVES, SUM);
            static_assert(bytes + 512 <= 64 * 1024, "what a workgroup may have without asking (512 bytes are the barrier's that counts votes)");
            p.tiles = (p.M + 15) / 16;
            p.col_tiles = p.N / (WAVES * 64);
            int rows = std::max(1, std::min(device_compute_units() * (8 / WAVES) / p.col_tiles, p.tiles)); // workgroups a column block (two wavefronts a SIMD)
            if (rows >= 8)
                rows = rows / 8 * 8;
            p.xcds = rows % 8 == 0 ? 8 : 1;
            conv_stream_kernel<C, WAVES, SUM, GATHER><<<static_cast<unsigned>(rows * p.col_tiles), WAVES * 64, bytes, s>>>(p);
            return check_launch("conv_stream_i8_16x16x64");
        }

        template <int C, int WAVES>
        int launch_stream_form(const StreamParams& p, bool gather, hipStream_t s)
        {
            if (p.sum)
                return gather ? launch_stream_kernel<C, WAVES, true, true>(p, s) : launch_stream_kernel<C, WAVES, true, false>(p, s);
            return gather ? launch_stream_kernel<C, WAVES, false, true>(p, s) : launch_stream_kernel<C, WAVES, false, false>(p, s);
        }
        template <int C>
        int launch_stream_width(const StreamParams& p, bool gather, hipStream_t s)
        {
            if (p.N % 512 == 0)
                return launch_stream_form<C, 8>(p, gather, s);
            if (p.N % 256 == 0)
                return launch_stream_form<C, 4>(p, gather, s);
            if constexpr (C <= 256)
                if (p.N % 128 == 0)
                    return launch_stream_form<C, 2>(p, gather, s);
            if constexpr (C <= 128)
                return launch_stream_form<C, 1>(p, gather, s);
            return HIPQ_ERR_UNSUPPORTED;
        }
    }

    bool conv_stream_eligible(const ConvGeom& g, const Epilogue& epi, const ZeroPoints& zp)
    {
        if (g.in[0] != 1 || g.taps() != 1 || g.st[0] != 1)
            return false;
        for (int i = 0; i < 3; ++i)
            if (g.dd[i] != 1 || g.pb[i] != 0 || (g.out[i] - 1) * g.st[i] >= g.in[i])
                return false;
        if (g.filter_t != HIPQ_I8 || (g.data_t != HIPQ_U8 && g.data_t != HIPQ_I8) || (g.out_t != HIPQ_U8 && g.out_t != HIPQ_I8))
            return false;
        if (epi.mode != EPI_FUSED || epi.post_scale != nullptr || zp.data_zp != nullptr || zp.filter_zp != nullptr)
            return false;
        if (g.data_layout != HIPQ_LAYOUT_NXC || g.out_layout != HIPQ_LAYOUT_NXC)
            return false;
        if ((reinterpret_cast<uintptr_t>(epi.sum_in) & 15) != 0) // (the tile kernels take a residual at any word)
            return false;
        if ((g.C != 64 && g.C != 128 && g.C != 256 && g.C != 512) || g.K % (g.C == 512 ? 256 : g.C == 256 ? 128 : 64) != 0 || g.K > 2048)
            return false;
        // From how many outputs a compute unit on: the weights' way into the registers has to be paid for, the more so the longer the
        // reduction.  Least multiples of 784 pixels and 64 channels for which this is faster, of 8 widths and 6 numbers of pixels each: 256
        // channels 12.8 M outputs (256 -> 512 over 25 088 pixels 12.2 us there, 12.5 here, over 50 176 18.1 and 16.6), 512 channels 26 M
        // (512 -> 1024 over 25 088 pixels 23.4 and 23.9, over 50 176 37.5 and 34.3), 128 channels 9 to 13 M (128 -> 512 over 12 544
        // pixels with a residual 7.9 and 8.8, over 25 088 9.6 and 9.5); 64 channels, or 128 at a stride, which the kernels there
        // look up pixel by pixel, from the smallest on (64 -> 64 over 6272 pixels 4.5 and 4.3 with the call, 128 -> 512 at stride 2
        // 7.1 and 6.5; worst of 60, 64 -> 512 over 12 544 with a residual, 7.2 and 7.4).
        const int64_t M = g.N * g.out[1] * g.out[2], units = device_compute_units();
        const bool strided = g.out[1] != g.in[1] || g.out[2] != g.in[2];
        const int64_t least = g.C == 64 || (g.C == 128 && strided) ? 0 : g.C == 128 ? 48 * 1024 : g.C == 256 ? 64 * 1024 : 128 * 1024;
        if (M < 16 * units || M * g.K < least * units || M * g.K >= (1ll << 31) || g.in_count() >= (1ll << 31))
            return false;
        return getenv("HIPQ_NO_PW64") == nullptr; // (the switch for the tile kernels)
    }

    int launch_conv_stream(const ConvGeom& g, const void* data, const void* packed, const Epilogue& epi, void* out, hipStream_t s)
    {
        HIPQ_REQUIRE((reinterpret_cast<uintptr_t>(data) & 15) == 0 && (reinterpret_cast<uintptr_t>(packed) & 15) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0,
                     "MFMA convolution needs 16-byte aligned tensors");
        StreamParams p;
        memset(&p, 0, sizeof(p));
        p.x = static_cast<const uint8_t*>(data);
        p.w = static_cast<const int8_t*>(packed);
        p.wsum = reinterpret_cast<const int32_t*>(static_cast<const uint8_t*>(packed) + align_up(static_cast<size_t>(g.K * g.C), 256));
        p.out = static_cast<uint8_t*>(out);
        p.sum = static_cast<const uint8_t*>(epi.sum_in);
        p.bias = epi.bias;
        p.scale = epi.scale;
        p.sum_scale = epi.sum_scale;
        p.x_bytes = static_cast<uint32_t>(g.in_count());
        p.M = static_cast<int32_t>(g.N * g.out[1] * g.out[2]);
        p.N = static_cast<int32_t>(g.K);
        p.x_unsigned = g.data_t == HIPQ_U8 ? 1 : 0;
        p.per_channel = epi.per_channel;
        p.relu = epi.relu;
        p.out_t = epi.out_t;
        p.sum_t = epi.sum_t;
        const bool gather = g.out[1] != g.in[1] || g.out[2] != g.in[2];
        p.PQ = static_cast<int32_t>(g.out[1] * g.out[2]);
        p.Q = static_cast<int32_t>(g.out[2]);
        p.by_pq = fast_div(p.PQ);
        p.by_q = fast_div(p.Q);
        p.image = static_cast<int32_t>(g.in[1] * g.in[2] * g.C);
        p.row_step = static_cast<int32_t>(g.st[1] * g.in[2] * g.C);
        p.col_step = static_cast<int32_t>(g.st[2] * g.C);
        switch (g.C)
        {
        case 64: return launch_stream_width<64>(p, gather, s);
        case 128: return launch_stream_width<128>(p, gather, s);
        case 256: return launch_stream_width<256>(p, gather, s);
        default: return launch_stream_width<512>(p, gather, s);
        }
    }
}
