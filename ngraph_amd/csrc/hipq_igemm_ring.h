// Products and implicit-GEMM convolutions of a hundred rows and more on tiles that fit the chip: one workgroup of eight
// wavefronts a compute unit, the tile chosen so that the fullest unit is done first (kRing*), operands in a ring of
// 128-byte reduction slices as deep as the LDS allows, loaded straight into it.
//
// What the kernel with four wavefronts a tile and three tiles a unit (igemm_pipe_kernel) spent its time on: half of
// each 64-byte slice waiting for LDS and for its barrier, partial sums of split reductions through memory where 128 x 128 tiles
// are few, and a last round of tiles that is nearly empty.  Here a slice has one barrier; the fragments of its second
// half are read while the first multiplies and the next slice's first half while the second does; the loads are issued
// between the products, a ring ahead, across tiles; the loop has no branch (a select that the compiler turns into one costs as much as
// its arithmetic saves: hence the masks in RingConv::advance), and every wait counts exactly what may still be in flight, stores of the tile
// before included.  A lane's four dwords of four neighbouring blocks are transposed among its lane group in
// registers (v_permlane*_swap) and leave as 16 bytes: no staging in LDS, no barrier for the epilogue.
//
// Measured on uniform random bytes, us, before (the better of igemm_pipe_kernel and igemm_wk_kernel) and here: 4096 x 768 x 2304 f32
// 23.9 -> 17.3, 4096 x 3072 x 768 f32 23.3 -> 17.0, 4096 x 768 x 768 f32 11.3 -> 9.6, 985 x 4096 x 768 27.6 -> 12.7; 3 x 3 over 256
// channels on 15 680 pixels 25.6 -> 14.5, over 512 on 2352 26.9 -> 17.1, inside ResNet-50 of 128 images 28.9 -> 24.0 and
// 33.7 -> 25.2 (the whole pass 1554 -> 1391).  What bounds it: see kRing*.
#pragma once
#include "hipq_igemm.h"

namespace hipq
{
    namespace
    {
        typedef int v4i_at4 __attribute__((ext_vector_type(4), aligned(4)));
        typedef int v4i_at1 __attribute__((ext_vector_type(4), aligned(1)));
        typedef uint32_t u32_at1 __attribute__((aligned(1)));
        constexpr int SL = 128; // reduction bytes of a slice: a row's piece is a whole cache line

        // 16 bytes a lane from `off` + soff of the buffer to LDS address lds_base + 16 * lane (zeros where off is out of range)
        __device__ __forceinline__ void ring_dma16(v4i rsrc, int32_t off, int32_t soff, uint32_t lds_base)
        {
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds_base), "v"(off), "s"(rsrc), "s"(soff));
        }
        __device__ __forceinline__ void ring_dma4(v4i rsrc, int32_t off, uint32_t lds_base)
        {
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"s"(lds_base), "v"(off), "s"(rsrc));
        }
        // every LDS access of this wavefront done, then the workgroup's barrier (loads into LDS stay in flight)
        __device__ __forceinline__ void ring_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

        // rows of a matrix
        struct RingRows
        {
            const uint8_t* x;
            uint32_t bytes;
            int32_t K;
            static constexpr bool kConv = false, kWhole = false; // kWhole: the reduction is whole slices
            struct Row
            {
                int32_t off; // of the lane's chunk, kOob beyond M
            };
            struct Cursor
            {
            };
            __device__ __forceinline__ void init_row(Row& r, int64_t m, int64_t M, int ch) const { r.off = m < M ? static_cast<int32_t>(m) * K + ch : kOob; }
            __device__ __forceinline__ void init_cursor(Cursor&, int) const {}
            __device__ __forceinline__ void advance(Cursor&) const {}
            __device__ __forceinline__ int32_t offset(const Row& r, const Cursor&) const { return r.off; }
            __device__ __forceinline__ bool oob(const Row&, const Cursor&) const { return false; }
            __device__ __forceinline__ int32_t direct(int64_t m, const int8_t* wrow, int32_t xzp, int32_t wzp, bool x_unsigned) const
            {
                return GemmX{x, K, bytes}.direct(m, wrow, xzp, wzp, x_unsigned);
            }
        };

        // windows over channels-last data, at most 32 taps, fewer than 2^31 output pixels
        struct RingWindow
        {
            const uint8_t* x; // [N][H][W][C]
            uint32_t bytes;
            int32_t H, W, C, Q, PQ, R, S, sh, sw, dh, dw, pbh, pbw;
            FastDiv by_pq, by_q;
            static constexpr bool kConv = true;
            struct Row
            {
                int32_t off;   // of the lane's chunk of the window's first tap (may lie before the image)
                uint32_t taps; // bit t: tap t lies inside the image
            };
            __device__ __forceinline__ void init_row(Row& rw, int64_t m, int64_t M, int ch) const
            {
                const bool valid = m < M;
                const uint32_t mm = valid ? static_cast<uint32_t>(m) : 0u;
                const int32_t n = static_cast<int32_t>(by_pq.div(mm));
                const int32_t rem = static_cast<int32_t>(mm) - n * PQ;
                const int32_t p = static_cast<int32_t>(by_q.div(static_cast<uint32_t>(rem)));
                const int32_t y0 = p * sh - pbh, x0 = (rem - p * Q) * sw - pbw;
                rw.off = ((n * H + y0) * W + x0) * C + ch;
                uint32_t xs = 0, all = 0;
                for (int32_t s = 0; s < S; ++s)
                    xs |= (static_cast<uint32_t>(x0 + s * dw) < static_cast<uint32_t>(W) ? 1u : 0u) << s;
                for (int32_t r = 0; r < R; ++r)
                    all |= (static_cast<uint32_t>(y0 + r * dh) < static_cast<uint32_t>(H) ? xs : 0u) << (r * S);
                rw.taps = valid ? all : 0u;
            }
            // exact accumulator of one output, any zero points
            __device__ __forceinline__ int32_t direct(int64_t m, const int8_t* wrow, int32_t xzp, int32_t wzp, bool x_unsigned) const
            {
                Row rw;
                init_row(rw, m, m + 1, 0);
                int32_t acc = 0;
                for (int32_t t = 0; t < R * S; ++t)
                {
                    if (((rw.taps >> t) & 1u) == 0)
                        continue;
                    const uint8_t* const p = x + rw.off + ((t / S) * dh * W + (t % S) * dw) * C;
                    const int8_t* const wp = wrow + t * C;
                    for (int32_t c = 0; c < C; ++c)
                    {
                        const int32_t a = x_unsigned ? static_cast<int32_t>(p[c]) : static_cast<int32_t>(static_cast<int8_t>(p[c]));
                        acc += (a - xzp) * (static_cast<int32_t>(wp[c]) - wzp);
                    }
                }
                return acc;
            }
        };

        // a multiple of 128 channels: a slice lies inside one tap, its cursor is the same for every lane
        struct RingConv : RingWindow
        {
            static constexpr bool kWhole = true;
            struct Cursor // the same for every lane
            {
                uint32_t bit;      // of the tap
                int32_t s, c, off; // tap's column, slice's first channel, and its distance from the window's first tap and channel
            };
            __device__ __forceinline__ void init_cursor(Cursor& c, int) const { c = Cursor{1u, 0, 0, 0}; }
            __device__ __forceinline__ void advance(Cursor& c) const
            {
                // (masks: a branch a slice costs more than the arithmetic)
                c.c += SL;
                const int32_t tap = ~((c.c - C) >> 31); // all ones: the next tap
                c.s -= tap;
                const int32_t row = ~((c.s - S) >> 31); // all ones: the next row of taps
                c.off += SL + (tap & ((dw - 1) * C)) + (row & ((dh * W - S * dw) * C));
                c.bit += c.bit & static_cast<uint32_t>(tap);
                c.s &= ~row;
                c.c &= ~tap;
            }
            __device__ __forceinline__ bool oob(const Row& r, const Cursor& c) const { return (r.taps & c.bit) == 0; }
            __device__ __forceinline__ int32_t offset(const Row& r, const Cursor& c) const { return oob(r, c) ? kOob : r.off + c.off; }
        };

        // a multiple of 16 channels: a lane's chunk lies inside one tap
        struct RingConvAny : RingWindow
        {
            static constexpr bool kWhole = false;
            FastDiv by_c, by_s;
            // a slice on: `taps` taps, `cols` of them beyond whole rows of taps, and `rest` channels; `step` bytes, `tap_step` and
            // `row_step` more where the channel or the column wraps
            int32_t taps, cols, rest, step, tap_step, row_step;
            struct Cursor // of the lane's chunk
            {
                uint32_t bit;      // of the tap
                int32_t s, c, off; // tap's column, chunk's channel, and its distance from where Row::off points, its place in the first slice
            };
            __device__ __forceinline__ void init_cursor(Cursor& cur, int ch) const
            {
                const int tap = static_cast<int>(by_c.div(static_cast<uint32_t>(ch)));
                const int r = static_cast<int>(by_s.div(static_cast<uint32_t>(tap)));
                cur.bit = tap < 32 ? 1u << tap : 0u;
                cur.s = tap - r * S;
                cur.c = ch - tap * C;
                cur.off = r * (dh * W * C) + cur.s * (dw * C) + cur.c - ch;
            }
            __device__ __forceinline__ void advance(Cursor& cur) const
            {
                cur.c += rest;
                const int32_t tap = ~((cur.c - C) >> 31); // all ones: one tap more
                cur.s += cols - tap;
                const int32_t row = ~((cur.s - S) >> 31); // all ones: the next row of taps
                cur.off += step + (tap & tap_step) + (row & row_step);
                cur.bit <<= taps - tap; // (31 + 8 at most: beyond the last tap, where nothing is asked for)
                cur.s -= row & S;
                cur.c -= tap & C;
            }
            __device__ __forceinline__ bool oob(const Row& r, const Cursor& c) const { return (r.taps & c.bit) == 0; }
            __device__ __forceinline__ int32_t offset(const Row& r, const Cursor& c) const { return oob(r, c) ? kOob : r.off + c.off; }
        };

        static inline RingWindow ring_window(const ConvX& cx)
        {
            return RingWindow{cx.x,  cx.bytes, cx.H,  cx.W,  cx.C,   cx.Q,   static_cast<int32_t>(cx.PQ), cx.R, cx.S, cx.sh,
                              cx.sw, cx.dh,    cx.dw, cx.pbh, cx.pbw, cx.by_pq, cx.by_q};
        }

        // where an output lies, for ANY (else row m, column n at m * N + n)
        struct RingMap
        {
            int32_t ncx; // [image][column][pixel]
            int32_t PQ;  // pixels of an image
            FastDiv by_pq;
        };

        // bytes of LDS
        constexpr int ring_wslots(int bn) { return (bn + 63) / 64; }
        constexpr int ring_stage(int bm, int bn) { return (bm + 64 * ring_wslots(bn)) * SL; }
        constexpr int ring_param_loads(int bn) { return (3 * ring_wslots(bn) + 7) / 8; } // a wavefront
        constexpr size_t ring_lds(int bm, int bn, int nbuf, bool sum)
        {
            return static_cast<size_t>(nbuf) * ring_stage(bm, bn) + (sum ? static_cast<size_t>(bm) * bn : 0) + static_cast<size_t>(ring_param_loads(bn)) * 8 * 256;
        }

        // ANY: any number of columns, any alignment of the output, channels-last or [image][channel][pixel] (`map`).  WGS: workgroups
        // that share a compute unit
        template <class XL, int WAVES_M, int WAVES_N, int A, int B, int NBUF, int MODE, bool HAS_SUM, int KIND, bool ANY = false, int WGS = 1>
        __global__ __launch_bounds__(512, 2 * WGS) void igemm_ring_kernel(XL xl, const int8_t* __restrict__ w, const int32_t* __restrict__ wsum, int64_t M, int32_t N, int32_t Kred, int32_t x_unsigned,
                                                                   int32_t m_tiles, int32_t n_tiles, FastDiv by_m_tiles, FastDiv by_group, int32_t group_shift, ZeroPoints zp, Epilogue epi,
                                                                   RingMap map, void* __restrict__ out)
        {
            static_assert(WAVES_M * WAVES_N == 8, "eight wavefronts per workgroup");
            constexpr int BM = WAVES_M * A * 16, BN = WAVES_N * B * 16;
            static_assert(BM % 64 == 0, "a load of the workgroup covers 64 rows of one operand");
            constexpr int XS = BM / 64, WS = ring_wslots(BN), L = XS + WS; // loads of a slice a lane
            constexpr int STAGE = ring_stage(BM, BN);
            constexpr int PL = ring_param_loads(BN);
            constexpr bool Q8 = KIND == OUT_Q8 || KIND == OUT_GELU_Q8;
            constexpr int QUADS = B / 4, LEFT = B % 4;                  // blocks of a row that leave as 16 bytes a lane, as 4
            constexpr int STORES = ANY ? 0 : Q8 ? A * (QUADS + LEFT) : A * B; // of a tile a lane that are sure to be issued
            constexpr bool RES_LDS = HAS_SUM && !ANY;                   // the residual comes through LDS, a tile ahead
            constexpr int RES = RES_LDS ? A * QUADS : 0;                // residual loads of a tile a lane
            static_assert(!HAS_SUM || (MODE == EPI_FUSED && KIND == OUT_Q8), "residuals: fused policy, 8-bit outputs");
            static_assert(!RES_LDS || (LEFT == 0 && NBUF <= 3), "residuals come 16 bytes a lane, and have landed once a tile's second slice has");
            static_assert(MODE == EPI_FUSED ? KIND != OUT_I32 : KIND == OUT_Q8 || (ANY && KIND == OUT_I32), "outputs of the policies");
            static_assert((NBUF - 1) * L + PL < 64 && (NBUF - 2) * L + RES + STORES < 64, "vmcnt is a 6-bit counter");
            extern __shared__ __attribute__((aligned(16))) uint8_t lds[]; // [NBUF][x | w], residual tile, [3][64 WS] wsum, bias, scale

            touch_arguments<sizeof(XL) + 72 + 2 * sizeof(FastDiv) + sizeof(ZeroPoints) + sizeof(Epilogue) + sizeof(RingMap)>(); // (72: 56 of arguments, then the grid)
            const int tid = threadIdx.x;
            const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
            const int wm = wave / WAVES_N, wn = wave % WAVES_N;
            const int r16 = lane & 15, kc = lane >> 4;
            const int grid = static_cast<int>(gridDim.x);
            // (consecutive workgroups go round-robin to the 8 compute dies: renumbered so that neighbouring tiles meet in one L2)
            const int total = m_tiles * n_tiles;
            const int vb = (grid & 7) == 0 ? (static_cast<int>(blockIdx.x) & 7) * (grid >> 3) + (static_cast<int>(blockIdx.x) >> 3) : static_cast<int>(blockIdx.x);
            if (vb >= total)
                return;
            const int my_tiles = (total - vb + grid - 1) / grid;
            HeadWords hw = head_scalars_load(zp, epi, wsum);
            const float post_scale = KIND == OUT_GELU_Q8 ? *epi.post_scale : 1.0f;
            const int32_t post_zp = KIND == OUT_GELU_Q8 ? load_zp(epi.post_zp, epi.post_t) : 0;
            // tile t: column blocks in groups of 2^group_shift, along the group first, then down the rows (as igemm_pipe_kernel)
            auto tile_origin = [&](int j, int64_t& m0, int32_t& n0) {
                const int t = vb + j * grid;
                const int g = static_cast<int>(by_group.div(static_cast<uint32_t>(t)));
                const int r = t - g * (m_tiles << group_shift);
                int mt, nt;
                if (((g + 1) << group_shift) <= n_tiles) // uniform
                {
                    mt = r >> group_shift;
                    nt = (g << group_shift) + (r & ((1 << group_shift) - 1));
                }
                else
                {
                    const int c = static_cast<int>(by_m_tiles.div(static_cast<uint32_t>(r)));
                    mt = r - c * m_tiles;
                    nt = (g << group_shift) + c;
                }
                m0 = static_cast<int64_t>(mt) * BM;
                n0 = nt * BN;
            };

            // ---- loader: the workgroup's slices, tile after tile, as one sequence --------------------------------
            v4i xrs = rsrc_words(xl.x, xl.bytes);
            v4i wrs = rsrc_words(w, static_cast<uint32_t>(N) * static_cast<uint32_t>(Kred));
            const int KT = (Kred + SL - 1) / SL;
            // load i of the workgroup covers rows 64 i .. 64 i + 63 of an operand, eight lanes a row; a lane's place in LDS
            // is fixed (chunk position lane % 8 of its row), so it reads the chunk that belongs there
            const int lrow = wave * 8 + (lane >> 3);
            const int ch = ((lane & 7) ^ ((lrow >> 1) & 7)) * 16;
            typename XL::Row xr[XS];
            typename XL::Cursor cur;
            int32_t woff[WS];
            int32_t kb = 0;
            int lj = 0;
            auto loader_tile = [&](int j) {
                int64_t m0;
                int32_t n0;
                tile_origin(j, m0, n0);
#pragma unroll
                for (int i = 0; i < XS; ++i)
                    xl.init_row(xr[i], m0 + lrow + 64 * i, M, ch);
                xl.init_cursor(cur, ch);
#pragma unroll
                for (int i = 0; i < WS; ++i)
                    woff[i] = (n0 + lrow + 64 * i < N && lrow + 64 * i < BN) ? (n0 + lrow + 64 * i) * Kred + ch : kOob;
                kb = 0;
            };
            const uint32_t lds_base = lds_address(lds);
            const uint32_t lds_wave = __builtin_amdgcn_readfirstlane(lds_base + static_cast<uint32_t>(wave) * 1024u);
            constexpr bool kFill = XL::kConv && MODE == EPI_INTERP; // taps in a padding hold the data zero point (fused policy: zero)
            uint32_t oob_queue = 0;                                 // which chunks of the slices in flight lie in the padding, XS bits a slice
            // loads [from, to) of the slice into buffer `buf`
            auto load_pieces = [&](int buf, int from, int to) {
                const uint32_t base = lds_wave + static_cast<uint32_t>(buf) * STAGE;
                const bool live = XL::kWhole || kb + ch < Kred; // (zeros beyond the reduction's end)
                const int32_t k = __builtin_amdgcn_readfirstlane(kb);
#pragma unroll
                for (int i = 0; i < L; ++i)
                    if (i >= from && i < to)
                    {
                        if (i < XS)
                            ring_dma16(xrs, live ? xl.offset(xr[i < XS ? i : 0], cur) : kOob, XL::kConv ? 0 : k, base + i * 8192);
                        else
                            ring_dma16(wrs, live ? woff[i < XS ? 0 : i - XS] : kOob, k, base + i * 8192);
                    }
            };
            auto loaded_slice = [&]() {
                if constexpr (kFill)
                {
                    uint32_t bits = 0;
#pragma unroll
                    for (int i = 0; i < XS; ++i)
                        bits |= (xl.oob(xr[i], cur) ? 1u : 0u) << i;
                    oob_queue = (oob_queue >> XS) | (bits << (XS * (NBUF - 1)));
                }
                kb += SL;
                xl.advance(cur);
            };
            auto loader_next = [&]() {
                if (++lj < my_tiles) // uniform
                    loader_tile(lj);
                else
                    xrs[2] = wrs[2] = 0; // behind the last slice: nothing in range, nothing read, zeros into the ring
            };
            int64_t cm0;
            int32_t cn0, params_n0;
            tile_origin(0, cm0, cn0);
            // per-channel constants of a column block, raw: wsum, bias, scale in pieces of 64 (a load a piece; absent arrays
            // and channels beyond N are zeros)
            const uint32_t params_at = lds_base + NBUF * STAGE + (RES_LDS ? BM * BN : 0);
            const int32_t* const params = reinterpret_cast<const int32_t*>(lds + NBUF * STAGE + (RES_LDS ? BM * BN : 0));
            auto load_params = [&](int32_t n0) {
#pragma unroll
                for (int p = 0; p < PL; ++p)
                {
                    const int piece = p * 8 + wave;
                    const int array = piece / WS, n = n0 + (piece - array * WS) * 64 + lane;
                    const void* const from = array == 0 ? static_cast<const void*>(wsum) : array == 1 ? static_cast<const void*>(epi.bias) : static_cast<const void*>(epi.scale);
                    const bool there = array == 0 || (MODE == EPI_FUSED && ((array == 1 && epi.bias != nullptr) || (array == 2 && epi.per_channel)));
                    ring_dma4(rsrc_words(from, there ? static_cast<uint32_t>(N) * 4u : 0u), n < N ? n * 4 : kOob, __builtin_amdgcn_readfirstlane(params_at + piece * 256));
                }
                params_n0 = n0;
            };
            load_params(cn0);
            loader_tile(0);
            {
                int k = 0;
#pragma unroll
                for (int i = 0; i < NBUF; ++i)
                {
                    if (k == KT) // uniform
                    {
                        loader_next();
                        k = 0;
                    }
                    load_pieces(i, 0, L);
                    loaded_slice();
                    ++k;
                }
            }
            const int cross = NBUF % KT == 0 ? 0 : KT - NBUF % KT; // the slice of a tile under which the loader, NBUF slices ahead, starts another tile
            head_scalars_settle(hw);
            const HeadScalars hs = head_scalars_finish(hw, zp, epi);
            const EpiConst ec = hs.ec;
            if (MODE == EPI_INTERP && hs.wzp != 0) // uniform across the grid; w - wzp does not fit a signed byte: exact, slow
            {
                wait_vmcnt<0>(); // nothing may still be on its way into LDS when the wavefront ends
                for (int j = 0; j < my_tiles; ++j)
                {
                    int64_t m0;
                    int32_t n0;
                    tile_origin(j, m0, n0);
                    slow_tile(xl, w, M, Kred, x_unsigned, hs.xzp, hs.wzp, epi, OutMap{ANY ? map.ncx : 0, N, ANY ? map.PQ : 1}, out, m0, n0, BM, BN);
                }
                return;
            }
            const int32_t mult = (x_unsigned ? 128 : 0) - hs.xzp;
            const int xor_mask = x_unsigned ? static_cast<int>(0x80808080u) : 0;
            const int fill = (hs.xzp & 0xFF) * 0x01010101;
            // slice `at` of the queue: its chunks in the padding become the data zero point (they arrived as zeros)
            auto fill_fix = [&](int buf, int at) {
                if constexpr (kFill)
                    if (fill != 0) // uniform
                    {
#pragma unroll
                        for (int i = 0; i < XS; ++i)
                            if ((oob_queue >> (XS * at + i)) & 1u)
                                *reinterpret_cast<v4i*>(lds + buf * STAGE + wave * 1024 + i * 8192 + lane * 16) = v4i{fill, fill, fill, fill};
                    }
            };

            // ---- consumer ----------------------------------------------------------------------------------------
            // fragment (16 rows x 64 bytes) of a 128-byte row pitch, chunk c of row r at position c ^ (r / 2 % 8): sixteen lanes
            // of one chunk index meet sixteen different 16-byte columns of the banks
            const int swz = (r16 >> 1) & 7;
            const int f0 = r16 * SL + ((kc ^ swz) << 4), f1 = r16 * SL + (((4 + kc) ^ swz) << 4);
            v4i acc[A][B], xf[2][A], wf[2][B];
            auto fragments = [&](auto half, int buf) {
                constexpr int h = decltype(half)::value;
                const uint8_t* const p = lds + buf * STAGE + (h ? f1 : f0);
#pragma unroll
                for (int j = 0; j < B; ++j)
                    wf[h][j] = *reinterpret_cast<const v4i*>(p + (BM + (wn * B + j) * 16) * SL);
#pragma unroll
                for (int i = 0; i < A; ++i)
                    xf[h][i] = *reinterpret_cast<const v4i*>(p + (wm * A + i) * 16 * SL);
            };
            auto multiply_row = [&](auto half, int i) {
                constexpr int h = decltype(half)::value;
                // (the data sits in LDS as it came: unsigned bytes become signed here)
                const v4i x = v4i{xf[h][i][0] ^ xor_mask, xf[h][i][1] ^ xor_mask, xf[h][i][2] ^ xor_mask, xf[h][i][3] ^ xor_mask};
#pragma unroll
                for (int j = 0; j < B; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[h][j], x, acc[i][j], 0, 0, 0);
            };
            // lane (r16, kc) of block (i, j): row 16 i + r16, channels 16 j + 4 kc .. + 3
            const int col0 = wn * B * 16 + 4 * kc;
            auto param4 = [&](int array, int j) { return *reinterpret_cast<const v4i*>(params + array * (64 * WS) + col0 + 16 * j); };
            const uint32_t res_at = lds_base + NBUF * STAGE + static_cast<uint32_t>(wave) * (RES * 1024);
            const v4i* const res = reinterpret_cast<const v4i*>(lds + NBUF * STAGE + wave * (RES * 1024)) + lane;
            // 16 bytes a lane of an 8-bit row block: piece kc of quad q, row 16 i + r16
            auto piece_offset = [&](int i, int q) -> int32_t {
                const int row = (wm * A + i) * 16 + r16, n = cn0 + (wn * B + 4 * q + kc) * 16;
                return cm0 + row < M && n < N ? row * N + n : kOob;
            };
            auto fetch_residual = [&]() {
                if constexpr (RES_LDS)
                {
                    const v4i srs = rsrc_words(static_cast<const uint8_t*>(epi.sum_in) + cm0 * N, static_cast<uint32_t>((M - cm0 < BM ? M - cm0 : BM) * N));
#pragma unroll
                    for (int i = 0; i < A; ++i)
#pragma unroll
                        for (int q = 0; q < QUADS; ++q)
                            ring_dma16(srs, piece_offset(i, q), 0, __builtin_amdgcn_readfirstlane(res_at + (i * QUADS + q) * 1024));
                }
            };
            // four blocks' dwords of lanes kc = 0 .. 3 <-> 16 bytes a lane: a 4 x 4 transposition (its own inverse)
            auto transpose4 = [](uint32_t (&d)[4]) {
                const auto a = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false);
                const auto b = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false);
                const auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
                const auto e = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
                d[0] = c[0];
                d[1] = c[1];
                d[2] = e[0];
                d[3] = e[1];
            };
            const float clamp_lo = fmaxf(ec.lo, ec.relu_floor);
            const float magic = 12582912.0f; // 1.5 * 2^23: adding it rounds half to even into the low mantissa bits
            const float away = interp_magic(ec);
            const bool fast_interp = fabsf(ec.scale) * (static_cast<float>(Kred) * (255.0f * 128.0f)) < kInterpSmallEnd;
            const GeluQuantize gelu = gelu_quantize_of(post_scale, post_zp, epi.post_t, epi.post_mode);
            auto epilogue = [&](auto to_u8) {
                constexpr bool PK_U8 = decltype(to_u8)::value;
                constexpr int ESZ = Q8 ? 1 : 4;
                const __amdgpu_buffer_rsrc_t ors = make_rsrc(static_cast<uint8_t*>(out) + cm0 * N * ESZ, static_cast<uint32_t>((M - cm0 < BM ? M - cm0 : BM) * N * ESZ));
                auto bias4 = [&](int j) -> v4f {
                    const v4i b = MODE == EPI_FUSED ? param4(1, j) : v4i{0, 0, 0, 0};
                    return v4f{static_cast<float>(b[0]), static_cast<float>(b[1]), static_cast<float>(b[2]), static_cast<float>(b[3])};
                };
                auto scale4 = [&](int j) -> v4f {
                    const v4f s = __builtin_bit_cast(v4f, param4(2, j));
                    return MODE == EPI_FUSED && epi.per_channel ? s : v4f{ec.scale, ec.scale, ec.scale, ec.scale};
                };
                if constexpr (KIND == OUT_F32)
                {
                    const bool relu = epi.relu != 0;
#pragma unroll
                    for (int j = 0; j < B; ++j)
                    {
                        const v4f b = bias4(j), s = scale4(j);
                        const int n = cn0 + col0 + 16 * j;
#pragma unroll
                        for (int i = 0; i < A; ++i)
                        {
                            const int row = (wm * A + i) * 16 + r16;
                            v4i v;
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                            {
                                const float x = __fmul_rn(__fadd_rn(static_cast<float>(acc[i][j][e]), b[e]), s[e]);
                                v[e] = __float_as_int(relu ? ((x > 0.0f) ? x : __fmul_rn(x, -0.0f)) : x);
                            }
                            if constexpr (ANY)
                            {
                                int32_t* const at = static_cast<int32_t*>(out) + (cm0 + row) * N + n;
                                if (cm0 + row < M && n + 3 < N)
                                    *reinterpret_cast<v4i_at4*>(at) = v;
                                else if (cm0 + row < M)
                                {
#pragma unroll
                                    for (int e = 0; e < 3; ++e)
                                        if (n + e < N)
                                            at[e] = v[e];
                                }
                            }
                            else
                                __builtin_amdgcn_raw_buffer_store_b128(v, ors, cm0 + row < M && n < N ? (row * N + n) * 4 : kOob, 0, 0);
                        }
                        asm volatile("" ::: "memory"); // (a block's constants are fetched when their turn comes: all at once they do not fit the registers)
                    }
                }
                else if constexpr (KIND == OUT_I32)
                {
                    int32_t* const o32 = static_cast<int32_t*>(out);
#pragma unroll
                    for (int i = 0; i < A; ++i)
                    {
                        const int64_t m = cm0 + (wm * A + i) * 16 + r16;
                        const int32_t img = map.ncx ? static_cast<int32_t>(map.by_pq.div(static_cast<uint32_t>(m))) : 0;
                        const int64_t pix = m - static_cast<int64_t>(img) * map.PQ;
#pragma unroll
                        for (int j = 0; j < B; ++j)
                        {
                            const int n = cn0 + col0 + 16 * j;
                            v4i v;
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                v[e] = epi_interp<OUT_I32>(ec, acc[i][j][e]);
                            if (m >= M)
                                continue;
                            if (!map.ncx && n + 3 < N)
                                *reinterpret_cast<v4i_at4*>(o32 + m * N + n) = v;
                            else
                            {
#pragma unroll
                                for (int e = 0; e < 4; ++e)
                                    if (n + e < N)
                                        o32[map.ncx ? (static_cast<int64_t>(img) * N + n + e) * map.PQ + pix : m * N + n + e] = v[e];
                            }
                        }
                    }
                }
                else if constexpr (Q8)
                {
                    // four channels of one row, as bytes
                    auto bytes4 = [&](const v4i& a, const v4f& b, const v4f& s, uint32_t sum) -> uint32_t {
                        uint32_t packed = 0;
                        if constexpr (KIND == OUT_GELU_Q8)
                        {
                            // the float result as the float kernels compute it, then the bytes of Gelu and Quantize
                            v4f y;
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                            {
                                y[e] = __fmul_rn(__fadd_rn(static_cast<float>(a[e]), b[e]), s[e]);
                                if (epi.relu) // uniform
                                    y[e] = (y[e] > 0.0f) ? y[e] : __fmul_rn(y[e], -0.0f);
                            }
                            return gelu_quantize4(y, gelu);
                        }
                        if constexpr (MODE == EPI_INTERP)
                        {
                            int32_t x[4];
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                            {
                                if (fast_interp) // uniform
                                    x[e] = interp_small(__fmul_rn(static_cast<float>(a[e]), ec.scale), away);
                                else
                                    x[e] = epi_interp<OUT_Q8>(ec, a[e]);
                            }
                            return (__builtin_amdgcn_perm(x[3], x[2], 0x0c0c0400u) << 16) | __builtin_amdgcn_perm(x[1], x[0], 0x0c0c0400u);
                        }
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                        {
                            float v = __fmul_rn(__fadd_rn(static_cast<float>(a[e]), b[e]), s[e]);
                            if (HAS_SUM)
                            {
                                const uint32_t byte = (sum >> (8 * e)) & 0xFFu;
                                v = fmaf(ec.sum_scale, epi.sum_t == HIPQ_I8 ? static_cast<float>(static_cast<int8_t>(byte)) : static_cast<float>(byte), v);
                            }
                            if constexpr (PK_U8)
                            {
                                packed = __builtin_amdgcn_cvt_pk_u8_f32(v, e, packed); // saturates, rounds half to even, packs (the ReLU is the lower bound)
                                continue;
                            }
                            v = __builtin_amdgcn_fmed3f(v, clamp_lo, ec.hi);
                            if (e == 0)
                                packed = __float_as_uint(__fadd_rn(v, magic)); // the bytes above are replaced below
                            else if (e == 1)
                                asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_1 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD" : "+v"(packed) : "v"(v), "v"(magic));
                            else if (e == 2)
                                asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_2 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD" : "+v"(packed) : "v"(v), "v"(magic));
                            else
                                asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_3 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD" : "+v"(packed) : "v"(v), "v"(magic));
                        }
                        return packed;
                    };
                    // four channels of four rows, a row a lane of a quad <-> the four rows of one channel (4 x 4 bytes, its own inverse)
                    auto quad_transpose = [&](uint32_t d) -> uint32_t {
                        const uint32_t sel = 0x0c0c0400u + 0x0101u * static_cast<uint32_t>(lane & 3);
                        const int x = static_cast<int>(d);
                        const uint32_t t0 = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(x, x, 0x00, 0xf, 0xf, false)), t1 = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(x, x, 0x55, 0xf, 0xf, false));
                        const uint32_t t2 = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(x, x, 0xaa, 0xf, 0xf, false)), t3 = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(x, x, 0xff, 0xf, 0xf, false));
                        return __builtin_amdgcn_perm(__builtin_amdgcn_perm(t3, t2, sel), __builtin_amdgcn_perm(t1, t0, sel), 0x05040100u);
                    };
                    // ANY: up to four bytes at any address, `left` of them there
                    auto put4 = [](uint8_t* at, uint32_t d, int left) {
                        if (left >= 4)
                            *reinterpret_cast<u32_at1*>(at) = d;
                        else
                        {
#pragma unroll
                            for (int e = 0; e < 3; ++e)
                                if (e < left)
                                    at[e] = static_cast<uint8_t>(d >> (8 * e));
                        }
                    };
                    auto get4 = [](const uint8_t* at, int left) -> uint32_t {
                        if (left >= 4)
                            return *reinterpret_cast<const u32_at1*>(at);
                        uint32_t d = 0;
#pragma unroll
                        for (int e = 0; e < 3; ++e)
                            if (e < left)
                                d |= static_cast<uint32_t>(at[e]) << (8 * e);
                        return d;
                    };
                    auto any_row = [&](int i, const v4f (&b)[B], const v4f (&s)[B]) {
                        uint8_t* const o8 = static_cast<uint8_t*>(out);
                        const uint8_t* const sum_in = static_cast<const uint8_t*>(epi.sum_in);
                        if (map.ncx) // uniform: a lane four pixels of one channel
                        {
                            const int64_t m = cm0 + (wm * A + i) * 16 + (r16 & ~3);
                            const int32_t img = static_cast<int32_t>(map.by_pq.div(static_cast<uint32_t>(m)));
                            const int32_t pix = static_cast<int32_t>(m - static_cast<int64_t>(img) * map.PQ);
                            const bool whole = pix + 4 <= map.PQ && m + 4 <= M;
                            // (pixel e of the four where they are not all of one image)
                            auto at_pixel = [&](int e, int n) -> int64_t {
                                const int32_t g = static_cast<int32_t>(map.by_pq.div(static_cast<uint32_t>(m + e)));
                                return (static_cast<int64_t>(g) * N + n) * map.PQ + (m + e - static_cast<int64_t>(g) * map.PQ);
                            };
                            uint32_t sum[B];
#pragma unroll
                            for (int j = 0; j < B; ++j)
                            {
                                sum[j] = 0;
                                const int n = cn0 + (wn * B + j) * 16 + 4 * kc + (lane & 3);
                                if (HAS_SUM && n < N)
                                {
                                    if (whole)
                                        sum[j] = *reinterpret_cast<const u32_at1*>(sum_in + (static_cast<int64_t>(img) * N + n) * map.PQ + pix);
                                    else
                                    {
#pragma unroll
                                        for (int e = 0; e < 4; ++e)
                                            if (m + e < M)
                                                sum[j] |= static_cast<uint32_t>(sum_in[at_pixel(e, n)]) << (8 * e);
                                    }
                                }
                            }
#pragma unroll
                            for (int j = 0; j < B; ++j)
                            {
                                const uint32_t d = quad_transpose(bytes4(acc[i][j], b[j], s[j], HAS_SUM ? quad_transpose(sum[j]) : 0u));
                                const int n = cn0 + (wn * B + j) * 16 + 4 * kc + (lane & 3);
                                if (n >= N)
                                    continue;
                                if (whole)
                                    *reinterpret_cast<u32_at1*>(o8 + (static_cast<int64_t>(img) * N + n) * map.PQ + pix) = d;
                                else
                                {
#pragma unroll
                                    for (int e = 0; e < 4; ++e)
                                        if (m + e < M)
                                            o8[at_pixel(e, n)] = static_cast<uint8_t>(d >> (8 * e));
                                }
                            }
                            return;
                        }
                        const int64_t m = cm0 + (wm * A + i) * 16 + r16;
                        uint32_t sum[B];
#pragma unroll
                        for (int j = 0; j < B; ++j)
                            sum[j] = HAS_SUM && m < M ? get4(sum_in + m * N + cn0 + col0 + 16 * j, N - (cn0 + col0 + 16 * j)) : 0u;
                        uint32_t d[B];
#pragma unroll
                        for (int j = 0; j < B; ++j)
                            d[j] = bytes4(acc[i][j], b[j], s[j], sum[j]);
#pragma unroll
                        for (int q = 0; q < QUADS; ++q)
                        {
                            uint32_t t[4] = {d[4 * q], d[4 * q + 1], d[4 * q + 2], d[4 * q + 3]};
                            transpose4(t);
                            const int n = cn0 + (wn * B + 4 * q + kc) * 16;
                            if (m >= M)
                                continue;
                            if (n + 16 <= N)
                                *reinterpret_cast<v4i_at1*>(o8 + m * N + n) = v4i{static_cast<int>(t[0]), static_cast<int>(t[1]), static_cast<int>(t[2]), static_cast<int>(t[3])};
                            else
                            {
#pragma unroll
                                for (int e = 0; e < 4; ++e)
                                    put4(o8 + m * N + n + 4 * e, t[e], N - (n + 4 * e));
                            }
                        }
#pragma unroll
                        for (int j = 4 * QUADS; j < B; ++j)
                            if (m < M)
                                put4(o8 + m * N + cn0 + col0 + 16 * j, d[j], N - (cn0 + col0 + 16 * j));
                    };
                    // row i of blocks, its accumulators in row `from`
                    auto row_of_blocks = [&](int i, int from, const v4f (&b)[B], const v4f (&s)[B]) {
#pragma unroll
                        for (int q = 0; q < QUADS; ++q)
                        {
                            uint32_t sum[4] = {0, 0, 0, 0};
                            if constexpr (RES_LDS)
                            {
                                const v4i r = res[(i * QUADS + q) * 64];
#pragma unroll
                                for (int e = 0; e < 4; ++e)
                                    sum[e] = static_cast<uint32_t>(r[e]);
                                transpose4(sum);
                            }
                            uint32_t d[4];
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                d[j] = bytes4(acc[from][4 * q + j], b[4 * q + j], s[4 * q + j], sum[j]);
                            transpose4(d);
                            __builtin_amdgcn_raw_buffer_store_b128(v4i{static_cast<int>(d[0]), static_cast<int>(d[1]), static_cast<int>(d[2]), static_cast<int>(d[3])}, ors, piece_offset(i, q), 0, 0);
                        }
#pragma unroll
                        for (int j = 4 * QUADS; j < B; ++j)
                        {
                            const int row = (wm * A + i) * 16 + r16, n = cn0 + col0 + 16 * j;
                            __builtin_amdgcn_raw_buffer_store_b32(static_cast<int>(bytes4(acc[from][j], b[j], s[j], 0u)), ors, cm0 + row < M && n < N ? row * N + n : kOob, 0, 0);
                        }
                    };
                    v4f b[B], s[B];
#pragma unroll
                    for (int j = 0; j < B; ++j)
                    {
                        b[j] = bias4(j);
                        s[j] = scale4(j);
                    }
                    if constexpr (ANY)
                    {
#pragma unroll
                        for (int i = 0; i < A; ++i)
                            any_row(i, b, s);
                    }
                    else if constexpr (KIND == OUT_GELU_Q8)
                    {
                        // (one row of blocks at a time through the same instructions: all rows' together are 12 KB and more, met
                        // once a tile, and wait for the instruction cache longer than moving the rows up takes)
#pragma unroll 1
                        for (int i = 0; i < A; ++i)
                        {
                            row_of_blocks(i, 0, b, s);
#pragma unroll
                            for (int k = 0; k + 1 < A; ++k)
#pragma unroll
                                for (int j = 0; j < B; ++j)
                                    acc[k][j] = acc[k + 1][j];
                        }
                    }
                    else
                    {
#pragma unroll
                        for (int i = 0; i < A; ++i)
                            row_of_blocks(i, i, b, s);
                    }
                }
            };

            int cb = 0; // buffer of the slice being multiplied
            // One slice.  Its second half's fragments are read while the first half multiplies, the next slice's first half's
            // while the second multiplies; one barrier, behind which this slice's buffer takes the loads of the slice NBUF on.
            // The wait in front of it is for the next slice: younger are NBUF - 2 slices and, in a tile's first slice, its
            // residual and the stores of the tile before (`first`, `stores`).
            auto slice = [&](auto first, bool stores) {
                fragments(std::integral_constant<int, 1>{}, cb);
                __builtin_amdgcn_sched_barrier(0); // (read first: a half's products are their time)
#pragma unroll
                for (int i = 0; i < A; ++i)
                    multiply_row(std::integral_constant<int, 0>{}, i);
                __builtin_amdgcn_sched_barrier(0); // (the products are issued ahead of the wait, not behind it)
                const int next = cb + 1 == NBUF ? 0 : cb + 1;
                constexpr int kYounger = (NBUF - 2) * L + (decltype(first)::value ? RES : 0);
                if (decltype(first)::value && stores) // uniform
                    wait_vmcnt<kYounger + (decltype(first)::value ? STORES : 0)>();
                else
                    wait_vmcnt<kYounger>();
                fill_fix(next, 1);
                ring_barrier();
                fragments(std::integral_constant<int, 0>{}, next);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < A; ++i)
                {
                    multiply_row(std::integral_constant<int, 1>{}, i);
                    load_pieces(cb, i * L / A, (i + 1) * L / A);
                    __builtin_amdgcn_sched_barrier(0); // (loads among the products, none of them behind)
                }
                loaded_slice();
                cb = next;
            };
            wait_vmcnt<(NBUF - 1) * L>();
            fill_fix(0, 0);
            ring_barrier();
            fragments(std::integral_constant<int, 0>{}, 0);
            for (int cj = 0; cj < my_tiles; ++cj)
            {
                if (cj > 0 && cn0 != params_n0) // uniform
                {
                    ring_barrier(); // every wavefront is past its last read of the constants
                    load_params(cn0);
                    wait_vmcnt<0>();
                    ring_barrier();
                }
                // the accumulators start from the zero-point correction of their channels (|wsum| < 2^23)
#pragma unroll
                for (int j = 0; j < B; ++j)
                {
                    const v4i s = param4(0, j);
                    const v4i c = v4i{__mul24(mult, s[0]), __mul24(mult, s[1]), __mul24(mult, s[2]), __mul24(mult, s[3])};
#pragma unroll
                    for (int i = 0; i < A; ++i)
                        acc[i][j] = c;
                }
                fetch_residual();
                if (cross == 0) // uniform
                    loader_next();
                slice(std::true_type{}, cj != 0);
                int kt = 1;
                for (; kt < cross; ++kt)
                    slice(std::false_type{}, false);
                if (cross > 0) // uniform
                    loader_next();
                for (; kt < KT; ++kt)
                    slice(std::false_type{}, false);
                if (KIND == OUT_Q8 && MODE == EPI_FUSED && epi.out_t == HIPQ_U8) // uniform
                    epilogue(std::true_type{});
                else
                    epilogue(std::false_type{});
                asm volatile("" ::: "memory"); // (the residual's region is read before the next tile's loads are issued)
                if (cj + 1 < my_tiles)
                    tile_origin(cj + 1, cm0, cn0);
            }
            wait_vmcnt<0>(); // (the loads behind the last slice write zeros into LDS)
        }
        template <class XL, int WAVES_M, int WAVES_N, int A, int B, int NBUF, int MODE, bool HAS_SUM, int KIND, bool ANY = false, int WGS = 1>
        int launch_ring_tile(const XL& xl, const int8_t* w, const int32_t* wsum, int64_t M, int32_t N, int32_t Kred, int x_unsigned, const ZeroPoints& zp, const Epilogue& epi, const RingMap& map, void* out,
                             hipStream_t s, const char* name)
        {
            constexpr int BM = WAVES_M * A * 16, BN = WAVES_N * B * 16;
            constexpr size_t lds_bytes = ring_lds(BM, BN, NBUF, HAS_SUM && !ANY);
            static_assert(WGS * lds_bytes <= 160 * 1024, "a compute unit's LDS");
            auto kernel = igemm_ring_kernel<XL, WAVES_M, WAVES_N, A, B, NBUF, MODE, HAS_SUM, KIND, ANY, WGS>;
            static bool configured[16] = {};
            int dev = 0;
            HIPQ_HIP(hipGetDevice(&dev));
            if (dev < 0 || dev >= 16 || !configured[dev])
            {
                HIPQ_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes)));
                if (dev >= 0 && dev < 16)
                    configured[dev] = true;
            }
            const int64_t m_tiles = (M + BM - 1) / BM, n_tiles = (N + BN - 1) / BN;
            HIPQ_REQUIRE(fits_i32(m_tiles * n_tiles + 1024), "too many tiles");
            const int64_t units = device_compute_units() * WGS, tiles = m_tiles * n_tiles;
            const unsigned grid = static_cast<unsigned>(tiles < units ? (tiles + 7) / 8 * 8 : units);
            int group_shift = 0;
            while (group_shift < 3 && (2ll << group_shift) <= n_tiles && grid % (2u << group_shift) == 0)
                ++group_shift;
            kernel<<<grid, 512, lds_bytes, s>>>(xl, w, wsum, M, N, Kred, x_unsigned, static_cast<int32_t>(m_tiles), static_cast<int32_t>(n_tiles), fast_div(m_tiles), fast_div(m_tiles << group_shift),
                                               group_shift, zp, epi, map, out);
            return check_launch(name);
        }

        // a tile's size, and what a slice and a round cost (see the lists); where two workgroups share a compute unit, that
        // of one alone there and of two at a time
        struct RingTile
        {
            int bm, bn;
            float slice, round;
            float pair_slice = 0.0f, pair_round = 0.0f;
        };
        template <int COUNT>
        int ring_choose(const RingTile (&tiles)[COUNT], int64_t M, int64_t N, int64_t K)
        {
            const int64_t units = device_compute_units(), slices = (K + SL - 1) / SL;
            const char* const forced = getenv("HIPQ_RING_TILE"); // (its place in the list, for tests)
            if (forced)
                return atoi(forced);
            int best = -1;
            float least = 0.0f;
            for (int i = 0; i < COUNT; ++i)
            {
                const RingTile& t = tiles[i];
                const int64_t rounds = (((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) + units - 1) / units, pairs = t.pair_slice > 0.0f ? rounds / 2 : 0;
                const float k = static_cast<float>(slices);
                const float cost = static_cast<float>(rounds - 2 * pairs) * (k * t.slice + t.round) + static_cast<float>(pairs) * (k * t.pair_slice + t.pair_round);
                if (best < 0 || cost < least)
                {
                    best = i;
                    least = cost;
                }
            }
            return best;
        }
    }
}
